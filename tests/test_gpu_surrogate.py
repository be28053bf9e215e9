"""GPU checks of the surrogate kernels against the numpy oracle
(oracle/sur_ref.py): the crop generator bit for bit, the BF16 MFMA forward
pass (hidden activations within two bfloat16 ulps on at most 0.1% of the
elements, output within float32 accumulation error), every gradient of the backward pass (relative
Frobenius error), that training on solver crops lowers the loss, and, with
the committed weights, the accepted surrogate blocks against the plain
method on the 2048^2 / 1024-cell monolayer.
"""
import sys

import numpy as np
import pytest
import torch

from pfh import params, sim2d, surrogate as su

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu-surrogate] {msg}", flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def R():
    from oracle import sur_ref
    return sur_ref


@pytest.fixture(scope="module")
def c1_after():
    wl = params.workload_c1()
    sim = sim2d.Sim2D(wl)
    sim.step(5)
    sim.sync()
    return sim


def _bits(t, shape):
    return t.cpu().numpy().view(np.uint16).reshape(shape)


def test_crop_matches_oracle(R, oracle, c1_after):
    sim = c1_after
    say("crops of C1 after 5 steps")
    ws = su.Workspace(sim.N, sim.dev)
    su.crop_sim(sim, ws)
    sim.sync()
    X, phic, origin = R.crops(sim.phi_now(), sim.cells(), sim.classes(), sim.S_now(), sim.L,
                              sim.P, oracle.sincosf)
    gX = _bits(ws.X0, (sim.N, 96, 96, 8))
    assert np.array_equal(gX, R.bf16_bits(X))
    assert np.array_equal(ws.phic.cpu().numpy().reshape(sim.N, 96, 96).view(np.uint32),
                          phic.view(np.uint32))
    assert np.array_equal(ws.origin.cpu().numpy().reshape(-1, 2), origin)
    assert phic.max() > 0.9


def _random_net(seed):
    net = su.Net(seed=seed)
    rng = np.random.default_rng(seed + 1)
    h = net.host()
    for k in ("b1", "b2", "b3"):
        h[k] = rng.normal(0, 0.05, h[k].shape).astype(np.float32)
    h["W4"] = rng.normal(0, 0.2, h["W4"].shape).astype(np.float32)
    h["b4"] = np.array([0.01], np.float32)
    net.set_host(h)
    return net


def _oracle_params(R, net):
    h = net.host()
    return R.Params(h["W1"].reshape(32, 9, 8), h["b1"], h["W2"].reshape(32, 9, 32), h["b2"],
                    h["W3"].reshape(32, 9, 32), h["b3"], h["W4"].reshape(9, 32), h["b4"][0])


def _gpu_forward_values(R, ws, n, N):
    """The kernels' own activations as float64 values."""
    fw = {"X0": R.bf16_value(_bits(ws.X0, (N, 96, 96, 8))[:n]).astype(np.float64)}
    for i, key in enumerate(("h1", "h2", "h3")):
        fw[key] = R.bf16_value(_bits(ws.h[i], (N, 96, 96, 32))[:n]).astype(np.float64)
    fw["dphi"] = ws.dphi.cpu().numpy().reshape(N, 96, 96)[:n].astype(np.float64)
    return fw


def test_forward_matches_oracle(R, c1_after):
    """Each layer of the kernels against the oracle applied to the kernels'
    own input of that layer."""
    sim = c1_after
    n = 4
    say("forward pass, 4 crops, random weights, layer by layer")
    ws = su.Workspace(sim.N, sim.dev)
    su.crop_sim(sim, ws)
    net = _random_net(11)
    su.forward(net, ws, n)
    torch.cuda.synchronize()
    p = _oracle_params(R, net)
    fw = _gpu_forward_values(R, ws, n, sim.N)
    prev = fw["X0"]
    for key, W, b in (("h1", p.W1, p.b1), ("h2", p.W2, p.b2), ("h3", p.W3, p.b3)):
        o = R.bf16_bits(np.maximum(R.conv(prev, W, b), 0.0)).astype(np.int32)
        g = R.bf16_bits(fw[key]).astype(np.int32)
        diff = np.abs(g - o)
        say(f"{key}: {np.count_nonzero(diff)} of {diff.size} differ, at most {diff.max()} "
            f"bf16 ulp")
        # fp32 (kernel) against fp64 (oracle) accumulation: sums that cancel
        # to near zero can round to neighbouring bf16 values
        assert diff.max() <= 2 and np.count_nonzero(diff) <= 1e-3 * diff.size
        assert np.count_nonzero(o) > 0.1 * o.size
        prev = fw[key]
    ref = R.conv(fw["h3"], p.W4)[..., 0] + p.b4
    err = np.abs(fw["dphi"] - ref).max()
    say(f"dphi max abs error {err:.3e} (|dphi| max {np.abs(ref).max():.3e})")
    assert err <= 1e-5 * np.abs(ref).max() + 1e-7
    # end to end, the oracle's own forward pass stays close
    full = R.forward(fw["X0"], p)
    rel = np.linalg.norm(full["dphi"] - fw["dphi"]) / np.linalg.norm(full["dphi"])
    say(f"end-to-end dphi relative L2 {rel:.2e}")
    assert rel <= 1e-2


def test_fused_inference_from_cells_equals_buffers(c1_after):
    """pfh_sur_infer_cells (crops built inside the kernel) gives bit for bit
    the origins and predictions of pfh_sur_crop followed by pfh_sur_infer."""
    sim = c1_after
    net = _random_net(7)
    a = su.Workspace(sim.N, sim.dev, hidden=False)
    su.crop_sim(sim, a)
    su.infer(net, a, sim.N)
    b = su.Workspace(sim.N, sim.dev, hidden=False)
    b.pred.fill_(float("nan"))
    su.infer_cells(net, sim, b)
    torch.cuda.synchronize()
    assert torch.equal(a.origin, b.origin)
    assert torch.equal(a.dphi, b.dphi)
    assert torch.equal(a.pred, b.pred)


def _w4_hi_lo(w4):
    """The fused kernel's output-layer weights: bf16 hi + bf16 lo parts."""
    from oracle import sur_ref as R
    w = np.asarray(w4, np.float32)
    hi = R.bf16_value(R.bf16_bits(w))
    lo = R.bf16_value(R.bf16_bits((w - hi).astype(np.float32)))
    return hi.astype(np.float64) + lo.astype(np.float64)


def test_hardware_bf16_rounding(R):
    """The conversion the fused kernel applies to hidden activations rounds
    to nearest even like the oracle, on ties (both parities), values just
    off ties, subnormals, the largest finite values, infinities and signed
    zeros; NaN stays NaN."""
    from pfh import abi
    rng = np.random.default_rng(4)
    hi = rng.integers(0, 1 << 16, 4096, dtype=np.uint32) << 16
    special = []
    for h in (0x3F80, 0x3F81, 0x0001, 0x0080, 0x7F7F, 0xBF80, 0x8001):
        for lo in (0x0000, 0x7FFF, 0x8000, 0x8001, 0xFFFF):
            special.append((h << 16) | lo)
    special += [0x00000001, 0x007FFFFF, 0x80000001, 0x7F7FFFFF, 0x7F800000, 0xFF800000,
                0x00000000, 0x80000000, 0x7FC00000, 0x7F800001]
    bits = np.concatenate([hi | rng.integers(0, 1 << 16, 4096, dtype=np.uint32),
                           np.array(special, np.uint32)])
    if bits.size % 2:
        bits = np.append(bits, np.uint32(0))
    x = bits.view(np.float32)
    xt = torch.from_numpy(x.copy()).cuda()
    yt = torch.zeros(x.size, dtype=torch.int16, device="cuda")
    abi.check(abi.load().pfh_sur_round_bf16(xt.data_ptr(), yt.data_ptr(), x.size, None),
              "round_bf16")
    got = yt.cpu().numpy().view(np.uint16)
    want = R.bf16_bits(x)
    nan = np.isnan(x)
    assert np.array_equal(got[~nan], want[~nan])
    assert np.all(np.isnan(R.bf16_value(got[nan])))


def test_fused_inference_matches(R, c1_after):
    """pfh_sur_infer (all layers in one kernel) against the layer-by-layer
    kernels and the oracle; the crops are repeated 20 times (320 crops) so
    that workgroups walk several crops, and every copy must agree bit for bit."""
    sim = c1_after
    n0, rep = sim.N, 20
    n = n0 * rep
    say(f"fused inference, {n} crops ({n0} distinct), random weights")
    one = su.Workspace(n0, sim.dev)
    su.crop_sim(sim, one)
    ws = su.Workspace(n, sim.dev)
    ws.X0.copy_(one.X0.repeat(rep))
    ws.phic.copy_(one.phic.repeat(rep))
    net = _random_net(11)
    su.forward(net, ws, n)
    d_layer = ws.dphi.clone()
    ws.dphi.fill_(float("nan"))
    ws.pred.fill_(float("nan"))
    su.infer(net, ws, n)
    torch.cuda.synchronize()
    d = ws.dphi.view(rep, -1)
    assert torch.isfinite(d).all()
    assert torch.equal(d, d[:1].expand_as(d)), "copies of one crop differ"
    assert torch.equal(ws.pred, ws.phic + ws.dphi)
    df = d[0].double().cpu().numpy()
    dl = d_layer.view(rep, -1)[0].double().cpu().numpy()
    rel_layer = np.linalg.norm(df - dl) / np.linalg.norm(dl)
    p = _oracle_params(R, net)
    p.W4 = _w4_hi_lo(net.host()["W4"]).reshape(1, 9, 32)
    X0 = R.bf16_value(_bits(one.X0, (n0, 96, 96, 8))).astype(np.float64)
    ref = R.forward(X0, p)["dphi"].reshape(-1)
    rel_oracle = np.linalg.norm(df - ref) / np.linalg.norm(ref)
    say(f"dphi relative L2: {rel_layer:.2e} vs layer-by-layer kernels, {rel_oracle:.2e} vs "
        f"oracle")
    # hidden maps round to bf16 in both; rare one-ulp flips (fp32 sums in
    # another order) propagate to the output
    assert rel_layer <= 2e-3
    assert rel_oracle <= 1e-2


def test_backward_matches_oracle(R, c1_after):
    """Every gradient against the oracle's backward pass over the kernels'
    own forward activations."""
    sim = c1_after
    n = 2
    say("backward pass, 2 crops, random weights")
    ws = su.Workspace(n, sim.dev, train=True)
    full = su.Workspace(sim.N, sim.dev)
    su.crop_sim(sim, full)
    ws.X0.copy_(full.X0[:n * su.PIX * su.C0])
    net = _random_net(5)
    rng = np.random.default_rng(2)
    target = rng.normal(0, 0.5, (n, 96, 96)).astype(np.float32)
    tg = torch.from_numpy(target.reshape(-1)).to(sim.dev)
    su.forward(net, ws, n, pred=False)
    loss = float(su.backward(net, ws, n, tg))
    torch.cuda.synchronize()
    p = _oracle_params(R, net)
    fw = _gpu_forward_values(R, ws, n, n)
    g = R.backward(fw, target.astype(np.float64), p)
    assert abs(loss - g["loss"]) <= 1e-5 * g["loss"]
    gv = {k: v.cpu().numpy() for k, v in net.gviews.items()}
    for k in ("W4", "b4", "W3", "b3", "W2", "b2", "W1", "b1"):
        ref = np.asarray(g[k], np.float64).reshape(-1)
        got = gv[k].astype(np.float64).reshape(-1)
        if k == "W1":   # the four zero input channels carry no information
            ref = ref.reshape(32, 9, 8)[:, :, :4].reshape(-1)
            got = got.reshape(32, 9, 8)[:, :, :4].reshape(-1)
        rel = np.linalg.norm(got - ref) / max(np.linalg.norm(ref), 1e-30)
        say(f"grad {k}: relative error {rel:.2e}")
        assert rel <= 1e-2, k


def test_training_lowers_loss():
    say("training on C2-style crops: loss decreases")
    X, D = su.make_dataset([1000], samples_per_seed=1, warm=100)
    net = su.Net(seed=0)
    n = D.numel() // su.PIX
    held = 128
    Xt, Dt = X[:(n - held) * su.PIX * su.C0], D[:(n - held) * su.PIX]
    hist = su.train(net, Xt, Dt, epochs=10, batch=32, lr=2e-3)
    say(f"loss history {hist}")
    # held-out crops: the network's increment beats predicting no change
    ws = su.Workspace(held, net.dev)
    ws.X0.copy_(X[(n - held) * su.PIX * su.C0:])
    su.forward(net, ws, held, pred=False)
    d_true = D[(n - held) * su.PIX:].double()
    d_net = ws.dphi.double() * net.scale
    e_net = float(torch.linalg.norm(d_net - d_true))
    e_id = float(torch.linalg.norm(d_true))
    say(f"held-out increment error: network {e_net:.4e}, no-change {e_id:.4e}")
    assert hist[-1] < 0.7 * hist[0]
    assert e_net < 0.7 * e_id


def test_accepted_block_commits_exactly():
    """An accepted block (tolerance forced open) leaves the aggregate S and
    the cell moments exactly as the plain path's own kernels rebuild them
    from the written field (k_scatter_all / k_init_moments), and the check
    error is finite."""
    from pfh import abi
    wl = params.workload_c1()
    sim = sim2d.Sim2D(wl)
    sim.step(20)
    net = _random_net(3)
    runner = su.SurrogateRunner(sim, net, K=8, tol=1e30, fallback="population")
    say("one accepted block on C1, then rebuild S and moments")
    runner.block()
    st = runner.stats()
    assert st["fallback_blocks"] == 0 and st["accepted_blocks"] == 1
    assert torch.isfinite(runner.err).all()
    e = sim.steps_done
    lib = abi.load()
    S_ref = torch.zeros(sim.words, dtype=torch.int32, device=sim.dev)
    flags = torch.zeros_like(sim.flags)
    abi.check(lib.pfh2d_scatter_all(sim.phi[e % 2].data_ptr(), sim.cell.data_ptr(),
                                    sim.cls.data_ptr(), S_ref.data_ptr(), sim.N, sim.L, sim.P,
                                    flags.data_ptr(), None), "scatter_all")
    cell_ref = sim.cell.clone()
    abi.check(lib.pfh2d_init_moments(cell_ref.data_ptr(), sim.cls.data_ptr(),
                                     sim.phi[e % 2].data_ptr(), sim.N, None), "init_moments")
    torch.cuda.synchronize()
    assert torch.equal(sim.S_slot(e % 3), S_ref)
    assert torch.equal(sim.cell, cell_ref)
    assert int(sim.S_slot(e % 3).count_nonzero()) > 0
    # and the plain method continues from the committed state
    sim.step(2)
    sim.sync()
    assert not sim.fatal()


def test_committed_weights_accuracy_and_acceptance():
    """The committed weights on the 2048^2 / 1024-cell monolayer (seed 7,
    not a training seed): 10 surrogate blocks of 8 steps from step 300, every
    block accepted, the field within 1e-3 relative L2 of the plain run on
    every cell's crop window."""
    from pfh import surrogate_train as st
    assert su.WEIGHTS_PATH.exists(), su.WEIGHTS_PATH
    net = su.Net.load(su.WEIGHTS_PATH)
    say("committed weights: 10 blocks on C2 against the plain method")
    r = st.evaluate(net, blocks=10)
    say(f"accepted {r['accepted_blocks']}/{r['blocks']}, rel L2 vs plain max "
        f"{r['rel_l2_vs_plain_max']:.3e} mean {r['rel_l2_vs_plain_mean']:.3e}, "
        f"speedup {r['speedup']:.3f}")
    assert not r["fatal"]
    assert r["fallback_blocks"] == 0
    assert r["rel_l2_vs_plain_max"] <= 1e-3


def test_committed_k16_weights_accuracy_and_acceptance():
    """The committed 16-step weights: 6 blocks (96 steps) from step 300 on the
    2048^2 / 1024-cell monolayer, every block accepted, within 1e-3 relative
    L2 of the plain run."""
    from pfh import surrogate_train as st
    assert su.WEIGHTS_PATH_K16.exists(), su.WEIGHTS_PATH_K16
    net = su.Net.load(su.WEIGHTS_PATH_K16)
    assert net.K == 16
    say("committed K=16 weights: 6 blocks on C2 against the plain method")
    r = st.evaluate(net, blocks=6, K=16)
    say(f"accepted {r['accepted_blocks']}/{r['blocks']}, rel L2 vs plain max "
        f"{r['rel_l2_vs_plain_max']:.3e}, speedup {r['speedup']:.3f}")
    assert not r["fatal"]
    assert r["fallback_blocks"] == 0
    assert r["rel_l2_vs_plain_max"] <= 1e-3


def _state(sim):
    return [sim.phi[0], sim.phi[1], sim.S, sim.cell, sim.cls, sim.stepc, sim.cursor, sim.flags]


def test_graph_blocks_equal_eager_blocks():
    """Captured block graphs, replayed over four blocks (all three residues
    of the step mod 6, one of them twice) with eager work between the
    replays, leave the state bit for bit equal to eager launches, for
    accepted blocks and for rejected blocks (gated fallback steps)."""
    wl = params.workload_c1()
    net = _random_net(3)
    for tol in (1e30, 0.0):
        sa, sb = sim2d.Sim2D(wl), sim2d.Sim2D(wl)
        sa.step(10)
        sb.step(10)
        ra = su.SurrogateRunner(sa, net, tol=tol, graphs=False, fallback="population")
        rb = su.SurrogateRunner(sb, net, tol=tol, graphs=True, fallback="population")
        for b in range(4):
            say(f"tol {tol:g}: block {b} from step {sa.steps_done}")
            ra.block()
            rb.block()
            sta, stb = ra.stats(), rb.stats()
            assert sta == stb
            assert sta["fallback_blocks"] == (0 if tol > 1.0 else b + 1)
            assert sa.steps_done == sb.steps_done
            for x, y in zip(_state(sa), _state(sb)):
                assert torch.equal(x, y)
            assert torch.equal(ra.err, rb.err)
            # eager work between replays
            sb.S_slot(0).sum()
        assert not sa.fatal()


def test_rejected_block_equals_plain_steps():
    """A rejected block (tolerance 0) leaves exactly the state of K plain
    steps: the gated launches change nothing and the host runs the plain
    steps; four rejected blocks in one chunk equal 32 plain steps."""
    wl = params.workload_c1()
    net = _random_net(3)
    sa, sb = sim2d.Sim2D(wl), sim2d.Sim2D(wl)
    sa.step(12)
    sb.step(12)
    r = su.SurrogateRunner(sa, net, tol=0.0, chunk=8, fallback="population")
    r.run(32)
    sb.step(32)
    torch.cuda.synchronize()
    st = r.stats()
    assert st["fallback_blocks"] == 4 and st["blocks"] == 4
    assert sa.steps_done == sb.steps_done
    for x, y in zip(_state(sa), _state(sb)):
        assert torch.equal(x, y)


class _SwitchingRunner(su.SurrogateRunner):
    """Eager runner whose first `n_ok` blocks are accepted and the rest
    rejected (tolerance switched per issued block)."""

    def __init__(self, *a, n_ok=2, **k):
        super().__init__(*a, graphs=False, **k)
        self.n_issued = 0
        self.n_ok = n_ok

    def _issue(self, s):
        self.tol = 1e30 if self.n_issued < self.n_ok else 0.0
        self.n_issued += 1
        super()._issue(s)


def test_abort_inside_chunk():
    """A rejection in the third block of a four-block chunk: the blocks
    after it do nothing, the host runs its plain steps and re-issues the
    last block, and the state equals two accepted surrogate blocks followed
    by 16 plain steps."""
    wl = params.workload_c1()
    net = _random_net(3)
    sa, sb = sim2d.Sim2D(wl), sim2d.Sim2D(wl)
    sa.step(12)
    sb.step(12)
    ra = _SwitchingRunner(sa, net, n_ok=2, chunk=4, fallback="population")
    ra.run(32)
    rb = su.SurrogateRunner(sb, net, tol=1e30, graphs=False, chunk=1,
                            fallback="population")
    rb.run(16)
    sb.step(16)
    torch.cuda.synchronize()
    st = ra.stats()
    say(f"stats {st}")
    assert st["blocks"] == 4 and st["fallback_blocks"] == 2
    assert sa.steps_done == sb.steps_done == 12 + 32
    for x, y in zip(_state(sa), _state(sb)):
        assert torch.equal(x, y)


def test_check_step_equals_gated_plain_step():
    """The surrogate's check step (pfh2d_launch_check_step_if: no moments,
    scatter, support box or flags) writes the same new field, window
    positions and classes, bit for bit, as the full step on the same
    private copies, on the default grid and on two workgroups."""
    import ctypes as C
    from pfh import abi
    wl = params.workload_c1()
    sim = sim2d.Sim2D(wl)
    sim.step(20)
    runner = su.SurrogateRunner(sim, _random_net(3), K=8, tol=1e30, graphs=False)
    lib, sp, N = abi.load(), sim._sp(), sim.N
    s = sim.steps_done
    go = su._ptr(runner.ctl)
    now = su._ptr(sim.stepc) + 8 * (s % 2)
    abi.check(lib.pfh_sur_prep(go, go + 4, su._ptr(sim.cell), su._ptr(runner.cell_chk),
                               su._ptr(sim.cls), su._ptr(runner.cls_chk), N, None, 0,
                               su._ptr(runner.cur_chk), su._ptr(runner.step_chk), now, sp),
              "prep")
    torch.cuda.synchronize()
    priv = [runner.cell_chk, runner.cls_chk, runner.cur_chk, runner.step_chk, runner.flags_chk]
    start = [t.clone() for t in priv]
    for grid in (sim.grid, 2):
        outs = []
        for check in (False, True):
            for t, t0 in zip(priv, start):
                t.copy_(t0)
            runner.phi_chk.zero_()
            a = runner._check_args(s)
            say(f"{'check' if check else 'full'} step from step {s} on {grid} workgroups")
            if check:
                abi.check(lib.pfh2d_launch_check_step_if(C.byref(a), go, grid, sp), "check")
            else:
                abi.check(lib.pfh2d_launch_step_if(C.byref(a), go, grid, sp), "full")
            torch.cuda.synchronize()
            cells = runner.cell_chk.cpu().numpy().view(abi.CELL_DTYPE)
            outs.append((runner.phi_chk.clone(), cells[["gx0", "gy0", "cls"]].copy(),
                         runner.cls_chk.clone(), runner.cur_chk.clone(),
                         runner.step_chk.clone()))
        (pa, ca, la, ua, sa), (pb, cb, lb, ub, sb) = outs
        assert torch.equal(pa.view(torch.int32), pb.view(torch.int32))
        assert np.array_equal(ca, cb)
        assert torch.equal(la, lb)
        assert torch.equal(ua, ub) and torch.equal(sa, sb)
        assert float(pa.abs().max()) > 0.9
    # a check step refuses an aggregate to scatter into
    a = runner._check_args(s)
    a.S_sc = sim._s_ptr(0)
    assert lib.pfh2d_launch_check_step_if(C.byref(a), go, sim.grid, sp) != 0


def test_block_finish_equals_tumble_and_advance():
    """pfh_sur_finish (the K polarity draws and the counter advance in one
    launch) leaves theta, tumble_ctr and the step counters of an accepted
    block exactly as pfh_sur_tumble applied to the block's starting cell
    states from its first step, on the 2048^2 / 1024-cell monolayer."""
    from pfh import abi
    wl = params.workload_c2()
    sim = sim2d.Sim2D(wl)
    sim.step(20)
    runner = su.SurrogateRunner(sim, _random_net(3), K=8, tol=1e30, graphs=False)
    lib = abi.load()
    s = sim.steps_done
    cell0 = sim.cell.clone()
    step0 = sim.stepc.clone()
    say(f"one accepted block from step {s}, draws against pfh_sur_tumble")
    runner.block()
    torch.cuda.synchronize()
    assert runner.stats()["accepted_blocks"] == 1
    ref = cell0.clone()
    abi.check(lib.pfh_sur_tumble(ref.data_ptr(), sim.N, step0.data_ptr() + 8 * (s % 2), 8,
                                 sim.p.polarity_stream(), sim.p.p_tumble(), None, None),
              "tumble")
    torch.cuda.synchronize()
    got = sim.cells()
    want = ref.cpu().numpy().view(abi.CELL_DTYPE)
    assert np.array_equal(got["theta"].view(np.uint32), want["theta"].view(np.uint32))
    assert np.array_equal(got["tumble_ctr"], want["tumble_ctr"])
    assert torch.equal(sim.stepc, step0 + 8)
    start = cell0.cpu().numpy().view(abi.CELL_DTYPE)
    expected = sim.p.p_tumble() * 8 * sim.N
    say(f"tumbles in the block: {int((got['tumble_ctr'] - start['tumble_ctr']).sum())} "
        f"(expected about {expected:.1f})")
    if expected > 5:
        assert (got["tumble_ctr"] != start["tumble_ctr"]).any()


def test_cell_fallback_commits_the_check_field():
    """Per-cell fallback with every cell rejected (tolerance 0): each cell
    takes the check step's field, window position and class, S and the
    moments are rebuilt from the committed fields exactly as the plain
    path's own kernels rebuild them, and the block advances K steps."""
    from pfh import abi
    wl = params.workload_c1()
    sim = sim2d.Sim2D(wl)
    sim.step(20)
    runner = su.SurrogateRunner(sim, _random_net(3), tol=0.0, graphs=False)
    s0 = sim.steps_done
    runner.block()
    torch.cuda.synchronize()
    st = runner.stats()
    assert st["fallback_cells"] == sim.N and st["accepted_cell_fraction"] == 0.0
    e = sim.steps_done
    assert e == s0 + 8 and int(sim.stepc[e % 2].item()) == e
    chk_cells = runner.cell_chk.cpu().numpy().view(abi.CELL_DTYPE)
    cells = sim.cells()
    assert np.array_equal(cells["gx0"], chk_cells["gx0"])
    assert np.array_equal(cells["gy0"], chk_cells["gy0"])
    assert np.array_equal(cells["cls"], chk_cells["cls"])
    phi = sim.phi[e % 2].view(sim.N, -1)
    chk = runner.phi_chk.view(sim.N, -1)
    for n in range(sim.N):
        wx, wy, tx0, ty0 = abi.CLASSES[int(cells["cls"][n])]
        a = phi[n].view(abi.TILE_PITCH, -1)[ty0:ty0 + wy, tx0:tx0 + wx]
        b = chk[n].view(abi.TILE_PITCH, -1)[ty0:ty0 + wy, tx0:tx0 + wx]
        assert torch.equal(a, b), n
    lib = abi.load()
    S_ref = torch.zeros(sim.words, dtype=torch.int32, device=sim.dev)
    flags = torch.zeros_like(sim.flags)
    abi.check(lib.pfh2d_scatter_all(sim.phi[e % 2].data_ptr(), sim.cell.data_ptr(),
                                    sim.cls.data_ptr(), S_ref.data_ptr(), sim.N, sim.L, sim.P,
                                    flags.data_ptr(), None), "scatter_all")
    cell_ref = sim.cell.clone()
    abi.check(lib.pfh2d_init_moments(cell_ref.data_ptr(), sim.cls.data_ptr(),
                                     sim.phi[e % 2].data_ptr(), sim.N, None), "init_moments")
    torch.cuda.synchronize()
    assert torch.equal(sim.S_slot(e % 3), S_ref)
    assert torch.equal(sim.cell, cell_ref)
    sim.step(2)
    sim.sync()
    assert not sim.fatal()


def test_cell_larger_than_the_crop_is_rejected():
    """The per-cell check counts the check field outside the 96-pixel crop:
    with a prediction equal to the check field on the crop, cells of radius
    20 (support about 66 pixels) pass at 1e-3, cells of radius 45 (support
    about 116 pixels, wider than the crop) fail, since committing the crop
    would cut their field off."""
    from pfh import abi
    lib = abi.load()
    for R, want_rejected in ((20.0, 0), (45.0, 16)):
        wl = params.monolayer(16, 768, R, 4, 4.0, 7, name=f"r{R:g}")
        sim = sim2d.Sim2D(wl)
        sim.step(40)
        r = su.SurrogateRunner(sim, _random_net(3), tol=1e30, tol_inc=1e30, budget=1e30,
                               graphs=False)
        s = sim.steps_done
        r.block()          # leaves the block's check field and crop origins behind
        torch.cuda.synchronize()
        pred = torch.zeros_like(r.ws.pred)
        abi.check(lib.pfh_sur_recrop(r.phi_chk.data_ptr(), r.cell_chk.data_ptr(),
                                     r.cls_chk.data_ptr(), r.ws.origin.data_ptr(), sim.N, sim.L,
                                     pred.data_ptr(), None), "recrop")
        acc = torch.zeros(sim.N, dtype=torch.float32, device=sim.dev)
        err = torch.zeros_like(acc)
        accept = torch.zeros(sim.N, dtype=torch.int32, device=sim.dev)
        rej = torch.zeros(1, dtype=torch.int32, device=sim.dev)
        pin = s % 2
        abi.check(lib.pfh_sur_check_cells(
            r.phi_chk.data_ptr(), r.cell_chk.data_ptr(), r.cls_chk.data_ptr(),
            sim.phi[pin].data_ptr(), sim.cell.data_ptr(), sim.cls.data_ptr(),
            r.ws.origin.data_ptr(), sim.N, sim.L, pred.data_ptr(), 1e-3, 1e30, 1e30,
            acc.data_ptr(), err.data_ptr(), accept.data_ptr(), rej.data_ptr(), None, None),
            "check cells")
        torch.cuda.synchronize()
        say(f"R={R:g}: rejected {int(rej.item())}, errors {err.min().item():.2e}.."
            f"{err.max().item():.2e}")
        assert int(rej.item()) == want_rejected
        assert not sim.fatal()


def test_long_run_stays_within_tolerance_of_plain():
    """1000 steps (125 blocks of 8) of surrogate + per-cell fallback from
    step 300 of the 2048^2 / 1024-cell monolayer (seed 7, not a training
    seed): every cell's field stays within 1e-3 relative L2 of the plain
    run, with the accumulated-error budget bounding the drift."""
    from pfh import surrogate_train as st
    net = su.Net.load(su.WEIGHTS_PATH)
    r = st.evaluate(net, blocks=125)
    say(f"1000 steps: rel L2 vs plain max {r['rel_l2_vs_plain_max']:.3e} mean "
        f"{r['rel_l2_vs_plain_mean']:.3e}, accepted cells {r['accepted_cell_fraction']:.3f}, "
        f"speedup {r['speedup']:.3f}")
    assert not r["fatal"]
    assert r["steps"] == 1000
    assert r["rel_l2_vs_plain_max"] <= 1e-3
    assert r["accepted_cell_fraction"] > 0.0



def _bf16(x: torch.Tensor) -> torch.Tensor:
    return x.to(torch.bfloat16)


@pytest.mark.parametrize("cin,crops,shift", [(8, 1, 0), (8, 3, 1), (32, 2, 0), (32, 3, 1)])
def test_training_kernels_on_odd_batches(cin, crops, shift):
    """The convolution (Y and the mask aligned for 16 B accesses or one
    element off), the weight gradients and the output layer's backward on 1-3
    crops, against plain fp64 sums on the CPU: corners, edges and every
    32-pixel block boundary included. Bounds: bf16 results one rounding
    (2^-8 of the value) plus fp32 sums; sums of n fp32 terms n 2^-24 of the sum
    of their magnitudes."""
    from pfh import abi
    lib, dev = abi.load(), "cuda:0"
    gen = torch.Generator().manual_seed(100 * cin + crops)
    rnd = lambda *s: _bf16(torch.randn(*s, generator=gen))          # noqa: E731
    X, W = rnd(crops, 96, 96, cin), _bf16(rnd(32, 9, cin) * 0.1)
    dY, H = rnd(crops, 96, 96, 32), rnd(crops, 96, 96, 32)
    bias, g = torch.randn(32, generator=gen), torch.randn(crops, 96, 96, generator=gen)
    W4 = torch.randn(9, 32, generator=gen)
    up = lambda t: t.contiguous().to(dev)                            # noqa: E731

    def taps(a):                         # [9, crops, 96, 96, c], a at p + off(tap)
        p = torch.nn.functional.pad(a.double(), (0, 0, 1, 1, 1, 1))
        return torch.stack([p[:, ky:ky + 96, kx:kx + 96] for ky in range(3) for kx in range(3)])

    # convolution, ReLU and mask
    Xd, Wd, bd = up(X), up(W), up(bias)
    room = torch.zeros(dY.numel() + 8, dtype=torch.bfloat16, device=dev)
    mask_room = torch.zeros_like(room)
    Y = room[shift:shift + dY.numel()]
    mask = mask_room[shift:shift + dY.numel()]
    mask.copy_(up(H).view(-1))
    abi.check(lib.pfh_sur_conv(cin, Xd.data_ptr(), Wd.data_ptr(), bd.data_ptr(),
                               mask.data_ptr(), Y.data_ptr(), crops, 1, None), "conv")
    xt = taps(X)
    ref = torch.einsum("tnyxi,oti->nyxo", xt, W.double()) + bias.double()
    mag = torch.einsum("tnyxi,oti->nyxo", xt.abs(), W.double().abs()) + bias.double().abs()
    ref = torch.where(H.double() > 0, ref, 0.0).clamp(min=0.0)
    err = (Y.view(ref.shape).cpu().double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + mag * (9 * cin * 2.0 ** -24)).all())
    assert float(room[:shift].abs().sum()) == 0.0 and float(room[shift + dY.numel():].abs().sum()) == 0.0

    # weight gradient, per crop
    width = 32 * 9 * cin + 32
    part = torch.zeros(crops * width, dtype=torch.float32, device=dev)
    dYd = up(dY)
    abi.check(lib.pfh_sur_wgrad(cin, dYd.data_ptr(), Xd.data_ptr(), part.data_ptr(), crops,
                                None), "wgrad")
    got = part.cpu().double().view(crops, width)
    dw = torch.einsum("nyxo,tnyxi->noti", dY.double(), xt)
    dm = torch.einsum("nyxo,tnyxi->noti", dY.double().abs(), xt.abs())
    lim = 9216 * 2.0 ** -24
    assert bool(((got[:, :-32].view(dw.shape) - dw).abs() <= lim * dm).all())
    db, bm = dY.double().sum((1, 2)), dY.double().abs().sum((1, 2))
    assert bool(((got[:, -32:] - db).abs() <= lim * bm).all())

    # output layer's backward
    gd, Hd, W4d = up(g), up(H), up(W4)
    dH = torch.zeros_like(Hd)
    p4 = torch.zeros(crops * 289, dtype=torch.float32, device=dev)
    abi.check(lib.pfh_sur_out_bwd(gd.data_ptr(), Hd.data_ptr(), W4d.data_ptr(), dH.data_ptr(),
                                  p4.data_ptr(), crops, None), "out_bwd")
    gt = taps(g[..., None]).flip(0)[..., 0]                          # g at q - off(tap)
    ref = torch.einsum("tnyx,tc->nyxc", gt, W4.double())
    mag = torch.einsum("tnyx,tc->nyxc", gt.abs(), W4.double().abs())
    ref = torch.where(H.double() > 0, ref, 0.0)
    err = (dH.cpu().double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + mag * (9 * 2.0 ** -24)).all())
    got = p4.cpu().double().view(crops, 289)
    dw4 = torch.einsum("tnyx,nyxc->ntc", gt, H.double())
    m4 = torch.einsum("tnyx,nyxc->ntc", gt.abs(), H.double().abs())
    assert bool(((got[:, :-1].view(dw4.shape) - dw4).abs() <= lim * m4).all())
    assert bool(((got[:, -1] - g.double().sum((1, 2))).abs()
                 <= lim * g.double().abs().sum((1, 2))).all())

    # the reduction over crops keeps the ascending order
    out = torch.zeros(289, dtype=torch.float32, device=dev)
    many = torch.randn(37 * 289, generator=gen).to(dev)
    abi.check(lib.pfh_sur_reduce(many.data_ptr(), 37, 289, out.data_ptr(), None), "reduce")
    acc = torch.zeros(289)
    for row in many.cpu().view(37, 289):
        acc = acc + row
    assert torch.equal(out.cpu(), acc)


@pytest.mark.parametrize("per_cell", [False, True])
def test_commit_in_one_call_equals_commit_in_parts(per_cell):
    """A population of more cells than compute units and its halves of fewer
    take different builds of the commit: the same fields, moments, aggregate
    and flags, over every class, with zeros, a value beyond the clamp and a
    NaN among the predictions, accepted and rejected cells."""
    from pfh import abi
    lib, dev = abi.load(), "cuda:0"
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    N, L, P, area = cus + 5, 1024, 1024, abi.TILE_AREA
    rng = np.random.default_rng(17)
    cells = np.zeros(N, abi.CELL_DTYPE)
    cells["gx0"], cells["gy0"] = rng.integers(0, L, (2, N))
    chk = cells.copy()
    chk["gx0"], chk["gy0"] = (cells["gx0"] + 2) % L, (cells["gy0"] - 1) % L
    cls, cls_chk = rng.integers(0, 6, (2, N)).astype(np.uint8)
    centre = np.array([72, 88, 72, 80, 112, 143])[cls]
    origin = np.stack([(cells["gx0"] + centre - 48) % L, (cells["gy0"] + centre - 48) % L], 1)
    pred = (0.05 * rng.random((N, 9216))).astype(np.float32)
    pred[:, ::7] = 0.0
    pred[3, 100], pred[N - 3, 200] = 2.5, np.nan
    accept = (rng.random(N) < 0.6).astype(np.int32)
    phi = (0.02 * rng.random((N, area))).astype(np.float32)
    phi_chk = (0.03 * rng.random((N, area))).astype(np.float32)
    up = lambda a: torch.from_numpy(                                          # noqa: E731
        np.ascontiguousarray(a).view(np.uint8).reshape(-1)).to(dev)
    fixed = [up(origin.astype(np.int32)), up(pred), up(accept), up(phi_chk), up(chk), up(cls_chk)]

    def commit(parts):
        d_phi, d_cells, d_cls = up(phi), up(cells), up(cls)
        S = torch.zeros(L * P, dtype=torch.int32, device=dev)
        flags = torch.zeros(abi.FLAG_COUNT, dtype=torch.int32, device=dev)
        for lo, hi in parts:
            at = lambda t: t.data_ptr() + lo * (t.numel() // N)                        # noqa: E731
            og, pr, ac, pc, cc, kc = (at(t) for t in fixed)
            if per_cell:
                abi.check(lib.pfh_sur_commit_cells(
                    at(d_phi), at(d_cells), at(d_cls), og, pr, ac, pc, cc, kc, 1, hi - lo, L, P,
                    S.data_ptr(), flags.data_ptr(), None), "commit_cells")
            else:
                abi.check(lib.pfh_sur_commit(at(d_phi), at(d_cells), at(d_cls), og, pr, hi - lo,
                                             L, P, S.data_ptr(), flags.data_ptr(), None, None),
                          "commit")
        return [t.cpu().numpy() for t in (d_phi, d_cells, d_cls, S, flags)]

    say(f"commit of {N} cells on {cus} compute units, per cell: {per_cell}")
    whole, parts = commit([(0, N)]), commit([(0, N // 2), (N // 2, N)])
    assert all(np.array_equal(a, b) for a, b in zip(whole, parts))
    assert whole[4].any()
    V = whole[1].view(abi.CELL_DTYPE)["V"]
    assert np.isnan(V).sum() == (1 if not per_cell or accept[N - 3] else 0)
    assert (V[~np.isnan(V)] > 0.0).all()


@pytest.mark.parametrize("cin", [8, 32])
def test_weight_gradient_of_values_that_are_not_finite(cin):
    """Infinities and NaN among the inputs, in rows on every side of the edges
    between the rows of two waves (12 rows each) and of the crop: an entry of
    the gradient is infinite, NaN or finite exactly where the sum of its own
    products is (finite ones within n 2^-24 of the sum of magnitudes, n fp32
    terms)."""
    from pfh import abi
    lib, dev = abi.load(), "cuda:0"
    gen = torch.Generator().manual_seed(cin)
    X, dY = (_bf16(torch.randn(5, 96, 96, c, generator=gen)) for c in (cin, 32))
    for n, (y, px, ch, v) in enumerate([(0, 3, 1, np.inf), (11, 95, 2, -np.inf), (12, 0, 3, np.inf),
                                        (95, 32, 0, np.nan)]):
        X[n, y, px, ch] = v
    dY[4, 24, 31, 7] = np.inf
    say(f"weight gradients of values that are not finite, {cin} channels")
    width = 32 * 9 * cin + 32
    part = torch.zeros(5 * width, dtype=torch.float32, device=dev)
    dYd, Xd = dY.to(dev), X.to(dev)
    abi.check(lib.pfh_sur_wgrad(cin, dYd.data_ptr(), Xd.data_ptr(), part.data_ptr(), 5, None),
              "wgrad")
    got = part.cpu().double().view(5, width)[:, :-32].reshape(5, 32, 9, cin)
    p = torch.nn.functional.pad(X.double(), (0, 0, 1, 1, 1, 1))
    taps = [p[:, ky:ky + 96, kx:kx + 96].reshape(5, 9216, cin)
            for ky in range(3) for kx in range(3)]
    dy = dY.double().reshape(5, 9216, 32).transpose(1, 2).contiguous()
    ref = torch.stack([torch.bmm(dy, t) for t in taps], 2)
    mag = torch.stack([torch.bmm(dy.abs(), t.abs()) for t in taps], 2)
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isposinf(), ref.isposinf())
    assert torch.equal(got.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    assert 0 < int((~ok).sum()) < ok.numel() // 4
    assert bool(((got - ref).abs()[ok] <= 9216 * 2.0 ** -24 * mag[ok]).all())


def test_output_gradient_of_weights_that_are_not_finite():
    """Infinite and NaN weights of the output layer reach a pixel only through
    a tap that lies in the crop: the gradient is infinite, NaN or finite
    exactly where the sum of its own products is (finite ones within one bf16
    rounding and the sums' 9 x 2^-24 of the magnitudes)."""
    from pfh import abi
    lib, dev = abi.load(), "cuda:0"
    gen = torch.Generator().manual_seed(4)
    g, W4 = torch.randn(2, 96, 96, generator=gen), torch.randn(9, 32, generator=gen)
    H = _bf16(torch.randn(2, 96, 96, 32, generator=gen))
    for t, ch, v in [(0, 3, np.inf), (8, 5, np.nan), (2, 7, -np.inf), (6, 7, np.inf),
                     (4, 9, np.inf)]:
        W4[t, ch] = v
    say("output gradients of weights that are not finite")
    dH = torch.zeros_like(H, device=dev)
    part = torch.zeros(2 * 289, dtype=torch.float32, device=dev)
    gd, Hd, Wd = g.to(dev), H.to(dev), W4.to(dev)
    abi.check(lib.pfh_sur_out_bwd(gd.data_ptr(), Hd.data_ptr(), Wd.data_ptr(), dH.data_ptr(),
                                  part.data_ptr(), 2, None), "out_bwd")
    ref = torch.zeros(2, 96, 96, 32, dtype=torch.float64)
    mag = torch.zeros_like(ref)
    for t in range(9):
        dy, dx = t // 3 - 1, t % 3 - 1                   # g at q - off(t)
        q = (slice(None), slice(max(dy, 0), 96 + min(dy, 0)), slice(max(dx, 0), 96 + min(dx, 0)))
        s = (slice(None), slice(max(-dy, 0), 96 + min(-dy, 0)),
             slice(max(-dx, 0), 96 + min(-dx, 0)))
        term = g.double()[s][..., None] * W4.double()[t]
        ref[q] += term
        mag[q] += term.abs()
    on = H.double() > 0                                  # masked entries are exactly zero
    ref, mag = torch.where(on, ref, 0.0), torch.where(on, mag, 0.0)
    got = dH.cpu().double()
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isposinf(), ref.isposinf())
    assert torch.equal(got.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    lim = ref.abs() * 2.0 ** -8 + mag * (9 * 2.0 ** -24)
    assert bool(((got - ref).abs()[ok] <= lim[ok]).all())
    assert bool(ok[:, 95, :, 3].all()) and not bool(ok[:, :95, :95, 3].all())   # tap (0, 0)
