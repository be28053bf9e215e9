// gfx950 kernels of the 2D per-cell phase-field update and their C ABI.
//
// The step is one persistent work-queue launch: two 8-wave workgroups per
// compute unit, or one of 16 waves where a cell would mostly be alone on its
// unit (one_cell_per_unit), take cells from a device cursor (reference
// step_body, src/kernels.cu:948-1024) and advance one cell at a time through:
//   A  a column walk with a 3x3 register stencil over rows that each wave
//      stages in LDS for itself; it gives the interaction integral terms and,
//      for every pixel, the passive right-hand side, which stays in VGPRs;
//   -  fixed-order fp64 reduction (64-lane tree, 16 logical waves ascending)
//      of the interaction integral and the cell velocity;
//   B  the explicit Euler update from the held terms plus advection, the
//      shifted store, the Q5.27 scatter into the next S with integer atomics,
//      and the moments/support/phi_max of the stored field;
//   -  a second fixed-order reduction and the CellState commit.
// Classes 0-3 take this walk; the rare classes 4 (224x224) and 5 (fallback)
// read the tile from global memory.
//
// Arithmetic: binary32 operations in the reference's order, each
// product-and-add of the update fused by an explicit fmaf (passive_head_of,
// with_repulsion, euler_update) and nothing contracted beyond that (the build
// passes -ffp-contract=off), fp64 reductions, Q5.27 integer scatter.
// Reference: process_cell src/kernels.cu:53-592, process_cell_fallback
// :604-937, init/verify/pack/morton :1044-1302.

#include <hip/hip_runtime.h>

#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "../../include/pfh.h"
#include "pfh_device.h"
#include "pfh_host.h"

namespace pfh {

// Control block written by thread 0 and read by the workgroup.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct Ctl {
    int sx, sy, gx0, gy0, gx0n, gy0n, dcls, zero_tile, fm, pctr, tumbled;
    int dwx, dwy, dtx0, dty0, no_margin;
    float gam, dwC, volC, vA, cosp, sinp, theta, mrel, vx, vy;
    // spatial velocity observer: 2 / V and the centroid of the step's input
    // (include/fused_moments.cuh:16-21)
    double og2iv, ocx, ocy;
};

// The cell a workgroup processes next: filled by the control wavefront
// during the previous cell, double-buffered.
struct Slot {
    int n, cls;
    Ctl ctl;
    // the cell's domain in a batched step: side, S pitch and the word
    // offset of its replica's S in each slot arena
    int L, P, s_off_lo, s_off_hi;
};

struct Smem {
    // LDS copy of the step arguments: the cell bodies make the few they use
    // per row wave-uniform; held in scalar registers all 54 words would spill
    pfh2d_step_args args;
    double vel[kWaves * 8];      // wave sums before the velocity
    double red[kWaves * 4];      // wave sums of the commit
    int ired[kWaves * 8];
    Slot slot[2];
    uint32_t csraw[2][48];       // CellState (192 B) of the next cell
    const pfh2d_replica* reps;   // batched step only: replica table
    const uint16_t* cell_rep;    // batched step only: replica of each cell
    int fm;                      // full-moment step (one in full_moment_every)
};

// The scalars of the next cell run on lane 0 of wave 1 (wave 0 fetches and
// commits).
constexpr int kScalarsThread = kWave;
constexpr int kFetchLanes = 48;                       // dwords of a CellState

#define PFH_LDS __attribute__((address_space(3)))

// threadIdx.x made opaque inside the persistent loop: without this, LICM
// hoists every per-thread index and address of the cell body out of the loop
// and keeps them all live (and spilled) across cells.
__device__ __forceinline__ int opaque_tid() {
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ __forceinline__ void flag_add(uint32_t* flags, int i, uint32_t v) {
    atomicAdd(&flags[i], v);
}
__device__ __forceinline__ void flag_or(uint32_t* flags, int i) {
    atomicOr(&flags[i], 1u);
}

// Barriers on the staged path order LDS only (lds_barrier): every value one
// thread passes to another there goes through LDS, and each thread's global
// stores and scatters are read back, if at all, by the same thread.

// Global (address space 1) views of the hot buffers: pointers read out of the
// argument struct are otherwise generic, and flat instructions would tie every
// LDS wait to outstanding memory operations.
#define PFH_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ PFH_GLOBAL T* gptr(T* p) {
    return (PFH_GLOBAL T*)p;
}
__device__ __forceinline__ uint32_t atomic_add_g(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_add(gptr(p), v, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
}

// The step arguments cell_scalars reads, passed by value so that the kernel
// argument block never has its address taken (which copies it to scratch).
struct ScalarArgs {
    const pfh_cell_state* cell;
    uint32_t* flags;
    unsigned long long polarity_seed;
    double p_tumble, vol_scale, A0;
    float bulk_scale;
    int L, parity_out;
    int fm;              // this launch's step is a full-moment step
};

__device__ __forceinline__ ScalarArgs scalar_args(const pfh2d_step_args& A, int fm) {
    ScalarArgs s;
    s.cell = A.cell;
    s.flags = A.flags;
    s.polarity_seed = A.polarity_seed;
    s.p_tumble = A.p_tumble;
    s.vol_scale = A.vol_scale;
    s.A0 = A.A0;
    s.bulk_scale = A.bulk_scale;
    s.L = A.L;
    s.parity_out = A.parity_out;
    s.fm = fm;
    return s;
}

// Per-cell scalars: tumble, polarity, coefficients, class hysteresis and the
// recentring shift (src/kernels.cu:93-191 and :624-711), from a copy of the
// cell's state. Out of line: its double-precision polynomial constants must
// not be hoisted out of the persistent loop into the update's registers.
__device__ __noinline__ void cell_scalars(const ScalarArgs A, const pfh_cell_state* csp,
                                         int CLS, unsigned long long step, Ctl* ctl) {
    const int WX = shape_of(CLS).wx, WY = shape_of(CLS).wy;
    const pfh_cell_state& cs = *csp;
    const Philox4 r = philox4x32_10(
        (uint32_t)(step & 0xFFFFFFFFull), (uint32_t)(step >> 32),
        (uint32_t)cs.global_id, 0xA5A5A5A5u,
        (uint32_t)(A.polarity_seed & 0xFFFFFFFFull),
        (uint32_t)(A.polarity_seed >> 32));
    float theta = cs.theta;
    int tumbled = 0;
    if (uniform53(r.v[0], r.v[1]) < A.p_tumble) {
        theta = (float)(2.0 * kPi * uniform53(r.v[2], r.v[3]));
        tumbled = 1;
    }
    double sd, cd;
    sincos_d((double)theta, &sd, &cd);
    const float gam = cs.gamma;
    const float dwC = A.bulk_scale * gam;
    const float volC = (float)(A.vol_scale * (A.A0 - cs.V));
    const float mrel = cs.M_pf * (float)(1.0 / 0.5);
    // the centroid (also the observers' reference point)
    const double cxr = cs.Cx / cs.V;
    const double cyr = cs.Cy / cs.V;
    ctl->og2iv = 2.0 / cs.V;
    ctl->ocx = cxr;
    ctl->ocy = cyr;

    const int ex = cs.bb_hi_x - cs.bb_lo_x + 1;
    const int ey = cs.bb_hi_y - cs.bb_lo_y + 1;
    int dcls = CLS, no_margin = 0;
    unsigned pctr = cs.promote_ctr;
    if (ex > 0) {
        if (ex + kPromoteSlack > WX || ey + kPromoteSlack > WY) {
            int grow = class_containing(ex, ey, kPromoteSlack);
            // a window must lie strictly inside the periodic domain: classes
            // as wide as the side are unavailable (the batched step's
            // 256-pixel replicas run without the 286-pixel fallback class)
            if (grow >= 0 && max(shape_of(grow).wx, shape_of(grow).wy) >= A.L) grow = -1;
            if (grow >= 0) {
                dcls = grow;
            } else if (CLS == kClassFallback && ex <= WX && ey <= WY) {
                no_margin = 1;
            } else {
                flag_add(A.flags, PFH_FLAG_CLASS_EXHAUSTED, 1u);
            }
            pctr = 0u;
        } else {
            const int small = class_containing(ex, ey, kDemoteSlack);
            if (small >= 0 && small != CLS &&
                shape_of(small).wx * shape_of(small).wy < WX * WY) {
                if (++pctr >= (unsigned)kDemoteDwell) { dcls = small; pctr = 0u; }
            } else {
                pctr = 0u;
            }
        }
    }
    const Shape dc = shape_of(dcls);
    int sx = 0, sy = 0;
    if (cs.V > 0.0) {
        sx = __double2int_rn(cxr - 0.5 * (double)(dc.wx - 1));
        sy = __double2int_rn(cyr - 0.5 * (double)(dc.wy - 1));
        if (dcls == CLS) {
            sx = max(-kMaxShiftPerStep, min(kMaxShiftPerStep, sx));
            sy = max(-kMaxShiftPerStep, min(kMaxShiftPerStep, sy));
        } else {
            sx = max(-WX, min(WX, sx));
            sy = max(-WY, min(WY, sy));
        }
    } else {
        flag_or(A.flags, PFH_FLAG_V_NONPOS);
    }
    ctl->sx = sx;
    ctl->sy = sy;
    ctl->gx0 = cs.gx0;
    ctl->gy0 = cs.gy0;
    ctl->gx0n = wrapi(cs.gx0 + sx, A.L);
    ctl->gy0n = wrapi(cs.gy0 + sy, A.L);
    ctl->dcls = dcls;
    ctl->zero_tile = (dcls != (int)cs.cls_written[A.parity_out]);
    ctl->fm = A.fm;
    ctl->pctr = (int)pctr;
    ctl->tumbled = tumbled;
    ctl->dwx = dc.wx;
    ctl->dwy = dc.wy;
    ctl->dtx0 = dc.tx0;
    ctl->dty0 = dc.ty0;
    ctl->no_margin = no_margin;
    ctl->gam = gam;
    ctl->dwC = dwC;
    ctl->volC = volC;
    ctl->vA = cs.v_A;
    ctl->cosp = (float)cd;
    ctl->sinp = (float)sd;
    ctl->theta = theta;
    ctl->mrel = mrel;
}

// Zero every tile pixel outside the destination window (class change). The
// window itself is fully rewritten by the update, so no ordering is needed.
template <int NT>
__device__ void zero_outside_window(float* tile, int dwx, int dwy, int dtx0,
                                    int dty0) {
    for (int i = opaque_tid(); i < kTileArea; i += NT) {
        const int x = i % kTilePitch, y = i / kTilePitch;
        if (!((unsigned)(x - dtx0) < (unsigned)dwx &&
              (unsigned)(y - dty0) < (unsigned)dwy))
            tile[i] = 0.0f;
    }
}

// ---- velocity observers (include/fused_moments.cuh:23-127,
// common/velocity_moments.h:42-100). Observation mode kObs: 0 none,
// 1 advection, 2 spatial. Nothing here changes the step's physics. ----

// Per-lane sums of the spatial observer: the interfacial (gx, gy) and
// overlap (kx, ky) centroid rates and the same-cell neighbour overlaps
// sum phi phi_east, sum phi phi_north (bx, by).
struct ObsSums {
    double gx = 0.0, gy = 0.0, kx = 0.0, ky = 0.0, bx = 0.0, by = 0.0;
};

// One pixel of the spatial observer (RelaxMoments::pixel,
// include/fused_moments.cuh:36-53, and the beta sums of
// src/kernels.cu:287-291): the pixel's weight 2 phi / V times its passive
// interfacial and overlap sources, in fp64 from the binary32 stencil, times
// its offset from the input centroid (g2iv = 2 / V, cx, cy).
__device__ __forceinline__ void observe_pixel(ObsSums& o, int x, int y, float c, float e,
                                              float w, float nn, float ss, float ne, float nw,
                                              float se, float sw, float other, float gam,
                                              float dwC, float repC, double g2iv, double cx,
                                              double cy) {
    const double v = (double)c;
    const double axial = (((double)nn + (double)ss) + (double)e) + (double)w;
    const double lap =
        (((((4.0 * axial + (double)ne) + (double)nw) + (double)se) + (double)sw) - 20.0 * v) /
        6.0;
    const double weight = g2iv * v;
    const double well = (((double)dwC * v) * (1.0 - v)) * (1.0 - 2.0 * v);
    const double interfacial = weight * ((double)gam * lap - well);
    const double dx = (double)x - cx, dy = (double)y - cy;
    o.gx += dx * interfacial;
    o.gy += dy * interfacial;
    const double overlap = (((-weight) * (double)repC) * v) * (double)other;
    o.kx += dx * overlap;
    o.ky += dy * overlap;
    o.bx += v * (double)e;
    o.by += v * (double)nn;
}

// Discrete linear-interpolation correction of a held rate
// (common/velocity_moments.h:80-85).
__device__ __forceinline__ double linear_correction(double dt, unsigned long long steps,
                                                    double first, double last) {
    return steps ? dt * 0.5 * (double)(steps - 1ull) * (last - first) : 0.0;
}

// Thread 0 after the velocity: the advection record of the step
// (record_advection, include/fused_moments.cuh:96-127) and, on a spatial
// step, the sample's bookkeeping (begin_spatial_sample,
// common/velocity_moments.h:59-77) and the new held rates
// (RelaxMoments::finish, include/fused_moments.cuh:55-88). red holds the
// wave sums: slots 2, 3 the neighbour overlaps, 4-7 gx, gy, kx, ky.
template <int kObs>
__device__ void record_observers(const pfh2d_step_args& A, int n, const Ctl& c, double sIx,
                                 double sIy, const double* red) {
    pfh_cell_state* cs = &A.cell[n];
    pfh_advection_accum& a = cs->advection;
    const double ax = (double)c.vA * (double)c.cosp;
    const double ay = (double)c.vA * (double)c.sinp;
    const double ix = (double)A.mot_coeff * sIx;
    const double iy = (double)A.mot_coeff * sIy;
    const double dt = A.physical_dt;
    if constexpr (kObs == 2) {
        pfh_moment_accum& m = A.moments[n];
        const double tot[4] = {a.q[0] + a.q[2], a.q[1] + a.q[3], a.q[4], a.q[5]};
        const unsigned long long interval = a.count - m.last_sample;
        if (m.spatial_count) {
            for (int j = 0; j < 4; ++j) m.q[4 + j] += (dt * (double)interval) * m.held[j];
            for (int xy = 0; xy < 2; ++xy) {
                const double beta = m.held[4 + xy];
                m.q[10 + xy] += (beta - 1.0) * (tot[xy] - m.last_totals[xy]) +
                                beta * (tot[2 + xy] - m.last_totals[2 + xy]);
            }
        }
        for (int j = 0; j < 4; ++j) m.last_totals[j] = tot[j];
        m.last_interval = interval;
        m.last_sample = a.count;
        ++m.spatial_count;
        double bx = 0.0, by = 0.0;
        for (int w = 0; w < kWaves; ++w) {
            bx += red[w * 8 + 2];
            by += red[w * 8 + 3];
        }
        m.held[4] = bx / cs->V;
        m.held[5] = by / cs->V;
    }
    a.q[0] += dt * ax;
    a.q[1] += dt * ay;
    a.q[2] += dt * ix;
    a.q[3] += dt * iy;
    a.q[4] += dt * (((double)c.vx - ax) - ix);
    a.q[5] += dt * (((double)c.vy - ay) - iy);
    ++a.count;
    if constexpr (kObs == 2) {
        pfh_moment_accum& m = A.moments[n];
        const double mrel = (double)cs->M_pf / 0.5;
        for (int j = 0; j < 4; ++j) {
            double rate = 0.0;
            for (int w = 0; w < kWaves; ++w) rate += red[w * 8 + 4 + j];
            // only the passive rates are held here; the area source has an
            // exactly zero centroid moment
            if (mrel != 1.0) rate *= mrel;
            if (m.spatial_count > 1)
                m.correction[j] += linear_correction(dt, m.last_interval, m.held[j], rate);
            m.held[j] = rate;
        }
    }
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// The spatial observer's wave sums (slots 2-7 of a logical wave's row).
__device__ __forceinline__ void publish_observer(Smem& sm, int lw, const ObsSums& ob) {
    const double v[2] = {wave_sum4(ob.bx, ob.by, ob.gx, ob.gy),
                         wave_sum4(ob.kx, ob.ky, ob.kx, ob.ky)};
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int j = 2 * ((lane >> 4) & 1) + (lane >> 5);   // lanes 0, 32, 16, 48: 0..3
    if ((lane & 15) == 0) {
        sm.vel[lw * 8 + 2 + j] = v[0];
        if (j < 2) sm.vel[lw * 8 + 6 + j] = v[1];
    }
}

// The wave sums of the interaction integral of a wave's VW logical waves.
template <int NW, int VW>
__device__ __forceinline__ void publish_velocity(Smem& sm, int wave, const double (&aIx)[VW],
                                                 const double (&aIy)[VW]) {
    const double v = wave_sum4(aIx[0], aIy[0], aIx[VW - 1], aIy[VW - 1]);
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int lw = wave + NW * (VW > 1 ? (lane >> 4) & 1 : 0);
    if ((lane & 15) == 0 && (VW > 1 || (lane & 16) == 0)) sm.vel[lw * 8 + (lane >> 5)] = v;
}

// Velocity from the interaction integral (src/kernels.cu:300-342), after the
// barrier that orders the wave sums: every wave adds the 16 wave sums in order
// itself, x on its even lanes and y on its odd ones (no second barrier to hand
// the result out); thread 0 and 1 store them, thread 0 runs the observer.
template <int kObs = 0>
__device__ __forceinline__ void finish_velocity(const pfh2d_step_args& A, int n, Smem& sm,
                                                Ctl& c, float& vx, float& vy) {
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int xy = lane & 1;
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += sm.vel[w * 8 + xy];
    const double vd = (double)c.vA * (double)(xy ? c.sinp : c.cosp)
                    + (double)A.mot_coeff * s;
    const uint32_t v = __float_as_uint((float)vd);
    vx = __uint_as_float(__builtin_amdgcn_readlane(v, 0));
    vy = __uint_as_float(__builtin_amdgcn_readlane(v, 1));
    if (threadIdx.x < 2) {
        pfh_cell_state* cs = &A.cell[n];
        (xy ? cs->vy : cs->vx) = __uint_as_float(v);
        (xy ? cs->Iy : cs->Ix) = s;
    }
    if constexpr (kObs != 0) {
        const double sIy = readlane_f64(s, 1);
        if (threadIdx.x == 0) {
            c.vx = vx;
            c.vy = vy;
            record_observers<kObs>(A, n, c, s, sIy, sm.vel);
        }
    }
}

// One logical wave's part of the commit: a lane's moments, support rows and
// phi_max, and the wave's support columns.
struct Part {
    double V = 0.0, Cx = 0.0, Cy = 0.0;
    int blox, bhix;                  // uniform
    int bloy, bhiy, pmaxb;
};
__device__ __forceinline__ void publish_part(Smem& sm, int lw, const Part& p) {
    const double m = wave_sum4(p.V, p.Cx, p.Cy, 0.0);
    const int b = wave_tree4(-p.bloy, p.bhiy, p.pmaxb, 0,
                             [](int x, int y) { return max(x, y); });
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int j = 2 * ((lane >> 4) & 1) + (lane >> 5);   // lanes 0, 32, 16: 0..2
    if ((lane & 15) == 0 && lane != 48) {
        sm.red[lw * 4 + j] = m;
        sm.ired[lw * 8 + 2 + j] = j == 0 ? -b : b;       // lo_y, hi_y, pmax
    }
    if (lane == 0) {
        sm.ired[lw * 8 + 0] = p.blox;
        sm.ired[lw * 8 + 1] = p.bhix;
    }
}

// The CellState commit (src/kernels.cu:542-591), on wave 0 after the barrier
// that orders publish_part: lanes 0-3 add the 16 wave partials of V, Cx, Cy
// and the perimeter, lanes 4-8 reduce the support box and phi_max, each in
// wave order from the same initial value. The other waves go on: the next
// cell's first barrier lies between this and the next publish_part.
// old_raw: the cell's CellState as fetched at the start of its turn (LDS),
// for the counters that the commit advances.
template <int CLS>
__device__ __forceinline__ void commit_cell(const pfh2d_step_args& A, int n, const Smem& sm,
                                            const Ctl& c, const uint32_t* old_raw) {
    const int lane = opaque_tid();
    double sl = 0.0;
    int ml = 0;
    if (lane < 4) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sl += sm.red[w * 4 + lane];
    } else if (lane < 9) {
        const int j = lane - 4;                  // 0 lo_x, 1 hi_x, 2 lo_y, 3 hi_y, 4 pmax
        const bool is_max = (j & 1) != 0 || j == 4;
        ml = j == 0 ? c.dwx : j == 2 ? c.dwy : j == 4 ? 0 : -1;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int v = sm.ired[w * 8 + j];
            ml = is_max ? max(ml, v) : min(ml, v);
        }
    }
    const double sV = readlane_f64(sl, 0), sCx = readlane_f64(sl, 1);
    const double sCy = readlane_f64(sl, 2), sPer = readlane_f64(sl, 3);
    const int Blox = __builtin_amdgcn_readlane(ml, 4);
    const int Bhix = __builtin_amdgcn_readlane(ml, 5);
    const int Bloy = __builtin_amdgcn_readlane(ml, 6);
    const int Bhiy = __builtin_amdgcn_readlane(ml, 7);
    const int Pmax = __builtin_amdgcn_readlane(ml, 8);
    const pfh_cell_state* old = reinterpret_cast<const pfh_cell_state*>(old_raw);
    if (lane == 0) {
        pfh_cell_state* cs = &A.cell[n];
        cs->gx0 = c.gx0n;
        cs->gy0 = c.gy0n;
        cs->cls = (uint8_t)c.dcls;
        cs->cls_written[A.parity_out] = (uint8_t)c.dcls;
        cs->theta = c.theta;
        cs->V = sV;
        cs->Cx = sCx;
        cs->Cy = sCy;
        if (c.fm) cs->perim = sPer;
        cs->bb_lo_x = Blox;
        cs->bb_hi_x = Bhix;
        cs->bb_lo_y = Bloy;
        cs->bb_hi_y = Bhiy;
        cs->promote_ctr = (uint32_t)c.pctr;
        cs->shift_ctr = old->shift_ctr + ((c.sx | c.sy) ? 1u : 0u);
        cs->tumble_ctr = old->tumble_ctr + (uint32_t)c.tumbled;
        cs->phi_max = __uint_as_float((uint32_t)Pmax);
        A.cell_cls[n] = (uint8_t)c.dcls;
        if (CLS == kClassFallback) {
            cs->reserved[0] = 1u;
            const bool edge = Bhix >= 0 && (Blox == 0 || Bhix == c.dwx - 1 ||
                                            Bloy == 0 || Bhiy == c.dwy - 1);
            if (c.no_margin || (c.dcls == kClassFallback && edge))
                cs->reserved[1] = old->reserved[1] + 1u;
        }
    }
}

// The check step's commit: the cell's new window position and class (all its
// consumer reads).
__device__ __forceinline__ void commit_position(const pfh2d_step_args& A, int n, const Ctl& c) {
    if (threadIdx.x == 0) {
        pfh_cell_state* cs = &A.cell[n];
        cs->gx0 = c.gx0n;
        cs->gy0 = c.gy0n;
        cs->cls = (uint8_t)c.dcls;
        cs->cls_written[A.parity_out] = (uint8_t)c.dcls;
        A.cell_cls[n] = (uint8_t)c.dcls;
    }
}

// -------------------------------------------------------------------------
// Next-cell fetch by wave 0, in four stages so that each stage only waits on
// a load issued one phase earlier:
//   1 the queue ticket (atomic on the cursor);
//   2 the cell id perm[ticket];
//   3 its class and its 192-byte CellState (a dword on each of 48 lanes);
//   4 the CellState copy into LDS, the slot, and the per-cell scalars.
// A workgroup's first cell is its own index; the cursor hands out the cells
// from gridDim.x on. An unsupported class id is flagged here (reference
// dispatch default, src/kernels.cu:1017-1021) and skipped by the dispatch.
// -------------------------------------------------------------------------
struct Fetch {
    unsigned long long tk;
    int nn, cls;
    uint32_t w;
};

__device__ __forceinline__ void fetch1(const pfh2d_step_args& A, Fetch& f) {
    if (threadIdx.x == 0) f.tk = atomicAdd(A.cursor_use, 1ull);
}

__device__ __forceinline__ void fetch2(const pfh2d_step_args& A, Fetch& f) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)f.tk);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(f.tk >> 32));
    const unsigned long long k =
        (((unsigned long long)hi << 32) | lo) + (unsigned long long)gridDim.x;
    f.nn = k < (unsigned long long)A.N ? (int)A.perm[k] : -1;
}

__device__ __forceinline__ void fetch3(const pfh2d_step_args& A, Fetch& f) {
    const int nn = __builtin_amdgcn_readfirstlane(f.nn);
    if (nn >= 0) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(A.cell + nn);
        f.cls = (int)A.cell_cls[nn];
        f.w = w[min((int)threadIdx.x, kFetchLanes - 1)];
    }
}

// 4a (wave 0): the CellState copy, the id and the class into LDS.
__device__ __forceinline__ void fetch4a(const pfh2d_step_args& A, Smem& sm, Fetch& f,
                                        int which) {
    const int j = (int)threadIdx.x;
    int cls = -1;
    if (f.nn >= 0) {
        if (j < kFetchLanes) sm.csraw[which][j] = f.w;
        cls = f.cls < kNumClasses ? f.cls : kNumClasses;
    }
    if (j == 0) {
        if (cls == kNumClasses) atomicAdd(&A.flags[PFH_FLAG_CLASS_UNSUPPORTED], 1u);
        sm.slot[which].n = f.nn;
        sm.slot[which].cls = cls;
    }
}

// 4b (one thread, after 4a is visible to it): the per-cell scalars.
template <bool kBatch>
__device__ __forceinline__ void fetch4b(const pfh2d_step_args& A, Smem& sm, int which,
                                        unsigned long long step) {
    const int cls = sm.slot[which].cls;
    if (cls >= 0 && cls < kNumClasses) {
        ScalarArgs s = scalar_args(A, sm.fm);
        if constexpr (kBatch) {
            // batched step: the cell's replica sets its domain and stream
            Slot& sl = sm.slot[which];
            const pfh2d_replica& rp = sm.reps[sm.cell_rep[sl.n]];
            s.L = rp.L;
            s.polarity_seed = rp.polarity_seed;
            sl.L = rp.L;
            sl.P = rp.P;
            sl.s_off_lo = (int)(uint32_t)rp.S_offset;
            sl.s_off_hi = (int)(uint32_t)(rp.S_offset >> 32);
        }
        cell_scalars(s, reinterpret_cast<const pfh_cell_state*>(sm.csraw[which]), cls, step,
                     &sm.slot[which].ctl);
    }
}

// Stages 2-4 at once (wave 0), where nothing is there to hide them behind.
template <bool kBatch>
__device__ __forceinline__ void fetch_rest(const pfh2d_step_args& A, Smem& sm, Fetch& f,
                                           int which, unsigned long long step) {
    fetch3(A, f);
    fetch4a(A, sm, f, which);
    if (threadIdx.x == 0) fetch4b<kBatch>(A, sm, which, step);
}
template <bool kBatch = false>
__device__ __forceinline__ void fetch_all(const pfh2d_step_args& A, Smem& sm, int which,
                                          unsigned long long step) {
    Fetch f;
    fetch1(A, f);
    fetch2(A, f);
    fetch_rest<kBatch>(A, sm, f, which, step);
}
// The workgroup's first cell.
template <bool kBatch = false>
__device__ __forceinline__ void fetch_first(const pfh2d_step_args& A, Smem& sm,
                                            unsigned long long step) {
    Fetch f;
    f.nn = (int)blockIdx.x < A.N ? (int)A.perm[blockIdx.x] : -1;
    fetch_rest<kBatch>(A, sm, f, 0, step);
}

// -------------------------------------------------------------------------
// Column-walk path: classes 0-3.
//
// Work split. A cell's pixels belong to 1024 logical threads (16 logical
// waves): thread t owns rows y0..y0+RB-1 of one column, x = (t - 16) % WX,
// band = (t - 16) / WX; the order of every fp64 sum follows that split. A
// workgroup has NW = 8 or 16 waves, and each wave walks 16 / NW logical
// waves one after the other. With NW = 8 two workgroups, two independent
// cells, share a compute unit, so that one cell's loads, reductions, scalars
// and barriers run under the other's arithmetic.
//
// Data path. A wave reads only the 64 columns of its logical wave (at most
// two runs of columns, in adjacent bands) and one halo column on each side:
// three rows are 57 groups of 16 B, one buffer load per lane, that goes
// through registers into rows private to the wave in LDS. No barrier is
// needed between staging and stencil. Groups outside the window (the halo of
// an edge column, rows past the window, the gap group between the two runs,
// columns of logical threads that own nothing) are past the descriptor's
// end, for which the buffer load returns zeros: the stencil has no edge test
// and a lane that owns nothing computes exact zeros. The rows of the last
// logical wave stay in LDS for the update; those of the other are read again
// (from L2).
//
// The S word of a pixel is requested at the start of the cell into the
// register that later holds the pixel's passive right-hand side, and the
// scatter's returned word replaces that right-hand side in the update.
//
// Exact shortcuts (phi never takes the value -0, so adding or subtracting a
// signed zero changes no sum or right-hand side):
//   - a wave-row where no lane overlaps another cell (S_other == 0) skips the
//     repulsion term and the fp64 interaction-integral terms, all zero.
// -------------------------------------------------------------------------
constexpr int kRowGroupsW = 19;                        // 16 groups, two halos, one gap
constexpr int kRowFloats = 4 * kRowGroupsW;
constexpr int kChunkRows = 3;                          // rows per buffer load
constexpr int kChunkFloats = kChunkRows * kRowFloats;
constexpr int kChunkLanes = kChunkRows * kRowGroupsW;  // 57 of 64
constexpr int kChunkSlots = 10;                        // chunks a wave holds in LDS
constexpr int kChunkDepth = 3;                         // chunk loads in flight
template <int NW> constexpr int kWindowFloats = NW * kChunkSlots * kChunkFloats;

struct Roll {
    float sW, sC, sE, cW, cC, cE, nW, nC, nE;
};

__device__ __forceinline__ void load_row(const PFH_LDS float* p, float& w, float& c, float& e) {
    w = p[-1];
    c = p[0];
    e = p[1];
}

__device__ __forceinline__ bool wave_any(bool v) {
    return __builtin_amdgcn_ballot_w64(v) != 0ull;
}

// First part of phase_field_rhs (include/kernels.cuh:127-136): every passive
// term but the repulsion, the reference's terms in its order with each
// product-and-add fused (one rounding where the reference's source has a
// multiply and an add): the 9-point Laplacian (edge sum x 4 + diagonal sum,
// then - 20 x centre, over 6), then gam x lap - dwC x phi(1 - phi)(1 - 2 phi),
// then + volC x phi.
__device__ __forceinline__ float passive_head_of(float nC, float sC, float cE, float cW,
                                                 float nE, float nW, float sE, float sW,
                                                 float cC, float gam, float dwC, float volC) {
    const float edge = nC + sC + cE + cW;
    const float diag = nE + nW + sE + sW;
    const float lap = fmaf(-20.0f, cC, fmaf(4.0f, edge, diag)) * (float)(1.0 / 6.0);
    const float dw = (cC * (1.0f - cC)) * fmaf(-2.0f, cC, 1.0f);
    return fmaf(volC, cC, fmaf(gam, lap, -(dwC * dw)));
}

__device__ __forceinline__ float passive_head(const Roll& q, float gam, float dwC,
                                              float volC) {
    return passive_head_of(q.nC, q.sC, q.cE, q.cW, q.nE, q.nW, q.sE, q.sW, q.cC, gam, dwC,
                           volC);
}

// The repulsion term: passive = head - repC x phi x S_other, fused.
__device__ __forceinline__ float with_repulsion(float head, float repC, float cC, float So) {
    return fmaf(-(repC * cC), So, head);
}

// The Euler update phi + dt (mrel x passive - (vx gx + vy gy)), fused. The
// reference takes passive - adv when mrel == 1 (include/kernels.cuh:118-138):
// 1 x passive is passive exactly, so one expression gives both.
__device__ __forceinline__ float euler_update(float cC, float gxv, float gyv, float pas,
                                              float vx, float vy, float mrel, float dt) {
    const float adv = fmaf(vy, gyv, vx * gxv);
    return fmaf(dt, fmaf(mrel, pas, -adv), cC);
}

// S_other, counting this lane's negative differences (the subtraction's
// borrow is added in with carry).
__device__ __forceinline__ float s_other_lane(uint32_t qS, float c, uint32_t& neg1) {
    const uint32_t qc = q_of(c);
    const bool neg = qS < qc;
    neg1 += (uint32_t)neg;
    return neg ? 0.0f : (float)(qS - qc) * kQInv;
}

// mask = 2 mask + (v > kSupportEps): the support rows of a column, one bit a
// row, the compare's bit shifted in by the add's carry.
__device__ __forceinline__ void push_support(uint32_t& mask, float v) {
    asm("v_cmp_gt_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
        : "+v"(mask) : "v"(v), "v"(kSupportEps) : "vcc");
}

// The cell's domain: the launch's own population or, in a batched step,
// its replica's side, S pitch and S offset, made wave-uniform.
struct Dom {
    int L, P;
    unsigned long long off;
};
template <bool kBatch>
__device__ __forceinline__ Dom cell_dom(const pfh2d_step_args& A, const Slot& c) {
    if constexpr (kBatch) {
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)c.s_off_lo);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)c.s_off_hi);
        return {__builtin_amdgcn_readfirstlane(c.L), __builtin_amdgcn_readfirstlane(c.P),
                ((unsigned long long)hi << 32) | lo};
    } else {
        return {__builtin_amdgcn_readfirstlane(A.L), __builtin_amdgcn_readfirstlane(A.P), 0ull};
    }
}

// Wave-uniform copies of values read from LDS (the out-of-line paths' arguments,
// the cell's scalars): they then live in scalar registers.
template <class T>
__device__ __forceinline__ T* uni_ptr(T* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T*)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float uni(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

// Raw buffer descriptors: a byte offset at or past the end reads zeros and
// stores nothing; on gfx950 the scalar offset takes part in that test. One
// covers the rows of a tile that a window occupies, so rows above and below the
// window need no test; kOffNone is past every one.
constexpr uint32_t kOffNone = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
constexpr uint32_t kTileRow = 4u * kTilePitch;         // bytes of a tile row

// phi_next of one source pixel from global memory, bit for bit as the walk
// computes it (the perimeter of a recentred cell needs values that the
// destination window does not hold).
struct NextArgs {
    const float* win;            // window origin in the input tile
    const uint32_t* S;
    int WX, WY, L, P, gx0, gy0;
    float gam, dwC, volC, repC, vx, vy, mrel, dt;
};
__device__ __noinline__ float next_at(const NextArgs a, int x, int y) {
    auto f = [&](int xx, int yy) -> float {
        return (unsigned)xx < (unsigned)a.WX && (unsigned)yy < (unsigned)a.WY
                   ? a.win[(size_t)yy * kTilePitch + xx] : 0.0f;
    };
    const float cC = f(x, y), cE = f(x + 1, y), cW = f(x - 1, y);
    const float nC = f(x, y + 1), sC = f(x, y - 1);
    uint32_t neg = 0u;
    const float So = s_other_lane(
        a.S[(size_t)wrapi(a.gy0 + y, a.L) * a.P + wrapi(a.gx0 + x, a.L)], cC, neg);
    const float pas = with_repulsion(
        passive_head_of(nC, sC, cE, cW, f(x + 1, y + 1), f(x - 1, y + 1), f(x + 1, y - 1),
                        f(x - 1, y - 1), cC, a.gam, a.dwC, a.volC), a.repC, cC, So);
    return euler_update(cC, 0.5f * (cE - cW), 0.5f * (nC - sC), pas, a.vx, a.vy, a.mrel, a.dt);
}

// One lane's share of logical wave lw: its column as a pixel, and the 16 B
// group it stages as a loader. Recomputed per pass (a few instructions on the
// lane index and scalars) rather than held.
template <int CLS>
struct Share {
    using G = Staged<CLS>;
    int lane, x0, split, band0;            // all but lane are uniform
    __device__ __forceinline__ explicit Share(int lw) {
        asm volatile("" : "+s"(lw));
        lane = opaque_tid() & (kWave - 1);
        const int pv = lw * kWave - kControlLanes + G::WX;   // >= 0
        const int row = pv / G::WX;
        band0 = row - 1;
        x0 = pv - row * G::WX;                               // first run's first column
        split = min(kWave, G::WX - x0);                      // lanes of the first run
    }
    __device__ __forceinline__ bool second() const { return lane >= split; }
    __device__ __forceinline__ int x() const { return lane + (second() ? -split : x0); }
    __device__ __forceinline__ int band() const { return band0 + (second() ? 1 : 0); }
    __device__ __forceinline__ bool active() const { return (unsigned)band() < (unsigned)G::NB; }
    // first row; band 0's or the last one's where the lane owns nothing
    __device__ __forceinline__ int y0() const {
        return min(max(band(), 0), G::NB - 1) * G::RB;
    }
    // the lane's column in a staged row (floats)
    __device__ __forceinline__ int col() const { return 4 + lane + (second() ? 4 : 0); }
    // byte offset, from the window's first row, of the lane's group in the
    // first chunk (rows -1, 0, 1 of the band)
    __device__ __forceinline__ uint32_t group() const {
        const int r = lane / kRowGroupsW, q = lane - r * kRowGroupsW;
        const int n1 = split / 4;
        const bool two = q > n1 + 1;
        const int xg = 4 * (q - 1) + (two ? -4 * (n1 + 1) : x0);
        const int bg = band0 + (two ? 1 : 0);
        const bool ok = lane < kChunkLanes && (unsigned)xg < (unsigned)G::WX &&
                        (unsigned)bg < (unsigned)G::NB && !(two && split == kWave);
        const int off = (bg * G::RB + r - 1) * (int)kTileRow + 4 * (G::TX0 + xg);
        return ok ? (uint32_t)off : kOffNone;
    }
};

// kCheck: a check step (the surrogate's acceptance field), which needs the
// new field and the cell's window position only: no scatter, moments,
// support, flags or perimeter, and a commit of the position alone.
// kStream: the new field bypasses the caches (see kStreamBytes).
template <int CLS, int NW, bool kCheck = false, bool kBatch = false, int kObs = 0,
          bool kStream = false>
__device__ void cell_walk(const pfh2d_step_args& A, int n, unsigned long long step, Smem& sm,
                          PFH_LDS float* win, Ctl& c, int nxt) {
    using G = Staged<CLS>;
    constexpr int WX = G::WX, WY = G::WY, TX0 = G::TX0, TY0 = G::TY0, RB = G::RB;
    constexpr int NT = NW * kWave, VW = kWaves / NW;
    constexpr int NCK = (RB + 2 + kChunkRows - 1) / kChunkRows;
    constexpr bool kKeep = NCK <= kChunkSlots;   // the last pass's rows stay for the update
    // chunk loads in order: the passes of phase A, then those of phase B that
    // find their rows gone
    constexpr int kLoads = (VW + (kKeep ? VW - 1 : VW)) * NCK;
    const int tid = opaque_tid();
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    Fetch nf;
    if (wave == 0) fetch1(A, nf);
    const Dom dm = cell_dom<kBatch>(A, sm.slot[nxt ^ 1]);
    const int L = dm.L, P = dm.P;
    const int gx0 = __builtin_amdgcn_readfirstlane(c.gx0);
    const int gy0 = __builtin_amdgcn_readfirstlane(c.gy0);
    PFH_LDS float* const rows = win + wave * (kChunkSlots * kChunkFloats);
    const __amdgpu_buffer_rsrc_t tin =
        rsrc_of(uni_ptr(A.phi_in) + (size_t)n * kTileArea + (size_t)TY0 * kTilePitch,
                WY * kTileRow);
    const uint32_t s_pitch = 4u * (uint32_t)P, s_wrap = s_pitch * (uint32_t)L;
    const __amdgpu_buffer_rsrc_t s_in = rsrc_of(uni_ptr(A.S_rd) + dm.off, s_wrap);
    // no row of the walk wraps around the domain (rows past the window included)
    const bool flat = gy0 + G::NB * RB <= L;

    auto lw_of = [&](int v) { return wave + NW * v; };
    // S byte offset of a lane's first row: 32 bits (4 P L < 2^32, checked at
    // launch); a wrapping column advances it row by row
    auto s_off_of = [&](int x, int y0) -> uint32_t {
        int gx = gx0 + x, gy = gy0 + y0;
        if (gx >= L) gx -= L;
        if (gy >= L) gy -= L;
        return (uint32_t)gy * s_pitch + 4u * (uint32_t)gx;
    };
    auto s_next = [&](uint32_t off) -> uint32_t {
        const uint32_t o = off + s_pitch;
        return min(o, o - s_wrap);               // o - s_wrap is huge below the wrap
    };

    // ---- chunk pipeline ----
    u32x4 pf[kChunkDepth];
    uint32_t group[VW];                          // the lane's group in each pass
#pragma unroll
    for (int v = 0; v < VW; ++v) group[v] = Share<CLS>(lw_of(v)).group();
    // logical wave of chunk load j
    auto v_of = [&](int j) {
        const int p = j / NCK;
        return p < VW ? p : (kKeep ? VW - 2 : VW - 1) - (p - VW);
    };
    auto issue = [&](int j) {                    // chunk j of the load order
        pf[j % kChunkDepth] = __builtin_amdgcn_raw_buffer_load_b128(
            tin, (int)(group[v_of(j)] + (uint32_t)(j % NCK) * (kChunkRows * kTileRow)), 0, 0);
    };
    auto chunk_at = [&](int j) -> PFH_LDS float* {
        return rows + (j % kChunkSlots) * kChunkFloats;
    };
    auto advance = [&](int j) {                  // chunk j into LDS, j + depth requested
        if (lane < kChunkLanes)
            *reinterpret_cast<PFH_LDS u32x4*>(chunk_at(j) + 4 * lane) = pf[j % kChunkDepth];
        __builtin_amdgcn_wave_barrier();
        if (j + kChunkDepth < kLoads) issue(j + kChunkDepth);
    };

#pragma unroll
    for (int j = 0; j < kChunkDepth; ++j) issue(j);
    uint32_t qS[VW][RB];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        const Share<CLS> g(lw_of(v));
        uint32_t off = s_off_of(g.x(), g.y0());
        if (flat) {
            uint32_t so = 0u;
#pragma unroll
            for (int k = 0; k < RB; ++k) {
                qS[v][k] = __builtin_amdgcn_raw_buffer_load_b32(s_in, (int)off, (int)so, 0);
                so += s_pitch;
                asm volatile("" : "+s"(so));     // one live offset, not one per row
            }
        } else {
#pragma unroll
            for (int k = 0; k < RB; ++k) {
                qS[v][k] = __builtin_amdgcn_raw_buffer_load_b32(s_in, (int)off, 0, 0);
                off = s_next(off);
            }
        }
    }

    const float gam = uni(c.gam), dwC = uni(c.dwC), volC = uni(c.volC);
    const float repC = uni(A.rep_coeff);
    if (c.zero_tile)
        zero_outside_window<NT>(A.phi_out + (size_t)n * kTileArea, c.dwx, c.dwy,
                                c.dtx0, c.dty0);

    // ---- phase A: interaction integral and the held passive RHS ----
    float pas[VW][RB];
    double aIx[VW], aIy[VW];
    uint32_t neg1 = 0u;
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        const int q0 = v * NCK;
        const Share<CLS> g(lw_of(v));
        const int col = g.col();
        auto row = [&](int kk) -> const PFH_LDS float* {
            return chunk_at(q0 + kk / kChunkRows) + (kk % kChunkRows) * kRowFloats + col;
        };
        aIx[v] = aIy[v] = 0.0;
        ObsSums ob;
        advance(q0);
        if (NCK > 1) advance(q0 + 1);
        Roll q;
        float fW, fC, fE;                        // the row after the next, on its way
        load_row(row(0), q.sW, q.sC, q.sE);
        load_row(row(1), q.cW, q.cC, q.cE);
        load_row(row(2), fW, fC, fE);
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            q.nW = fW; q.nC = fC; q.nE = fE;
            if (k + 1 < RB) load_row(row(k + 3), fW, fC, fE);
            const float head = passive_head(q, gam, dwC, volC);
            const float So = s_other_lane(qS[v][k], q.cC, neg1);
            if constexpr (kObs == 2)
                observe_pixel(ob, g.x(), g.y0() + k, q.cC, q.cE, q.cW, q.nC, q.sC, q.nE, q.nW,
                              q.sE, q.sW, So, gam, dwC, repC, c.og2iv, c.ocx, c.ocy);
            // added up here: sunk to the end of the pass, the sums would keep
            // every row's stencil live
            if constexpr (kObs == 2)
                asm volatile("" : "+v"(ob.gx), "+v"(ob.gy), "+v"(ob.kx), "+v"(ob.ky),
                                  "+v"(ob.bx), "+v"(ob.by));
            if (wave_any(So != 0.0f)) {
                pas[v][k] = with_repulsion(head, repC, q.cC, So);
                const float gxv = 0.5f * (q.cE - q.cW);
                const float gyv = 0.5f * (q.nC - q.sC);
                aIx[v] += (double)(q.cC * gxv * So);
                aIy[v] += (double)(q.cC * gyv * So);
            } else {
                pas[v][k] = head;
            }
            q.sW = q.cW; q.sC = q.cC; q.sE = q.cE;
            q.cW = q.nW; q.cC = q.nC; q.cE = q.nE;
            if (k % kChunkRows == kChunkRows - 1 && (k + 4) / kChunkRows < NCK)
                advance(q0 + (k + 4) / kChunkRows);
            if (v == 0 && k == RB / 3 && wave == 0) fetch2(A, nf);
            if (v == 0 && k == 2 * RB / 3 && wave == 0) fetch3(A, nf);
            // One row per scheduling region keeps the walk's register
            // footprint at one row instead of the whole column.
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kObs == 2) publish_observer(sm, lw_of(v), ob);
    }
    publish_velocity<NW, VW>(sm, wave, aIx, aIy);
    // two events per negative pixel (the reference evaluates S_other once
    // per pass)
    if (neg1) flag_add(A.flags, PFH_FLAG_S_NEGATIVE, 2u * neg1);
    if (wave == 0) fetch4a(A, sm, nf, nxt);     // visible after the barrier
    lds_barrier();
    float vx, vy;
    finish_velocity<kObs>(A, n, sm, c, vx, vy);

    // ---- phase B: Euler update, shifted store, scatter, moments ----
    const float mrel = uni(c.mrel), dt = uni(A.dt);
    const int sx = __builtin_amdgcn_readfirstlane(c.sx);
    const int sy = __builtin_amdgcn_readfirstlane(c.sy);
    const int dwx = __builtin_amdgcn_readfirstlane(c.dwx);
    const int dwy = __builtin_amdgcn_readfirstlane(c.dwy);
    const int dtx0 = __builtin_amdgcn_readfirstlane(c.dtx0);
    const int dty0 = __builtin_amdgcn_readfirstlane(c.dty0);
    const int dcls = __builtin_amdgcn_readfirstlane(c.dcls);
    const bool moved = (sx | sy) != 0 || dcls != CLS;
    float* const tout_p = uni_ptr(A.phi_out) + (size_t)n * kTileArea;
    PFH_GLOBAL float* const tout = gptr(tout_p);
    const __amdgpu_buffer_rsrc_t tst =
        rsrc_of(tout_p + (size_t)dty0 * kTilePitch, (uint32_t)dwy * kTileRow);
    // a step without a scatter (S_sc NULL) has an empty aggregate
    uint32_t* const S_sc_p = uni_ptr(A.S_sc);
    const __amdgpu_buffer_rsrc_t s_out = rsrc_of(S_sc_p + dm.off, S_sc_p ? s_wrap : 0u);
    uint32_t olds[VW][RB];
    bool nonfin = false, clampf = false, ovf = false;

    // One pass: kGen handles recentred cells, class changes, columns that wrap
    // around the domain and lanes that own nothing; without it a destination
    // pixel is its source.
    auto pass_b = [&](auto gen, int v) {
        constexpr bool kGen = decltype(gen)::value;
        const bool loads = !(kKeep && v == VW - 1);
        // first chunk of this pass in the ring
        const int q0 = !loads ? v * NCK
                              : (VW + (kKeep ? VW - 2 - v : VW - 1 - v)) * NCK;
        const Share<CLS> g(lw_of(v));
        const int col = g.col();
        auto row = [&](int kk) -> const PFH_LDS float* {
            return chunk_at(q0 + kk / kChunkRows) + (kk % kChunkRows) * kRowFloats + col;
        };
        const int y0 = g.y0();
        const int a = kGen ? g.x() - sx : g.x();
        const bool ain = !kGen || (g.active() && (unsigned)a < (unsigned)dwx);
        const int b0 = kGen ? y0 - sy : y0;
        uint32_t st = (uint32_t)(b0 * (int)kTileRow + 4 * ((kGen ? dtx0 : TX0) + a));
        if (kGen && !ain) st = kOffNone;
        uint32_t s_off = s_off_of(g.x(), y0), so = 0u;
        Part p;
        p.blox = dwx; p.bhix = -1; p.bloy = dwy; p.bhiy = -1; p.pmaxb = 0;
        uint32_t sup = 0u, pmax = 0u;
        double bd = (double)b0;
        const double ad = (double)a;
        if (loads) {
            advance(q0);
            if (NCK > 1) advance(q0 + 1);
        }
        float sC = row(0)[0];
        float cW, cC, cE, fW, fC, fE;
        load_row(row(1), cW, cC, cE);
        load_row(row(2), fW, fC, fE);
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            const float nW = fW, nC = fC, nE = fE;
            if (k + 2 < RB) load_row(row(k + 3), fW, fC, fE);
            else if (k + 1 < RB) fC = row(k + 3)[0];
            const float gxv = 0.5f * (cE - cW);
            const float gyv = 0.5f * (nC - sC);
            const float pn = euler_update(cC, gxv, gyv, pas[v][k], vx, vy, mrel, dt);
            // rows past the destination window are past the descriptor's end;
            // rows past the source window hold no pixel of the cell (shifted,
            // they could land inside)
            if constexpr (kGen) {
                uint32_t o = st + (uint32_t)k * kTileRow;
                if (k >= G::RFULL) o = y0 + k < WY ? o : kOffNone;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(pn), tst, (int)o, 0,
                                                      kStream ? 2 : 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(pn), tst, (int)st,
                                                      (int)(k * kTileRow), kStream ? 2 : 0);
            }
            if constexpr (!kCheck) {
                // A lane whose destination is outside the window contributes
                // an exact zero to every sum below. Rows below RFULL exist in
                // every band, so only the last band's tail rows are tested
                // without a shift.
                float pv = pn;
                if (kGen)
                    pv = ain && y0 + k < WY && (unsigned)(b0 + k) < (unsigned)dwy ? pn : 0.0f;
                else if (k >= G::RFULL)
                    pv = y0 + k < WY ? pn : 0.0f;
                const float sq = pv * pv;
                pmax = max(pmax, __float_as_uint(fabsf(pv)));
                uint32_t w = __float2uint_rn(fminf(sq, kQClampPhiSq) * kQScale);
                const bool add = w != 0u;
                asm volatile("" : "+v"(w));  // the old word takes the addend's register
                if (add)
                    w = (uint32_t)__builtin_amdgcn_raw_ptr_buffer_atomic_add_i32(
                        (int)w, s_out, (int)s_off, (int)so, 0);
                olds[v][k] = w;
                const double d = (double)pv * (double)pv;
                p.V += d;
                p.Cy += d * bd;
                bd += 1.0;
                push_support(sup, pv);
                // added up here: sunk to the end of the pass, the sums would
                // keep every row's value live
                asm volatile("" : "+v"(p.V), "+v"(p.Cy), "+v"(pmax));
                if (kGen) {
                    s_off = s_next(s_off);
                } else {
                    so += s_pitch;
                    asm volatile("" : "+s"(so));
                }
            }
            sC = cC;
            cW = nW; cC = nC; cE = nE;
            if (loads && k % kChunkRows == kChunkRows - 1 && (k + 4) / kChunkRows < NCK)
                advance(q0 + (k + 4) / kChunkRows);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!kCheck) {
            p.Cx = p.V * ad;               // every pixel of this lane has column a
            if (sup) {                     // bit RB - 1 - k: row k
                p.bloy = b0 + (RB - 32) + __clz((int)sup);
                p.bhiy = b0 + RB - __ffs((int)sup);
            }
            // columns of the two runs: the second run's lie left of the first's
            const uint64_t m = __builtin_amdgcn_ballot_w64(sup != 0u);
            const uint64_t m2 = g.split < kWave ? m >> g.split : 0ull;
            const uint64_t m1 = g.split < kWave ? m & ((1ull << g.split) - 1ull) : m;
            if (m) {
                const int sh = kGen ? sx : 0;
                p.blox = (m2 ? __builtin_ctzll(m2) : g.x0 + __builtin_ctzll(m1)) - sh;
                p.bhix = (m1 ? g.x0 + 63 - __builtin_clzll(m1) : 63 - __builtin_clzll(m2)) - sh;
            }
            p.pmaxb = (int)pmax;
            nonfin |= pmax >= 0x7F800000u;
            // sq grows with |phi|; a NaN hides the lane's other values, which
            // are then read back
            const float pm = __uint_as_float(pmax);
            clampf |= pm * pm > kQClampPhiSq;
            if (pmax > 0x7F800000u) {
                for (int k = 0; k < RB; ++k) {
                    const int b = b0 + k;
                    if (ain && y0 + k < WY && (unsigned)b < (unsigned)dwy) {
                        const float t = tout[(size_t)(dty0 + b) * kTilePitch + dtx0 + a];
                        clampf |= t * t > kQClampPhiSq;
                    }
                }
            }
            publish_part(sm, lw_of(v), p);
        }
    };
    // a logical wave with lanes that own nothing takes the general pass too
    auto whole = [&](int lw) {
        return lw > 0 && (lw + 1) * kWave - kControlLanes <= G::NB * WX;
    };
#pragma unroll
    for (int v = VW - 1; v >= 0; --v) {
        if (moved || !flat || !whole(lw_of(v))) pass_b(std::true_type{}, v);
        else pass_b(std::false_type{}, v);
    }
    if constexpr (!kCheck) {
        // Exact S_overflow test: every addend is at most 2^29, so a wrap needs
        // old >= 2^32 - 2^29; only such candidates recompute q from this
        // thread's own stored value.
        uint32_t big = 0u;
#pragma unroll
        for (int v = 0; v < VW; ++v)
#pragma unroll
            for (int k = 0; k < RB; ++k) big = max(big, olds[v][k]);
        if (big >= 0xE0000000u) {
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                const Share<CLS> g(lw_of(v));
                const PFH_GLOBAL float* mine =
                    tout + (ptrdiff_t)(dty0 + g.y0() - sy) * kTilePitch + dtx0 + g.x() - sx;
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    if (olds[v][k] >= 0xE0000000u) {
                        const uint32_t qv = q_of(mine[k * kTilePitch]);
                        ovf |= olds[v][k] > 0xFFFFFFFFu - qv;
                    }
                }
            }
        }
        if (nonfin) flag_or(A.flags, PFH_FLAG_NONFINITE);
        if (clampf) flag_or(A.flags, PFH_FLAG_Q_CLAMP);
        if (ovf) flag_or(A.flags, PFH_FLAG_S_OVERFLOW);
    }

    // Destination pixels whose source lies outside the window are zero.
    if (moved) {
        if (dcls == CLS) {
            const int ny = sy > 0 ? sy : -sy, nx = sx > 0 ? sx : -sx;
            const int nrow = ny * dwx, total = nrow + nx * dwy;
            for (int i = tid; i < total; i += NT) {
                int aa, b;
                if (i < nrow) {
                    const int rr = i / dwx;
                    aa = i - rr * dwx;
                    b = sy > 0 ? dwy - sy + rr : rr;
                } else {
                    const int j = i - nrow, cc = j / dwy;
                    b = j - cc * dwy;
                    aa = sx > 0 ? dwx - sx + cc : cc;
                }
                tout[(size_t)(dty0 + b) * kTilePitch + dtx0 + aa] = 0.0f;
            }
        } else {
            for (int i = tid; i < dwx * dwy; i += NT) {
                const int b = i / dwx, aa = i - (i / dwx) * dwx;
                const int ii = aa + sx, jj = b + sy;
                if (!((unsigned)ii < (unsigned)WX && (unsigned)jj < (unsigned)WY))
                    tout[(size_t)(dty0 + b) * kTilePitch + dtx0 + aa] = 0.0f;
            }
        }
    }

    // Perimeter on full-moment steps (one step in full_moment_every) from the
    // new field in the source layout with source-window zeros (the staged
    // semantics, src/kernels.cu:512-538): read back from the stored tile, or
    // recomputed where a recentred window does not hold it.
    if (!kCheck && c.fm) {
        __threadfence();          // stores reach L2; L1 lines are invalidated
        __syncthreads();
        const NextArgs na{A.phi_in + (size_t)n * kTileArea + (size_t)TY0 * kTilePitch + TX0,
                          A.S_rd + dm.off, WX, WY, L, P, c.gx0, c.gy0, c.gam, c.dwC, c.volC,
                          A.rep_coeff, vx, vy, mrel, dt};
        auto value = [&](int ii, int jj) -> float {
            return moved ? next_at(na, ii, jj)
                         : tout[(size_t)(TY0 + jj) * kTilePitch + TX0 + ii];
        };
        for (int v = 0; v < VW; ++v) {
            double aPer = 0.0;
            for (int i = tid + v * NT; i < dwx * dwy; i += kNT) {
                const int b = i / dwx, aa = i - (i / dwx) * dwx;
                const int ii = aa + sx, jj = b + sy;
                const bool iin = (unsigned)ii < (unsigned)WX;
                const bool jin = (unsigned)jj < (unsigned)WY;
                float e = 0.0f, w = 0.0f, nn = 0.0f, ss = 0.0f;
                if (jin) {
                    if ((unsigned)(ii + 1) < (unsigned)WX) e = value(ii + 1, jj);
                    if ((unsigned)(ii - 1) < (unsigned)WX) w = value(ii - 1, jj);
                }
                if (iin) {
                    if ((unsigned)(jj + 1) < (unsigned)WY) nn = value(ii, jj + 1);
                    if ((unsigned)(jj - 1) < (unsigned)WY) ss = value(ii, jj - 1);
                }
                const float pgx = 0.5f * (e - w), pgy = 0.5f * (nn - ss);
                aPer += (double)sqrtf(pgx * pgx + pgy * pgy);
            }
            aPer = wave_sum(aPer);
            if (lane == 0) sm.red[lw_of(v) * 4 + 3] = aPer;
        }
    }
    // The next cell's scalars, then the commit by wave 0. The other waves go
    // on to the next cell: its first barrier orders their next partials.
    if (tid == kScalarsThread) fetch4b<kBatch>(A, sm, nxt, step);
    lds_barrier();
    if constexpr (kCheck) {
        commit_position(A, n, c);
    } else {
        if (wave == 0) commit_cell<CLS>(A, n, sm, c, sm.csraw[nxt ^ 1]);
    }
}

// -------------------------------------------------------------------------
// Global-memory path: class 4 (window zeros synthesized) and the fallback
// class 5 (the tile's own one-pixel zero ring), src/kernels.cu:604-937.
// Logical thread t owns pixels t, t + 1024, ...
// -------------------------------------------------------------------------
template <int CLS, int NW, bool kBatch = false, int kObs = 0>
__device__ void cell_global(const pfh2d_step_args& A, int n,
                            unsigned long long step, Smem& sm, Ctl& c, int nxt) {
    constexpr int WX = kShapes[CLS].wx, WY = kShapes[CLS].wy;
    constexpr int TX0 = kShapes[CLS].tx0, TY0 = kShapes[CLS].ty0;
    constexpr int NT = NW * kWave, VW = kWaves / NW;
    const int tid = opaque_tid();
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const Dom dm = cell_dom<kBatch>(A, sm.slot[nxt ^ 1]);
    const int L = dm.L, P = dm.P;
    const uint32_t* S_rd = A.S_rd + dm.off;
    uint32_t* S_sc = A.S_sc ? A.S_sc + dm.off : nullptr;
    if (wave == 0) fetch_all<kBatch>(A, sm, nxt, step);
    const int gx0 = c.gx0, gy0 = c.gy0;
    const float* tin = A.phi_in + (size_t)n * kTileArea;
    float* tout = A.phi_out + (size_t)n * kTileArea;
    auto pin = [&](int xx, int yy) -> float {
        if (CLS != kClassFallback &&
            !((unsigned)xx < (unsigned)WX && (unsigned)yy < (unsigned)WY))
            return 0.0f;
        return tin[(size_t)(TY0 + yy) * kTilePitch + TX0 + xx];
    };
    if (c.zero_tile) zero_outside_window<NT>(tout, c.dwx, c.dwy, c.dtx0, c.dty0);

    uint32_t negc = 0u;
    double aIxv[VW], aIyv[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        double aIx = 0.0, aIy = 0.0;
        ObsSums ob;
        for (int p = tid + v * NT; p < WX * WY; p += kNT) {
            const int y = p / WX, x = p - (p / WX) * WX;
            const float cc = pin(x, y);
            const float gxv = 0.5f * (pin(x + 1, y) - pin(x - 1, y));
            const float gyv = 0.5f * (pin(x, y + 1) - pin(x, y - 1));
            const uint32_t qS = S_rd[(size_t)wrapi(gy0 + y, L) * P + wrapi(gx0 + x, L)];
            const uint32_t qc = q_of(cc);
            float So = 0.0f;
            if (qS >= qc) So = (float)(qS - qc) * kQInv;
            else negc += 1u;
            aIx += (double)(cc * gxv * So);
            aIy += (double)(cc * gyv * So);
            if constexpr (kObs == 2)
                observe_pixel(ob, x, y, cc, pin(x + 1, y), pin(x - 1, y), pin(x, y + 1),
                              pin(x, y - 1), pin(x + 1, y + 1), pin(x - 1, y + 1),
                              pin(x + 1, y - 1), pin(x - 1, y - 1), So, c.gam, c.dwC,
                              A.rep_coeff, c.og2iv, c.ocx, c.ocy);
        }
        aIxv[v] = aIx;
        aIyv[v] = aIy;
        if constexpr (kObs == 2) publish_observer(sm, wave + NW * v, ob);
    }
    publish_velocity<NW, VW>(sm, wave, aIxv, aIyv);
    lds_barrier();
    float vx, vy;
    finish_velocity<kObs>(A, n, sm, c, vx, vy);

    const float gam = c.gam, dwC = c.dwC, volC = c.volC, repC = A.rep_coeff;
    const float mrel = c.mrel, dt = A.dt;
    const int sx = c.sx, sy = c.sy, dwx = c.dwx, dwy = c.dwy;
    const int dtx0 = c.dtx0, dty0 = c.dty0;
    for (int p = tid; p < WX * WY; p += NT) {
        const int y = p / WX, x = p - (p / WX) * WX;
        const float cC = pin(x, y);
        const float cE = pin(x + 1, y), cW = pin(x - 1, y);
        const float nC = pin(x, y + 1), sC = pin(x, y - 1);
        const float nE = pin(x + 1, y + 1), nW = pin(x - 1, y + 1);
        const float sE = pin(x + 1, y - 1), sW = pin(x - 1, y - 1);
        const float gxv = 0.5f * (cE - cW);
        const float gyv = 0.5f * (nC - sC);
        const uint32_t qS = S_rd[(size_t)wrapi(gy0 + y, L) * P + wrapi(gx0 + x, L)];
        const uint32_t qc = q_of(cC);
        float So = 0.0f;
        if (qS >= qc) So = (float)(qS - qc) * kQInv;
        else negc += 1u;
        const float passive = with_repulsion(
            passive_head_of(nC, sC, cE, cW, nE, nW, sE, sW, cC, gam, dwC, volC), repC, cC, So);
        const float pn = euler_update(cC, gxv, gyv, passive, vx, vy, mrel, dt);
        const int a = x - sx, b = y - sy;
        if ((unsigned)a < (unsigned)dwx && (unsigned)b < (unsigned)dwy)
            tout[(size_t)(dty0 + b) * kTilePitch + dtx0 + a] = pn;
    }
    if (negc) flag_add(A.flags, PFH_FLAG_S_NEGATIVE, negc);
    for (int i = tid; i < dwx * dwy; i += NT) {
        const int b = i / dwx, a = i - (i / dwx) * dwx;
        const int ii = a + sx, jj = b + sy;
        if (!((unsigned)ii < (unsigned)WX && (unsigned)jj < (unsigned)WY))
            tout[(size_t)(dty0 + b) * kTilePitch + dtx0 + a] = 0.0f;
    }
    __threadfence();      // stores reach L2; L1 lines are invalidated
    __syncthreads();

    const int gx0n = c.gx0n, gy0n = c.gy0n, fm = c.fm;
    bool nonfin = false, clampf = false, ovf = false;
    for (int v = 0; v < VW; ++v) {
        double aPer = 0.0;
        Part pt;
        pt.blox = dwx; pt.bhix = -1; pt.bloy = dwy; pt.bhiy = -1; pt.pmaxb = 0;
        for (int i = tid + v * NT; i < dwx * dwy; i += kNT) {
            const int b = i / dwx, a = i - (i / dwx) * dwx;
            const size_t row = (size_t)(dty0 + b) * kTilePitch + dtx0;
            const float pn = tout[row + a];
            nonfin |= !isfinite(pn);
            clampf |= (pn * pn > kQClampPhiSq);
            pt.pmaxb = max(pt.pmaxb, (int)__float_as_uint(fabsf(pn)));
            const uint32_t q = q_of(pn);
            if (q && S_sc) {
                const uint32_t old = atomicAdd(
                    &S_sc[(size_t)wrapi(gy0n + b, L) * P + wrapi(gx0n + a, L)], q);
                ovf |= old > 0xFFFFFFFFu - q;
            }
            const double d = (double)pn * (double)pn;
            pt.V += d;
            pt.Cx += d * (double)a;
            pt.Cy += d * (double)b;
            if (pn > kSupportEps) {
                pt.blox = min(pt.blox, a); pt.bhix = max(pt.bhix, a);
                pt.bloy = min(pt.bloy, b); pt.bhiy = max(pt.bhiy, b);
            }
            if (fm) {
                const float e = a + 1 < dwx ? tout[row + a + 1] : 0.0f;
                const float w = a > 0 ? tout[row + a - 1] : 0.0f;
                const float nn = b + 1 < dwy ? tout[row + kTilePitch + a] : 0.0f;
                const float ss = b > 0 ? tout[row - kTilePitch + a] : 0.0f;
                const float pgx = 0.5f * (e - w), pgy = 0.5f * (nn - ss);
                aPer += (double)sqrtf(pgx * pgx + pgy * pgy);
            }
        }
        pt.blox = __builtin_amdgcn_readfirstlane(wave_min(pt.blox));
        pt.bhix = __builtin_amdgcn_readfirstlane(wave_max(pt.bhix));
        publish_part(sm, wave + NW * v, pt);
        if (fm) {
            aPer = wave_sum(aPer);
            if ((tid & (kWave - 1)) == 0) sm.red[(wave + NW * v) * 4 + 3] = aPer;
        }
    }
    if (nonfin) flag_or(A.flags, PFH_FLAG_NONFINITE);
    if (clampf) flag_or(A.flags, PFH_FLAG_Q_CLAMP);
    if (ovf) flag_or(A.flags, PFH_FLAG_S_OVERFLOW);
    lds_barrier();
    if (wave == 0) commit_cell<CLS>(A, n, sm, c, sm.csraw[nxt ^ 1]);
}

// Classes other than the round class 0 run out of line, with their own
// register allocation, so their longer per-thread columns (up to 29 rows) do
// not raise the pressure of the hot class-0 path.
template <int CLS, int NW, bool kBatch = false, int kObs = 0>
__device__ __noinline__ void cell_cold(const pfh2d_step_args* A, int n, unsigned long long step,
                                       Smem* sm, PFH_LDS float* win, int cur) {
    n = __builtin_amdgcn_readfirstlane(n);
    if constexpr (CLS <= kClassStagedMax)
        cell_walk<CLS, NW, false, kBatch, kObs>(*A, n, step, *sm, win, sm->slot[cur].ctl, cur ^ 1);
    else
        cell_global<CLS, NW, kBatch, kObs>(*A, n, step, *sm, sm->slot[cur].ctl, cur ^ 1);
}

// -------------------------------------------------------------------------
// The persistent step kernel (src/kernels.cu:948-1030).
// -------------------------------------------------------------------------
// Batched form (kBatch): A describes the whole ensemble as one population
// (tiles, cell states, classes and the queue order over every replica's
// cells; each S slot one arena holding every replica's aggregate; the
// clear-ahead sweeps the whole arena), and each cell's side, S pitch, S
// offset and polarity stream come from its replica's record.
template <int NW, bool kCheck, bool kBatch = false, int kObs = 0, bool kStream = false>
__global__ __launch_bounds__(NW * kWave, 4) void k_step(const pfh2d_step_args A,
                                                        const int* run_if,
                                                        const pfh2d_replica* reps,
                                                        const uint16_t* cell_rep) {
    constexpr int NT = NW * kWave;
    __shared__ Smem sm;
    __shared__ __attribute__((aligned(16))) float window[kWindowFloats<NW>];
    PFH_LDS float* const win = (PFH_LDS float*)window;
    const int tid = (int)threadIdx.x;
    if (run_if != nullptr && *run_if == 0) return;   // gated-off launch: no effect

    const unsigned long long step = *A.step_rd;
    if (tid == 0) {
        sm.args = A;
        sm.fm = (A.full_moment_every > 0 &&
                 ((step + 1ull) % (unsigned long long)A.full_moment_every) == 0ull) ? 1 : 0;
        if constexpr (kBatch) {
            sm.reps = reps;
            sm.cell_rep = cell_rep;
        }
    }
    // Wave 0 fetches each next cell one cell ahead (ticket, id, class,
    // CellState) while it computes, so the queue's global round trips stay
    // off the critical path.
    if (tid < kWave) fetch_first<kBatch>(A, sm, step);
    // Clear S[(step+2)%3] ahead: this slot is neither read nor scattered
    // into by this launch. Non-temporal stores keep it out of the caches.
    if (A.clear_ahead_words > 0ull) {
        u32x4* dst = reinterpret_cast<u32x4*>(A.S_cl);
        const u32x4 zero4 = {0u, 0u, 0u, 0u};
        const size_t nvec = (size_t)(A.clear_ahead_words >> 2);
        const size_t stride = (size_t)gridDim.x * NT;
        for (size_t i = (size_t)blockIdx.x * NT + tid; i < nvec; i += stride)
            __builtin_nontemporal_store(zero4, &dst[i]);
        for (size_t i = (nvec << 2) + (size_t)blockIdx.x * NT + tid;
             i < (size_t)A.clear_ahead_words; i += stride)
            A.S_cl[i] = 0u;
    }
    // Cursor and step slots alternate with the phi parity; the kernel
    // boundary orders the reset and publication for the next launch.
    if (blockIdx.x == 0 && tid == 0) {
        *A.cursor_clear = 0ull;
        *A.step_wr = step + 1ull;
    }
    lds_barrier();
    int cur = 0;
    for (;;) {
        const int cls = __builtin_amdgcn_readfirstlane(sm.slot[cur].cls);
        const int n = __builtin_amdgcn_readfirstlane(sm.slot[cur].n);
        if (cls < 0) break;
        switch (cls) {
            case 0:
                cell_walk<0, NW, kCheck, kBatch, kObs, kStream>(sm.args, n, step, sm, win,
                                                                sm.slot[cur].ctl, cur ^ 1);
                break;
            case 1: cell_cold<1, NW, kBatch, kObs>(&sm.args, n, step, &sm, win, cur); break;
            case 2: cell_cold<2, NW, kBatch, kObs>(&sm.args, n, step, &sm, win, cur); break;
            case 3: cell_cold<3, NW, kBatch, kObs>(&sm.args, n, step, &sm, win, cur); break;
            case 4: cell_cold<4, NW, kBatch, kObs>(&sm.args, n, step, &sm, win, cur); break;
            case 5: cell_cold<5, NW, kBatch, kObs>(&sm.args, n, step, &sm, win, cur); break;
            default:                       // unsupported id, flagged at fetch
                if (tid < kWave) fetch_all<kBatch>(sm.args, sm, cur ^ 1, step);
                lds_barrier();
                break;
        }
        cur ^= 1;
    }
}

// -------------------------------------------------------------------------
// Initial condition, verification, trajectory, ordering.
//
// Layout shared by these kernels: a tile row is 72 groups of 16 B; work is
// spread over (cell, band of rows) workgroups so that a small population
// still fills the chip, every global access is a 16 B vector or a lane per
// word of one row, and flag words take at most one atomic per wave.
// -------------------------------------------------------------------------
constexpr int kRowGroups = kTilePitch / 4;          // 16 B groups per tile row
constexpr int kInitBandRows = 32;                   // 288 = 9 bands
constexpr int kInitBands = kTilePitch / kInitBandRows;
constexpr int kScatterBandRows = 16;
constexpr int kScatterBands = (286 + kScatterBandRows - 1) / kScatterBandRows;

__device__ __forceinline__ float f4_get(const float4& v, int k) {
    return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w;
}

// Fill n words with v: 16 B stores on the aligned body, words at both ends.
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t head = (size_t)((0u - (uint32_t)(uintptr_t)p) & 15u) >> 2;
    if (head > n) head = n;
    if (tid < head) p[tid] = v;
    u32x4* body = reinterpret_cast<u32x4*>(p + head);
    const size_t nv = (n - head) >> 2;
    const u32x4 v4 = {v, v, v, v};
    for (size_t i = tid; i < nv; i += stride) body[i] = v4;
    const size_t done = head + 4 * nv;
    if (tid < n - done) p[done + tid] = v;
}

// Smoothed disk of one window pixel (k_init_tiles' profile,
// src/kernels.cu:1072-1085): binary32 distance with minimum-image wrap,
// 0.5 (1 - tanh(k (r - R_eff))).
__device__ __forceinline__ float disk_value(int gx0, int gy0, int a, int b, float cx,
                                            float cy, int L, float radius_eff,
                                            float kappa_iface) {
    const float half = 0.5f * (float)L;
    float dx = (float)(gx0 + a) - cx;
    float dy = (float)(gy0 + b) - cy;
    if (dx > half) dx -= (float)L;
    if (dx < -half) dx += (float)L;
    if (dy > half) dy -= (float)L;
    if (dy < -half) dy += (float)L;
    const float r = sqrtf(dx * dx + dy * dy);
    const float t = (float)tanh_d((double)(kappa_iface * (r - radius_eff)));
    return 0.5f * (1.0f - t);
}

// grid (N, 9): workgroup (n, band) writes tile rows band*32 .. band*32+31 of
// both tiles of cell n in one pass of 16 B stores: the disk inside the class
// window, zeros elsewhere (phi_b all zeros). Band 0 records the origin.
__global__ __launch_bounds__(256) void k_init_tiles(float* phi_a, float* phi_b,
                                                    pfh_cell_state* cell,
                                                    const uint8_t* clsv, int L,
                                                    const float* seed_cx,
                                                    const float* seed_cy,
                                                    float radius_eff, float kappa_iface) {
    const int n = (int)blockIdx.x;
    const int cls = (int)clsv[n];
    const Shape sc = shape_of(cls);
    const float cx = seed_cx[n], cy = seed_cy[n];
    const int gx0 = wrapi((int)rintf(cx - 0.5f * (float)(sc.wx - 1)), L);
    const int gy0 = wrapi((int)rintf(cy - 0.5f * (float)(sc.wy - 1)), L);
    float4* ta = reinterpret_cast<float4*>(phi_a + (size_t)n * kTileArea);
    float4* tb = reinterpret_cast<float4*>(phi_b + (size_t)n * kTileArea);
    const int row0 = (int)blockIdx.y * kInitBandRows;
    const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int g = (int)threadIdx.x; g < kInitBandRows * kRowGroups; g += (int)blockDim.x) {
        const int ty = row0 + g / kRowGroups, gx = g % kRowGroups;
        const int b = ty - sc.ty0;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if ((unsigned)b < (unsigned)sc.wy) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int a = 4 * gx + k - sc.tx0;
                if ((unsigned)a < (unsigned)sc.wx)
                    v[k] = disk_value(gx0, gy0, a, b, cx, cy, L, radius_eff, kappa_iface);
            }
        }
        const size_t o = (size_t)ty * kRowGroups + gx;
        ta[o] = make_float4(v[0], v[1], v[2], v[3]);
        tb[o] = zero4;
    }
    if (blockIdx.y == 0 && threadIdx.x == 0) {
        pfh_cell_state* cs = &cell[n];
        cs->gx0 = gx0;
        cs->gy0 = gy0;
        cs->cls = (uint8_t)cls;
        cs->cls_written[0] = (uint8_t)cls;
        cs->cls_written[1] = (uint8_t)cls;
    }
}

// Moments of the stored field with the update's thread mapping (column bands
// for the LDS classes, flat pixel index for classes 4-5).
__global__ __launch_bounds__(kNT) void k_init_moments(pfh_cell_state* cell,
                                                      const uint8_t* clsv,
                                                      const float* phi, int N) {
    const int n = blockIdx.x;
    if (n >= N) return;
    const int cls = (int)clsv[n];
    const Shape sc = shape_of(cls);
    const float* t = phi + (size_t)n * kTileArea + (size_t)sc.ty0 * kTilePitch + sc.tx0;
    const WindowMoments m = stored_moments(cls, t);
    if (threadIdx.x == 0) store_moments(&cell[n], m);
}

// grid (N, 18): workgroup (n, band) adds q(phi) of window rows band*16 ..
// band*16+15 of cell n into S; wave w takes rows w, w+4, ..., its lanes one
// word of the row each (coalesced loads, atomics only where q != 0). All of a
// wave's rows are requested, then added, then tested: a load and a returning
// atomic for each row one after the other took 49 us for 1024 windows of
// 144 x 144, together 29 us (118 MB). Flag conditions are collected per lane
// and raised by one atomic per wave.
__global__ __launch_bounds__(256) void k_scatter_all(const float* phi,
                                                     const pfh_cell_state* cell,
                                                     const uint8_t* clsv, uint32_t* S,
                                                     int L, int P, uint32_t* flags) {
    const int n = (int)blockIdx.x;
    const Shape sc = shape_of((int)clsv[n]);
    const int r0 = (int)blockIdx.y * kScatterBandRows;
    if (r0 >= sc.wy) return;
    const int r1 = min(r0 + kScatterBandRows, sc.wy);
    const int gx0 = cell[n].gx0, gy0 = cell[n].gy0;
    const int lane = (int)threadIdx.x & (kWave - 1), wave = (int)threadIdx.x / kWave;
    const float* win = phi + (size_t)n * kTileArea + (size_t)sc.ty0 * kTilePitch + sc.tx0;
    uint32_t overflow = 0u, clamp = 0u;
    constexpr int kRows = kScatterBandRows / 4, kWords = 3;
    for (int a0 = lane; a0 < sc.wx; a0 += kWords * kWave) {
        float v[kRows][kWords];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int w = 0; w < kWords; ++w) {
                const int b = r0 + wave + 4 * r, a = a0 + w * kWave;
                v[r][w] = b < r1 && a < sc.wx ? win[(size_t)b * kTilePitch + a] : 0.0f;
            }
        uint32_t old[kRows][kWords];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            uint32_t* srow = S + (size_t)wrapi(gy0 + r0 + wave + 4 * r, L) * (size_t)P;
#pragma unroll
            for (int w = 0; w < kWords; ++w) {
                const uint32_t q = q_of(v[r][w]);
                old[r][w] = 0u;
                if (q)
                    old[r][w] = __hip_atomic_fetch_add(&srow[wrapi(gx0 + a0 + w * kWave, L)], q,
                                                       __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int w = 0; w < kWords; ++w) {
                const float pn = v[r][w];
                const uint32_t q = q_of(pn);
                overflow |= old[r][w] > 0xFFFFFFFFu - q;
                clamp |= q && pn * pn > kQClampPhiSq;
            }
    }
    const bool any_overflow = __ballot(overflow) != 0ull;
    const bool any_clamp = __ballot(clamp) != 0ull;
    if (lane == 0) {
        if (any_overflow) atomicOr(&flags[PFH_FLAG_S_OVERFLOW], 1u);
        if (any_clamp) atomicOr(&flags[PFH_FLAG_Q_CLAMP], 1u);
    }
}

// Per cell: V of the stored window in the update's reduction order (the
// moments pass), and max |phi| over the tile outside the window (a 16 B sweep
// of the whole tile). Sim::verify compares V with CellState.V.
__global__ __launch_bounds__(kNT) void k_verify_cells(const float* phi,
                                                      const uint8_t* clsv,
                                                      double* out_V,
                                                      float* out_outside_max) {
    __shared__ float wmax[kWaves];
    const int n = (int)blockIdx.x;
    const int cls = (int)clsv[n];
    const Shape sc = shape_of(cls);
    const float* tile = phi + (size_t)n * kTileArea;
    const float4* t4 = reinterpret_cast<const float4*>(tile);
    float omax = 0.0f;
    for (int g = (int)threadIdx.x; g < kTileArea / 4; g += kNT) {
        const int y = g / kRowGroups, x0 = 4 * (g % kRowGroups);
        const float4 v = t4[g];
        const bool row_in = (unsigned)(y - sc.ty0) < (unsigned)sc.wy;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (!(row_in && (unsigned)(x0 + k - sc.tx0) < (unsigned)sc.wx))
                omax = fmaxf(omax, fabsf(f4_get(v, k)));
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) omax = fmaxf(omax, __shfl_xor(omax, d, kWave));
    if (((int)threadIdx.x & (kWave - 1)) == 0) wmax[threadIdx.x / kWave] = omax;
    const float* win = tile + (size_t)sc.ty0 * kTilePitch + sc.tx0;
    const WindowMoments m =
        stored_moments(cls, win);
    if (threadIdx.x == 0) {
        float o = 0.0f;
        for (int w = 0; w < kWaves; ++w) o = fmaxf(o, wmax[w]);
        out_V[n] = m.V;
        out_outside_max[n] = o;
    }
}

// Plain streaming copy: the known-size reference kernel used to calibrate
// hardware byte counters against bytes actually moved.
__global__ __launch_bounds__(256) void k_stream_copy(u32x4* dst, const u32x4* src,
                                                     size_t nvec) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec;
         i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Max word of S into *out_max: 16 B loads on the aligned body, a per-wave
// maximum, then one atomic per wave that saw a nonzero word.
__global__ __launch_bounds__(256) void k_verify_S(const uint32_t* S, size_t n,
                                                  uint32_t* out_max) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t head = (size_t)((0u - (uint32_t)(uintptr_t)S) & 15u) >> 2;
    if (head > n) head = n;
    uint32_t m = tid < head ? S[tid] : 0u;
    const u32x4* body = reinterpret_cast<const u32x4*>(S + head);
    const size_t nv = (n - head) >> 2;
    for (size_t i = tid; i < nv; i += stride) {
        const u32x4 v = body[i];
        m = max(m, max(max(v.x, v.y), max(v.z, v.w)));
    }
    const size_t done = head + 4 * nv;
    if (tid < n - done) m = max(m, S[done + tid]);
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d, kWave));
    if (((int)threadIdx.x & (kWave - 1)) == 0 && m) atomicMax(out_max, m);
}

// Trajectory records (k_pack_traj's fields, src/kernels.cu:1242-1265) of 64
// cells per one-wave workgroup: the 64 CellStates (12 KiB) arrive in LDS by
// 16 B loads, lane c packs cell c into LDS, and the 3 KiB of records leave by
// 16 B stores (write-combined when out is mapped host memory).
constexpr int kCellVecs = (int)(sizeof(pfh_cell_state) / 16);
constexpr int kTrajVecs = (int)(sizeof(pfh_traj_packed_cell) / 16);
static_assert(sizeof(pfh_cell_state) % 16 == 0 && sizeof(pfh_traj_packed_cell) % 16 == 0,
              "16 B record vectors");

__global__ __launch_bounds__(kWave) void k_pack_traj(const pfh_cell_state* cell,
                                                     const uint8_t* clsv,
                                                     pfh_traj_packed_cell* out, int N,
                                                     int L) {
    __shared__ u32x4 in[kWave * kCellVecs];
    __shared__ u32x4 rec[kWave * kTrajVecs];
    const int lane = (int)threadIdx.x;
    const int base = (int)blockIdx.x * kWave;
    const int cnt = min(kWave, N - base);
    const u32x4* src = reinterpret_cast<const u32x4*>(cell + base);
    for (int i = lane; i < cnt * kCellVecs; i += kWave) in[i] = src[i];
    __syncthreads();
    if (lane < cnt) {
        const pfh_cell_state& cs = *reinterpret_cast<const pfh_cell_state*>(&in[lane * kCellVecs]);
        pfh_traj_packed_cell& t = *reinterpret_cast<pfh_traj_packed_cell*>(&rec[lane * kTrajVecs]);
        const double V = cs.V > 0.0 ? cs.V : 1.0;
        const double Ld = (double)L;
        const double cx = (double)cs.gx0 + cs.Cx / V;
        const double cy = (double)cs.gy0 + cs.Cy / V;
        t.global_id = cs.global_id;
        t.cls = (int)clsv[base + lane];
        t.cx = (float)(cx - floor(cx / Ld) * Ld);
        t.cy = (float)(cy - floor(cy / Ld) * Ld);
        t.vx = cs.vx;
        t.vy = cs.vy;
        t.theta = cs.theta;
        t.volume = (float)cs.V;
        t.perim = (float)cs.perim;
        t.gamma = cs.gamma;
        t.v_A = cs.v_A;
        t.phi_max = cs.phi_max;
    }
    __syncthreads();
    u32x4* dst = reinterpret_cast<u32x4*>(out + base);
    for (int i = lane; i < cnt * kTrajVecs; i += kWave) dst[i] = rec[i];
}

// ---- Morton ordering of the cell queue ----
// Key of cell i: 2D Morton code (x in the even bits, y in the odd bits, 16
// bits each) of its truncated centroid, wrapped into the domain
// (src/kernels.cu:1271-1279). The queue is the cells sorted by (key, i).
//
// One workgroup of 1024 threads: a stable least-significant-digit radix sort
// of the indices on 4-bit digits, entirely in LDS. Per pass, each wave ranks
// its 64 elements in their digit bucket with 16 ballots, the per-(digit,
// round, wave) counts are scanned in that order (stable across waves and
// rounds of 1024 elements), and the indices move to their bucket positions.
// Only as many passes run as the domain's coordinates have bits.
constexpr int kMortonMax = 16384;
constexpr int kMortonRounds = kMortonMax / kNT;
constexpr int kDigitBits = 4;
constexpr int kBuckets = 1 << kDigitBits;
constexpr int kCountSlots = kBuckets * kMortonRounds * kWaves;   // 4096

__device__ __forceinline__ uint32_t spread_bits16(uint32_t v) {
    // bit i of v -> bit 2i of the result (v < 2^16)
    uint32_t r = 0u;
#pragma unroll
    for (int i = 0; i < 16; ++i) r |= ((v >> i) & 1u) << (2 * i);
    return r;
}

__global__ __launch_bounds__(kNT) void k_morton_sort(const pfh_cell_state* cell,
                                                     uint32_t* perm, int N, int L,
                                                     int passes) {
    __shared__ uint32_t key[kMortonMax];
    __shared__ uint16_t idx[2][kMortonMax];
    __shared__ uint32_t cnt[kCountSlots];
    __shared__ uint32_t wsum[kWaves];
    const int tid = (int)threadIdx.x;
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    const int rounds = (N + kNT - 1) / kNT;
    for (int i = tid; i < N; i += kNT) {
        const pfh_cell_state& cs = cell[i];
        const double V = cs.V > 0.0 ? cs.V : 1.0;
        const uint32_t x = (uint32_t)wrapi(cs.gx0 + (int)(cs.Cx / V), L);
        const uint32_t y = (uint32_t)wrapi(cs.gy0 + (int)(cs.Cy / V), L);
        key[i] = spread_bits16(x & 0xFFFFu) | (spread_bits16(y & 0xFFFFu) << 1);
        idx[0][i] = (uint16_t)i;
    }
    __syncthreads();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
    int cur = 0;
    for (int pass = 0; pass < passes; ++pass) {
        const int shift = pass * kDigitBits;
        uint32_t digit[kMortonRounds], rank[kMortonRounds];
        // 1. per-wave digit counts and ranks within the wave
#pragma unroll
        for (int r = 0; r < kMortonRounds; ++r) {
            if (r >= rounds) break;
            const int i = r * kNT + tid;
            const uint32_t d = i < N ? (key[idx[cur][i]] >> shift) & (kBuckets - 1)
                                     : (uint32_t)kBuckets;
            uint64_t mine = 0ull;
            uint32_t c = 0u;
#pragma unroll
            for (int k = 0; k < kBuckets; ++k) {
                const uint64_t m = __ballot(d == (uint32_t)k);
                if (d == (uint32_t)k) mine = m;
                if (lane == k) c = (uint32_t)__popcll(m);
            }
            digit[r] = d;
            rank[r] = (uint32_t)__popcll(mine & lt_mask);
            if (lane < kBuckets) cnt[(lane * rounds + r) * kWaves + wave] = c;
        }
        __syncthreads();
        // 2. exclusive scan of the counts in (digit, round, wave) order
        const int slots = kBuckets * rounds * kWaves;
        const int per = (slots + kNT - 1) / kNT;
        uint32_t local = 0u;
        for (int k = 0; k < per; ++k) {
            const int s = tid * per + k;
            if (s < slots) local += cnt[s];
        }
        uint32_t incl = local;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, d, kWave);
            if (lane >= d) incl += o;
        }
        if (lane == kWave - 1) wsum[wave] = incl;
        __syncthreads();
        uint32_t run = incl - local;
        for (int w = 0; w < wave; ++w) run += wsum[w];
        for (int k = 0; k < per; ++k) {
            const int s = tid * per + k;
            if (s < slots) {
                const uint32_t c = cnt[s];
                cnt[s] = run;
                run += c;
            }
        }
        __syncthreads();
        // 3. stable moves into the other index buffer
#pragma unroll
        for (int r = 0; r < kMortonRounds; ++r) {
            if (r >= rounds) break;
            const int i = r * kNT + tid;
            if (i < N)
                idx[cur ^ 1][cnt[(digit[r] * rounds + r) * kWaves + wave] + rank[r]] =
                    idx[cur][i];
        }
        __syncthreads();
        cur ^= 1;
    }
    for (int i = tid; i < N; i += kNT) perm[i] = idx[cur][i];
}

// -------------------------------------------------------------------------
// Independent dense velocity observer (src/velocity_moments.cu:43-128): one
// 256-thread workgroup per cell, straight from the step's input field and
// aggregate in global memory (no window staging, no shift, no class
// hysteresis: none of the step's code paths), two passes over the window:
// the interaction force, then the centroid rates of the four velocity
// sources (passive interfacial, overlap, area; advection) in fp64.
// Lane-strided sums, 64-lane trees, waves in ascending order.
// -------------------------------------------------------------------------
constexpr int kObsNT = 256, kObsWaves = kObsNT / kWave;

template <int K>
__device__ void obs_block_sum(double (&v)[K], double* sh) {
    const int lane = (int)threadIdx.x & (kWave - 1), wave = (int)threadIdx.x / kWave;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        v[j] = wave_sum(v[j]);
        if (lane == 0) sh[j * kObsWaves + wave] = v[j];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            double t = 0.0;
            for (int w = 0; w < kObsWaves; ++w) t += sh[j * kObsWaves + w];
            sh[j * kObsWaves] = t;
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(kObsNT) void k_velocity_observe(const pfh2d_step_args A,
                                                             pfh_moment_accum* out,
                                                             double pdt) {
    __shared__ double sh[8 * kObsWaves];
    __shared__ double vel[4];
    const int n = (int)blockIdx.x;
    const pfh_cell_state& c = A.cell[n];
    const Shape sc = shape_of((int)c.cls);
    const int L = A.L, P = A.P, gx0 = c.gx0, gy0 = c.gy0;
    const float* tile = A.phi_in + (size_t)n * kTileArea;
    auto at = [&](int x, int y) -> float {
        return ((unsigned)x < (unsigned)sc.wx && (unsigned)y < (unsigned)sc.wy)
            ? tile[(size_t)(sc.ty0 + y) * kTilePitch + sc.tx0 + x] : 0.0f;
    };
    // S_other at a window pixel; an invalid aggregate (S below the cell's own
    // share) gives NaN, so the sample is refused downstream
    auto other = [&](int x, int y, float p) -> float {
        const uint32_t all = A.S_rd[(size_t)wrap_once(gy0 + y, L) * P + wrap_once(gx0 + x, L)];
        const uint32_t self = q_of(p);
        return all >= self ? (float)(all - self) * kQInv : __int_as_float(0x7fc00000);
    };
    const int W = sc.wx * sc.wy;
    double f[2] = {0.0, 0.0};
    for (int k = (int)threadIdx.x; k < W; k += kObsNT) {
        const int y = k / sc.wx, x = k - y * sc.wx;
        const float p = at(x, y);
        const float gx = 0.5f * (at(x + 1, y) - at(x - 1, y));
        const float gy = 0.5f * (at(x, y + 1) - at(x, y - 1));
        const float so = other(x, y, p);
        // the same binary32 product as the step's interaction integrand
        f[0] += (double)(p * gx * so);
        f[1] += (double)(p * gy * so);
    }
    obs_block_sum(f, sh);
    if (threadIdx.x == 0) {
        const unsigned long long step = *A.step_rd;
        const Philox4 r = philox4x32_10(
            (uint32_t)(step & 0xFFFFFFFFull), (uint32_t)(step >> 32), (uint32_t)c.global_id,
            0xA5A5A5A5u, (uint32_t)(A.polarity_seed & 0xFFFFFFFFull),
            (uint32_t)(A.polarity_seed >> 32));
        float theta = c.theta;
        if (uniform53(r.v[0], r.v[1]) < A.p_tumble)
            theta = (float)(2.0 * kPi * uniform53(r.v[2], r.v[3]));
        double sd, cd;
        sincos_d((double)theta, &sd, &cd);
        vel[0] = (double)c.v_A * (double)(float)cd;
        vel[1] = (double)c.v_A * (double)(float)sd;
        vel[2] = (double)A.mot_coeff * sh[0];
        vel[3] = (double)A.mot_coeff * sh[kObsWaves];
    }
    __syncthreads();
    const double cx = c.Cx / c.V, cy = c.Cy / c.V;
    const double dw = (double)(A.bulk_scale * c.gamma);
    const double vol = (double)(float)(A.vol_scale * (A.A0 - c.V));
    const double mob = (double)(c.M_pf / 0.5f);
    // the advection uses the stored (binary32) velocity
    const double vx = (double)(float)(vel[0] + vel[2]);
    const double vy = (double)(float)(vel[1] + vel[3]);
    double m[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int k = (int)threadIdx.x; k < W; k += kObsNT) {
        const int y = k / sc.wx, x = k - y * sc.wx;
        const double p = (double)at(x, y);
        const double e = at(x + 1, y), w = at(x - 1, y);
        const double nn = at(x, y + 1), ss = at(x, y - 1);
        const double ne = at(x + 1, y + 1), nw = at(x - 1, y + 1);
        const double se = at(x + 1, y - 1), sw = at(x - 1, y - 1);
        const double lap =
            (((((4.0 * (((nn + ss) + e) + w) + ne) + nw) + se) + sw) - 20.0 * p) / 6.0;
        const double so = (double)other(x, y, (float)p);
        double src[4] = {(double)c.gamma * lap - ((dw * p) * (1.0 - p)) * (1.0 - 2.0 * p),
                         -((double)A.rep_coeff * p) * so, vol * p,
                         -(vx * (0.5 * (e - w)) + vy * (0.5 * (nn - ss)))};
        // the mobility scales the passive sources, never the advection
        if (mob != 1.0) {
            src[0] *= mob;
            src[1] *= mob;
            src[2] *= mob;
        }
        const double wxp = ((2.0 * ((double)x - cx)) * p) / c.V;
        const double wyp = ((2.0 * ((double)y - cy)) * p) / c.V;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m[2 * j] += wxp * src[j];
            m[2 * j + 1] += wyp * src[j];
        }
    }
    obs_block_sum(m, sh);
    if (threadIdx.x == 0) {
        pfh_moment_accum& z = out[n];
        for (int j = 0; j < 4; ++j) z.q[j] += pdt * vel[j];
        for (int j = 0; j < 6; ++j) z.q[4 + j] += pdt * sh[j * kObsWaves];
        z.q[10] += pdt * ((sh[6 * kObsWaves] - vel[0]) - vel[2]);
        z.q[11] += pdt * ((sh[7 * kObsWaves] - vel[1]) - vel[3]);
        ++z.count;
    }
}

}  // namespace pfh

// -------------------------------------------------------------------------
// C ABI
// -------------------------------------------------------------------------
namespace {
thread_local char g_last_error[256] = {0};
}  // namespace

namespace pfh_host {
int hip_status(hipError_t e, const char* what) {
    if (e == hipSuccess) return PFH_OK;
    snprintf(g_last_error, sizeof(g_last_error), "%s: %s", what,
             hipGetErrorString(e));
    return PFH_ERR_HIP;
}
int launch_status(const char* what) {
    return hip_status(hipGetLastError(), what);
}
int invalid(const char* what) {
    snprintf(g_last_error, sizeof(g_last_error), "invalid argument: %s", what);
    return PFH_ERR_INVALID;
}
int unsupported(const char* what) {
    snprintf(g_last_error, sizeof(g_last_error), "%s", what);
    return PFH_ERR_UNSUPPORTED;
}
}  // namespace pfh_host
using namespace pfh_host;

namespace {
// While the step after this one finds the field in the 256 MiB Infinity Cache,
// its stores go through the caches; larger populations store it
// non-temporally and leave the cache to the aggregate. us per step, cached /
// non-temporal: 1024 cells (162 MiB for both fields) 80.7 / 82.1, 1536 (243 MiB)
// 115.9 / 114.4, 2048 161.4 / 155.6, 4096 299.8 / 285.6. The line, 1314 cells, is
// where the two differences interpolate to none. It counts class-0 windows for
// every cell, and only class 0 has a body that streams: a population of larger
// windows is stored through the caches whatever its size.
constexpr size_t kStreamBytes = (size_t)208 << 20;
constexpr size_t kCellFieldBytes =
    2u * sizeof(float) * (size_t)pfh::kShapes[0].wx * (size_t)pfh::kShapes[0].wy;

// grid compute units: two 8-wave workgroups on each, or one of 16 waves where a
// cell would mostly be alone on its unit: no more cells than units, or three
// rounds of them, which pairs would take as two rounds of which the second is
// half empty. us per step on 256 units, pairs / 16 waves, cells of radius 20 and
// of radius 45 (larger classes among them):
//    256  28.9 / 25.1   32.1 / 31.2      768  69.5 / 60.8   81.4 / 72.3
//    288  38.5 / 36.4   40.7 / 41.6      896  74.6 / 71.1   86.6 / 84.4
//    384  39.7 / 39.0   45.0 / 46.2     1024  75.9 / 76.5   90.6 / 96.2
//    512  43.4 / 42.0   51.3 / 51.4     1280  94.5 / 101    113 / 119
//    560  63.6 / 51.8   71.3 / 59.1     2048   149 / 159    174 / 189
// Two rounds are pairs for the larger cells' sake; small ones lose 1 to 8% by
// it, and four rounds of up to 900 cells 3 to 9%. The check step and the ensemble
// behave as the plain step (check: 640 cells 51.0 / 42.5, 1024 57.3 / 58.4;
// ensemble: 666 cells 72.0 / 59.6, 1155 91.1 / 97.3). The spatial observer does
// not: its 8-wave build spills 49 registers where the other spills 10, and is
// the slower one at every size (288 cells 72.3 / 58.4, 1024 141 / 120).
bool one_cell_per_unit(int N, int grid) {
    const long long rounds = ((long long)N + grid - 1) / grid;
    return rounds <= 1 || rounds == 3;
}

template <bool kCheck, bool kBatch, int kObs>
void launch_k_step(const pfh2d_step_args& a, const int* run_if, const pfh2d_replica* reps,
                   const uint16_t* cell_rep, int grid, void* stream) {
    const dim3 pairs(2u * (unsigned)grid), threads8(8 * pfh::kWave);
    if (one_cell_per_unit(a.N, grid)) {
        hipLaunchKernelGGL((pfh::k_step<16, kCheck, kBatch, kObs>), dim3((unsigned)grid),
                           dim3(16 * pfh::kWave), 0, as_stream(stream), a, run_if, reps,
                           cell_rep);
        return;
    }
    if constexpr (!kCheck && kObs == 0) {
        if ((size_t)a.N * kCellFieldBytes > kStreamBytes) {
            hipLaunchKernelGGL((pfh::k_step<8, kCheck, kBatch, kObs, true>), pairs, threads8, 0,
                               as_stream(stream), a, run_if, reps, cell_rep);
            return;
        }
    }
    hipLaunchKernelGGL((pfh::k_step<8, kCheck, kBatch, kObs>), pairs, threads8, 0,
                       as_stream(stream), a, run_if, reps, cell_rep);
}
}  // namespace

extern "C" {

int pfh_abi_version(void) { return 10000; }

const char* pfh_last_error(void) { return g_last_error; }

int pfh2d_configure_step(void) {
    // k_step uses static LDS only; nothing to opt into on gfx950.
    return PFH_OK;
}

int pfh2d_configure_morton(int smem_bytes) {
    // The sort keeps its keys and index buffers in static LDS (sized for
    // 16384 cells); there is nothing to opt into on gfx950.
    if (smem_bytes <= 0 || smem_bytes > 160 * 1024) return invalid("morton smem");
    return PFH_OK;
}

int pfh2d_step_grid(int device) {
    int cus = 0;
    const int st = hip_status(
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device),
        "hipDeviceGetAttribute(multiProcessorCount)");
    if (st != PFH_OK) return st;
    return cus > 0 ? cus : 1;
}

namespace {
int step_launch(const pfh2d_step_args* a, const int* run_if, int grid, void* stream,
                bool check = false, int observation = PFH_OBSERVE_DISABLED) {
    if (!a) return invalid("args");
    if (observation == PFH_OBSERVE_SPATIAL && !a->moments)
        return invalid("a spatial observation needs the moment accumulators (moments)");
    if (grid <= 0 || a->N < 0 || a->L <= 0 || a->P < a->L || !a->phi_in ||
        !a->phi_out || !a->S_rd || !a->cell || !a->cell_cls ||
        !a->perm || !a->cursor_use || !a->cursor_clear || !a->step_rd ||
        !a->step_wr || !a->flags || (a->clear_ahead_words && !a->S_cl) ||
        a->parity_out < 0 || a->parity_out > 1)
        return invalid("step args");
    // Every window must fit strictly inside the periodic domain
    // (include/params.cuh:666-680), or S self-subtraction is not exact.
    if (a->L <= 286) return invalid("domain side must exceed 286");
    // the step addresses S with 32-bit byte offsets
    if (4ull * (unsigned long long)a->P * (unsigned long long)a->L > 0xFFFFFFFFull)
        return invalid("aggregate larger than 4 GiB");
    const pfh2d_replica* no_reps = nullptr;
    const uint16_t* no_map = nullptr;
    if (check)
        launch_k_step<true, false, 0>(*a, run_if, no_reps, no_map, grid, stream);
    else if (observation == PFH_OBSERVE_ADVECTION)
        launch_k_step<false, false, 1>(*a, run_if, no_reps, no_map, grid, stream);
    else if (observation == PFH_OBSERVE_SPATIAL)
        launch_k_step<false, false, 2>(*a, run_if, no_reps, no_map, grid, stream);
    else
        launch_k_step<false, false, 0>(*a, run_if, no_reps, no_map, grid, stream);
    return launch_status("k_step");
}
}  // namespace

int pfh2d_launch_step(const pfh2d_step_args* a, int grid, void* stream,
                      const void* l2_base, size_t l2_bytes, float l2_hit_ratio,
                      int observation) {
    (void)l2_base; (void)l2_bytes; (void)l2_hit_ratio;
    if (!a) return invalid("args");
    if (observation < PFH_OBSERVE_DISABLED || observation > PFH_OBSERVE_SPATIAL)
        return invalid("observation is 0 (disabled), 1 (advection) or 2 (spatial)");
    return step_launch(a, nullptr, grid, stream, false, observation);
}

int pfh2d_velocity_moments(const pfh2d_step_args* a, pfh_moment_accum* out,
                           double physical_dt, void* stream) {
    if (!a || !out) return invalid("velocity_moments: args and out are required");
    if (a->N <= 0 || a->L <= 286 || a->P < a->L || !a->phi_in || !a->S_rd || !a->cell ||
        !a->step_rd)
        return invalid("velocity_moments: step args");
    hipLaunchKernelGGL(pfh::k_velocity_observe, dim3((unsigned)a->N), dim3(pfh::kObsNT), 0,
                       as_stream(stream), *a, out, physical_dt);
    return launch_status("k_velocity_observe");
}

int pfh2d_launch_step_if(const pfh2d_step_args* a, const int* run_if, int grid,
                         void* stream) {
    return step_launch(a, run_if, grid, stream);
}

int pfh2d_launch_check_step_if(const pfh2d_step_args* a, const int* run_if, int grid,
                               void* stream) {
    if (a && a->S_sc) return invalid("a check step scatters nothing: S_sc must be NULL");
    return step_launch(a, run_if, grid, stream, true);
}

int pfh2d_launch_batch_step(const pfh2d_step_args* a, const pfh2d_replica* replicas,
                            const uint16_t* cell_replica, int num_replicas, int max_side,
                            int max_pitch, int grid, void* stream) {
    if (!a || !replicas || !cell_replica) return invalid("batch step: null argument");
    if (num_replicas <= 0 || num_replicas > 65536 || grid <= 0 || a->N <= 0 ||
        !a->phi_in || !a->phi_out || !a->S_rd || !a->S_sc || !a->cell || !a->cell_cls ||
        !a->perm || !a->cursor_use || !a->cursor_clear || !a->step_rd || !a->step_wr ||
        !a->flags || (a->clear_ahead_words && !a->S_cl) || a->parity_out < 0 ||
        a->parity_out > 1)
        return invalid("batch step args");
    // every replica's side must exceed the classes it can use: 256 is the
    // smallest side (class 4, 224 wide, still fits; the 286-wide fallback
    // class is then unavailable and a cell that needs it is flagged)
    if (max_side < 256 || max_pitch < max_side)
        return invalid("batch step: replica sides must be at least 256");
    if (4ull * (unsigned long long)max_pitch * (unsigned long long)max_side > 0xFFFFFFFFull)
        return invalid("aggregate larger than 4 GiB");
    launch_k_step<false, true, 0>(*a, nullptr, replicas, cell_replica, grid, stream);
    return launch_status("k_step (batched)");
}

int pfh2d_query_step_stats(int device, pfh_kernel_stats* out) {
    if (!out) return invalid("out");
    hipFuncAttributes fa{};
    int st = hip_status(hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(pfh::k_step<8, false>)),
                        "hipFuncGetAttributes(k_step)");
    if (st != PFH_OK) return st;
    int blocks = 0;
    st = hip_status(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                        &blocks, reinterpret_cast<const void*>(pfh::k_step<8, false>),
                        8 * pfh::kWave, 0),
                    "hipOccupancyMaxActiveBlocksPerMultiprocessor(k_step)");
    if (st != PFH_OK) return st;
    int max_threads = 0;
    if (hipDeviceGetAttribute(&max_threads, hipDeviceAttributeMaxThreadsPerMultiProcessor,
                              device) != hipSuccess || max_threads <= 0)
        max_threads = 2048;
    memset(out, 0, sizeof(*out));
    out->regs = fa.numRegs;
    out->local_bytes = fa.localSizeBytes;
    out->static_smem = (int)fa.sharedSizeBytes;
    out->dynamic_smem = 0;
    out->ctas_per_sm = blocks;
    out->warps_per_sm = blocks * 8;
    out->occupancy = (double)(blocks * 8 * pfh::kWave) / (double)max_threads;
    return PFH_OK;
}

int pfh2d_init_tiles(float* phi_a, float* phi_b, pfh_cell_state* cell,
                     const uint8_t* cls, int N, int L, const float* seed_cx,
                     const float* seed_cy, float radius_eff, float kappa_iface,
                     void* stream) {
    if (N < 0 || L <= 0 || (N > 0 && (!phi_a || !phi_b || !cell || !cls ||
                                      !seed_cx || !seed_cy)))
        return invalid("init_tiles");
    if (N == 0) return PFH_OK;
    if ((uintptr_t)phi_a % 16 || (uintptr_t)phi_b % 16)
        return invalid("init_tiles: tiles must be 16 B aligned");
    hipLaunchKernelGGL(pfh::k_init_tiles, dim3((unsigned)N, pfh::kInitBands), dim3(256), 0,
                       as_stream(stream), phi_a, phi_b, cell, cls, L, seed_cx, seed_cy,
                       radius_eff, kappa_iface);
    return launch_status("k_init_tiles");
}

int pfh2d_init_moments(pfh_cell_state* cell, const uint8_t* cls,
                       const float* phi, int N, void* stream) {
    if (N < 0 || (N > 0 && (!cell || !cls || !phi))) return invalid("init_moments");
    if (N == 0) return PFH_OK;
    hipLaunchKernelGGL(pfh::k_init_moments, dim3(N), dim3(pfh::kNT), 0,
                       as_stream(stream), cell, cls, phi, N);
    return launch_status("k_init_moments");
}

int pfh2d_scatter_all(const float* phi, const pfh_cell_state* cell,
                      const uint8_t* cls, uint32_t* S, int N, int L, int P,
                      uint32_t* flags, void* stream) {
    if (N < 0 || L <= 0 || P < L ||
        (N > 0 && (!phi || !cell || !cls || !S || !flags)))
        return invalid("scatter_all");
    if (N == 0) return PFH_OK;
    hipLaunchKernelGGL(pfh::k_scatter_all, dim3((unsigned)N, pfh::kScatterBands), dim3(256), 0,
                       as_stream(stream), phi, cell, cls, S, L, P, flags);
    return launch_status("k_scatter_all");
}

int pfh2d_zero_u32(uint32_t* p, size_t n, void* stream) {
    if (n == 0) return PFH_OK;
    if (!p) return invalid("zero_u32");
    size_t blocks = (n / 4 + 255) / 256 + 1;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(pfh::k_fill_u32, dim3((unsigned)blocks), dim3(256), 0,
                       as_stream(stream), p, n, 0u);
    return launch_status("k_fill_u32");
}

int pfh2d_verify_cells(const float* phi, const pfh_cell_state* cell,
                       const uint8_t* cls, int N, double* out_V,
                       float* out_outside_max, void* stream) {
    if (N < 0 || (N > 0 && (!phi || !cell || !cls || !out_V || !out_outside_max)))
        return invalid("verify_cells");
    if (N == 0) return PFH_OK;
    if ((uintptr_t)phi % 16) return invalid("verify_cells: tiles must be 16 B aligned");
    hipLaunchKernelGGL(pfh::k_verify_cells, dim3((unsigned)N), dim3(pfh::kNT), 0,
                       as_stream(stream), phi, cls, out_V, out_outside_max);
    return launch_status("k_verify_cells");
}

int pfh2d_verify_S(const uint32_t* S, size_t n, uint32_t* out_max, void* stream) {
    if (!out_max || (n > 0 && !S)) return invalid("verify_S");
    if (n == 0) return PFH_OK;
    size_t blocks = (n / 4 + 255) / 256 + 1;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(pfh::k_verify_S, dim3((unsigned)blocks), dim3(256), 0,
                       as_stream(stream), S, n, out_max);
    return launch_status("k_verify_S");
}

int pfh_stream_copy(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return PFH_OK;
    if (!dst || !src || (bytes & 15u) || ((uintptr_t)dst & 15u) || ((uintptr_t)src & 15u))
        return invalid("stream_copy needs 16 B aligned pointers and sizes");
    const size_t nvec = bytes / 16;
    size_t blocks = (nvec + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(pfh::k_stream_copy, dim3((unsigned)blocks), dim3(256), 0,
                       as_stream(stream), reinterpret_cast<pfh::u32x4*>(dst),
                       reinterpret_cast<const pfh::u32x4*>(src), nvec);
    return launch_status("k_stream_copy");
}

int pfh2d_pack_traj(const pfh_cell_state* cell, const uint8_t* cls,
                    pfh_traj_packed_cell* out, int N, int L, void* stream) {
    if (N < 0 || L <= 0 || (N > 0 && (!cell || !cls || !out))) return invalid("pack_traj");
    if (N == 0) return PFH_OK;
    if ((uintptr_t)out % 16 || (uintptr_t)cell % 16)
        return invalid("pack_traj: cell and out must be 16 B aligned");
    hipLaunchKernelGGL(pfh::k_pack_traj, dim3((unsigned)((N + pfh::kWave - 1) / pfh::kWave)),
                       dim3(pfh::kWave), 0, as_stream(stream), cell, cls, out, N, L);
    return launch_status("k_pack_traj");
}

int pfh2d_morton_sort(const pfh_cell_state* cell, uint32_t* perm, int N, int M,
                      int L, void* stream) {
    if (N <= 0 || M < N || (M & (M - 1)) != 0 || M > pfh::kMortonMax || L <= 0 || !cell ||
        !perm)
        return invalid("morton_sort");
    // Digit passes needed for the key bits the domain can produce: both
    // coordinates are below min(L, 2^16).
    int coord_bits = 0;
    while (coord_bits < 16 && ((L - 1) >> coord_bits) != 0) ++coord_bits;
    const int passes = (2 * coord_bits + pfh::kDigitBits - 1) / pfh::kDigitBits;
    hipLaunchKernelGGL(pfh::k_morton_sort, dim3(1), dim3(pfh::kNT), 0, as_stream(stream),
                       cell, perm, N, L, passes);
    return launch_status("k_morton_sort");
}

}  // extern "C"
