// Strict FP64 kernels: no FMA contraction, one IEEE operation per NumPy
// operation of the reference, so every result equals the FP64 oracle bit for bit.
#include "pp_internal.h"
#include "pp_bvh.inc"

#pragma clang fp contract(off)

#define PP_STRICT 1

namespace pp_strict {

#include "pp_fp64.inc"

// ---- per-step kernels with per-particle fields (the reference's Numba batch
// kernels) and the elementwise stages of _rk4_step_batch / the field algebra.

__global__ void __launch_bounds__(256) k_batch(const BatchArgs q) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= q.m) return;
    const d3 A = load3(q.a, i);
    d3 r;
    switch (q.which) {
        case PP_BK_POS:                                   // position_update_batch, pusher.py:402
            r = A + load3(q.b, i) * q.s1;
            break;
        case PP_BK_BORIS:                                 // boris_push_batch, pusher.py:376
            r = boris_kick(A, load3(q.b, i), load3(q.c, i), q.s1, q.qm);
            break;
        case PP_BK_VAY:                                   // vay_push_batch, pusher.py:389
            r = vay_rel_kick(A, load3(q.b, i), load3(q.c, i), q.s1, q.qm, q.c2, q.clight, q.vclamp);
            break;
        case PP_BK_RK4REL:                                // rk4_rel_dbetagamma_dt_batch, pusher.py:326
            r = rk4_rel_deriv(A, load3(q.b, i), load3(q.c, i), q.qm, q.c2);
            break;
        case PP_BK_LORENTZ:                               // pusher.py:828-829
            r = lorentz(A, load3(q.b, i), load3(q.c, i), q.qm);
            break;
        case PP_BK_AXPY: {                                // r + 0.5*dt*k  (pusher.py:834-835 ...)
            const double sc = q.s_pp ? q.s_pp[i] : q.s1;
            r = A + sc * load3(q.b, i);
            break;
        }
        case PP_BK_RK4COMB: {                             // pusher.py:882-883
            const double w = q.s_pp ? q.s_pp[i] : q.s1;
            r = A + w * (((load3(q.b, i) + 2.0 * load3(q.c, i)) + 2.0 * load3(q.d, i)) + load3(q.e, i));
            break;
        }
        case PP_BK_CLAMP:                                 // pusher.py:886-890
            r = clamp_speed(A, q.vclamp);
            break;
        default: {                                        // PP_BK_SCALEOFF, field.py:690
            r = A;
            if (q.f1) r = q.s1 * r;
            if (q.f2) r = r + mk3(q.s2, q.s2, q.s2);
            break;
        }
    }
    q.out[3 * i] = r.x;
    q.out[3 * i + 1] = r.y;
    q.out[3 * i + 2] = r.z;
}

__global__ void __launch_bounds__(256) k_util(int which, double* a, double* b, double* c, double* aos, int64_t m,
                                              double c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    if (which == PP_UT_AOS2SOA) {
        a[i] = aos[3 * i];
        b[i] = aos[3 * i + 1];
        c[i] = aos[3 * i + 2];
    } else if (which == PP_UT_SOA2AOS) {
        aos[3 * i] = a[i];
        aos[3 * i + 1] = b[i];
        aos[3 * i + 2] = c[i];
    } else if (which == PP_UT_V2U) {
        const d3 v = mk3(a[i], b[i], c[i]);
        const d3 u = rgamma(v, c2) * v;
        a[i] = u.x;
        b[i] = u.y;
        c[i] = u.z;
    } else {
        const d3 v = v_from_u(mk3(a[i], b[i], c[i]), c2);
        a[i] = v.x;
        b[i] = v.y;
        c[i] = v.z;
    }
}

DEV bool holds_u(const pp_bunch& b) { return b.algorithm == PP_ALG_BORIS_REL || b.algorithm == PP_ALG_VAY; }

__global__ void __launch_bounds__(256) k_velocity_rows(const double* __restrict__ vx, const double* __restrict__ vy,
                                                       const double* __restrict__ vz, const uint8_t* __restrict__ alive,
                                                       int ustate, const pp_bunch* __restrict__ bunches,
                                                       const int32_t* __restrict__ group, int64_t n, double c2,
                                                       double* __restrict__ aos) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || (alive && !alive[i])) return;
    d3 v = mk3(vx[i], vy[i], vz[i]);
    if (ustate || (bunches && holds_u(bunches[group[i]]))) v = v_from_u(v, c2);
    aos[3 * i] = v.x;
    aos[3 * i + 1] = v.y;
    aos[3 * i + 2] = v.z;
}

__global__ void __launch_bounds__(256) k_velocity_convert(double* vx, double* vy, double* vz,
                                                          const pp_bunch* __restrict__ bunches,
                                                          const int32_t* __restrict__ group, int64_t n, double c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !holds_u(bunches[group[i]])) return;
    const d3 v = mk3(vx[i], vy[i], vz[i]);
    const d3 u = rgamma(v, c2) * v;
    vx[i] = u.x;
    vy[i] = u.y;
    vz[i] = u.z;
}

// Host rows (mapped pinned memory) to state slots, v as u where ustate; and state slots back to host rows.
__global__ void __launch_bounds__(64) k_rows_to_state(const double* __restrict__ rows, StateView st, int64_t n, int ustate,
                                                      double c2) {
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    const d3 r = load3(rows, i);
    d3 v = load3(rows + 3 * n, i);
    if (ustate) v = rgamma(v, c2) * v;
    st.x[i] = r.x;
    st.y[i] = r.y;
    st.z[i] = r.z;
    st.vx[i] = v.x;
    st.vy[i] = v.y;
    st.vz[i] = v.z;
}

__global__ void __launch_bounds__(64) k_state_to_rows(StateView st, double* __restrict__ rows, int64_t n, int ustate,
                                                      double c2) {
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    d3 v = mk3(st.vx[i], st.vy[i], st.vz[i]);
    if (ustate) v = v_from_u(v, c2);
    rows[3 * i] = st.x[i];
    rows[3 * i + 1] = st.y[i];
    rows[3 * i + 2] = st.z[i];
    double* w = rows + 3 * n;
    w[3 * i] = v.x;
    w[3 * i + 1] = v.y;
    w[3 * i + 2] = v.z;
}

__global__ void k_add_i64(int64_t* p, int64_t v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p += v;
}

__global__ void __launch_bounds__(256) k_fill(double* p, double v, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Node table [node][ncomp] from z columns [cols][nz] of the components' grids (a periodic z axis gets node 0 again
// as its last).  Writes are contiguous; reads run along ncomp streams.
__global__ void __launch_bounds__(256) k_interleave(const MapParts src, const MapDesc d, int64_t cols,
                                                    double* __restrict__ raw) {
    const int64_t ngz = d.ng[2], nz = d.n[2], n = cols * ngz * d.ncomp;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t node = t / d.ncomp, comp = t - node * d.ncomp;
        const int64_t col = node / ngz, k = node - col * ngz;
        raw[t] = src.comp[comp][col * nz + (k < nz ? k : 0)];
    }
}

// Per-cell trilinear coefficients of every component from the raw node table.
__global__ void __launch_bounds__(256) k_build_coef(const MapDesc d, double* __restrict__ c64, float* __restrict__ c32) {
    const int64_t ncell = (int64_t)d.nc[0] * d.nc[1] * d.nc[2];
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ncell * d.ncomp) return;
    const int comp = (int)(t % d.ncomp);
    const int64_t cell = t / d.ncomp;
    const int k = (int)(cell % d.nc[2]);
    const int j = (int)((cell / d.nc[2]) % d.nc[1]);
    const int i = (int)(cell / ((int64_t)d.nc[2] * d.nc[1]));
    const int64_t ngz = d.ng[2], ngy = d.ng[1];
    const int i1 = d.n[0] > 1 ? i + 1 : i;
    const int j1 = d.n[1] > 1 ? j + 1 : j;
    const int k1 = d.n[2] > 1 ? k + 1 : k;   // periodic maps carry the wrap node at k = nz
    const double* v = d.raw + comp;
    auto at = [&](int a, int b, int c) { return v[(((int64_t)a * ngy + b) * ngz + c) * d.ncomp]; };
    const double c000 = at(i, j, k), c100 = at(i1, j, k), c010 = at(i, j1, k), c110 = at(i1, j1, k);
    const double c001 = at(i, j, k1), c101 = at(i1, j, k1), c011 = at(i, j1, k1), c111 = at(i1, j1, k1);
    double q[8];
    q[0] = c000;
    q[1] = c100 - c000;
    q[2] = c010 - c000;
    q[3] = c001 - c000;
    q[4] = (c110 - c100) - (c010 - c000);
    q[5] = (c101 - c100) - (c001 - c000);
    q[6] = (c011 - c010) - (c001 - c000);
    q[7] = ((c111 - c110) - (c101 - c100)) - ((c011 - c010) - (c001 - c000));
    const int64_t o = (cell * d.ncomp + comp) * 8;
    for (int e = 0; e < 8; ++e) {
        if (c64) c64[o + e] = q[e];
        if (c32) c32[o + e] = (float)q[e];
    }
}

// ---- few particles through a fused map: one particle per row of 16 lanes ---------------------------------
//
// A track of a few particles is one wavefront's chain of dependent lookups: with a lane per particle a gather was
// 126 FP64 operations for the interpolation and 48 loads behind six node reads in a chain (2.4 us of gather and
// step, whatever the number of particles).  Here lane c of a row interpolates component c (E 0..2, B 3..5) and
// lanes 8..13 do the same at a second position, so the two lookups of a pair run as one; the values reach all lanes
// by row broadcasts in registers.  RK4's second position r + dt/2 v is known with its first, and its third and
// fourth (r + dt/2 v2, r + dt v3) are both known once the first two derivatives are: two gathers in the chain per
// step, not four.  Corners are loaded at the guessed cell together with its nodes; lanes whose guess is off repeat.
// Every value goes through the same operations in the same order as in k_push64, so results are the same bits.

template <int LANE>
DEV double row_bcast(double v) {
    // row_newbcast: lane LANE of each row of 16 to the whole row
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + LANE, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + LANE, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// What one lane of a row interpolates: its component of the map and that component's chain of factors.
struct RowFE64 {
    const PushParams& p;
    const double* __restrict__ values;      // this lane's component of node 0
    double scale1, scale2, offset;
    int32_t has_offset, rf;
    bool second;                            // lanes 8..15: the second position

    DEV RowFE64(const PushParams& q, int lane16) : p(q) {
        second = lane16 >= 8;
        const int c = (lane16 & 7) < 6 ? (lane16 & 7) : 5;
        const bool b = c >= 3;
        const int comp = b ? q.B.comp0 + (c - 3) : q.E.comp0 + c;
        const MapDesc& m = q.E.map;
        values = m.raw + comp;
        scale1 = b ? q.B.scale1 : q.E.scale1;
        const int has2 = b ? q.B.has_scale2 : q.E.has_scale2;
        scale2 = has2 ? (b ? q.B.scale2 : q.E.scale2) : 1.0;        // a product with 1 changes no bit
        has_offset = b ? q.B.has_offset : q.E.has_offset;
        offset = b ? q.B.offset : q.E.offset;
        rf = b ? q.B.rf : q.E.rf;
    }

    // the corners of cell `base` in lerp8 order: x fastest, then y, then z
    DEV void corners(int64_t base, double f[8]) const {
        const MapDesc& m = p.E.map;
        const double* v = values + 6 * base;
        const int64_t sz = 6, sy = 6 * (int64_t)m.ng[2], sx = sy * m.ng[1];
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = v[(k & 1 ? sx : 0) + (k & 2 ? sy : 0) + (k & 4 ? sz : 0)];
    }

    // this lane's component at (x, y, z)
    DEV double value(double x, double y, double z, int64_t gs, int stage) const {
        const MapDesc& m = p.E.map;
        const double rfv = rf != PP_RF_NONE ? rf_factor(p, gs, stage, rf) : 1.0;
        if (m.periodic) z = wrap_periodic(z, m.lo[2], m.L, m.inv_d[2] * m.inv_nz);
        const AxisGuess qx = guess_axis(m, 0, x), qy = guess_axis(m, 1, y), qz = guess_axis(m, 2, z);
        StrictCell c;
        c.base = ((int64_t)qx.i * m.ng[1] + qy.i) * m.ng[2] + qz.i;
        double f[8];
        corners(c.base, f);
        if (guess_is_off(m, 0, qx, x) || guess_is_off(m, 1, qy, y) || guess_is_off(m, 2, qz, z)) {
            c = strict_locate_wrapped<true>(m, x, y, z);
            corners(c.base, f);
        } else {
            const double wx = (x - qx.g0) / (qx.g1 - qx.g0), wy = (y - qy.g0) / (qy.g1 - qy.g0),
                         wz = (z - qz.g0) / (qz.g1 - qz.g0);
            c.tx = dmax(0.0, dmin(wx, 1.0));
            c.ty = dmax(0.0, dmin(wy, 1.0));
            c.tz = dmax(0.0, dmin(wz, 1.0));
        }
        double raw = lerp8(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], c);
        const bool out = x < m.lo[0] || x > m.hi[0] || y < m.lo[1] || y > m.hi[1] || z < m.lo[2] || z > m.hi[2];
        raw = out ? m.fill : raw;
        double r = scale1 * raw;
        r = scale2 * r;
        r = has_offset ? r + offset : r;
        return r * rfv;
    }

    // E, B at the position of lanes 0..7 and of lanes 8..15
    DEV void pair(d3 r1, d3 r2, int64_t gs, int stage1, d3& E1, d3& B1, d3& E2, d3& B2) const {
        const double f = value(second ? r2.x : r1.x, second ? r2.y : r1.y, second ? r2.z : r1.z, gs,
                               second ? stage1 + 1 : stage1);
        E1 = mk3(row_bcast<0>(f), row_bcast<1>(f), row_bcast<2>(f));
        B1 = mk3(row_bcast<3>(f), row_bcast<4>(f), row_bcast<5>(f));
        E2 = mk3(row_bcast<8>(f), row_bcast<9>(f), row_bcast<10>(f));
        B2 = mk3(row_bcast<11>(f), row_bcast<12>(f), row_bcast<13>(f));
    }

    // the evaluator step64 and kick64 take: both halves of the row look up the same position
    DEV void operator()(int64_t, double x, double y, double z, int64_t gs, int stage, d3& E, d3& B) const {
        const double f = value(x, y, z, gs, stage);
        E = mk3(row_bcast<0>(f), row_bcast<1>(f), row_bcast<2>(f));
        B = mk3(row_bcast<3>(f), row_bcast<4>(f), row_bcast<5>(f));
    }
};

// The RK4 step of step64 with its four gathers in two pairs.
template <int ALG>
DEV void rk4_row_step(d3& r, d3& v, double dt, int64_t gs, const RowFE64& fe, const AlgConst& p) {
    constexpr bool REL = (ALG == PP_ALG_RK4_REL);
    auto deriv = [&](d3 vv, d3 ee, d3 bb) {
        if constexpr (REL) return rk4_rel_deriv(vv, ee, bb, p.qm, p.c2);
        else return lorentz(vv, ee, bb, p.qm);
    };
    const double hdt = 0.5 * dt;
    d3 E1, B1, E2, B2;
    const d3 r2 = r + hdt * v;
    fe.pair(r, r2, gs, 0, E1, B1, E2, B2);
    const d3 k1v = deriv(v, E1, B1);
    const d3 v2 = v + hdt * k1v;
    const d3 k2v = deriv(v2, E2, B2);
    const d3 v3 = v + hdt * k2v;
    const d3 r3 = r + hdt * v2;
    const d3 r4 = r + dt * v3;
    fe.pair(r3, r4, gs, 2, E1, B1, E2, B2);
    const d3 k3v = deriv(v3, E1, B1);
    const d3 v4 = v + dt * k3v;
    const d3 k4v = deriv(v4, E2, B2);
    const double w = dt / 6.0;
    r = r + w * (((v + 2.0 * v2) + 2.0 * v3) + v4);
    v = v + w * (((k1v + 2.0 * k2v) + 2.0 * k3v) + k4v);
    if constexpr (REL) v = clamp_speed(v, p.vclamp);
}

// One wavefront per block: four particles, spread over as many CUs as there are blocks.  Rows beyond the last
// particle repeat it and write nothing, so every lane takes part in the broadcasts.
template <int ALG>
__global__ void __launch_bounds__(64) k_push64_row(const PushParams p) {
    const int lane16 = threadIdx.x & 15;
    const int64_t at = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 4);
    const bool live = at < p.n;
    const int64_t i = live ? at : p.n - 1;
    const RowFE64 fe(p, lane16);
    const AlgConst ac = alg_const(p);
    const double dt = p.dt_pp ? p.dt_pp[i] : p.dt;
    d3 r = mk3(p.x[i], p.y[i], p.z[i]);
    d3 v = mk3(p.vx[i], p.vy[i], p.vz[i]);
    d3 vrec = v;
    if (p.kick_only) {
        if constexpr (ALG == PP_ALG_BORIS || ALG == PP_ALG_BORIS_REL || ALG == PP_ALG_VAY)
            v = kick64<ALG>(i, r, v, dt, p.step0, fe, ac);
    } else {
        const int64_t row = p.ids ? (int64_t)p.ids[i] : i;
        const bool writes = p.r_hist != nullptr && live && lane16 < 6 && row >= 0 && row < p.hist_rows;
        double* out = (lane16 < 3 ? p.r_hist + lane16 : p.v_hist + (lane16 - 3));
        int64_t rec_left = p.rec_every - (p.step0 % p.rec_every);
        int64_t rec_idx = p.step0 / p.rec_every + 1;
        for (int64_t s = 0; s < p.nsteps; ++s) {
            if constexpr (ALG == PP_ALG_RK4 || ALG == PP_ALG_RK4_REL) {
                rk4_row_step<ALG>(r, v, dt, p.step0 + s, fe, ac);
                vrec = v;
            } else {
                step64<ALG>(i, r, v, vrec, dt, p.step0 + s, fe, ac);
            }
            if (--rec_left == 0) {
                rec_left = p.rec_every;
                if (writes && rec_idx < p.n_records) {
                    const d3 w = lane16 < 3 ? r : vrec;
                    const int c = lane16 < 3 ? lane16 : lane16 - 3;
                    out[(rec_idx * p.hist_rows + row) * 3] = c == 0 ? w.x : (c == 1 ? w.y : w.z);
                }
                ++rec_idx;
            }
        }
    }
    if (live && lane16 == 0) {
        p.x[i] = r.x;
        p.y[i] = r.y;
        p.z[i] = r.z;
        p.vx[i] = v.x;
        p.vy[i] = v.y;
        p.vz[i] = v.z;
    }
}

// Launches k_push64_row takes: one 3-D six-component map of evenly spaced axes, no alive mask, and few enough
// particles that the rows' redundant arithmetic costs less than the chain it shortens.  A SIMD holds 3 (RK4) or 1
// wavefronts of rows there.  100 steps through a 97 x 81 x 113 map, rows / a lane per particle in ms:
//   rk4    1: 0.17 / 0.46   4096: 0.19 / 0.60   8192: 0.28 / 0.60   16384: 0.53 / 0.56   32768: 1.01 / 0.58
//   vay    1: 0.15 / 0.20   4096: 0.17 / 0.24   8192: 0.28 / 0.24   16384: 0.52 / 0.24
//   boris  1: 0.10 / 0.14   4096: 0.12 / 0.19   8192: 0.17 / 0.19   16384: 0.30 / 0.18
// (1000 RK4 steps of 7 particles with a record per step: 9.6 -> 1.75 ms of device time.)
constexpr int64_t kRowMaxRk4 = 12288, kRowMaxSingle = 4096;

static bool row_route(int alg, const PushParams& p) {
    if (p.mesh || p.alive || !p.fused || !p.E.map.uniform || !fused_3d(p)) return false;
    return p.n <= (alg == PP_ALG_RK4 || alg == PP_ALG_RK4_REL ? kRowMaxRk4 : kRowMaxSingle);
}

static inline unsigned grid_for(int64_t n, int block) { return (unsigned)((n + block - 1) / block); }

#define PP_STRICT_SINGLE(L, U)                                                                                \
    case PP_ALG_LEAPFROG: hipLaunchKernelGGL((k_push64<PP_ALG_LEAPFROG, L, U>), g, b, 0, s, p); break;       \
    case PP_ALG_BORIS: hipLaunchKernelGGL((k_push64<PP_ALG_BORIS, L, U>), g, b, 0, s, p); break;             \
    case PP_ALG_YOSHIDA: hipLaunchKernelGGL((k_push64<PP_ALG_YOSHIDA, L, U>), g, b, 0, s, p); break;         \
    case PP_ALG_VAY_REL: hipLaunchKernelGGL((k_push64<PP_ALG_VAY_REL, L, U>), g, b, 0, s, p); break;         \
    case PP_ALG_YOSHIDA_REL: hipLaunchKernelGGL((k_push64<PP_ALG_YOSHIDA_REL, L, U>), g, b, 0, s, p); break; \
    case PP_ALG_BORIS_REL: hipLaunchKernelGGL((k_push64<PP_ALG_BORIS_REL, L, U>), g, b, 0, s, p); break;     \
    case PP_ALG_VAY: hipLaunchKernelGGL((k_push64<PP_ALG_VAY, L, U>), g, b, 0, s, p); break;

#define PP_STRICT_RK4(L, U)                                                                                   \
    case PP_ALG_RK4: hipLaunchKernelGGL((k_push64<PP_ALG_RK4, L, U>), g, b, 0, s, p); break;                 \
    case PP_ALG_RK4_REL: hipLaunchKernelGGL((k_push64<PP_ALG_RK4_REL, L, U>), g, b, 0, s, p); break;

#define PP_STRICT_CASES(L, U)                                                                                 \
    switch (alg) {                                                                                            \
        PP_STRICT_SINGLE(L, U)                                                                                \
        PP_STRICT_RK4(L, U)                                                                                   \
        default: return hipErrorInvalidValue;                                                                 \
    }

// The general build of terms that share no map: with all corners of a lookup in flight it holds two wavefronts per
// SIMD, plane by plane three or four.  Over the former build (all corners, the fused map's code in it too), 100 Boris
// steps through an E map and a constant B / a B map of its own: 0.96 / 1.01 at 1e4 particles, 0.96 / 1.01 at 1e5 (all
// corners), 0.88 / 0.87 at 2e5, 0.83 / 0.82 at 1e6 (plane by plane; 2.56 -> 2.13 and 3.92 -> 3.22 ms); RK4, which
// holds two wavefronts either way, keeps all corners (0.90 / 0.92 at 1e6).
constexpr int64_t kGeneralAll = 2 * 4 * 256 * 64;

template <int ALG>
static void launch_row(const PushParams& p, hipStream_t s) {
    hipLaunchKernelGGL(k_push64_row<ALG>, dim3(grid_for(p.n, 4)), dim3(64), 0, s, p);
}

static hipError_t launch_push_row(int alg, const PushParams& p, hipStream_t s) {
    switch (alg) {
        case PP_ALG_LEAPFROG: launch_row<PP_ALG_LEAPFROG>(p, s); break;
        case PP_ALG_BORIS: launch_row<PP_ALG_BORIS>(p, s); break;
        case PP_ALG_RK4: launch_row<PP_ALG_RK4>(p, s); break;
        case PP_ALG_YOSHIDA: launch_row<PP_ALG_YOSHIDA>(p, s); break;
        case PP_ALG_VAY_REL: launch_row<PP_ALG_VAY_REL>(p, s); break;
        case PP_ALG_RK4_REL: launch_row<PP_ALG_RK4_REL>(p, s); break;
        case PP_ALG_YOSHIDA_REL: launch_row<PP_ALG_YOSHIDA_REL>(p, s); break;
        case PP_ALG_BORIS_REL: launch_row<PP_ALG_BORIS_REL>(p, s); break;
        case PP_ALG_VAY: launch_row<PP_ALG_VAY>(p, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_push(int alg, const PushParams& p, int block, hipStream_t s) {
    if (row_route(alg, p)) return launch_push_row(alg, p, s);
    if (block <= 0) block = 256;
    const dim3 g(grid_for(p.n, block)), b(block);
    const int fields = fields_case(p);
    if (p.mesh) {
        if (fields == kFieldsMap3dAny) PP_STRICT_CASES(true, kFieldsMap3dAny)
        else if (fields == kFieldsMap3dAnyRF) PP_STRICT_CASES(true, kFieldsMap3dAnyRF)
        else if (fields == kFieldsFusedStatic) PP_STRICT_CASES(true, kFieldsFusedStatic)
        else if (fields == kFieldsFusedRF) PP_STRICT_CASES(true, kFieldsFusedRF)
        else PP_STRICT_CASES(true, kFieldsGeneral)
    } else if (fields == kFieldsUniform) {
        PP_STRICT_CASES(false, kFieldsUniform)
    } else if (fields == kFieldsMap3d) {
        PP_STRICT_CASES(false, kFieldsMap3d)
    } else if (fields == kFieldsMap3dRF) {
        PP_STRICT_CASES(false, kFieldsMap3dRF)
    } else if (fields == kFieldsMap3dAny) {
        PP_STRICT_CASES(false, kFieldsMap3dAny)
    } else if (fields == kFieldsMap3dAnyRF) {
        PP_STRICT_CASES(false, kFieldsMap3dAnyRF)
    } else if (fields == kFieldsFusedStatic) {
        PP_STRICT_CASES(false, kFieldsFusedStatic)
    } else if (fields == kFieldsFusedRF) {
        PP_STRICT_CASES(false, kFieldsFusedRF)
    } else if (p.n > kGeneralAll) {
        switch (alg) {
            PP_STRICT_SINGLE(false, kFieldsGeneralMany)
            PP_STRICT_RK4(false, kFieldsGeneral)
            default: return hipErrorInvalidValue;
        }
    } else {
        PP_STRICT_CASES(false, kFieldsGeneral)
    }
    return hipGetLastError();
}

hipError_t launch_push_sum(int alg, const PushParams& p, const SumParams& t, int block, hipStream_t s) {
    if (block <= 0) block = 256;
    const dim3 g(grid_for(p.n, block)), b(block);
    switch (alg) {
        case PP_ALG_LEAPFROG: hipLaunchKernelGGL(k_push64_sum<PP_ALG_LEAPFROG>, g, b, 0, s, p, t); break;
        case PP_ALG_BORIS: hipLaunchKernelGGL(k_push64_sum<PP_ALG_BORIS>, g, b, 0, s, p, t); break;
        case PP_ALG_RK4: hipLaunchKernelGGL(k_push64_sum<PP_ALG_RK4>, g, b, 0, s, p, t); break;
        case PP_ALG_YOSHIDA: hipLaunchKernelGGL(k_push64_sum<PP_ALG_YOSHIDA>, g, b, 0, s, p, t); break;
        case PP_ALG_VAY_REL: hipLaunchKernelGGL(k_push64_sum<PP_ALG_VAY_REL>, g, b, 0, s, p, t); break;
        case PP_ALG_RK4_REL: hipLaunchKernelGGL(k_push64_sum<PP_ALG_RK4_REL>, g, b, 0, s, p, t); break;
        case PP_ALG_YOSHIDA_REL: hipLaunchKernelGGL(k_push64_sum<PP_ALG_YOSHIDA_REL>, g, b, 0, s, p, t); break;
        case PP_ALG_BORIS_REL: hipLaunchKernelGGL(k_push64_sum<PP_ALG_BORIS_REL>, g, b, 0, s, p, t); break;
        case PP_ALG_VAY: hipLaunchKernelGGL(k_push64_sum<PP_ALG_VAY>, g, b, 0, s, p, t); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_field_eval(const FieldDev& f, const double* pts, int64_t m, double rf, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_field_eval64, dim3(grid_for(m, 256)), dim3(256), 0, s, f, pts, m, rf, out);
    return hipGetLastError();
}

hipError_t launch_batch_kernel(const BatchArgs& args, hipStream_t s) {
    hipLaunchKernelGGL(k_batch, dim3(grid_for(args.m, 256)), dim3(256), 0, s, args);
    return hipGetLastError();
}

hipError_t launch_util(int which, double* a, double* b, double* c, double* aos, int64_t m, double c2, hipStream_t s) {
    hipLaunchKernelGGL(k_util, dim3(grid_for(m, 256)), dim3(256), 0, s, which, a, b, c, aos, m, c2);
    return hipGetLastError();
}

hipError_t launch_velocity_rows(const double* vx, const double* vy, const double* vz, const uint8_t* alive, bool ustate,
                                const pp_bunch* bunches, const int32_t* group, int64_t n, double c2, double* aos,
                                hipStream_t s) {
    hipLaunchKernelGGL(k_velocity_rows, dim3(grid_for(n, 256)), dim3(256), 0, s, vx, vy, vz, alive, ustate ? 1 : 0,
                       bunches, group, n, c2, aos);
    return hipGetLastError();
}

hipError_t launch_velocity_convert(double* vx, double* vy, double* vz, const pp_bunch* bunches, const int32_t* group,
                                   int64_t n, double c2, hipStream_t s) {
    hipLaunchKernelGGL(k_velocity_convert, dim3(grid_for(n, 256)), dim3(256), 0, s, vx, vy, vz, bunches, group, n, c2);
    return hipGetLastError();
}

hipError_t launch_rows_to_state(const double* rows, const StateView& st, int64_t n, bool ustate, double c2,
                                hipStream_t s) {
    hipLaunchKernelGGL(k_rows_to_state, dim3(grid_for(n, 64)), dim3(64), 0, s, rows, st, n, ustate ? 1 : 0, c2);
    return hipGetLastError();
}

hipError_t launch_state_to_rows(const StateView& st, double* rows, int64_t n, bool ustate, double c2, hipStream_t s) {
    hipLaunchKernelGGL(k_state_to_rows, dim3(grid_for(n, 64)), dim3(64), 0, s, st, rows, n, ustate ? 1 : 0, c2);
    return hipGetLastError();
}

hipError_t launch_fill(double* p, double v, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

hipError_t launch_add_i64(int64_t* p, int64_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_add_i64, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}

hipError_t launch_interleave(const MapParts& src, const MapDesc& d, int64_t cols, double* raw, hipStream_t s) {
    const unsigned g = loop_blocks(cols * d.ng[2] * d.ncomp);
    hipLaunchKernelGGL(k_interleave, dim3(g), dim3(256), 0, s, src, d, cols, raw);
    return hipGetLastError();
}

hipError_t launch_build_coef(const MapDesc& d, double* c64, float* c32, hipStream_t s) {
    const int64_t work = (int64_t)d.nc[0] * d.nc[1] * d.nc[2] * d.ncomp;
    hipLaunchKernelGGL(k_build_coef, dim3(grid_for(work, 256)), dim3(256), 0, s, d, c64, c32);
    return hipGetLastError();
}

}  // namespace pp_strict
