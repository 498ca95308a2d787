// mm_stage.h -- the fused stage kernel: inverse x transform of the demag
// spectrum, the per-cell epilogue (field terms, LLG, stage combination) and
// the next stage input's x transform.  Device records, the kernels and the
// launch functions, which mm_stage.hip instantiates per precision and physics
// class (one object file each, so that they compile side by side).
#ifndef MM_STAGE_H
#define MM_STAGE_H

#include <hip/hip_runtime.h>

#include <cstddef>

#include "mm_cell.h"
#include "mm_conv.h"
#include "mm_reduce.h"

// device control block
struct StepCtl {
    double t, h, h_last;
    long long attempts, rejections, accepted, target;
    int cur;                       // index of the current y buffer
    int stop;                      // accepted == target: remaining launches exit
    // relaxation stop rule, checked on the first attempt from every
    // check_every-th accepted state (condition.py:169-200 checks state.step)
    int relax_mode;                // MM_RELAX_NONE / _DMDT / _DEG_PER_NS
    int relax_every;
    int relaxed;                   // the current state satisfied the rule
    int have_last;                 // relax_last holds a previous deg/ns value
    double relax_thr, relax_value, relax_last;
    long long last_check;          // accepted count of the last check
    // end time (RungeKutta.evolve's t_max, runge_kutta.py:74-78): an accepted
    // step past t_max is redone from the same state with h = t_max - t and
    // taken without error check (forced); the controller's h resumes after it
    int tmax_on, forced;
    double t_max, h_saved;
    // stop time without clipping (the solver loop's stop conditions on t,
    // solver.py:110-112 with condition.py:145-157, which name no time of
    // interest): the run stops after the first accepted step that ends at
    // t >= t_stop, and that step keeps its full length
    int tstop_on;
    double t_stop;
};

// a per-cell parameter that is either uniform (p == null) or an array
template <typename T> struct Param {
    const T *p;
    T u;
    __device__ __forceinline__ T at(size_t i) const { return p ? gfield(p)[i] : u; }
};
template <typename T> struct VParam {
    const T *p; // 3n SoA or null
    T u[3];
    __device__ __forceinline__ V3<T> at(size_t n, size_t i) const
    {
        return p ? v3<T>(gfield(p)[i], gfield(p)[n + i], gfield(p)[2 * n + i]) : v3<T>(u[0], u[1], u[2]);
    }
};

enum { FORM_SUM = 0, FORM_SEQ = 1 };

// Physics compiled into a stage kernel beyond uniform exchange, uniaxial
// anisotropy and Zeeman field.  GEN_CUB: cubic anisotropy.  GEN_ALL: that,
// exchange with per-cell Ms/A and 64-bit addresses.
// Cubic anisotropy ran in GEN_ALL before, whose FP32 inner stage spilled
// registers at 8 waves per SIMD: 512x512x32 FP32 inner stages 344 -> 300 us,
// final 392 -> 374 us, 1 ps 124 -> 116 ms.
enum StageGen { GEN_NONE = 0, GEN_ALL = 1, GEN_CUB = 2 };

template <typename T> struct SysDev {
    MeshDev m;
    size_t n;
    T dx, dy, dz;
    T wx, wy, wz, coef_ex, mu0, cm2mu0, mu_b, e_charge;
    Param<T> Ms, A, f1, f2, alpha, kuni, kcub, P, xi;
    VParam<T> axis1, axis2, j;
    int has_exch, has_uni, has_cub, has_zee, has_stt, do_precess;
    T hext[3];
    // alternating Zeeman field: hoff + ac_amp sin(t ac_freq + ac_phase)
    int has_ac;
    double hoff[3], ac_amp[3], ac_freq[3], ac_phase[3];
    int Ms_uniform;
    double Ms_u;
    // exchange with uniform, non-zero Ms and uniform A: no masking, no
    // per-neighbour Ms loads; H = exch_f * sum_j w_j (M_j - M_i) with
    // exch_f = 2 A / (mu0 Ms^2), the reference's (2A/(mu0 Ms)) sum (m_j - m_i) w
    int exch_uniform;
    T exch_f;
    // rows of the stage launch in XCD-contiguous ranges (xcd_tile): the
    // exchange stencil's neighbour rows are then read from the same L2
    int xcd_remap;
    // tile_zcol > 0: tiles of rpw rows align with the z planes (tile_zcol =
    // ny / rpw tiles per plane) and consecutive tiles walk a column of
    // planes (same y range, z = 0 .. nz-1) before moving on in y.  The
    // z +- 1 neighbour rows of the exchange stencil are then read by tiles
    // that run next to each other, while still in L2; in plane order they
    // come back only after a whole plane of tiles, which evicts them.
    int tile_zcol;
    // Zeeman field from a host function (has_fn): fn_tab[3 slot + c] is the
    // field of stage record `slot`, evaluated on the host at that
    // evaluation's time before the launch
    int has_fn;
    const double *fn_tab;
    // uniaxial anisotropy with uniform k, Ms (non-zero) and axis:
    // H = uni_c (M.a) a with uni_c = 2 k / (mu0 Ms^2), the reference's
    // 2 k (m.a) / (mu0 Ms) a with m = M / Ms; energy density uni_e |a x M|^2,
    // uni_e = k / Ms^2 (no per-cell divisions)
    int uni_fast;
    T uni_c, uni_e;
    // Zhang-Li torque with uniform P, xi, Ms (non-zero), alpha and j: the
    // factors f1, f2 of fdm_zhangli_cpu.cpp:95-114 and the inverse cell sizes
    // computed once (no per-cell divisions)
    int stt_fast;
    T stt_f1, stt_f2, inv_d[3];
};

// Zhang-Li torque of cell (x,y,z) with the precomputed uniform factors
// (zhangli_cell with its divisions hoisted): gradients central inside,
// one-sided at the faces, zero along axes of one cell
template <typename T>
__device__ __forceinline__ V3<T> zhangli_cell_uniform(const MeshDev &m, int x, int y, int z, size_t i, size_t n,
                                                      const T *inv_d, T f1, T f2, const V3<T> &j,
                                                      const T *__restrict__ M)
{
    const long li = (long)i;
    auto grad = [&](int pos, int dim, long st, T id) -> V3<T> {
        if (dim <= 1) return v3<T>(0, 0, 0);
        long a = li - st, b = li + st;
        T f = id * (T)0.5;
        if (pos == 0) {
            a = li;
            f = id;
        } else if (pos == dim - 1) {
            b = li;
            f = id;
        }
        return v3<T>((M[b] - M[a]) * f, (M[n + b] - M[n + a]) * f, (M[2 * n + b] - M[2 * n + a]) * f);
    };
    const V3<T> gx = grad(x, m.nx, 1, inv_d[0]);
    const V3<T> gy = grad(y, m.ny, m.nx, inv_d[1]);
    const V3<T> gz = grad(z, m.nz, (long)m.nx * m.ny, inv_d[2]);
    const V3<T> jg = v3<T>(j.x * gx.x + j.y * gy.x + j.z * gz.x, j.x * gx.y + j.y * gy.y + j.z * gz.y,
                           j.x * gx.z + j.y * gy.z + j.z * gz.z);
    const V3<T> Mv = v3<T>(M[li], M[n + li], M[2 * n + li]);
    const V3<T> B = cross3(Mv, jg);
    const V3<T> Av = cross3(Mv, B);
    return v3<T>(f1 * Av.x + f2 * B.x, f1 * Av.y + f2 * B.y, f1 * Av.z + f2 * B.z);
}

// exchange field of cell i for uniform Ms and A (see exch_uniform).  Each
// direction's neighbour is the periodic image or, at an open boundary, the
// cell itself (M_i - M_i adds an exact zero), so the six neighbours load
// without branches, in one batch, and sum in the fixed order -x, +x, -y, +y,
// -z, +z.
template <typename T>
__device__ __forceinline__ V3<T> exchange_cell_uniform(const MeshDev &m, int x, int y, int z, size_t i, size_t n,
                                                       T wx, T wy, T wz, T f, const T *__restrict__ M)
{
    const long li = (long)i, sy = m.nx, sz = (long)m.nx * m.ny;
    long j[6];
    j[0] = x > 0 ? li - 1 : (m.px ? li + (m.nx - 1) : li);
    j[1] = x < m.nx - 1 ? li + 1 : (m.px ? li - (m.nx - 1) : li);
    j[2] = y > 0 ? li - sy : (m.py ? li + sy * (m.ny - 1) : li);
    j[3] = y < m.ny - 1 ? li + sy : (m.py ? li - sy * (m.ny - 1) : li);
    j[4] = z > 0 ? li - sz : (m.pz ? li + sz * (m.nz - 1) : li);
    j[5] = z < m.nz - 1 ? li + sz : (m.pz ? li - sz * (m.nz - 1) : li);
    T a[6][3];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        a[q][0] = M[j[q]];
        a[q][1] = M[n + j[q]];
        a[q][2] = M[2 * n + j[q]];
    }
    const V3<T> mi = v3<T>(M[i], M[n + i], M[2 * n + i]);
    const T w[6] = {wx, wx, wy, wy, wz, wz};
    V3<T> s = v3<T>(0, 0, 0);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        s.x += (a[q][0] - mi.x) * w[q];
        s.y += (a[q][1] - mi.y) * w[q];
        s.z += (a[q][2] - mi.z) * w[q];
    }
    return v3<T>(f * s.x, f * s.y, f * s.z);
}

// 32-bit byte-offset access for arrays under 4 GiB: base is a pointer the
// whole workgroup shares (held in SGPRs), off a per-lane byte offset, so the
// access is one global load/store with an SGPR base and a 32-bit VGPR offset
// (no 64-bit address arithmetic per element).
template <typename T> __device__ __forceinline__ T ld32(const T *__restrict__ base, unsigned off)
{
    return *(const T *)((const char *)base + off);
}
template <typename T> __device__ __forceinline__ void st32(T *__restrict__ base, unsigned off, T v)
{
    *(T *)((char *)base + off) = v;
}

// exchange_cell_uniform with byte offsets: ib = i sizeof(T), nb = n sizeof(T)
// (3 nb < 2^32); same neighbours, loads and summation order
template <typename T>
__device__ __forceinline__ V3<T> exchange_cell_uniform32(const MeshDev &m, int x, int y, int z, unsigned ib,
                                                         unsigned nb, T wx, T wy, T wz, T f, const V3<T> &mi,
                                                         const T *__restrict__ M)
{
    constexpr unsigned sx = sizeof(T);
    const unsigned sy = (unsigned)m.nx * sx, sz = (unsigned)m.nx * (unsigned)m.ny * sx;
    unsigned j[6];
    j[0] = x > 0 ? ib - sx : (m.px ? ib + sx * (unsigned)(m.nx - 1) : ib);
    j[1] = x < m.nx - 1 ? ib + sx : (m.px ? ib - sx * (unsigned)(m.nx - 1) : ib);
    j[2] = y > 0 ? ib - sy : (m.py ? ib + sy * (unsigned)(m.ny - 1) : ib);
    j[3] = y < m.ny - 1 ? ib + sy : (m.py ? ib - sy * (unsigned)(m.ny - 1) : ib);
    j[4] = z > 0 ? ib - sz : (m.pz ? ib + sz * (unsigned)(m.nz - 1) : ib);
    j[5] = z < m.nz - 1 ? ib + sz : (m.pz ? ib - sz * (unsigned)(m.nz - 1) : ib);
    T a[6][3];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        a[q][0] = ld32(M, j[q]);
        a[q][1] = ld32(M, j[q] + nb);
        a[q][2] = ld32(M, j[q] + 2 * nb);
    }
    const T w[6] = {wx, wx, wy, wy, wz, wz};
    V3<T> s = v3<T>(0, 0, 0);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        s.x += (a[q][0] - mi.x) * w[q];
        s.y += (a[q][1] - mi.y) * w[q];
        s.z += (a[q][2] - mi.z) * w[q];
    }
    return v3<T>(f * s.x, f * s.y, f * s.z);
}

// zhangli_cell_uniform with byte offsets (as exchange_cell_uniform32)
template <typename T>
__device__ __forceinline__ V3<T> zhangli_cell_uniform32(const MeshDev &m, int x, int y, int z, unsigned ib,
                                                        unsigned nb, const T *inv_d, T f1, T f2, const V3<T> &j,
                                                        const V3<T> &Mv, const T *__restrict__ M)
{
    // one-sided differences at the ends, central inside; a dimension of one
    // cell has a = b (difference 0).  All 18 loads are unconditional and go
    // out together (with a branch per axis the compiler waited for each
    // axis's loads before issuing the next axis's).
    T gv[3][2][3], f[3];
    auto fetch = [&](int d, int pos, int dim, unsigned st, T id) {
        const bool lo = pos == 0, hi = pos == dim - 1;
        const unsigned a = lo ? ib : ib - st, b = hi ? ib : ib + st;
        f[d] = (lo || hi) ? id : id * (T)0.5;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            gv[d][0][c] = ld32(M, a + (unsigned)c * nb);
            gv[d][1][c] = ld32(M, b + (unsigned)c * nb);
        }
    };
    constexpr unsigned sx = sizeof(T);
    fetch(0, x, m.nx, sx, inv_d[0]);
    fetch(1, y, m.ny, (unsigned)m.nx * sx, inv_d[1]);
    fetch(2, z, m.nz, (unsigned)m.nx * (unsigned)m.ny * sx, inv_d[2]);
    auto grad = [&](int d) -> V3<T> {
        return v3<T>((gv[d][1][0] - gv[d][0][0]) * f[d], (gv[d][1][1] - gv[d][0][1]) * f[d],
                     (gv[d][1][2] - gv[d][0][2]) * f[d]);
    };
    const V3<T> gx = grad(0), gy = grad(1), gz = grad(2);
    const V3<T> jg = v3<T>(j.x * gx.x + j.y * gy.x + j.z * gz.x, j.x * gx.y + j.y * gy.y + j.z * gz.y,
                           j.x * gx.z + j.y * gy.z + j.z * gz.z);
    const V3<T> B = cross3(Mv, jg);
    const V3<T> Av = cross3(Mv, B);
    return v3<T>(f1 * Av.x + f2 * B.x, f1 * Av.y + f2 * B.y, f1 * Av.z + f2 * B.z);
}

// stored stage vectors one stage combination reads at most (DP54's last
// stage: k_0 .. k_5)
#define MM_STAGE_MAXK 6
// rows of the host-evaluated Zeeman table (stage records: at most 7 stages,
// dM/dt and energy)
#define MM_FN_SLOTS 16

template <typename T> struct StageDev {
    const T *Ys;          // stage input (null: y[cur])
    T *yb0, *yb1;         // the two y buffers
    T *kout;              // k_s (null: not stored)
    T *Hout;              // H_tot (null: not stored)
    // next stage input: out = base + (h*) sum coef_j k_j  (k_s last, from registers)
    int prep;             // 0 none, 1 prepare next stage, 2 final combine
    int form;             // FORM_SUM / FORM_SEQ
    T *prep_out;
    int nk;               // number of stored k_j used (j < s)
    const T *kin[MM_STAGE_MAXK];
    double b[MM_STAGE_MAXK];  // coefficients for kin
    double bself;             // coefficient for k_s
    double ec[MM_STAGE_MAXK], ecself;  // error coefficients (final stage)
    int want_dydt;        // reduce max|k_s| (stage 0)
    int norm_mode;
    // FSAL (dp54, rk23): the last stage takes max|k_0| from kin[0] and then
    // overwrites k_0 with its own k_s for the next attempt (runge_kutta.py:97-101,131-134)
    int dydt_from_k0;
    T *fsal_out;
    // prep == 1 with the demag field: the epilogue also transforms the next
    // stage input along x (rows into S1), so that stage needs no x pass
    int fwd;
    C2<T> *fwd_S1;
    // per-block maxima, rows [0] |err|^2 (final stage), [1] |k0|^2 scaled,
    // [2] |k0|^2, [3] |y|^2, one entry per block of the launch; the
    // controller reduces them (no same-address atomics across the grid)
    double *mpart;
    // node a_s of this stage: the stage is evaluated at t + a_s h (the
    // alternating Zeeman field depends on it)
    double tnode;
    // index of this record (stages 0..ns-1, then dM/dt, then energy): its
    // row of the host-evaluated Zeeman table
    int slot;
};


template <typename T> __device__ __forceinline__ double dotd(const V3<T> &a, const V3<T> &b)
{
    return (double)a.x * b.x + (double)a.y * b.y + (double)a.z * b.z;
}

// per-thread maxima of one stage launch (squared norms, FP64)
struct StageRed {
    double err;   // |err|^2 (/Ms^2 when Ms is not uniform)
    double dydt;  // |k0|^2 (/Ms^2 when Ms is not uniform)
    double draw;  // |k0|^2
    double mraw;  // |y|^2 of the attempt's start state
};

// per-thread sums of M.H per term (energy launches only), compensated
struct EnergyAcc {
    Dd demag, exch, aniso, zee;
};

// Per-cell epilogue: everything after the demag field of one cell.  STT:
// the Zhang-Li term is compiled in; GEN (StageGen): which of cubic anisotropy
// and the exchange with per-cell Ms/A are compiled in (without them the
// epilogue is shorter and needs fewer registers).  Except in GEN_ALL the state
// arrays are addressed by 32-bit byte offsets from their (workgroup-uniform)
// bases, which the host guarantees by taking GEN_ALL for state arrays of
// 4 GiB or more.
template <typename T, bool EN, bool STT, int GEN, bool P1S = false>
__device__ __forceinline__ void stage_cell(const SysDev<T> &S, const StageDev<T> &G, const StepCtl *ctl,
                                           const T *__restrict__ Y, int x, int y, int z, const V3<T> &Hd,
                                           const V3<T> &hz, StageRed &red, EnergyAcc &ea, T *nxt)
{
    constexpr bool O32 = GEN != GEN_ALL, CUB = GEN != GEN_NONE;
    const size_t n = S.n;
    const size_t i = (size_t)x + (size_t)S.m.nx * ((size_t)y + (size_t)S.m.ny * z);
    // byte offsets of cell i and of one component plane (O32 only)
    const unsigned ib = O32 ? ((unsigned)x + (unsigned)S.m.nx * ((unsigned)y + (unsigned)S.m.ny * (unsigned)z)) *
                                  (unsigned)sizeof(T)
                            : 0u;
    const unsigned nb = O32 ? (unsigned)n * (unsigned)sizeof(T) : 0u;
    auto ldv = [&](const T *__restrict__ a) -> V3<T> {
        if constexpr (O32) return v3<T>(ld32(a, ib), ld32(a, ib + nb), ld32(a, ib + 2 * nb));
        else return v3<T>(a[i], a[n + i], a[2 * n + i]);
    };
    auto stv = [&](T *__restrict__ a, const V3<T> &v) {
        if constexpr (O32) {
            st32(a, ib, v.x);
            st32(a, ib + nb, v.y);
            st32(a, ib + 2 * nb, v.z);
        } else {
            store3<T>(a, n, i, v);
        }
    };
    // the record's flags and uniform parameters of this cell's path, read in
    // one block (merged scalar loads, one wait) instead of inside each
    // guarded section
    const int Ms_uniform = S.Ms_uniform, has_exch = S.has_exch, has_uni = S.has_uni, uni_fast = S.uni_fast;
    const int has_zee = S.has_zee;
    const T Ms_u = S.Ms.u, wx = S.wx, wy = S.wy, wz = S.wz, exch_f = S.exch_f, uni_c = S.uni_c;
    const T ax0 = S.axis1.u[0], ax1 = S.axis1.u[1], ax2 = S.axis1.u[2];
    const T *const f1p = S.f1.p, *const f2p = S.f2.p;
    const T f1u = S.f1.u, f2u = S.f2.u;
    const T ms = Ms_uniform ? Ms_u : (O32 ? ld32(gfield(S.Ms.p), ib) : S.Ms.at(i));
    const V3<T> Mv = ldv(Y);
    V3<T> H = Hd;
    if (EN) dd_add(ea.demag, dotd<T>(Mv, Hd));
    if (has_exch && ms != (T)0) {
        V3<T> he;
        if constexpr (O32) {
            he = exchange_cell_uniform32<T>(S.m, x, y, z, ib, nb, wx, wy, wz, exch_f, Mv, Y);
        } else {
            he = S.exch_uniform
                     ? exchange_cell_uniform<T>(S.m, x, y, z, i, n, S.wx, S.wy, S.wz, S.exch_f, Y)
                     : exchange_cell_batch<T>(S.m, x, y, z, i, n, S.wx, S.wy, S.wz, S.coef_ex, gfield(S.Ms.p),
                                              gfield(S.A.p), Y, ms);
        }
        if constexpr (GEN == GEN_CUB) {
            // rounded before the sum, as GEN_ALL has it (there the field comes
            // from one of two branches): the same bits in both classes
#pragma clang fp contract(off)
            H.x += he.x;
            H.y += he.y;
            H.z += he.z;
        } else {
            H.x += he.x;
            H.y += he.y;
            H.z += he.z;
        }
        if (EN) dd_add(ea.exch, dotd<T>(Mv, he));
    }
    if (has_uni || (CUB && S.has_cub)) {
        T e0 = (T)0, e1 = (T)0;
        V3<T> ha = v3<T>(0, 0, 0);
        if (CUB && S.has_cub) ha = cubic_cell<T>(Mv, S.axis1.at(n, i), S.axis2.at(n, i), S.kcub.at(i), ms, S.cm2mu0, &e1);
        if (has_uni) {
            V3<T> hu;
            if (uni_fast) {
                const V3<T> ax = v3<T>(ax0, ax1, ax2);
                const T f = uni_c * dot3(Mv, ax);
                hu = v3<T>(f * ax.x, f * ax.y, f * ax.z);
                if (EN) {
                    const V3<T> c = cross3(ax, Mv);
                    e0 = S.uni_e * dot3(c, c);
                }
            } else {
                hu = uniaxial_cell<T>(Mv, S.axis1.at(n, i), S.kuni.at(i), ms, S.mu0, &e0);
            }
            if (EN) dd_add(ea.aniso, (double)e0);
            if (CUB && S.has_cub) {
                ha.x += hu.x;
                ha.y += hu.y;
                ha.z += hu.z;
            } else {
                ha = hu;
            }
        }
        if (EN && CUB && S.has_cub) dd_add(ea.aniso, (double)e1);
        H.x += ha.x;
        H.y += ha.y;
        H.z += ha.z;
    }
    if (has_zee) {
        H.x += hz.x;
        H.y += hz.y;
        H.z += hz.z;
        if (EN) dd_add(ea.zee, (double)Mv.x * hz.x + (double)Mv.y * hz.y + (double)Mv.z * hz.z);
    }
    if (EN) return;
    V3<T> k = llge_cell<T>(Mv, H, f1p ? gfield(f1p)[i] : f1u, f2p ? gfield(f2p)[i] : f2u);
    if (STT && S.has_stt) {
        V3<T> st;
        if (O32 && S.stt_fast)
            st = zhangli_cell_uniform32<T>(S.m, x, y, z, ib, nb, S.inv_d, S.stt_f1, S.stt_f2,
                                           v3<T>(S.j.u[0], S.j.u[1], S.j.u[2]), Mv, Y);
        else if (S.stt_fast)
            st = zhangli_cell_uniform<T>(S.m, x, y, z, i, n, S.inv_d, S.stt_f1, S.stt_f2,
                                         v3<T>(S.j.u[0], S.j.u[1], S.j.u[2]), Y);
        else
            st = zhangli_cell<T>(S.m, x, y, z, i, n, S.dx, S.dy, S.dz, S.do_precess != 0, S.P.at(i), S.xi.at(i), ms,
                                 S.alpha.at(i), S.j.at(n, i), Y, S.mu_b, S.e_charge);
        k.x += st.x;
        k.y += st.y;
        k.z += st.z;
    }
    if (G.kout) stv(gfield(G.kout), k);
    if (G.Hout) stv(gfield(G.Hout), H);
    if (G.want_dydt) {
        const double a = k.x, b = k.y, c = k.z;
        double q = a * a + b * b + c * c;
        red.draw = fmax(red.draw, q);
        red.mraw = fmax(red.mraw, (double)Mv.x * Mv.x + (double)Mv.y * Mv.y + (double)Mv.z * Mv.z);
        if (!S.Ms_uniform) {
            const double s = ms;
            q = s == 0.0 ? 0.0 : q / (s * s);
        }
        red.dydt = fmax(red.dydt, q);
    }
    if (!P1S && !G.prep) return;
    // the combination's inputs (stored stage vectors, the attempt's start
    // state) load in one batch of independent loads before any arithmetic
    // (loading them here rather than at the top keeps them out of the field
    // computation's live registers)
    const T *yc = ctl->cur ? gfield(G.yb1) : gfield(G.yb0);
    T kv[MM_STAGE_MAXK][3], ycv[3];
    {
        const V3<T> v = ldv(yc);
        ycv[0] = v.x;
        ycv[1] = v.y;
        ycv[2] = v.z;
    }
#pragma unroll
    for (int q = 0; q < MM_STAGE_MAXK; ++q)
        if (q < G.nk) {
            const V3<T> v = ldv(gfield(G.kin[q]));
            kv[q][0] = v.x;
            kv[q][1] = v.y;
            kv[q][2] = v.z;
        }
    const double h = ctl->h;
    // stage vectors outermost, components inside: each tableau coefficient is
    // read once per cell (with the components outermost, the guarded loops
    // loaded every coefficient again per component); per component the sums
    // keep the order q = 0, 1, ..., self
    const int nk = G.nk, form = P1S ? FORM_SUM : G.form, prep = P1S ? 1 : G.prep;
    const T kc[3] = {k.x, k.y, k.z};
    T out[3];
    double er[3] = {0.0, 0.0, 0.0};
    if (form == FORM_SUM) {
        T sum[3];
        double e[3];
#pragma unroll
        for (int q = 0; q < MM_STAGE_MAXK; ++q) {
            if (q < nk) {
                const T bq = (T)G.b[q];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const T term = bq * kv[q][c];
                    sum[c] = q == 0 ? term : sum[c] + term;
                }
                if (prep == 2) {
                    const double ecq = G.ec[q];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const double term = ecq * (double)kv[q][c];
                        e[c] = q == 0 ? term : e[c] + term;
                    }
                }
            }
        }
        const T bself = (T)G.bself;
        const double ecself = G.ecself;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T ts = bself * kc[c];
            const T sc = nk == 0 ? ts : sum[c] + ts;
            out[c] = ycv[c] + (T)h * sc;
            if (prep == 2) {
                const double tse = ecself * (double)kc[c];
                er[c] = h * (nk == 0 ? tse : e[c] + tse);
            }
        }
    } else {
        T v[3] = {ycv[0], ycv[1], ycv[2]};
#pragma unroll
        for (int q = 0; q < MM_STAGE_MAXK; ++q) {
            if (q < nk) {
                const T f = (T)(h * G.b[q]);
                const double fe = prep == 2 ? h * G.ec[q] : 0.0;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const T kq = kv[q][c];
                    v[c] += kq * f;
                    if (prep == 2) er[c] += (double)kq * fe;
                }
            }
        }
        const T fs = (T)(h * G.bself);
        const double fes = h * G.ecself;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v[c] += kc[c] * fs;
            if (prep == 2) er[c] += (double)kc[c] * fes;
            out[c] = v[c];
        }
    }
    if (prep == 1) {
        stv(gfield(G.prep_out), v3<T>(out[0], out[1], out[2]));
        nxt[0] = out[0];
        nxt[1] = out[1];
        nxt[2] = out[2];
        return;
    }
    // final stage: error norm and normalised new state into the other buffer
    if (G.dydt_from_k0) {
        const V3<T> k0 = ldv(gfield(G.kin[0]));
        const double a = k0.x, b = k0.y, c = k0.z;
        double q = a * a + b * b + c * c;
        red.draw = fmax(red.draw, q);
        const double y0 = ycv[0], y1 = ycv[1], y2 = ycv[2];
        red.mraw = fmax(red.mraw, y0 * y0 + y1 * y1 + y2 * y2);
        if (!S.Ms_uniform) {
            const double s = ms;
            q = s == 0.0 ? 0.0 : q / (s * s);
        }
        red.dydt = fmax(red.dydt, q);
    }
    if (G.fsal_out) stv(gfield(G.fsal_out), k);
    {
        double q = er[0] * er[0] + er[1] * er[1] + er[2] * er[2];
        if (!S.Ms_uniform) {
            const double s = ms;
            q = s == 0.0 ? 0.0 : q / (s * s);
        }
        red.err = fmax(red.err, q);
    }
    T *yn = ctl->cur ? gfield(G.yb0) : gfield(G.yb1);
    double norm;
    if (G.norm_mode == 0) {
        norm = float_cast_norm((double)out[0], (double)out[1], (double)out[2]);
    } else {
        norm = fp64_norm((double)out[0], (double)out[1], (double)out[2]);
    }
    if (norm != 0.0) {
        const double sc = (double)ms / norm;
        out[0] = (T)(out[0] * sc);
        out[1] = (T)(out[1] * sc);
        out[2] = (T)(out[2] * sc);
    }
    stv(yn, v3<T>(out[0], out[1], out[2]));
}

// x inverse of the demag spectrum rows + epilogue.  rpw rows per block, all
// three components of a row in the same block.  has_demag: 0 no stray field,
// 1 inverse x transform of S1 rows in LDS, 2 H_demag read from Hdem (lines
// too long for three in one workgroup's LDS).  EN: instead of the stage
// epilogue, per-block compensated sums of M.H per term: the pair of term q
// at epart[2q nblk + blk] (s) and epart[(2q+1) nblk + blk] (e).  blk: this
// workgroup's index among the nblk of the system's launch; remap: order the
// tiles by xcd_tile(blk, nblk) (the single-system launch; a batched launch
// orders its global workgroups before it picks the system).
template <typename T, bool EN, int LC, bool STT, int GEN, bool P1S = false>
__device__ __forceinline__ void stage_body(const SysDev<T> *__restrict__ Sp, const StageDev<T> *__restrict__ Gp,
                                           StepCtl *ctl, const C2<T> *__restrict__ S1, const FftPlanDev &p, int Hx,
                                           int Hp, int rpw, int has_demag, double *__restrict__ epart,
                                           const T *__restrict__ Hdem, int blk, int nblk, bool remap)
{
    // the system and stage records live in device memory (read where used)
    // rather than in the kernel arguments: by value they need ~160 SGPRs,
    // and the compiler spilled most of them to VGPR lanes
    const SysDev<T> &S = *Sp;
    const StageDev<T> &G = *Gp;
    constexpr int SK = MM_SKEW_X;
    // stages of an attempt (prep != 0) do nothing once the run has stopped;
    // evaluations outside attempts (dM/dt, energies) always run
    if (!EN && (P1S || G.prep) && ctl->stop) return;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int nx = S.m.nx, ny = S.m.ny, nz = S.m.nz;
    const int nrows = ny * nz;
    int tile = (remap && S.xcd_remap) ? xcd_tile(blk, nblk) : blk;
    if (S.tile_zcol > 0) {
        const int ty = tile / nz;
        tile = (tile - ty * nz) * S.tile_zcol + ty;
    }
    const int row0 = tile * rpw;
    const T *Y = G.Ys ? gfield(G.Ys) : (ctl->cur ? gfield(G.yb1) : gfield(G.yb0));
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L), TL = PlanC<LC>::tline(p);
    // Rows are transformed in pairs, two real rows per complex line: line
    // l = (component c, pair q) holds rows gr0 = row0 + 2q (real part) and
    // gr0 + 1 (imaginary part).  With has_demag == 1, rpw is even.
    const int np = rpw >> 1;
    C2<T> *twl = sm + (size_t)3 * np * LP;
    if (has_demag == 1) {
        const TwFetch<T> twf = TwFetch<T>::fetch(p);
        // inverse: Z = X0 + i X1 with both half spectra extended Hermitian
        // (X[L-k] = conj X[k]; X[0], X[L/2] taken real), so that Re and Im of
        // the inverse transform are the two rows
        const int l = threadIdx.x / TL, t = threadIdx.x % TL;
        const int c = np == 1 ? l : l / (np > 0 ? np : 1), q = np == 1 ? 0 : l % (np > 0 ? np : 1);
        const int gr0 = row0 + 2 * q;
        const bool active = (l < 3 * np) && gr0 < nrows;
        const bool has1 = gr0 + 1 < nrows;
        C2<T> *line = sm + (size_t)l * LP;
        const C2<T> *src0 = S1 + ((size_t)c * nrows + (active ? gr0 : 0)) * Hp;
        const C2<T> *src1 = src0 + (has1 ? Hp : 0);
        const LineMap m = {t, active};
        fft_line<T, true, true, false, LC, SK>(
            p, twl, line, m, line, m,
            [&](int k) {
                const bool lo = k < Hx;
                const int kk = lo ? k : L - k;
                // both loads unconditional (src1 is src0 for an absent second
                // row) and the cases folded into a factor f (0 at k = 0 and
                // L/2, +1 below Hx, -1 above; f*v is exact): with branches
                // around the loads, the compiler waited for every element's
                // loads before issuing the next element's
                const C2<T> a = src0[kk];
                const C2<T> b = src1[kk];
                const T bx = has1 ? b.x : (T)0, by = has1 ? b.y : (T)0;
                const T f = ((k == 0) | (2 * k == L)) ? (T)0 : (lo ? (T)1 : (T)-1);
                return cmk<T>(a.x - f * by, bx + f * a.y);
            },
            [](int, C2<T>) {}, [&] { twf.store(twl); });
    }
    StageRed red = {0.0, 0.0, 0.0, 0.0};
    EnergyAcc ea = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
    const bool fused = !EN && has_demag == 1 && G.fwd;
    // Zeeman field of this evaluation (alternating_field.py:57-84), at the
    // stage time t + a_s h
    V3<T> hz = v3<T>(S.hext[0], S.hext[1], S.hext[2]);
    if (S.has_zee && S.has_ac) {
        const double ts = ctl->t + G.tnode * ctl->h;
        hz = v3<T>((T)(S.hoff[0] + S.ac_amp[0] * sin(ts * S.ac_freq[0] + S.ac_phase[0])),
                   (T)(S.hoff[1] + S.ac_amp[1] * sin(ts * S.ac_freq[1] + S.ac_phase[1])),
                   (T)(S.hoff[2] + S.ac_amp[2] * sin(ts * S.ac_freq[2] + S.ac_phase[2])));
    } else if (S.has_zee && S.has_fn) {
        const double *f = gfield(S.fn_tab) + 3 * G.slot;
        hz = v3<T>((T)f[0], (T)f[1], (T)f[2]);
    }
    // The epilogue's cells: rows of nx cells over groups of whole waves.  A
    // group takes the waves one row fills (at most the workgroup) and the
    // groups take the rows in turn, so that short rows do not leave most of
    // the workgroup idle while it walks the rows one after another; the row
    // stays uniform per wave (scalar y, z and tile edges).  48 systems of
    // 32..256 cells per row, batched: stage 211 -> 162 us (MI355X, FP32).
    // The loops step unsigned: with a signed step, which cannot wrap, the
    // compiler turned the addresses of every array into induction variables of
    // the x loop (FP32 77 -> 88 to 101 VGPRs, FP64 110 -> 128 and spilled).
    const int nwv = (int)(blockDim.x >> 6);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rw = min(nwv, (nx + 63) >> 6), ngr = nwv / rw, grp = wv / rw;
    // rows of the group in (y, z): once, then stepped (no per-cell division)
    int yr = (row0 + grp) % ny, zr = (row0 + grp) / ny;
    for (int r = grp < ngr ? grp : rpw; r < rpw; r += ngr, yr += ngr) {
        while (yr >= ny) {
            yr -= ny;
            ++zr;
        }
        const int gr = row0 + r;
        const int q = r >> 1, hi = r & 1;
        for (int x = (int)(threadIdx.x - (unsigned)(grp * rw * 64)); x < nx; x = (int)((unsigned)x + (unsigned)(rw * 64))) {
            if (gr >= nrows) {
                // the absent second row of a pair transforms as zeros
                if (fused)
                    for (int c = 0; c < 3; ++c) reinterpret_cast<T *>(&sm[(c * np + q) * LP + sk<SK>(x)])[hi] = (T)0;
                continue;
            }
            V3<T> Hd = v3<T>(0, 0, 0);
            if (has_demag == 1) {
                T h3[3];
                for (int c = 0; c < 3; ++c) h3[c] = reinterpret_cast<const T *>(&sm[(c * np + q) * LP + sk<SK>(x)])[hi];
                Hd = v3<T>(h3[0], h3[1], h3[2]);
            } else if (has_demag == 2) {
                const size_t i = (size_t)gr * nx + x;
                Hd = v3<T>(Hdem[i], Hdem[S.n + i], Hdem[2 * S.n + i]);
            }
            T nxt[3];
            stage_cell<T, EN, STT, GEN, P1S>(S, G, ctl, Y, x, yr, zr, Hd, hz, red, ea, nxt);
            // the half slot (row, x) of the three lines is this thread's
            // alone: the next stage input replaces H_demag in place
            if (fused)
                for (int c = 0; c < 3; ++c) reinterpret_cast<T *>(&sm[(c * np + q) * LP + sk<SK>(x)])[hi] = nxt[c];
        }
    }
    if (fused) {
        // the zeros that extend the lines, and below the spectra, line by
        // line over the same kind of wave groups
        {
            const int lw = min(nwv, (L - nx + 63) >> 6), nlg = lw > 0 ? nwv / lw : 1, lg = lw > 0 ? wv / lw : 0;
            if (lg < nlg)
                for (int l = lg; l < 3 * np; l += nlg)
                    for (int x = (int)((unsigned)nx + threadIdx.x - (unsigned)(lg * lw * 64)); x < L; x = (int)((unsigned)x + (unsigned)(lw * 64)))
                        sm[(size_t)l * LP + sk<SK>(x)] = cmk<T>((T)0, (T)0);
        }
        __syncthreads();
        {
            const int l = threadIdx.x / TL, t = threadIdx.x % TL;
            const bool active = (l < 3 * np) && row0 + 2 * (np == 1 ? 0 : l % np) < nrows;
            C2<T> *line = sm + (size_t)l * LP;
            const LineMap m = {t, active};
            fft_line<T, false, false, false, LC, SK>(
                p, twl, line, m, line, m, [](int) { return cmk<T>((T)0, (T)0); }, [](int, C2<T>) {});
        }
        // forward: Z = FFT(x0 + i x1); X0[k] = (Z[k] + conj Z[L-k]) / 2,
        // X1[k] = (Z[k] - conj Z[L-k]) / 2i for k < Hx.  The thread of k = 0
        // also writes k = L/2 of an even line, so that 2^m columns take 2^m
        // threads and not another, nearly empty round.
        const int kh = (L & 1) ? Hx : Hx - 1;
        const int lw = max(1, min(nwv, (kh + 63) >> 6)), nlg = nwv / lw, lg = wv / lw;
        for (int l = lg < nlg ? lg : 3 * np; l < 3 * np; l += nlg) {
            const int c = l / np, q = l % np;
            const int gr0 = row0 + 2 * q;
            if (gr0 >= nrows) continue;
            const bool has1 = gr0 + 1 < nrows;
            const C2<T> *ln = sm + (size_t)l * LP;
            C2<T> *d0 = gfield(G.fwd_S1) + ((size_t)c * nrows + gr0) * Hp;
            for (int k = (int)(threadIdx.x - (unsigned)(lg * lw * 64)); k < kh; k = (int)((unsigned)k + (unsigned)(lw * 64))) {
                const C2<T> zk = ln[sk<SK>(k)], zm = ln[sk<SK>(k == 0 ? 0 : L - k)];
                d0[k] = cmk<T>((zk.x + zm.x) * (T)0.5, (zk.y - zm.y) * (T)0.5);
                if (has1) d0[(size_t)Hp + k] = cmk<T>((zk.y + zm.y) * (T)0.5, (zm.x - zk.x) * (T)0.5);
                if (k == 0 && kh < Hx) {
                    const C2<T> zh = ln[sk<SK>(kh)];
                    d0[kh] = cmk<T>(zh.x, (T)0);
                    if (has1) d0[(size_t)Hp + kh] = cmk<T>(zh.y, (T)0);
                }
            }
        }
    }
    __shared__ double wred[4][16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (int)((blockDim.x + 63) >> 6);
    if (EN) {
        __shared__ double wsum[8][16];
        const Dd a = wave_sum_dd(ea.demag), b = wave_sum_dd(ea.exch), c = wave_sum_dd(ea.aniso),
                 d = wave_sum_dd(ea.zee);
        if (lane == 0) {
            wsum[0][w] = a.s;
            wsum[1][w] = a.e;
            wsum[2][w] = b.s;
            wsum[3][w] = b.e;
            wsum[4][w] = c.s;
            wsum[5][w] = c.e;
            wsum[6][w] = d.s;
            wsum[7][w] = d.e;
        }
        __syncthreads();
        if (threadIdx.x < 4) {
            const int q = threadIdx.x;
            Dd acc = {wsum[2 * q][0], wsum[2 * q + 1][0]};
            for (int v = 1; v < nw; ++v) {
                const Dd o = {wsum[2 * q][v], wsum[2 * q + 1][v]};
                acc = dd_merge(acc, o);
            }
            epart[(size_t)(2 * q) * nblk + blk] = acc.s;
            epart[(size_t)(2 * q + 1) * nblk + blk] = acc.e;
        }
        return;
    }
    if ((!P1S && (G.prep == 2 || G.dydt_from_k0)) || G.want_dydt) {
        const double a = wave_max(red.err), b = wave_max(red.dydt), c = wave_max(red.draw), d = wave_max(red.mraw);
        if (lane == 0) {
            wred[0][w] = a;
            wred[1][w] = b;
            wred[2][w] = c;
            wred[3][w] = d;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double ea0 = wred[0][0], eb = wred[1][0], ec = wred[2][0], ed = wred[3][0];
            for (int q = 1; q < nw; ++q) {
                ea0 = fmax(ea0, wred[0][q]);
                eb = fmax(eb, wred[1][q]);
                ec = fmax(ec, wred[2][q]);
                ed = fmax(ed, wred[3][q]);
            }
            double *mp = gfield(G.mpart);
            if (!P1S && G.prep == 2) mp[blk] = ea0;
            if (G.want_dydt || (!P1S && G.dydt_from_k0)) {
                mp[(size_t)nblk + blk] = eb;
                mp[2 * (size_t)nblk + blk] = ec;
                mp[3 * (size_t)nblk + blk] = ed;
            }
        }
    }
}

// P1S: the record is an inner stage with a summed combination (prep 1,
// FORM_SUM, no FSAL reads), so the final-stage code and its record reads
// are compiled out (RKF45 / CC45: five of the six stage launches).  In FP32
// that kernel needs 55-59 VGPRs and is held to 7 waves per SIMD by its 106
// SGPRs; asking for 8 (SGPRs 78, the rest spilled to VGPR lanes, no
// scratch) lets a CU hold 8 of its 256-thread workgroups, one round for
// 256x256x16 cells: stage 32.4 -> 30.7 us (MI355X, same-run A/B).  The other
// FP32 kernels ask for 6 (80 VGPRs, 81 to 83 without; none to three spilled,
// in spin torque with cubic anisotropy, all mixed lengths and runtime plans):
// 24 waves a CU, two workgroups of 768 threads on 1024-cell rows.
template <typename T, bool EN, int LC, bool STT, int GEN, bool P1S = false>
__global__ void __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? (P1S ? 8 : (EN ? 1 : 6)) : 1))) k_stage(const SysDev<T> *__restrict__ Sp, const StageDev<T> *__restrict__ Gp, StepCtl *ctl,
                        const C2<T> *__restrict__ S1, FftPlanDev p, int Hx, int Hp, int rpw, int has_demag,
                        double *__restrict__ epart, const T *__restrict__ Hdem)
{
    stage_body<T, EN, LC, STT, GEN, P1S>(Sp, Gp, ctl, S1, p, Hx, Hp, rpw, has_demag, epart, Hdem, (int)blockIdx.x,
                                    (int)gridDim.x, true);
}

// Per-system records of the batched stage and controller launches (the conv
// passes' records are in mm_conv.h).  The global workgroup index in XCD order
// picks the system through the pass's tile table, as in the conv passes.
template <typename T> struct BStageDesc {
    const SysDev<T> *S;
    const StageDev<T> *G0;  // the system's stage records; the launch picks stage st
    StepCtl *ctl;
    const C2<T> *S1;
    int Hx, Hp, rpw, nb, tbase;
    FftPlanDev p;
};

template <typename T, int LC, bool STT, int GEN, bool P1S = false>
__global__ void kb_stage(const BStageDesc<T> *__restrict__ D, const int *__restrict__ tsys, int st)
{
    const int gi = block_tile(1);
    const BStageDesc<T> &d = D[tsys[gi]];
    stage_body<T, false, LC, STT, GEN, P1S>(gfield(d.S), gfield(d.G0) + st, gfield(d.ctl), gfield(d.S1), d.p, d.Hx, d.Hp,
                                      d.rpw, 1, nullptr, nullptr, gi - d.tbase, d.nb, false);
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
// One stage launch of a single system.  len: the x transform inside the
// kernel (0: none); generic: runtime FFT plans.
template <typename T> struct StageArgs {
    int grid, threads;
    size_t lds;
    hipStream_t s;
    const SysDev<T> *sys;
    const StageDev<T> *rec;
    StepCtl *ctl;
    const C2<T> *S1;
    FftPlanDev p;
    int Hx, Hp, rpw, demag, len;
    bool generic;
    double *epart;
    const T *Hdem;
};
// the kernel of a physics class: EN the energy sums, STT Zhang-Li torque, GEN
// the StageGen class, P1S inner stages with a summed combination
template <typename T, bool EN, bool STT, int GEN, bool P1S> void stage_run(const StageArgs<T> &a);
// workgroups of the (non-energy) kernel that one CU holds
template <typename T, bool STT, int GEN> int stage_blocks_per_cu(int len, bool generic, int threads, size_t lds);
// stage st of every system of a batch
template <typename T, bool STT, int GEN, bool P1S> void stage_run_batch(const BatchPass &bp, hipStream_t s, int st);

#endif
