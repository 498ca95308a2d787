// mm_conv_passes.hip -- FFT demag convolution on gfx950: the passes, for one
// precision (MM_CONV_T; the Makefile builds one object per precision).
//
// Replaces SymmetricMatrixVectorConvolution_FFT / MatrixVectorConvolution_FFT
// (src/magneto/math/conv/MatrixVectorConvolution_FFT.cpp:110-375) with five
// LDS-staged passes per evaluation instead of thirteen:
//
//   x fwd  : real rows of M (x < nx) zero-extended to Px, complex FFT,
//            keep kx < Hx = Px/2+1                    M  -> S1[c][z][y][kx]
//   y fwd  : columns of S1 (y < ny) zero-extended to Py  S1 -> S2[c][z][ky][kx]
//   z      : lines of S2 (z < nz) zero-extended to Pz, FFT, 3x3 multiply with
//            the real octant-stored Fourier kernel, inverse FFT, keep z < nz
//   y inv  : inverse FFT of S2 columns, keep y < ny     S2 -> S1
//   x inv  : Hermitian extension, inverse FFT, keep x < nx  S1 -> H
//
// 2-D meshes (nz == 1) fuse y fwd + multiply + y inv into one pass on S1.
// No transpose passes: strided passes load tiles of adjacent kx columns so
// every global access is a contiguous row segment, and the zero padding is
// never stored (only nonzero input rows are read, only kept outputs written).
//
// Fourier kernel: the padded tensor is even/odd in every axis, so its
// transform is real; only kx < Hx, ky <= Py/2, kz <= Pz/2 are stored (6 real
// planes, sign flips for the odd components on the other octants).  It is
// computed once on the device in FP64 with the same passes and cast to the
// working precision.  The reference keeps the full complex kernel; the
// dropped imaginary parts are rounding noise (~1e-17 relative).
#include "mm_conv.h"
#include "mm_cell.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

// Dynamic LDS above 64 KB needs no opt-in on gfx950 (the device reports its
// per-workgroup maximum); launches are error-checked.  Kept as the single
// place that validates a request against that maximum.
template <typename K> static void set_lds(K, size_t bytes)
{
    MM_REQUIRE(bytes <= (size_t)mm_max_lds_bytes(), "LDS request exceeds the device maximum");
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------

// x forward: rows (c, z, y); input rows of nx_in reals with row stride nx_in;
// workgroup blk takes lines blk lpw .. (blk + 1) lpw - 1 (threads beyond the
// lpw lines stay idle)
template <typename T, typename TIN, int LC = 0>
__device__ __forceinline__ void xfwd_body(const TIN *__restrict__ in, size_t in_cstride, C2<T> *__restrict__ out,
                                          size_t out_cstride, int Hx, int Hp, int ny, int nz, int nrows, int nx_in,
                                          const FftPlanDev &p, int lpw, int blk)
{
    constexpr int SK = MM_SKEW_X;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L), TL = PlanC<LC>::tline(p);
    // two real rows per complex line: line l of the block holds rows
    // 2 g and 2 g + 1 (g = blockIdx.x lpw + l) as real and imaginary part
    const int l = threadIdx.x / TL, t = threadIdx.x % TL;
    const int g0 = 2 * (blk * lpw + l);
    const bool active = l < lpw && g0 < nrows;
    const bool has1 = g0 + 1 < nrows;
    C2<T> *line = sm + (size_t)l * LP;
    C2<T> *twl = sm + (size_t)lpw * LP;
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    const int rows_c = ny * nz;
    auto row_src = [&](int g) { return in + (g / rows_c) * in_cstride + (size_t)(g % rows_c) * nx_in; };
    const TIN *src0 = row_src(active ? g0 : 0);
    const TIN *src1 = row_src(active && has1 ? g0 + 1 : 0);
    const LineMap m = {t, active};
    fft_line<T, false, true, false, LC, SK>(
        p, twl, line, m, line, m,
        [&](int x) {
            const bool in_row = x < nx_in;
            return cmk<T>(in_row ? (T)src0[x] : (T)0, in_row && has1 ? (T)src1[x] : (T)0);
        },
        [](int, C2<T>) {}, [&] { twf.store(twl); });
    xfwd_store<T>(sm, LP, L, lpw, blk, nrows, Hx, [&](int h) { return out + (h / rows_c) * out_cstride + (size_t)(h % rows_c) * Hp; });
}

// sel (may be null): device index choosing in (0) or in_alt (1)
template <typename T, typename TIN, int LC = 0>
__global__ void k_xfwd(const TIN *__restrict__ in, size_t in_cstride, C2<T> *__restrict__ out,
                       size_t out_cstride, int Hx, int Hp, int ny, int nz, int nrows, int nx_in,
                       FftPlanDev p, int lpw, const TIN *__restrict__ in_alt = nullptr,
                       const int *__restrict__ sel = nullptr)
{
    if (sel && *sel) in = in_alt;
    xfwd_body<T, TIN, LC>(in, in_cstride, out, out_cstride, Hx, Hp, ny, nz, nrows, nx_in, p, lpw, (int)blockIdx.x);
}

// y forward: columns kx of planes (c, z); rows y < ny_in read, Py written.
// O32: both arrays under 4 GiB and a row under 16 MiB: 32-bit byte offsets
// from the kernel-argument bases, rows stepped by 24-bit multiplies
// tile: (kx tile, z, c) with the kx tile fastest, ntx kx tiles per plane
template <typename T, int LC = 0, bool O32 = false>
__device__ __forceinline__ void yfwd_body(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp,
                                          int ny_in, int nzl, const FftPlanDev &p, int tk, int tile, int ntx,
                                          unsigned mtx, unsigned mzl)
{
    constexpr int SK = MM_SKEW_Y;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L);
    // tk is a power of two
    const int ltk = __ffs(tk) - 1;
    const int q1 = (int)udiv((unsigned)tile, (unsigned)ntx, mtx), c = (int)udiv((unsigned)q1, (unsigned)nzl, mzl);
    const int kx0 = (tile - q1 * ntx) * tk;
    const int z = q1 - c * nzl;
    const C2<T> *src = in + ((size_t)c * nzl + z) * (size_t)ny_in * Hp;
    C2<T> *dst = out + ((size_t)c * nzl + z) * (size_t)L * Hp;
    C2<T> *twl = sm + (size_t)tk * LP;
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    // global passes: columns fastest across the threads (row segments of tk
    // values per load); LDS passes: one line per group of tline threads
    const int lg = threadIdx.x & (tk - 1), ls = threadIdx.x / PlanC<LC>::tline(p);
    const int tg = (int)(threadIdx.x >> ltk);
    const LineMap mg = {tg, tg < PlanC<LC>::tline(p)}, ms = {(int)(threadIdx.x % PlanC<LC>::tline(p)), ls < tk};
    const int kx = kx0 + lg;
    constexpr unsigned CS = sizeof(C2<T>);
    const unsigned rs = (unsigned)Hp * CS, pl = ((unsigned)c * nzl + z);
    const unsigned sb = O32 ? (pl * (unsigned)ny_in * Hp + kx) * CS : 0u, db = O32 ? (pl * (unsigned)L * Hp + kx) * CS : 0u;
    fft_line<T, false, true, true, LC, SK>(
        p, twl, sm + (size_t)lg * LP, mg, sm + (size_t)ls * LP, ms,
        [&](int y) {
            if (!(y < ny_in && kx < Hx)) return cmk<T>((T)0, (T)0);
            if constexpr (O32) return *(const C2<T> *)((const char *)in + (sb + __umul24((unsigned)y, rs)));
            else return src[(size_t)y * Hp + kx];
        },
        [&](int y, C2<T> v) {
            if (kx < Hx) {
                if constexpr (O32) *(C2<T> *)((char *)out + (db + __umul24((unsigned)y, rs))) = v;
                else dst[(size_t)y * Hp + kx] = v;
            }
        }, [&] { twf.store(twl); });
}

template <typename T, int LC = 0, bool O32 = false>
__global__ void k_yfwd(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp, int ny_in,
                       int nzl, FftPlanDev p, int tk, int remap, unsigned mtx, unsigned mzl)
{
    yfwd_body<T, LC, O32>(in, out, Hx, Hp, ny_in, nzl, p, tk, block_tile(remap), (int)gridDim.x, mtx, mzl);
}

// y inverse: columns of S2 planes (c, z), all Py rows read, y < ny_out
// written; O32 as k_yfwd
template <typename T, int LC = 0, bool O32 = false>
__device__ __forceinline__ void yinv_body(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp,
                                          int ny_out, int nzl, const FftPlanDev &p, int tk, int tile, int ntx,
                                          unsigned mtx, unsigned mzl)
{
    constexpr int SK = MM_SKEW_Y;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L);
    const int ltk = __ffs(tk) - 1;
    const int q1 = (int)udiv((unsigned)tile, (unsigned)ntx, mtx), c = (int)udiv((unsigned)q1, (unsigned)nzl, mzl);
    const int kx0 = (tile - q1 * ntx) * tk;
    const int z = q1 - c * nzl;
    const C2<T> *src = in + ((size_t)c * nzl + z) * (size_t)L * Hp;
    C2<T> *dst = out + ((size_t)c * nzl + z) * (size_t)ny_out * Hp;
    C2<T> *twl = sm + (size_t)tk * LP;
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    const int lg = threadIdx.x & (tk - 1), ls = threadIdx.x / PlanC<LC>::tline(p);
    const int tg = (int)(threadIdx.x >> ltk);
    const LineMap mg = {tg, tg < PlanC<LC>::tline(p)}, ms = {(int)(threadIdx.x % PlanC<LC>::tline(p)), ls < tk};
    const int kx = kx0 + lg;
    constexpr unsigned CS = sizeof(C2<T>);
    const unsigned rs = (unsigned)Hp * CS, pl = ((unsigned)c * nzl + z);
    const unsigned sb = O32 ? (pl * (unsigned)L * Hp + kx) * CS : 0u, db = O32 ? (pl * (unsigned)ny_out * Hp + kx) * CS : 0u;
    fft_line<T, true, true, true, LC, SK>(
        p, twl, sm + (size_t)lg * LP, mg, sm + (size_t)ls * LP, ms,
        [&](int y) {
            if (!(kx < Hx)) return cmk<T>((T)0, (T)0);
            if constexpr (O32) return *(const C2<T> *)((const char *)in + (sb + __umul24((unsigned)y, rs)));
            else return src[(size_t)y * Hp + kx];
        },
        [&](int y, C2<T> v) {
            if (y < ny_out && kx < Hx) {
                if constexpr (O32) *(C2<T> *)((char *)out + (db + __umul24((unsigned)y, rs))) = v;
                else dst[(size_t)y * Hp + kx] = v;
            }
        }, [&] { twf.store(twl); });
}

template <typename T, int LC = 0, bool O32 = false>
__global__ void k_yinv(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp, int ny_out,
                       int nzl, FftPlanDev p, int tk, int remap, unsigned mtx, unsigned mzl)
{
    yinv_body<T, LC, O32>(in, out, Hx, Hp, ny_out, nzl, p, tk, block_tile(remap), (int)gridDim.x, mtx, mzl);
}

// Pruned y transforms for zero-padded lines (P = 2h even, data only in
// y < ny <= h).  Forward: X[2m] = DFT_h(x)[m], X[2m+1] = DFT_h(x W_P^n)[m];
// inverse: x[n] = IDFT_h(X_even)[n] + W_P^-n IDFT_h(X_odd)[n] for n < h.
// Two half-length transforms per line halve the LDS per line, which lets a
// workgroup take 128-byte column tiles.  twP: the length-P twiddle table.
// Each thread keeps the elements e = tid + q*blockDim (col = e % tk,
// n = e / tk) of its tile in registers between the two halves; blockDim =
// tk * tline with tline >= h/8 gives at most 8 per thread.
template <typename T>
__global__ void k_yfwd_pr(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp, int ny_in,
                          int nzl, FftPlanDev ph, const C2<T> *__restrict__ twP, int tk)
{
    constexpr int SK = MM_SKEW_Y;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int h = ph.L, LP = lds_len<SK>(h);
    const int kx0 = blockIdx.x * tk;
    const int z = blockIdx.y, c = blockIdx.z;
    const C2<T> *src = in + ((size_t)c * nzl + z) * (size_t)ny_in * Hp;
    C2<T> *dst = out + ((size_t)c * nzl + z) * (size_t)(2 * h) * Hp;
    C2<T> *twl = sm + (size_t)tk * LP;
    load_twiddles<T>(twl, ph);
    constexpr int MAXE = 8;
    C2<T> xr[MAXE];
#pragma unroll
    for (int q = 0; q < MAXE; ++q) {
        const int e = threadIdx.x + q * blockDim.x;
        const int col = e % tk, n = e / tk, kx = kx0 + col;
        xr[q] = cmk<T>((T)0, (T)0);
        if (e < tk * h) {
            if (n < ny_in && kx < Hx) xr[q] = src[(size_t)n * Hp + kx];
            sm[col * LP + sk<SK>(n)] = xr[q];
        }
    }
    __syncthreads();
    const int l = threadIdx.x / ph.tline, t = threadIdx.x % ph.tline;
    lds_fft<T, false, SK>(sm + (size_t)l * LP, ph, t, l < tk, twl);
    for (int e = threadIdx.x; e < tk * h; e += blockDim.x) {
        const int col = e % tk, m = e / tk, kx = kx0 + col;
        if (kx < Hx) dst[(size_t)(2 * m) * Hp + kx] = sm[col * LP + sk<SK>(m)];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MAXE; ++q) {
        const int e = threadIdx.x + q * blockDim.x;
        const int col = e % tk, n = e / tk;
        if (e < tk * h) sm[col * LP + sk<SK>(n)] = cmul<T>(xr[q], twP[n]);
    }
    __syncthreads();
    lds_fft<T, false, SK>(sm + (size_t)l * LP, ph, t, l < tk, twl);
    for (int e = threadIdx.x; e < tk * h; e += blockDim.x) {
        const int col = e % tk, m = e / tk, kx = kx0 + col;
        if (kx < Hx) dst[(size_t)(2 * m + 1) * Hp + kx] = sm[col * LP + sk<SK>(m)];
    }
}

template <typename T>
__global__ void k_yinv_pr(const C2<T> *__restrict__ in, C2<T> *__restrict__ out, int Hx, int Hp, int ny_out,
                          int nzl, FftPlanDev ph, const C2<T> *__restrict__ twP, int tk)
{
    constexpr int SK = MM_SKEW_Y;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int h = ph.L, LP = lds_len<SK>(h);
    const int kx0 = blockIdx.x * tk;
    const int z = blockIdx.y, c = blockIdx.z;
    const C2<T> *src = in + ((size_t)c * nzl + z) * (size_t)(2 * h) * Hp;
    C2<T> *dst = out + ((size_t)c * nzl + z) * (size_t)ny_out * Hp;
    const int l = threadIdx.x / ph.tline, t = threadIdx.x % ph.tline;
    C2<T> *twl = sm + (size_t)tk * LP;
    load_twiddles<T>(twl, ph);
    constexpr int MAXE = 8;
    C2<T> ar[MAXE];
    for (int e = threadIdx.x; e < tk * h; e += blockDim.x) {
        const int col = e % tk, m = e / tk, kx = kx0 + col;
        sm[col * LP + sk<SK>(m)] = (kx < Hx) ? src[(size_t)(2 * m) * Hp + kx] : cmk<T>((T)0, (T)0);
    }
    __syncthreads();
    lds_fft<T, true, SK>(sm + (size_t)l * LP, ph, t, l < tk, twl);
#pragma unroll
    for (int q = 0; q < MAXE; ++q) {
        const int e = threadIdx.x + q * blockDim.x;
        const int col = e % tk, n = e / tk;
        ar[q] = (e < tk * h) ? sm[col * LP + sk<SK>(n)] : cmk<T>((T)0, (T)0);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < tk * h; e += blockDim.x) {
        const int col = e % tk, m = e / tk, kx = kx0 + col;
        sm[col * LP + sk<SK>(m)] = (kx < Hx) ? src[(size_t)(2 * m + 1) * Hp + kx] : cmk<T>((T)0, (T)0);
    }
    __syncthreads();
    lds_fft<T, true, SK>(sm + (size_t)l * LP, ph, t, l < tk, twl);
#pragma unroll
    for (int q = 0; q < MAXE; ++q) {
        const int e = threadIdx.x + q * blockDim.x;
        const int col = e % tk, n = e / tk, kx = kx0 + col;
        if (e < tk * h && n < ny_out && kx < Hx)
            dst[(size_t)n * Hp + kx] = cadd<T>(ar[q], cmul<T>(sm[col * LP + sk<SK>(n)], cconj<T>(twP[n])));
    }
}

// real octant-stored kernel entry e at (kx, ky, kz) of the full spectrum
template <typename T>
__device__ __forceinline__ void kernel_at(const T *__restrict__ K, size_t plane, int Hp, int Hy2,
                                          int Py, int Pz, int kx, int ky, int kz, T k[6])
{
    const bool fy = ky > Py / 2, fz = kz > Pz / 2;
    const int kyf = fy ? Py - ky : ky;
    const int kzf = fz ? Pz - kz : kz;
    const size_t o = ((size_t)kzf * Hy2 + kyf) * Hp + kx;
    const T sy = fy ? (T)-1 : (T)1, sz = fz ? (T)-1 : (T)1;
    k[0] = K[o];
    k[1] = sy * K[plane + o];
    k[2] = sz * K[2 * plane + o];
    k[3] = K[3 * plane + o];
    k[4] = sy * sz * K[4 * plane + o];
    k[5] = K[5 * plane + o];
}

// kernel items (column, kz pair) per thread of the z pass
#define ZM_ITEMS 2

// z pass (3-D): forward over z (nz rows, zero-extended), multiply, inverse,
// keep z < nz.  Lines: 3 components x tk columns for one ky.
// O32: S2 and K are under 4 GiB and a z step of S2 under 16 MiB (zsb bytes),
// so every access is a 32-bit byte offset from the kernel-argument base
// (global_load with an SGPR base: no 64-bit address arithmetic per element;
// the offsets' z steps are 24-bit multiplies); pb: bytes of one K plane.
template <typename T, int LC = 0, bool O32 = false>
__device__ __forceinline__ void zmi_body(C2<T> *__restrict__ S2, const T *__restrict__ K, size_t plane, int Hx,
                                         int Hp, int Hy2, int Py, int nz, const FftPlanDev &p, int tk, int remap,
                                         int tile, int ntx, unsigned mtx, unsigned zsb, unsigned pb)
{
    constexpr int SK = MM_SKEW_Z;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L);
    // tiles (kx tile, m), kx tile fastest.  With remap, rows come in the order
    // 0, 1, Py-1, 2, Py-2, ...: ky and Py-ky read the same kernel row
    // tk is a power of two
    const int ltk = __ffs(tk) - 1;
    const int m = (int)udiv((unsigned)tile, (unsigned)ntx, mtx), hm = (m + 1) >> 1;
    const int kx0 = (tile - m * ntx) * tk;
    const int ky = !remap || m == 0 ? m : ((m & 1) ? hm : Py - hm);
    const size_t cstride = (size_t)nz * Py * Hp;
    const size_t zstride = (size_t)Py * Hp;
    C2<T> *base = S2 + (size_t)ky * Hp;
    C2<T> *twl = sm + (size_t)3 * tk * LP;
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    // global passes: columns fastest, then components; LDS passes: one line
    // (component c, column) per group of tline threads
    const int colg = threadIdx.x & (tk - 1), cg = (int)(threadIdx.x >> ltk) % 3;
    const int tg = (int)(threadIdx.x >> ltk) / 3;
    const LineMap mg = {tg, tg < PlanC<LC>::tline(p)};
    C2<T> *lineG = sm + (size_t)(cg * tk + colg) * LP;
    const int l = threadIdx.x / PlanC<LC>::tline(p), t = threadIdx.x % PlanC<LC>::tline(p);
    const LineMap ms = {t, l < 3 * tk};
    C2<T> *line = sm + (size_t)l * LP;
    const int kxg = kx0 + colg;
    C2<T> *colp = base + cg * cstride + kxg;
    const unsigned cb = O32 ? (unsigned)(((size_t)cg * cstride + (size_t)ky * Hp + kxg) * sizeof(C2<T>)) : 0u;
    auto col_at = [&](int z) -> C2<T> & {
        if constexpr (O32) return *(C2<T> *)((char *)S2 + (cb + __umul24((unsigned)z, zsb)));
        else return colp[z * zstride];
    };
    // The kernel entries this thread multiplies load before the forward
    // transform, so their latency hides behind it.  Items (col, kzf) with
    // kzf <= L/2 each serve kz = kzf and the mirror kz = L - kzf, whose xz
    // and yz entries change sign (real octant storage, as kernel_at); at most
    // ZM_ITEMS per thread (the host checks).
    const int nitems = tk * (L / 2 + 1);
    const bool fy = ky > Py / 2;
    const int kyf = fy ? Py - ky : ky;
    const T sy = fy ? (T)-1 : (T)1;
    T kk[ZM_ITEMS][6];
#pragma unroll
    for (int j = 0; j < ZM_ITEMS; ++j) {
        const int e = threadIdx.x + j * blockDim.x;
        const int col = e & (tk - 1), kzf = e >> ltk, kx = kx0 + col;
        if (e < nitems && kx < Hx) {
            const size_t o = ((size_t)kzf * Hy2 + kyf) * Hp + kx;
            if constexpr (O32) {
                const unsigned ob = (unsigned)o * (unsigned)sizeof(T);
#pragma unroll
                for (int q = 0; q < 6; ++q) kk[j][q] = *(const T *)((const char *)K + (ob + (unsigned)q * pb));
            } else {
#pragma unroll
                for (int q = 0; q < 6; ++q) kk[j][q] = K[q * plane + o];
            }
        }
    }
    fft_line<T, false, true, false, LC, SK>(
        p, twl, lineG, mg, line, ms,
        [&](int z) { return (z < nz && kxg < Hx) ? col_at(z) : cmk<T>((T)0, (T)0); },
        [](int, C2<T>) {}, [&] { twf.store(twl); });
#pragma unroll
    for (int j = 0; j < ZM_ITEMS; ++j) {
        const int e = threadIdx.x + j * blockDim.x;
        const int col = e & (tk - 1), kzf = e >> ltk, kx = kx0 + col;
        if (e < nitems && kx < Hx) {
            const T k[6] = {kk[j][0], sy * kk[j][1], kk[j][2], kk[j][3], sy * kk[j][4], kk[j][5]};
            C2<T> *l0 = sm + (size_t)(0 * tk + col) * LP, *l1 = sm + (size_t)(1 * tk + col) * LP,
                  *l2 = sm + (size_t)(2 * tk + col) * LP;
            mult3<T>(l0[sk<SK>(kzf)], l1[sk<SK>(kzf)], l2[sk<SK>(kzf)], k);
            const int kz2 = L - kzf;
            if (kzf > 0 && kz2 != kzf) mult3_mirror<T>(l0[sk<SK>(kz2)], l1[sk<SK>(kz2)], l2[sk<SK>(kz2)], k);
        }
    }
    __syncthreads();
    fft_line<T, true, false, true, LC, SK>(
        p, twl, lineG, mg, line, ms, [](int) { return cmk<T>((T)0, (T)0); },
        [&](int z, C2<T> v) {
            if (z < nz && kxg < Hx) col_at(z) = v;
        });
}

template <typename T, int LC = 0, bool O32 = false>
__global__ void k_zmi(C2<T> *__restrict__ S2, const T *__restrict__ K, size_t plane, int Hx, int Hp, int Hy2,
                      int Py, int nz, FftPlanDev p, int tk, int remap, unsigned mtx, unsigned zsb, unsigned pb)
{
    zmi_body<T, LC, O32>(S2, K, plane, Hx, Hp, Hy2, Py, nz, p, tk, remap, block_tile(remap), (int)gridDim.x, mtx,
                         zsb, pb);
}

// 2-D: y forward (ny rows, zero-extended) + multiply (kz = 0) + y inverse,
// keep y < ny, in place on S1 planes [c][y][kx].
template <typename T, int LC = 0>
__device__ __forceinline__ void ymi2d_body(C2<T> *__restrict__ S1, const T *__restrict__ K, size_t plane, int Hx,
                                           int Hp, int Hy2, int ny, const FftPlanDev &p, int tk, int blk)
{
    constexpr int SK = MM_SKEW_Y;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p), LP = lds_len<SK>(L);
    const int kx0 = blk * tk;
    const size_t cstride = (size_t)ny * Hp;
    C2<T> *twl = sm + (size_t)3 * tk * LP;
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    const int colg = threadIdx.x % tk, cg = (threadIdx.x / tk) % 3;
    const int tg = (int)(threadIdx.x / (3 * tk));
    const LineMap mg = {tg, tg < PlanC<LC>::tline(p)};
    C2<T> *lineG = sm + (size_t)(cg * tk + colg) * LP;
    const int l = threadIdx.x / PlanC<LC>::tline(p), t = threadIdx.x % PlanC<LC>::tline(p);
    const LineMap ms = {t, l < 3 * tk};
    C2<T> *line = sm + (size_t)l * LP;
    const int kxg = kx0 + colg;
    C2<T> *colp = S1 + cg * cstride + kxg;
    fft_line<T, false, true, false, LC, SK>(
        p, twl, lineG, mg, line, ms,
        [&](int y) { return (y < ny && kxg < Hx) ? colp[(size_t)y * Hp] : cmk<T>((T)0, (T)0); },
        [](int, C2<T>) {}, [&] { twf.store(twl); });
    for (int e = threadIdx.x; e < tk * L; e += blockDim.x) {
        const int col = e % tk, ky = e / tk, kx = kx0 + col;
        if (kx < Hx) {
            T k[6];
            kernel_at<T>(K, plane, Hp, Hy2, L, 1, kx, ky, 0, k);
            mult3<T>(sm[(0 * tk + col) * LP + sk<SK>(ky)], sm[(1 * tk + col) * LP + sk<SK>(ky)], sm[(2 * tk + col) * LP + sk<SK>(ky)], k);
        }
    }
    __syncthreads();
    fft_line<T, true, false, true, LC, SK>(
        p, twl, lineG, mg, line, ms, [](int) { return cmk<T>((T)0, (T)0); },
        [&](int y, C2<T> v) {
            if (y < ny && kxg < Hx) colp[(size_t)y * Hp] = v;
        });
}

template <typename T, int LC = 0>
__global__ void k_ymi2d(C2<T> *__restrict__ S1, const T *__restrict__ K, size_t plane, int Hx, int Hp, int Hy2,
                        int ny, FftPlanDev p, int tk)
{
    ymi2d_body<T, LC>(S1, K, plane, Hx, Hp, Hy2, ny, p, tk, (int)blockIdx.x);
}

// x inverse (C2R): rows (c, z, y) of S1, Hermitian extension, keep x < nx
template <typename T, typename TOUT, int LC = 0>
__global__ void k_xinv(const C2<T> *__restrict__ in, TOUT *__restrict__ out, size_t out_cstride, int Hx,
                       int Hp, int ny, int nz, int nrows, int nx, FftPlanDev p, int lpw)
{
    constexpr int SK = MM_SKEW_X;
    extern __shared__ char smem_raw[];
    C2<T> *sm = reinterpret_cast<C2<T> *>(smem_raw);
    const int L = PlanC<LC>::L(p);
    const int l = threadIdx.x / PlanC<LC>::tline(p), t = threadIdx.x % PlanC<LC>::tline(p);
    const int g = blockIdx.x * lpw + l;
    const bool active = g < nrows;
    C2<T> *line = sm + (size_t)l * lds_len<SK>(L);
    C2<T> *twl = sm + (size_t)lpw * lds_len<SK>(L);
    const TwFetch<T> twf = TwFetch<T>::fetch(p);
    const int c = active ? g / (ny * nz) : 0, r = active ? g % (ny * nz) : 0;
    const C2<T> *src = in + (size_t)(active ? g : 0) * Hp;
    TOUT *dst = out + c * out_cstride + (size_t)r * nx;
    const LineMap m = {t, active};
    fft_line<T, true, true, true, LC, SK>(
        p, twl, line, m, line, m,
        [&](int k) {
            // one unconditional load per element (the conjugate by an exact
            // sign): a load in each arm of a branch made the compiler wait
            // for every element's load before issuing the next
            const bool lo = k < Hx;
            const C2<T> v = src[lo ? k : L - k];
            return cmk<T>(v.x, (lo ? (T)1 : (T)-1) * v.y);
        },
        [&](int x, C2<T> v) {
            if (x < nx) dst[x] = (TOUT)v.x;
        }, [&] { twf.store(twl); });
}

// setup: forward z over full lines (no multiply), all Pz outputs stored
static __global__ void k_zfwd_setup(double2 *__restrict__ S, int Hx, int Hp, int Py, FftPlanDev p, int tk)
{
    constexpr int SK = MM_SKEW_Z;
    extern __shared__ char smem_raw[];
    double2 *sm = reinterpret_cast<double2 *>(smem_raw);
    const int L = p.L, LP = lds_len<SK>(L);
    const int kx0 = blockIdx.x * tk, ky = blockIdx.y;
    const size_t zstride = (size_t)Py * Hp;
    double2 *base = S + (size_t)ky * Hp;
    double2 *twl = sm + (size_t)tk * LP;
    load_twiddles<double>(twl, p);
    for (int e = threadIdx.x; e < tk * L; e += blockDim.x) {
        const int col = e % tk, z = e / tk, kx = kx0 + col;
        sm[col * LP + sk<SK>(z)] = kx < Hx ? base[z * zstride + kx] : cmk<double>(0.0, 0.0);
    }
    __syncthreads();
    const int l = threadIdx.x / p.tline, t = threadIdx.x % p.tline;
    lds_fft<double, false, SK>(sm + (size_t)l * LP, p, t, l < tk, twl);
    for (int e = threadIdx.x; e < tk * L; e += blockDim.x) {
        const int col = e % tk, z = e / tk, kx = kx0 + col;
        if (kx < Hx) base[z * zstride + kx] = sm[col * LP + sk<SK>(z)];
    }
}

// setup: real part of the octant ky <= Py/2, kz <= Pz/2, scaled
template <typename T>
__global__ void k_extract_kernel(const double2 *__restrict__ S, T *__restrict__ K, int Hx, int Hp, int Py,
                                 int Hy2, int Hz2, double scale)
{
    const size_t n = (size_t)Hx * Hy2 * Hz2;
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const int kx = (int)(q % Hx);
        const size_t r = q / Hx;
        const int ky = (int)(r % Hy2), kz = (int)(r / Hy2);
        K[((size_t)kz * Hy2 + ky) * Hp + kx] = (T)(scale * S[((size_t)kz * Py + ky) * Hp + kx].x);
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int grid_1d(size_t n, int bs)
{
    size_t b = (n + bs - 1) / bs;
    return (int)std::min<size_t>(b, 65535 * 64);
}

template <typename T>
void ConvImpl<T>::init(const double *N_host, int nx, int ny, int nz, int ex, int ey, int ez)
{
    MM_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1, "bad mesh size");
    g.nx = nx; g.ny = ny; g.nz = nz;
    g.Px = mm_fft_size_for(nx, ex);
    g.Py = mm_fft_size_for(ny, ey);
    g.Pz = mm_fft_size_for(nz, ez);
    g.Hx = g.Px / 2 + 1;
    // spectral row pitch: a multiple of 16 complex values, so that rows and
    // the column tiles of the y/z passes start on 128-byte boundaries
    g.Hp = (g.Hx + 15) / 16 * 16;
    g.Hy2 = g.Py / 2 + 1;
    g.Hz2 = g.Pz / 2 + 1;
    g.is2d = (nz == 1 && g.Pz == 1);
    px.build(g.Px);
    py.build(g.Py);
    pz.build(g.Pz);
    // MM_FFT_GENERIC=1: runtime FFT plans for every length, single and batched
    // (tests compare them with the compiled plans)
    fft_generic = env_int("MM_FFT_GENERIC", 0) != 0;
    if (fft_generic)
        for (FftPlanHost *p : {&px, &py, &pz}) p->no_compiled();
    else if (!mm_plan_z(g.Pz))
        pz.no_compiled();
    // The narrow y plans once the wide ones, whose tiles hold one column (2-D)
    // or two to four (3-D), fill the chip: there the row segments count, and
    // fewer workgroups finish sooner with more threads to a line.  Field, wide
    // -> narrow, MI355X: 256x450x1 (900 points, 257 workgroups) FP64 55.0 ->
    // 41.7 us, FP32 33.0 -> 32.3; 450x450x8 FP64 401 -> 356, FP32 196 -> 162;
    // 500x500x1 FP64 80.5 -> 70.2; 270x270x8 FP64 136 -> 129, FP32 81.4 ->
    // 81.3; below, 64x450x1 (65 workgroups) FP32 22.7 -> 27.1, 64x270x1 FP64
    // 21.9 -> 23.9.
    {
        const int cols = floor_pow2(1024 / ((g.is2d ? 3 : 1) * py.tline));
        const size_t wgs = (size_t)((g.Hx + cols - 1) / cols) * (g.is2d ? 1 : 3 * nz);
        pyn = py.narrow();
        y_narrow = !fft_generic && pyn.id > 0 && wgs >= (size_t)mm_num_cus();
        if (y_narrow) tk_yn = mm_choose_launch(g, px, pyn, pz, sizeof(C2<T>)).tk_y;
    }
    ln = mm_choose_launch(g, px, py, pz, sizeof(C2<T>));
    // MM_WIDE_INDEX=1: the general forms of the index arithmetic (integer
    // division, 64-bit element addressing) that grids beyond the 32-bit
    // ranges take, for any grid (tests compare both; the results are equal)
    wide = env_int("MM_WIDE_INDEX", 0) != 0;
    // MM_XCD_REMAP=0: hardware workgroup order for the tiles (measurements)
    xcd_remap = env_int("MM_XCD_REMAP", 1) != 0 ? 1 : 0;
    // pruned y transforms when the padding is at least half of the line
    {
        // measured on MI355X (256x256x16 cells): slower than the full-length
        // y transforms in FP32 (48 vs 38 us per launch), equal in FP64; opt-in
        const char *e = std::getenv("MM_PRUNE_Y");
        const bool want = e && std::atoi(e) != 0;
        prune_y = want && !g.is2d && g.Py % 2 == 0 && ny <= g.Py / 2 && g.Py / 2 >= 8;
        if (prune_y) {
            pyh.build(g.Py / 2);
            pyh.no_compiled();
            const int lds = mm_max_lds_bytes();
            const size_t cs = sizeof(C2<T>);
            int tk = env_int("MM_TK_YP", (int)(128 / cs));
            while (tk > 1 && ((size_t)tk * pyh.tline > 1024 || lines_lds<MM_SKEW_Y>(tk, pyh.L, cs) > (size_t)lds)) tk /= 2;
            tk_yp = tk;
        }
    }
    MM_REQUIRE((size_t)px.tline <= 1024, "x transform length too large");

    // re-embed the tensor into the radix-friendly padded grid
    const int Px = g.Px, Py = g.Py, Pz = g.Pz;
    auto map_axis = [](int X, int e, int n, int P) -> int {
        if (X < n) return X;
        if (X > e - n) return P - (e - X);
        return -1;
    };
    const size_t plane_full = (size_t)Px * Py * Pz;
    std::vector<double> Nr((size_t)6 * plane_full, 0.0);
    for (int Z = 0; Z < ez; ++Z) {
        const int z2 = map_axis(Z, ez, nz, Pz);
        if (z2 < 0) continue;
        for (int Y = 0; Y < ey; ++Y) {
            const int y2 = map_axis(Y, ey, ny, Py);
            if (y2 < 0) continue;
            for (int X = 0; X < ex; ++X) {
                const int x2 = map_axis(X, ex, nx, Px);
                if (x2 < 0) continue;
                const double *src = N_host + 6 * ((size_t)X + (size_t)ex * ((size_t)Y + (size_t)ey * Z));
                const size_t dst = (size_t)x2 + (size_t)Px * ((size_t)y2 + (size_t)Py * z2);
                for (int e = 0; e < 6; ++e) Nr[e * plane_full + dst] = src[e];
            }
        }
    }

    // Fourier transform of each component in FP64 on the device
    const size_t plane = (size_t)g.Hp * g.Hy2 * g.Hz2;
    kern_elems = 6 * plane;
    MM_HIP(hipMalloc(&kern, sizeof(T) * kern_elems));
    MM_HIP(hipMemset(kern, 0, sizeof(T) * kern_elems));
    double *dN = nullptr;
    double2 *T1 = nullptr, *T2 = nullptr;
    const size_t nspec = (size_t)g.Hp * Py * Pz;
    MM_HIP(hipMalloc(&dN, sizeof(double) * plane_full));
    MM_HIP(hipMalloc(&T1, sizeof(double2) * nspec));
    MM_HIP(hipMalloc(&T2, sizeof(double2) * nspec));
    const int lds = mm_max_lds_bytes();
    const FftPlanDev dx = px.dev_loop<double>(), dy = py.dev_loop<double>(), dz = pz.dev_loop<double>();
    int lpw = std::max(1, 256 / dx.tline);
    while (lpw > 1 && lines_lds<MM_SKEW_X>(lpw, dx.L, 16) > (size_t)lds) --lpw;
    int tky = 8;
    while (tky > 1 && ((size_t)tky * dy.tline > 1024 || lines_lds<MM_SKEW_Y>(tky, dy.L, 16) > (size_t)lds)) tky /= 2;
    int tkz = 8;
    while (tkz > 1 && ((size_t)tkz * dz.tline > 1024 || lines_lds<MM_SKEW_Z>(tkz, dz.L, 16) > (size_t)lds)) tkz /= 2;
    const size_t shx = lines_lds<MM_SKEW_X>(lpw, dx.L, 16), shy = lines_lds<MM_SKEW_Y>(tky, dy.L, 16),
                 shz = lines_lds<MM_SKEW_Z>(tkz, dz.L, 16);
    set_lds(k_xfwd<double, double>, shx);
    set_lds(k_yfwd<double>, shy);
    set_lds(k_zfwd_setup, shz);
    const double scale = 1.0 / ((double)Px * (double)Py * (double)Pz);
    for (int e = 0; e < 6; ++e) {
        MM_HIP(hipMemcpy(dN, Nr.data() + e * plane_full, sizeof(double) * plane_full, hipMemcpyHostToDevice));
        const int nrows = Py * Pz;
        hipLaunchKernelGGL((k_xfwd<double, double>), dim3(((nrows + 1) / 2 + lpw - 1) / lpw), dim3(lpw * dx.tline), shx, 0,
                           dN, 0, T1, 0, g.Hx, g.Hp, Py, Pz, nrows, Px, dx, lpw, (const double *)nullptr,
                           (const int *)nullptr);
        MM_HIP(hipGetLastError());
        const unsigned ntyk = (unsigned)((g.Hx + tky - 1) / tky), nbk = ntyk * Pz;
        hipLaunchKernelGGL((k_yfwd<double>), dim3(ntyk, Pz, 1), dim3(tky * dy.tline), shy, 0, T1, T2, g.Hx, g.Hp, Py,
                           Pz, dy, tky, 0, mdiv(ntyk, nbk), mdiv((unsigned)Pz, nbk));
        MM_HIP(hipGetLastError());
        if (Pz > 1) {
            hipLaunchKernelGGL(k_zfwd_setup, dim3((g.Hx + tkz - 1) / tkz, Py, 1), dim3(tkz * dz.tline), shz, 0,
                               T2, g.Hx, g.Hp, Py, dz, tkz);
            MM_HIP(hipGetLastError());
        }
        hipLaunchKernelGGL((k_extract_kernel<T>), dim3(grid_1d(plane, 256)), dim3(256), 0, 0, T2, kern + e * plane,
                           g.Hx, g.Hp, Py, g.Hy2, g.Hz2, scale);
        MM_HIP(hipGetLastError());
    }
    MM_HIP(hipDeviceSynchronize());
    (void)hipFree(dN);
    (void)hipFree(T1);
    (void)hipFree(T2);

    MM_HIP(hipMalloc(&S1, sizeof(C2<T>) * 3 * (size_t)nz * ny * g.Hp));
    if (!g.is2d) MM_HIP(hipMalloc(&S2, sizeof(C2<T>) * 3 * (size_t)nz * Py * g.Hp));

    const size_t cs = sizeof(C2<T>);
    set_lds(k_xfwd<T, T>, lines_lds<MM_SKEW_X>(ln.lpw_x, px.L, cs));
    set_lds(k_xinv<T, T>, lines_lds<MM_SKEW_X>(ln.lpw_x, px.L, cs));
    if (g.is2d) {
        set_lds(k_ymi2d<T>, lines_lds<MM_SKEW_Y>(3 * ln.tk_y, py.L, cs));
    } else {
        set_lds(k_yfwd<T>, lines_lds<MM_SKEW_Y>(ln.tk_y, py.L, cs));
        set_lds(k_yinv<T>, lines_lds<MM_SKEW_Y>(ln.tk_y, py.L, cs));
        set_lds(k_zmi<T>, lines_lds<MM_SKEW_Z>(3 * ln.tk_z, pz.L, cs));
    }
}

template <typename T> void ConvImpl<T>::release()
{
    if (kern) (void)hipFree(kern);
    if (S1) (void)hipFree(S1);
    if (S2) (void)hipFree(S2);
    kern = nullptr;
    S1 = S2 = nullptr;
    px.release();
    py.release();
    pz.release();
    pyh.release();
}

// algorithmic HBM bytes per launch (each array read or written once)
template <typename T> static double conv_bytes(const ConvGeom &g, int cls)
{
    const double b = sizeof(T), c = 2.0 * sizeof(T);
    const double N = (double)g.nx * g.ny * g.nz;
    const double s1 = 3.0 * c * g.Hx * g.ny * g.nz;  // S1 planes
    const double s2 = 3.0 * c * g.Hx * g.Py * g.nz;  // S2 planes
    const double K = 6.0 * b * g.Hx * g.Hy2 * g.Hz2;  // real octant kernel
    switch (cls) {
    case KC_XFWD: return 3.0 * b * N + s1;
    case KC_YFWD: return s1 + s2;
    case KC_ZMI: return 2.0 * s2 + K;
    case KC_YINV: return s2 + s1;
    case KC_YMI2D: return 2.0 * s1 + K;
    default: return 0.0;
    }
}

template <typename T> void ConvImpl<T>::forward_x(const T *M, hipStream_t s, const T *M_alt, const int *sel)
{
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    const int nrows = 3 * g.ny * g.nz;
    const size_t sh = lines_lds<MM_SKEW_X>(ln.lpw_x, px.L, sizeof(C2<T>));
    mm_with_len(px.L, fft_generic, [&](auto lc) {
        hipLaunchKernelGGL((k_xfwd<T, T, decltype(lc)::value>), dim3(((nrows + 1) / 2 + ln.lpw_x - 1) / ln.lpw_x),
                           dim3(ln.lpw_x * px.tline), sh, s, M, n, S1, (size_t)g.ny * g.nz * g.Hp, g.Hx, g.Hp, g.ny,
                           g.nz, nrows, g.nx, px.dev<T>(), ln.lpw_x, M_alt, sel);
    });
    MM_HIP(hipGetLastError());
    if (klog) klog->mark(s, KC_XFWD, conv_bytes<T>(g, KC_XFWD));
}

template <typename T> void ConvImpl<T>::spectral(hipStream_t s)
{
    const size_t cs = sizeof(C2<T>);
    const size_t plane = (size_t)g.Hp * g.Hy2 * g.Hz2;
    if (g.is2d) {
        const int tk = ln.tk_y;
        const size_t sh = lines_lds<MM_SKEW_Y>(3 * tk, py.L, cs);
        if (y_narrow) mm_narrow_ymi2d<T>(*this, s);
        else mm_with_len(py.L, fft_generic, [&](auto lc) {
            hipLaunchKernelGGL((k_ymi2d<T, decltype(lc)::value>), dim3((g.Hx + tk - 1) / tk), dim3(3 * tk * py.tline),
                               sh, s, S1, kern, plane, g.Hx, g.Hp, g.Hy2, g.ny, py.dev<T>(), tk);
        });
        MM_HIP(hipGetLastError());
        if (klog) klog->mark(s, KC_YMI2D, conv_bytes<T>(g, KC_YMI2D));
        return;
    }
    const int tk = ln.tk_y;
    const size_t shy = lines_lds<MM_SKEW_Y>(tk, py.L, cs);
    const bool y_o32 = y_offsets32();
    const int tkp = tk_yp;
    const size_t shyp = lines_lds<MM_SKEW_Y>(tkp, pyh.L, cs);
    if (prune_y) {
        hipLaunchKernelGGL((k_yfwd_pr<T>), dim3((g.Hx + tkp - 1) / tkp, g.nz, 3), dim3(tkp * pyh.tline), shyp, s, S1, S2,
                           g.Hx, g.Hp, g.ny, g.nz, pyh.dev<T>(), (const C2<T> *)py.plain<T>(), tkp);
    } else if (y_narrow) {
        mm_narrow_yfwd<T>(*this, s);
    } else {
        mm_with_len(py.L, fft_generic, [&](auto lc) {
            const unsigned ntx = (unsigned)((g.Hx + tk - 1) / tk), nb = ntx * g.nz * 3;
            if (y_o32)
                hipLaunchKernelGGL((k_yfwd<T, decltype(lc)::value, true>), dim3(ntx, g.nz, 3), dim3(tk * py.tline), shy,
                                   s, S1, S2, g.Hx, g.Hp, g.ny, g.nz, py.dev<T>(), tk, xcd_remap, mdiv(ntx, nb, wide),
                                   mdiv((unsigned)g.nz, nb, wide));
            else
                hipLaunchKernelGGL((k_yfwd<T, decltype(lc)::value, false>), dim3(ntx, g.nz, 3), dim3(tk * py.tline),
                                   shy, s, S1, S2, g.Hx, g.Hp, g.ny, g.nz, py.dev<T>(), tk, xcd_remap, mdiv(ntx, nb, wide),
                                   mdiv((unsigned)g.nz, nb, wide));
        });
    }
    MM_HIP(hipGetLastError());
    if (klog) klog->mark(s, KC_YFWD, conv_bytes<T>(g, KC_YFWD));
    const int tz = ln.tk_z;
    const size_t shz = lines_lds<MM_SKEW_Z>(3 * tz, pz.L, cs);
    MM_REQUIRE((size_t)tz * (pz.L / 2 + 1) <= (size_t)ZM_ITEMS * 3 * tz * pz.tline, "z pass items per thread");
    const unsigned ntz = (unsigned)((g.Hx + tz - 1) / tz);
    const unsigned mtz = mdiv(ntz, (size_t)ntz * g.Py, wide);
    const size_t zsb = (size_t)g.Py * g.Hp * cs;
    const bool o32 = zsb < (1u << 24) && 3 * (size_t)g.nz * zsb < (1ull << 32) &&
                     kern_elems * sizeof(T) < (1ull << 32) && !wide;
    if (zreg()) mm_zreg_pass<T>(*this, s);
    else mm_with_len<MM_LC_Z>(pz.L, fft_generic, [&](auto lc) {
        if (o32)
            hipLaunchKernelGGL((k_zmi<T, decltype(lc)::value, true>), dim3(ntz, g.Py), dim3(3 * tz * pz.tline), shz, s,
                               S2, kern, plane, g.Hx, g.Hp, g.Hy2, g.Py, g.nz, pz.dev<T>(), tz, xcd_remap, mtz,
                               (unsigned)zsb, (unsigned)(plane * sizeof(T)));
        else
            hipLaunchKernelGGL((k_zmi<T, decltype(lc)::value, false>), dim3(ntz, g.Py), dim3(3 * tz * pz.tline), shz,
                               s, S2, kern, plane, g.Hx, g.Hp, g.Hy2, g.Py, g.nz, pz.dev<T>(), tz, xcd_remap, mtz, 0u,
                               0u);
    });
    MM_HIP(hipGetLastError());
    if (klog) klog->mark(s, KC_ZMI, conv_bytes<T>(g, KC_ZMI));
    if (prune_y) {
        hipLaunchKernelGGL((k_yinv_pr<T>), dim3((g.Hx + tkp - 1) / tkp, g.nz, 3), dim3(tkp * pyh.tline), shyp, s, S2, S1,
                           g.Hx, g.Hp, g.ny, g.nz, pyh.dev<T>(), (const C2<T> *)py.plain<T>(), tkp);
    } else if (y_narrow) {
        mm_narrow_yinv<T>(*this, s);
    } else {
        mm_with_len(py.L, fft_generic, [&](auto lc) {
            const unsigned ntx = (unsigned)((g.Hx + tk - 1) / tk), nb = ntx * g.nz * 3;
            if (y_o32)
                hipLaunchKernelGGL((k_yinv<T, decltype(lc)::value, true>), dim3(ntx, g.nz, 3), dim3(tk * py.tline), shy,
                                   s, S2, S1, g.Hx, g.Hp, g.ny, g.nz, py.dev<T>(), tk, xcd_remap, mdiv(ntx, nb, wide),
                                   mdiv((unsigned)g.nz, nb, wide));
            else
                hipLaunchKernelGGL((k_yinv<T, decltype(lc)::value, false>), dim3(ntx, g.nz, 3), dim3(tk * py.tline),
                                   shy, s, S2, S1, g.Hx, g.Hp, g.ny, g.nz, py.dev<T>(), tk, xcd_remap, mdiv(ntx, nb, wide),
                                   mdiv((unsigned)g.nz, nb, wide));
        });
    }
    MM_HIP(hipGetLastError());
    if (klog) klog->mark(s, KC_YINV, conv_bytes<T>(g, KC_YINV));
}

template <typename T> void ConvImpl<T>::inverse_x(T *H, hipStream_t s)
{
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    const int nrows = 3 * g.ny * g.nz;
    const size_t sh = lines_lds<MM_SKEW_X>(ln.lpw_x, px.L, sizeof(C2<T>));
    mm_with_len(px.L, fft_generic, [&](auto lc) {
        hipLaunchKernelGGL((k_xinv<T, T, decltype(lc)::value>), dim3((nrows + ln.lpw_x - 1) / ln.lpw_x),
                           dim3(ln.lpw_x * px.tline), sh, s, S1, H, n, g.Hx, g.Hp, g.ny, g.nz, nrows, g.nx,
                           px.dev<T>(), ln.lpw_x);
    });
    MM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// batched passes
// ---------------------------------------------------------------------------
template <typename T>
int ConvImpl<T>::batch_x(BxDesc<T> &d, int threads, size_t &lds, const T *y0, const T *y1, const int *sel,
                         const int *stop) const
{
    const size_t cs = sizeof(C2<T>);
    MM_REQUIRE(threads >= px.tline, "batch launch has fewer threads than one x line needs");
    int lpw = std::max(1, threads / px.tline);
    while (lpw > 1 && lines_lds<MM_SKEW_X>(lpw, px.L, cs) > (size_t)mm_max_lds_bytes()) --lpw;
    const int nrows = 3 * g.ny * g.nz;
    d.y0 = y0;
    d.y1 = y1;
    d.sel = sel;
    d.stop = stop;
    d.S1 = S1;
    d.in_cstride = (size_t)g.nx * g.ny * g.nz;
    d.out_cstride = (size_t)g.ny * g.nz * g.Hp;
    d.Hx = g.Hx;
    d.Hp = g.Hp;
    d.ny = g.ny;
    d.nz = g.nz;
    d.nrows = nrows;
    d.nx = g.nx;
    d.lpw = lpw;
    d.tbase = 0;
    d.p = px.template dev<T>();
    lds = lines_lds<MM_SKEW_X>(lpw, px.L, cs);
    return ((nrows + 1) / 2 + lpw - 1) / lpw;
}

template <typename T>
int ConvImpl<T>::batch_y(ByDesc<T> &d, int threads, size_t &lds, bool &o32, const int *stop) const
{
    const size_t cs = sizeof(C2<T>);
    MM_REQUIRE(!g.is2d && threads >= py.tline, "batch y pass: 2-D system or too few threads");
    int tk = std::min(16, floor_pow2(std::max(1, threads / py.tline)));
    while (tk > 1 && lines_lds<MM_SKEW_Y>(tk, py.L, cs) > (size_t)mm_max_lds_bytes()) tk /= 2;
    const unsigned ntx = (unsigned)((g.Hx + tk - 1) / tk), nb = ntx * g.nz * 3;
    d.S1 = S1;
    d.S2 = S2;
    d.stop = stop;
    d.Hx = g.Hx;
    d.Hp = g.Hp;
    d.ny = g.ny;
    d.nz = g.nz;
    d.tk = tk;
    d.ntx = (int)ntx;
    d.tbase = 0;
    d.mtx = mdiv(ntx, nb);
    d.mzl = mdiv((unsigned)g.nz, nb);
    d.p = py.template dev<T>();
    o32 = (size_t)g.Hp * cs < (1u << 24) && (size_t)3 * g.nz * g.Py * g.Hp * cs < (1ull << 32);
    lds = lines_lds<MM_SKEW_Y>(tk, py.L, cs);
    return (int)nb;
}

template <typename T>
int ConvImpl<T>::batch_z(BzDesc<T> &d, int threads, size_t &lds, bool &o32, const int *stop) const
{
    const size_t cs = sizeof(C2<T>);
    MM_REQUIRE(!g.is2d && threads >= 3 * pz.tline, "batch z pass: 2-D system or too few threads");
    // the system's own z tile width (wide for short z lines), within the
    // launch's threads
    int tz = std::min(ln.tk_z, floor_pow2(std::max(1, threads / (3 * pz.tline))));
    while (tz > 1 && lines_lds<MM_SKEW_Z>(3 * tz, pz.L, cs) > (size_t)mm_max_lds_bytes()) tz /= 2;
    MM_REQUIRE((size_t)tz * (pz.L / 2 + 1) <= (size_t)ZM_ITEMS * threads, "z pass items per thread");
    const unsigned ntz = (unsigned)((g.Hx + tz - 1) / tz), nb = ntz * (unsigned)g.Py;
    const size_t plane = (size_t)g.Hp * g.Hy2 * g.Hz2;
    const size_t zsb = (size_t)g.Py * g.Hp * cs;
    d.S2 = S2;
    d.K = kern;
    d.plane = plane;
    d.stop = stop;
    d.Hx = g.Hx;
    d.Hp = g.Hp;
    d.Hy2 = g.Hy2;
    d.Py = g.Py;
    d.nz = g.nz;
    d.tk = tz;
    d.ntx = (int)ntz;
    d.tbase = 0;
    d.mtx = mdiv(ntz, nb);
    d.zsb = (unsigned)zsb;
    d.pb = (unsigned)(plane * sizeof(T));
    d.p = pz.template dev<T>();
    o32 = zsb < (1u << 24) && 3 * (size_t)g.nz * zsb < (1ull << 32) && kern_elems * sizeof(T) < (1ull << 32);
    lds = lines_lds<MM_SKEW_Z>(3 * tz, pz.L, cs);
    return (int)nb;
}

template <typename T> int ConvImpl<T>::batch_2d(B2Desc<T> &d, int threads, size_t &lds, const int *stop) const
{
    const size_t cs = sizeof(C2<T>);
    MM_REQUIRE(g.is2d && threads >= 3 * py.tline, "batch 2-D pass: 3-D system or too few threads");
    int tk = std::min(16, floor_pow2(std::max(1, threads / (3 * py.tline))));
    while (tk > 1 && lines_lds<MM_SKEW_Y>(3 * tk, py.L, cs) > (size_t)mm_max_lds_bytes()) tk /= 2;
    d.S1 = S1;
    d.K = kern;
    d.plane = (size_t)g.Hp * g.Hy2 * g.Hz2;
    d.stop = stop;
    d.Hx = g.Hx;
    d.Hp = g.Hp;
    d.Hy2 = g.Hy2;
    d.ny = g.ny;
    d.tk = tk;
    d.tbase = 0;
    d.p = py.template dev<T>();
    lds = lines_lds<MM_SKEW_Y>(3 * tk, py.L, cs);
    return (g.Hx + tk - 1) / tk;
}

// The batched kernels: the global workgroup index in XCD order picks the
// system (tsys) and that system's workgroup; descriptor fields are read
// through global-address-space pointer types (gfield) so that the accesses
// through them are global, not flat, operations.
template <typename T, int LC> __global__ void kb_xfwd(const BxDesc<T> *__restrict__ D, const int *__restrict__ tsys)
{
    const int gi = block_tile(1);
    const BxDesc<T> &d = D[tsys[gi]];
    if (gfield(d.stop)[0]) return;
    const T *in = gfield(d.sel)[0] ? gfield(d.y1) : gfield(d.y0);
    xfwd_body<T, T, LC>(in, d.in_cstride, gfield(d.S1), d.out_cstride, d.Hx, d.Hp, d.ny, d.nz, d.nrows, d.nx, d.p,
                       d.lpw, gi - d.tbase);
}

template <typename T, bool INV, int LC, bool O32>
__global__ void kb_y(const ByDesc<T> *__restrict__ D, const int *__restrict__ tsys)
{
    const int gi = block_tile(1);
    const ByDesc<T> &d = D[tsys[gi]];
    if (gfield(d.stop)[0]) return;
    if (INV)
        yinv_body<T, LC, O32>(gfield(d.S2), gfield(d.S1), d.Hx, d.Hp, d.ny, d.nz, d.p, d.tk, gi - d.tbase, d.ntx,
                             d.mtx, d.mzl);
    else
        yfwd_body<T, LC, O32>(gfield(d.S1), gfield(d.S2), d.Hx, d.Hp, d.ny, d.nz, d.p, d.tk, gi - d.tbase, d.ntx,
                             d.mtx, d.mzl);
}

template <typename T, int LC, bool O32> __global__ void kb_zmi(const BzDesc<T> *__restrict__ D, const int *__restrict__ tsys)
{
    const int gi = block_tile(1);
    const BzDesc<T> &d = D[tsys[gi]];
    if (gfield(d.stop)[0]) return;
    zmi_body<T, LC, O32>(gfield(d.S2), gfield(d.K), d.plane, d.Hx, d.Hp, d.Hy2, d.Py, d.nz, d.p, d.tk, 1, gi - d.tbase,
                        d.ntx, d.mtx, d.zsb, d.pb);
}

template <typename T, int LC> __global__ void kb_ymi2d(const B2Desc<T> *__restrict__ D, const int *__restrict__ tsys)
{
    const int gi = block_tile(1);
    const B2Desc<T> &d = D[tsys[gi]];
    if (gfield(d.stop)[0]) return;
    ymi2d_body<T, LC>(gfield(d.S1), gfield(d.K), d.plane, d.Hx, d.Hp, d.Hy2, d.ny, d.p, d.tk, gi - d.tbase);
}

// f(compiled plans, 32-bit offsets) of the launch
template <int ANY, typename F> static void batch_kind(const BatchPass &bp, F &&f)
{
    if (bp.o32) {
        if (bp.compiled) f(std::integral_constant<int, ANY>(), std::true_type());
        else f(std::integral_constant<int, 0>(), std::true_type());
    } else {
        if (bp.compiled) f(std::integral_constant<int, ANY>(), std::false_type());
        else f(std::integral_constant<int, 0>(), std::false_type());
    }
}
template <typename T> void mm_batch_xfwd(const BatchPass &bp, hipStream_t s)
{
    batch_kind<MM_LC_ANY>(bp, [&](auto lc, auto) {
        hipLaunchKernelGGL((kb_xfwd<T, decltype(lc)::value>), dim3(bp.ntiles), dim3(bp.threads), bp.lds, s,
                           (const BxDesc<T> *)bp.desc, (const int *)bp.tsys);
    });
    MM_HIP(hipGetLastError());
}
template <typename T, bool INV> static void batch_y_pass(const BatchPass &bp, hipStream_t s)
{
    batch_kind<MM_LC_ANY>(bp, [&](auto lc, auto o32) {
        hipLaunchKernelGGL((kb_y<T, INV, decltype(lc)::value, decltype(o32)::value>), dim3(bp.ntiles),
                           dim3(bp.threads), bp.lds, s, (const ByDesc<T> *)bp.desc, (const int *)bp.tsys);
    });
    MM_HIP(hipGetLastError());
}
template <typename T> void mm_batch_yfwd(const BatchPass &bp, hipStream_t s) { batch_y_pass<T, false>(bp, s); }
template <typename T> void mm_batch_yinv(const BatchPass &bp, hipStream_t s) { batch_y_pass<T, true>(bp, s); }
template <typename T> void mm_batch_zmi(const BatchPass &bp, hipStream_t s)
{
    batch_kind<MM_LC_Z>(bp, [&](auto lc, auto o32) {
        hipLaunchKernelGGL((kb_zmi<T, decltype(lc)::value, decltype(o32)::value>), dim3(bp.ntiles), dim3(bp.threads),
                           bp.lds, s, (const BzDesc<T> *)bp.desc, (const int *)bp.tsys);
    });
    MM_HIP(hipGetLastError());
}
template <typename T> void mm_batch_ymi2d(const BatchPass &bp, hipStream_t s)
{
    batch_kind<MM_LC_ANY>(bp, [&](auto lc, auto) {
        hipLaunchKernelGGL((kb_ymi2d<T, decltype(lc)::value>), dim3(bp.ntiles), dim3(bp.threads), bp.lds, s,
                           (const B2Desc<T> *)bp.desc, (const int *)bp.tsys);
    });
    MM_HIP(hipGetLastError());
}
template struct ConvImpl<MM_CONV_T>;
template void mm_batch_xfwd<MM_CONV_T>(const BatchPass &, hipStream_t);
template void mm_batch_yfwd<MM_CONV_T>(const BatchPass &, hipStream_t);
template void mm_batch_yinv<MM_CONV_T>(const BatchPass &, hipStream_t);
template void mm_batch_zmi<MM_CONV_T>(const BatchPass &, hipStream_t);
template void mm_batch_ymi2d<MM_CONV_T>(const BatchPass &, hipStream_t);

// y passes of narrow plans.  Behind everything else: between the other kernels
// of this file they moved those, whose times hang on where their code lies
// (150x90x14 FP32 y inverse 7.3 -> 7.8 us with the same code).
template <typename T, bool INV> static void narrow_y(const ConvImpl<T> &c, hipStream_t s)
{
    const ConvGeom &g = c.g;
    const int tk = c.tk_yn;
    const size_t sh = lines_lds<MM_SKEW_Y>(tk, c.pyn.L, sizeof(C2<T>));
    const unsigned ntx = (unsigned)((g.Hx + tk - 1) / tk), nb = ntx * g.nz * 3;
    const dim3 grid(ntx, g.nz, 3), block(tk * c.pyn.tline);
    const FftPlanDev p = c.pyn.template dev<T>();
    const unsigned mx = mdiv(ntx, nb, c.wide), mz = mdiv((unsigned)g.nz, nb, c.wide);
    auto go = [&](auto o32) {
        constexpr bool O32 = decltype(o32)::value;
        if constexpr (INV)
            hipLaunchKernelGGL((k_yinv<T, MM_LC_NARROW, O32>), grid, block, sh, s, c.S2, c.S1, g.Hx, g.Hp, g.ny, g.nz,
                               p, tk, c.xcd_remap, mx, mz);
        else
            hipLaunchKernelGGL((k_yfwd<T, MM_LC_NARROW, O32>), grid, block, sh, s, c.S1, c.S2, g.Hx, g.Hp, g.ny, g.nz,
                               p, tk, c.xcd_remap, mx, mz);
    };
    if (c.y_offsets32()) go(std::true_type());
    else go(std::false_type());
    MM_HIP(hipGetLastError());
}
template <typename T> void mm_narrow_yfwd(const ConvImpl<T> &c, hipStream_t s) { narrow_y<T, false>(c, s); }
template <typename T> void mm_narrow_yinv(const ConvImpl<T> &c, hipStream_t s) { narrow_y<T, true>(c, s); }
template <typename T> void mm_narrow_ymi2d(const ConvImpl<T> &c, hipStream_t s)
{
    const ConvGeom &g = c.g;
    const int tk = c.tk_yn;
    hipLaunchKernelGGL((k_ymi2d<T, MM_LC_NARROW>), dim3((g.Hx + tk - 1) / tk), dim3(3 * tk * c.pyn.tline),
                       lines_lds<MM_SKEW_Y>(3 * tk, c.pyn.L, sizeof(C2<T>)), s, c.S1, c.kern,
                       (size_t)g.Hp * g.Hy2 * g.Hz2, g.Hx, g.Hp, g.Hy2, g.ny, c.pyn.template dev<T>(), tk);
    MM_HIP(hipGetLastError());
}
template void mm_narrow_yfwd<MM_CONV_T>(const ConvImpl<MM_CONV_T> &, hipStream_t);
template void mm_narrow_yinv<MM_CONV_T>(const ConvImpl<MM_CONV_T> &, hipStream_t);
template void mm_narrow_ymi2d<MM_CONV_T>(const ConvImpl<MM_CONV_T> &, hipStream_t);
