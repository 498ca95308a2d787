// mm_conv_zreg.hip -- z pass of short lines in registers, for one precision
// (MM_CONV_T; the Makefile builds one object per precision).
//
// The LDS form (zmi_body, mm_conv_passes.hip) spreads a line over L/8 threads
// and takes six barriers; at 4 to 12 points it waits for those and for few
// loads in flight, not for memory.  Here nothing is exchanged between threads:
// every read of a thread is issued at its start, the rest is arithmetic, so
// the pass is bound by the spectra's traffic.  200x200x5 FP64 (12 points): 27
// -> 14 us, 58 MB.  Registers set the limit: 3 L complex values and the
// kernel entries take 103 / 158 / 204 VGPRs at 8 / 12 / 16 points in FP32 and
// 204 / 312 at 8 / 12 in FP64 (4, 3, 2 and 2, 1 waves per SIMD).
#include "mm_conv.h"
#include "mm_cell.h"

// The transform of a line in one thread's registers: the passes, twiddles and
// roundings of fft_line (SPLIT as its last inverse pass, which stores), no
// LDS, no barriers.  tw is the plan's per-pass table in global memory; its
// indices are constants and its base is uniform, so the twiddles come in by
// scalar loads.
template <typename T, bool INV, int LC, int PS = 0, int NS = 1>
__device__ __forceinline__ void fft_reg(C2<T> (&v)[LC], const C2<T> *__restrict__ tw)
{
    using F = FftLen<LC>;
    if constexpr (PS < F::npass) {
        constexpr int R = F::radix(PS), nb = LC / R;
        constexpr bool SPLIT = INV && PS == F::npass - 1;
        C2<T> o[LC];
#pragma unroll
        for (int b = 0; b < nb; ++b) {
            const int k = b % NS;
            C2<T> u[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                u[r] = v[b + r * nb];
                if (r > 0 && k > 0) u[r] = cmul_tw<T, INV>(u[r], tw[F::toff(PS) + (r - 1) * NS + k]);
            }
            dftR<R, T, INV, SPLIT>(u);
#pragma unroll
            for (int r = 0; r < R; ++r) o[(b / NS) * NS * R + k + r * NS] = u[r];
        }
#pragma unroll
        for (int j = 0; j < LC; ++j) v[j] = o[j];
        fft_reg<T, INV, LC, PS + 1, NS * R>(v, tw);
    }
}

// One thread holds the z lines of the three components of one (kx, ky).
// Threads run over the rows' whole pitch, so a
// wave's accesses are contiguous; (c, z) planes and kernel planes have uniform
// bases and the thread's offset in a plane is one 32-bit value.  Needs
// nz <= (LC + 1) / 2 (lines at least half zeros), so the upper half of a line
// is never read.  Loads beyond nz take the last plane, so that no branch
// parts them, and are replaced by zeros.
template <typename T, int LC>
__device__ __forceinline__ void zmir_body(C2<T> *__restrict__ S2, const T *__restrict__ K, size_t plane, int Hx,
                                          int Hp, int Hy2, int Py, int nz, const C2<T> *__restrict__ tw, int remap,
                                          unsigned cell, unsigned mhp)
{
    constexpr int NIN = (LC + 1) / 2;
    const int m = (int)udiv(cell, (unsigned)Hp, mhp), kx = (int)cell - m * Hp;
    if (m >= Py || kx >= Hx) return;
    const int hm = (m + 1) >> 1;
    // rows in the order of zmi_body: ky and Py - ky read the same kernel row
    const int ky = !remap || m == 0 ? m : ((m & 1) ? hm : Py - hm);
    const size_t zstride = (size_t)Py * Hp;
    const unsigned so = ((unsigned)ky * Hp + kx) * (unsigned)sizeof(C2<T>);
    auto at = [&](int c, int z) -> C2<T> & {
        return *(C2<T> *)((char *)(S2 + ((size_t)c * nz + z) * zstride) + so);
    };
    C2<T> v[3][LC];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int z = 0; z < LC; ++z)
            v[c][z] = z < NIN ? at(c, min(z, nz - 1)) : cmk<T>((T)0, (T)0);
    }
    const bool fy = ky > Py / 2;
    const int kyf = fy ? Py - ky : ky;
    const T sy = fy ? (T)-1 : (T)1;
    const unsigned ko = ((unsigned)kyf * Hp + kx) * (unsigned)sizeof(T);
    T kk[LC / 2 + 1][6];
#pragma unroll
    for (int kz = 0; kz <= LC / 2; ++kz) {
#pragma unroll
        for (int q = 0; q < 6; ++q)
            kk[kz][q] = *(const T *)((const char *)(K + q * plane + (size_t)kz * Hy2 * Hp) + ko);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int z = 1; z < NIN; ++z)
            if (z >= nz) v[c][z] = cmk<T>((T)0, (T)0);
        fft_reg<T, false, LC>(v[c], tw);
    }
#pragma unroll
    for (int kz = 0; kz <= LC / 2; ++kz) {
        const T k[6] = {kk[kz][0], sy * kk[kz][1], kk[kz][2], kk[kz][3], sy * kk[kz][4], kk[kz][5]};
        mult3<T>(v[0][kz], v[1][kz], v[2][kz], k);
        if (kz > 0 && LC - kz != kz) mult3_mirror<T>(v[0][LC - kz], v[1][LC - kz], v[2][LC - kz], k);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        fft_reg<T, true, LC>(v[c], tw);
#pragma unroll
        for (int z = 0; z < NIN; ++z)
            if (z < nz) at(c, z) = v[c][z];
    }
}

template <typename T, int LC>
__global__ __launch_bounds__(256) void k_zmir(C2<T> *__restrict__ S2, const T *__restrict__ K, size_t plane, int Hx,
                                              int Hp, int Hy2, int Py, int nz, const C2<T> *__restrict__ tw,
                                              int remap, unsigned mhp)
{
    const unsigned cell = (unsigned)block_tile(remap) * blockDim.x + threadIdx.x;
    zmir_body<T, LC>(S2, K, plane, Hx, Hp, Hy2, Py, nz, tw, remap, cell, mhp);
}

template <typename T> void mm_zreg_pass(const ConvImpl<T> &c, hipStream_t s)
{
    const ConvGeom &g = c.g;
    MM_REQUIRE(c.zreg(), "z pass has no register form of this line");
    const size_t plane = (size_t)g.Hp * g.Hy2 * g.Hz2, cells = (size_t)g.Py * g.Hp;
    // Workgroups of one wave spread evenly over the CUs; of four once there are
    // enough of them, up to 8 points: longer FP64 lines leave one wave per SIMD,
    // and a workgroup of four waits for a whole CU.  Field, 64 -> 256 threads:
    // 1024x1024x2 FP32 202.9 -> 200.9 us, 512x512x4 FP64 173.8 -> 174.4;
    // 512x512x5 FP64 207.6 -> 214.7, FP32 102.4 -> 103.1; 40x30x5 FP64 23.2 -> 24.0.
    const unsigned bs = cells < 262144 || g.Pz > 8 ? 64u : 256u, nb = (unsigned)((cells + bs - 1) / bs);
    const unsigned mhp = mdiv((unsigned)g.Hp, (size_t)nb * bs, c.wide);
    const C2<T> *tw = (const C2<T> *)c.pz.template dev<T>().tw;
    switch (g.Pz) {
#define MM_FFT_X(N)                                                                                               \
    case N:                                                                                                       \
        hipLaunchKernelGGL((k_zmir<T, N>), dim3(nb), dim3(bs), 0, s, c.S2, c.kern, plane, g.Hx, g.Hp, g.Hy2, g.Py, \
                           g.nz, tw, c.xcd_remap, mhp);                                                           \
        break;
    MM_FFT_X(4) MM_FFT_X(6) MM_FFT_X(8) MM_FFT_X(10) MM_FFT_X(12) MM_FFT_X(16)
#undef MM_FFT_X
    default: throw mm_error(MM_ERR_RUNTIME, "z pass in registers: length");
    }
    MM_HIP(hipGetLastError());
}
template void mm_zreg_pass<MM_CONV_T>(const ConvImpl<MM_CONV_T> &, hipStream_t);

// Batched form: systems of one-pass lines, which need no twiddles.  A wider
// choice of lengths would give every system the registers of the longest.
template <typename T>
__global__ __launch_bounds__(MM_ZREG_BATCH_THREADS) void kb_zmir(const BzDesc<T> *__restrict__ D,
                                                                 const int *__restrict__ tsys)
{
    const int gi = block_tile(1);
    const BzDesc<T> &d = D[tsys[gi]];
    if (gfield(d.stop)[0]) return;
    const unsigned cell = (unsigned)(gi - d.tbase) * blockDim.x + threadIdx.x;
    if (d.p.L == 4)
        zmir_body<T, 4>(gfield(d.S2), gfield(d.K), d.plane, d.Hx, d.Hp, d.Hy2, d.Py, d.nz, nullptr, 1, cell, d.mtx);
    else if (d.p.L == 8)
        zmir_body<T, 8>(gfield(d.S2), gfield(d.K), d.plane, d.Hx, d.Hp, d.Hy2, d.Py, d.nz, nullptr, 1, cell, d.mtx);
}

template <typename T> int mm_zreg_desc(const ConvImpl<T> &c, BzDesc<T> &d, const int *stop)
{
    const ConvGeom &g = c.g;
    MM_REQUIRE(c.zreg_batch(), "system has no batched register form of the z pass");
    const size_t cells = (size_t)g.Py * g.Hp;
    const int nb = (int)((cells + MM_ZREG_BATCH_THREADS - 1) / MM_ZREG_BATCH_THREADS);
    d = BzDesc<T>();
    d.S2 = c.S2;
    d.K = c.kern;
    d.plane = (size_t)g.Hp * g.Hy2 * g.Hz2;
    d.stop = stop;
    d.Hx = g.Hx;
    d.Hp = g.Hp;
    d.Hy2 = g.Hy2;
    d.Py = g.Py;
    d.nz = g.nz;
    d.mtx = mdiv((unsigned)g.Hp, (size_t)nb * MM_ZREG_BATCH_THREADS, c.wide);
    d.p = c.pz.template dev<T>();
    return nb;
}

template <typename T> void mm_batch_zreg(const BatchPass &bp, hipStream_t s)
{
    hipLaunchKernelGGL((kb_zmir<T>), dim3(bp.ntiles), dim3(bp.threads), 0, s, (const BzDesc<T> *)bp.desc,
                       (const int *)bp.tsys);
    MM_HIP(hipGetLastError());
}
template int mm_zreg_desc<MM_CONV_T>(const ConvImpl<MM_CONV_T> &, BzDesc<MM_CONV_T> &, const int *);
template void mm_batch_zreg<MM_CONV_T>(const BatchPass &, hipStream_t);
