// mm_conv.h -- FFT demag convolution objects (host side of mm_conv.hip).
#ifndef MM_CONV_H
#define MM_CONV_H

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>
#include <vector>

#include "mm_fft_device.h"
#include "mm_internal.h"

#define MM_HIP(call)                                                                      \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            throw mm_error(MM_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// host plan of one FFT length: radix list, threads per line, twiddle tables
struct FftPlanHost {
    int L = 1;
    int tline = 1;
    std::vector<int> rad;
    void *tw32 = nullptr;  // float2[L], exp(-2 pi i m / L)
    void *tw64 = nullptr;  // double2[L]
    void *twp32 = nullptr; // float2[ntw], per-pass layout (FftPlanDev)
    void *twp64 = nullptr; // double2[ntw]
    int ntw = 0;
    int id = 0;             // compiled plan (mm_plan_id), 0: none
    void build(int len);
    // the plan as kernels that run the passes in a loop take it (the same
    // passes and twiddles, L/8 threads per line)
    static int tline_loop(int len) { return len > MM_FFT_EPT ? (len + MM_FFT_EPT - 1) / MM_FFT_EPT : 1; }
    void no_compiled()
    {
        id = 0;
        tline = tline_loop(L);
    }
    // the narrow plan of a length that has one (id 0 if not), on the same tables
    FftPlanHost narrow() const
    {
        FftPlanHost n = *this;
        n.id = mm_plan_id(L, true);
        if (n.id > 0) n.tline = mm_plan_tline(L, true);
        return n;
    }
    template <typename T> FftPlanDev dev_loop() const
    {
        FftPlanDev d = dev<T>();
        d.tline = tline_loop(L);
        d.id = 0;
        return d;
    }
    void release();
    template <typename T> FftPlanDev dev() const
    {
        FftPlanDev d;
        d.L = L;
        d.tline = tline;
        d.npass = (int)rad.size();
        d.radices = 0u;
        for (int i = 0; i < d.npass; ++i) d.radices |= (unsigned)rad[i] << (4 * i);
        d.tw = sizeof(T) == 4 ? twp32 : twp64;
        d.ntw = ntw;
        d.pow2 = (L & (L - 1)) == 0 ? 1 : 0;
        d.id = id;
        return d;
    }
    // the plain table exp(-2 pi i m / L), m < L
    template <typename T> const void *plain() const { return sizeof(T) == 4 ? tw32 : tw64; }
};

// Calls f(std::integral_constant<int, LC>()) with the kernel instantiation for
// lines of length L: LC = L for powers of two 2..2048, MM_LC_ANY (MM_LC_Z for
// the z pass) for the other compiled lengths, else and with `generic` 0, the
// runtime plan.
template <int ANY = MM_LC_ANY, typename F> void mm_with_len(int L, bool generic, F &&f)
{
    if (!generic) {
        switch (L) {
#define MM_FFT_X(N) case N: f(std::integral_constant<int, N>()); return;
        MM_FFT_POW2(MM_FFT_X)
#undef MM_FFT_X
        default: break;
        }
        if (mm_plan_id(L) > 0 && (ANY != MM_LC_Z || mm_plan_z(L))) {
            f(std::integral_constant<int, ANY>());
            return;
        }
    }
    f(std::integral_constant<int, 0>());
}

bool mm_is_smooth(int n);                  // n has no prime factor > 5
int mm_fft_size_for(int n, int given);     // radix-friendly padded size for n cells

// Geometry of a convolution: physical (nx,ny,nz), padded FFT sizes (Px,Py,Pz).
struct ConvGeom {
    int nx, ny, nz, Px, Py, Pz, Hx, Hy2, Hz2;
    int Hp;  // row pitch of the spectra and the kernel planes (>= Hx)
    bool is2d;
};

// Tile widths (lines per workgroup) for the strided passes.
struct ConvLaunch {
    int lpw_x;  // x lines per WG (plain x passes)
    int tk_y;   // kx columns per WG, y passes
    int tk_z;   // kx columns per WG, z pass (3 components each)
};

// End of the x forward passes: the lpw lines of workgroup blk (two real rows
// per complex line, transformed in LDS) as half spectra
// X0[k] = (Z[k] + conj Z[L-k]) / 2, X1[k] = (Z[k] - conj Z[L-k]) / 2i.
// row(h): where row h of the nrows rows goes.  Short spectra take several
// lines at a time; the thread of k = 0 also writes k = L/2 of an even line.
template <typename T, typename ROW>
__device__ __forceinline__ void xfwd_store(const C2<T> *sm, int LP, int L, int lpw, int blk, int nrows, int Hx,
                                           ROW row)
{
    constexpr int SK = MM_SKEW_X;
    const int nt = (int)blockDim.x, t = (int)threadIdx.x;
    const int kh = (L & 1) ? Hx : Hx - 1;
    const int ng = max(1, nt / kh), g = ng == 1 ? 0 : t / kh;
    for (int l2 = g < ng ? g : lpw; l2 < lpw; l2 += ng) {
        const int h0 = 2 * (blk * lpw + l2);
        if (h0 >= nrows) break;
        const C2<T> *ln = sm + (size_t)l2 * LP;
        C2<T> *d0 = row(h0), *d1 = h0 + 1 < nrows ? row(h0 + 1) : nullptr;
        for (int k = t - g * kh; k < kh; k += ng == 1 ? nt : kh) {
            const C2<T> zk = ln[sk<SK>(k)], zm = ln[sk<SK>(k == 0 ? 0 : L - k)];
            d0[k] = cmk<T>((zk.x + zm.x) * (T)0.5, (zk.y - zm.y) * (T)0.5);
            if (d1) d1[k] = cmk<T>((zk.y + zm.y) * (T)0.5, (zm.x - zk.x) * (T)0.5);
            if (k == 0 && kh < Hx) {
                const C2<T> zh = ln[sk<SK>(kh)];
                d0[kh] = cmk<T>(zh.x, (T)0);
                if (d1) d1[kh] = cmk<T>(zh.y, (T)0);
            }
        }
    }
}

// multiplier for udiv: n / d for every n < nmax (0: not exact, divide;
// wide: always divide)
static inline unsigned mdiv(unsigned d, size_t nmax, bool wide = false)
{
    MM_REQUIRE(d >= 1, "zero divisor");
    if (d == 1 || (unsigned long long)nmax * d >= (1ull << 32) || wide) return 0u;
    return (unsigned)((1ull << 32) / d + 1);
}

// n / d for the tile indices of a launch without an integer division (the
// GPU has none; the compiler emits some twenty instructions for one):
// m = floor(2^32 / d) + 1 gives floor(n / d) = umulhi(n, m) exactly when
// n * d < 2^32.  mdiv returns 0 where that does not hold, and the division
// is then done the long way.
__device__ __forceinline__ unsigned udiv(unsigned n, unsigned d, unsigned m)
{
    return d == 1 ? n : (m ? __umulhi(n, m) : n / d);
}

// Fourier kernel times spectrum of one point; k: xx, xy, xz, yy, yz, zz.  The
// roundings are spelled out, as those of the DFTs.
template <typename T>
__device__ __forceinline__ void mult3(C2<T> &mx, C2<T> &my, C2<T> &mz, const T k[6])
{
    auto row = [](T a, T x, T b, T y, T c, T z) { return fma(c, z, fma(a, x, b * y)); };
    const C2<T> x = mx, y = my, z = mz;
    mx = cmk<T>(row(k[0], x.x, k[1], y.x, k[2], z.x), row(k[0], x.y, k[1], y.y, k[2], z.y));
    my = cmk<T>(row(k[1], x.x, k[3], y.x, k[4], z.x), row(k[1], x.y, k[3], y.y, k[4], z.y));
    mz = cmk<T>(row(k[2], x.x, k[4], y.x, k[5], z.x), row(k[2], x.y, k[4], y.y, k[5], z.y));
}

// ... at the point mirrored in z of the one k belongs to: xz and yz change sign
template <typename T>
__device__ __forceinline__ void mult3_mirror(C2<T> &mx, C2<T> &my, C2<T> &mz, const T k[6])
{
    auto row = [](T a, T x, T b, T y, T c, T z) { return fma(-c, z, fma(a, x, b * y)); };
    auto last = [](T a, T x, T b, T y, T c, T z) { return fma(c, z, fma(-b, y, -(a * x))); };
    const C2<T> x = mx, y = my, z = mz;
    mx = cmk<T>(row(k[0], x.x, k[1], y.x, k[2], z.x), row(k[0], x.y, k[1], y.y, k[2], z.y));
    my = cmk<T>(row(k[1], x.x, k[3], y.x, k[4], z.x), row(k[1], x.y, k[3], y.y, k[4], z.y));
    mz = cmk<T>(last(k[2], x.x, k[4], y.x, k[5], z.x), last(k[2], x.y, k[4], y.y, k[5], z.y));
}

static inline int floor_pow2(int v) { return v < 1 ? 1 : 1 << (31 - __builtin_clz((unsigned)v)); }

static inline int env_int(const char *name, int dflt)
{
    const char *v = std::getenv(name);
    return (v && *v) ? std::atoi(v) : dflt;
}

// LDS bytes of `nlines` transform lines of length L plus the plan's twiddle table
template <int SK> inline size_t lines_lds(int nlines, int L, size_t csize)
{
    return ((size_t)nlines * lds_len<SK>(L) + (size_t)L) * csize;
}

// Launch shapes: x passes take several rows per workgroup; the strided y and
// z passes take tiles of adjacent kx columns (row segments of tile*16 or
// tile*8 bytes).  Tiles are sized for several resident workgroups per CU so
// that global loads of one overlap the FFT of another.  MM_LPW_X, MM_TK_Y and
// MM_TK_Z override the choice (launch-shape sweeps).
ConvLaunch mm_choose_launch(const ConvGeom &g, const FftPlanHost &px, const FftPlanHost &py, const FftPlanHost &pz,
                            size_t csize);

// Optional per-launch event log used by the measurement entry point: after
// every kernel the owner records an event tagged with the kernel class.
enum {
    KC_XFWD = 0, KC_YFWD = 1, KC_ZMI = 2, KC_YINV = 3, KC_YMI2D = 4, KC_STAGE = 5, KC_CTRL = 6, KC_NCLASS = 7
};
struct KernelLog {
    std::vector<hipEvent_t> ev;
    std::vector<int> cls;
    std::vector<double> bytes;
    size_t used = 0;
    void reserve(size_t n)
    {
        while (ev.size() < n) {
            hipEvent_t e;
            MM_HIP(hipEventCreate(&e));
            ev.push_back(e);
        }
        cls.resize(n);
        bytes.resize(n);
    }
    void mark(hipStream_t s, int c, double b)
    {
        MM_REQUIRE(used < ev.size(), "kernel log full");
        MM_HIP(hipEventRecord(ev[used], s));
        cls[used] = c;
        bytes[used] = b;
        ++used;
    }
    ~KernelLog()
    {
        for (auto e : ev) (void)hipEventDestroy(e);
    }
};

// ---- batched passes: one launch runs one pass for many systems ----------
// Each system of a batch has a descriptor per pass; the launch's global
// workgroup g (in XCD order, xcd_tile) belongs to system tsys[g] and is that
// system's workgroup g - tbase.  A system whose stop flag is set skips the
// pass.  Lengths differ between systems, so each workgroup selects its
// system's compiled plan (or all run the runtime plans, if one has no such
// length).
template <typename T> struct BxDesc {  // x forward of the current state y[*sel]
    const T *y0, *y1;
    const int *sel, *stop;
    C2<T> *S1;
    size_t in_cstride, out_cstride;
    int Hx, Hp, ny, nz, nrows, nx, lpw, tbase;
    FftPlanDev p;
};
template <typename T> struct ByDesc {  // y forward S1 -> S2 and inverse S2 -> S1
    C2<T> *S1, *S2;
    const int *stop;
    int Hx, Hp, ny, nz, tk, ntx, tbase;
    unsigned mtx, mzl;
    FftPlanDev p;
};
template <typename T> struct BzDesc {  // z forward, multiply, z inverse on S2
    C2<T> *S2;
    const T *K;
    size_t plane;
    const int *stop;
    int Hx, Hp, Hy2, Py, nz, tk, ntx, tbase;
    unsigned mtx, zsb, pb;
    FftPlanDev p;
};
template <typename T> struct B2Desc {  // 2-D: y forward, multiply, y inverse on S1
    C2<T> *S1;
    const T *K;
    size_t plane;
    const int *stop;
    int Hx, Hp, Hy2, ny, tk, tbase;
    FftPlanDev p;
};

// One pass of a batch: descriptors and tile table in device memory, the
// launch's workgroups, threads per workgroup and dynamic LDS.  o32: every
// system's spectra fit the 32-bit offset forms.
struct BatchPass {
    void *desc = nullptr;
    int *tsys = nullptr;
    int ntiles = 0, threads = 0;
    size_t lds = 0;
    bool o32 = true;
    bool compiled = true;  // every system's lines have a compiled length
};

template <typename T>
struct ConvImpl {
    KernelLog *klog = nullptr;
    ConvGeom g;
    ConvLaunch ln;
    FftPlanHost px, py, pz;
    FftPlanHost pyh;        // length Py/2, for the pruned y transforms
    bool fft_generic = false;  // runtime FFT plans only (no compile-time lengths)
    int xcd_remap = 1;         // XCD-contiguous tile order (xcd_tile)
    bool prune_y = false;
    bool wide = false;         // general index arithmetic only (MM_WIDE_INDEX)
    int tk_yp = 1;          // kx columns per WG of the pruned y transforms
    // The y passes run py's narrow plan.  Single launches only: a batch's
    // workgroups select their lengths in one kernel.
    bool y_narrow = false;
    FftPlanHost pyn;
    int tk_yn = 1;
    int tk_y() const { return y_narrow ? tk_yn : ln.tk_y; }
    // the y passes address by 32-bit offsets (S2, 3 nz Py rows, is the larger
    // of their two arrays)
    bool y_offsets32() const
    {
        const size_t cs = sizeof(C2<T>);
        return (size_t)g.Hp * cs < (1u << 24) && (size_t)3 * g.nz * g.Py * g.Hp * cs < (1ull << 32) && !wide;
    }
    T *kern = nullptr;      // 6 real planes [e][kz<Hz2][ky<Hy2][kx<Hx], pitch Hp, scaled 1/(PxPyPz)
    C2<T> *S1 = nullptr;    // [c][z<nz][y<ny][kx<Hx], pitch Hp
    C2<T> *S2 = nullptr;    // [c][z<nz][ky<Py][kx<Hx], pitch Hp   (3-D only)
    size_t kern_elems = 0;

    void init(const double *N_host, int nx, int ny, int nz, int ex, int ey, int ez);
    void release();
    // spectral part: pad+x forward .. x inverse up to S1 holding the result
    // spectrum rows; then x inverse into H.
    void forward_x(const T *M, hipStream_t s, const T *M_alt = nullptr, const int *sel = nullptr);
    void spectral(hipStream_t s);  // y fwd, z fwd*mult*inv / 2-D fused, y inv
    void inverse_x(T *H, hipStream_t s);
    void execute(const T *M, T *H, hipStream_t s)
    {
        forward_x(M, s);
        spectral(s);
        inverse_x(H, s);
    }
    // this system's part of a batched pass launched with `threads` threads
    // per workgroup: its descriptor (tbase left to the caller), workgroup
    // count, the dynamic LDS it needs and whether it fits the 32-bit offset
    // forms.  Tile widths follow the batch's thread count.
    int batch_x(BxDesc<T> &d, int threads, size_t &lds, const T *y0, const T *y1, const int *sel,
                const int *stop) const;
    int batch_y(ByDesc<T> &d, int threads, size_t &lds, bool &o32, const int *stop) const;
    int batch_z(BzDesc<T> &d, int threads, size_t &lds, bool &o32, const int *stop) const;
    int batch_2d(B2Desc<T> &d, int threads, size_t &lds, const int *stop) const;
    // The z pass takes its register form (mm_conv_zreg.hip).  Both forms on
    // MI355X, field evaluation, LDS form -> register form: 200x200x5 (12
    // points) FP32 49.6 -> 43.8 us, FP64 74.3 -> 60.0; 256x256x5 FP64 86.1 ->
    // 66.0; 256x256x4 (8 points) FP32 41.0 -> 40.4, FP64 54.1 -> 53.4;
    // 256x256x8 (16 points) FP32 58.9 -> 56.8, 99x85x8 28.3 -> 29.0: with
    // less than a wave per SIMD the longer chain of one thread shows, and at
    // 16 points it costs more than the barriers it saves.  FP64 lines of 16
    // points leave one wave per SIMD (200x200x8: 83.9 -> 87.7), 20 and more
    // likewise in FP32 (99x85x9: 29.7 -> 31.5, 256x256x16: 93.7 -> 105).
    // Up to 12 points the mesh may be as small as it likes: 24x24x5 FP64 23.9
    // -> 24.7, 40x30x5 25.2 -> 25.9, 64x64x5 26.0 -> 25.9, 100x100x5 33.8 ->
    // 31.2 (launch-bound below), FP32 level there.
    bool zreg() const
    {
        const int L = g.Pz;
        const size_t cells = (size_t)g.Py * g.Hp;
        const bool len = L == 4 || L == 6 || L == 8 || L == 10 || L == 12 ||
                         (L == 16 && sizeof(T) == 4 && cells >= 65536);
        return len && !g.is2d && !fft_generic && g.nz <= (L + 1) / 2 && cells * sizeof(C2<T>) < (1ull << 32);
    }
    // ... and of a batched launch, whose kernel holds the lines of one pass (4
    // and 8 points, 2 to 4 layers).  Both forms give the same bits at every
    // length, so that a member is a single stepper bit for bit.
    bool zreg_batch() const { return zreg() && (g.Pz == 4 || g.Pz == 8); }
    // threads per workgroup this system's passes need at least
    int batch_threads_x() const { return px.tline; }
    int batch_threads_y() const { return (g.is2d ? 3 : 1) * py.tline; }
    int batch_threads_z() const { return 3 * pz.tline; }
};

// y passes of narrow plans (ConvImpl::y_narrow): 3-D forward and inverse, 2-D
template <typename T> void mm_narrow_yfwd(const ConvImpl<T> &c, hipStream_t s);
template <typename T> void mm_narrow_yinv(const ConvImpl<T> &c, hipStream_t s);
template <typename T> void mm_narrow_ymi2d(const ConvImpl<T> &c, hipStream_t s);

// z pass in registers (ConvImpl::zreg)
template <typename T> void mm_zreg_pass(const ConvImpl<T> &c, hipStream_t s);
// a system's descriptor and workgroup count in the batched form (zreg_batch),
// and the launch of all of them
#define MM_ZREG_BATCH_THREADS 256
template <typename T> int mm_zreg_desc(const ConvImpl<T> &c, BzDesc<T> &d, const int *stop);
template <typename T> void mm_batch_zreg(const BatchPass &bp, hipStream_t s);

// batched launches (all systems of bp in one launch on stream s)
template <typename T> void mm_batch_xfwd(const BatchPass &bp, hipStream_t s);
template <typename T> void mm_batch_yfwd(const BatchPass &bp, hipStream_t s);
template <typename T> void mm_batch_yinv(const BatchPass &bp, hipStream_t s);
template <typename T> void mm_batch_zmi(const BatchPass &bp, hipStream_t s);
template <typename T> void mm_batch_ymi2d(const BatchPass &bp, hipStream_t s);

// device-side FFT kernels reused by the fused stepper
template <typename T> size_t conv_lds_xinv(const ConvImpl<T> &c, int lines) { return (size_t)lines * (c.px.L + 1) * sizeof(C2<T>); }

struct mm_conv {
    int precision;
    ConvImpl<float> *c32 = nullptr;
    ConvImpl<double> *c64 = nullptr;
};

void mm_lds_attr_once();
int mm_max_lds_bytes();
int mm_num_cus();  // of the current device

// Launch shapes of a mesh (0: not set, the built-in choice applies): x lines
// per workgroup, kx columns per workgroup of the y and z passes, rows per
// stage workgroup and stage threads.  Tuned shapes live in a process-wide
// table keyed by mesh size, precision and device (the counterpart of the
// reference's FFTW wisdom, Magneto.cpp:151-190).  mm_shape_for gives the
// shape in force for a new convolution or stepper: the tuner's candidate
// while it measures one (this thread), else the table's entry.  The MM_LPW_X,
// MM_TK_Y, MM_TK_Z, MM_RPW and MM_STAGE_THREADS variables override both.
struct MmShape {
    int lpw_x, tk_y, tk_z, rpw, stage_threads;
};
MmShape mm_shape_for(int nx, int ny, int nz, size_t real_bytes);
void mm_shape_set_candidate(const MmShape *s);
void mm_wisdom_put(int nx, int ny, int nz, size_t real_bytes, const MmShape &s);

#endif
