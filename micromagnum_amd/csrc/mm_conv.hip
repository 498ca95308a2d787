// mm_conv.hip -- FFT demag convolution on gfx950, host side: transform plans,
// padded sizes, launch shapes and their table, the C ABI, and the direct sum.
// The passes are in mm_conv_passes.hip.
#include "mm_conv.h"
#include "mm_cell.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>

// ---------------------------------------------------------------------------
// FFT plan
// ---------------------------------------------------------------------------
void FftPlanHost::build(int len)
{
    MM_REQUIRE(len >= 1, "FFT length must be positive");
    L = len;
    const FftRadices f = mm_plan_radices(len);
    if (f.n == 0 && len != 1)
        throw mm_error(MM_ERR_UNSUPPORTED, "FFT length " + std::to_string(len) + " has a prime factor > 5");
    MM_REQUIRE(f.n <= MM_FFT_MAX_PASSES, "FFT length needs too many passes");
    rad.assign(f.r, f.r + f.n);
    id = mm_plan_id(len);
    tline = id > 0 ? mm_plan_tline(len) : tline_loop(len);
    if (tline > 1024) throw mm_error(MM_ERR_UNSUPPORTED, "FFT length " + std::to_string(len) + " above 8192");
    std::vector<float2> t32(L);
    std::vector<double2> t64(L);
    for (int m = 0; m < L; ++m) {
        const long double a = -2.0L * MM_PI_L * (long double)m / (long double)L;
        const long double c = cosl(a), s = sinl(a);
        t64[m].x = (double)c;
        t64[m].y = (double)s;
        t32[m].x = (float)c;
        t32[m].y = (float)s;
    }
    MM_HIP(hipMalloc(&tw32, sizeof(float2) * L));
    MM_HIP(hipMalloc(&tw64, sizeof(double2) * L));
    MM_HIP(hipMemcpy(tw32, t32.data(), sizeof(float2) * L, hipMemcpyHostToDevice));
    MM_HIP(hipMemcpy(tw64, t64.data(), sizeof(double2) * L, hipMemcpyHostToDevice));
    // per-pass layout: pass p (radix R, Ns > 1) holds W_{Ns R}^{r k} at
    // (r-1) Ns + k, copied from the plain table at index r k L / (Ns R)
    std::vector<float2> p32;
    std::vector<double2> p64;
    int Ns = 1;
    for (int R : rad) {
        if (Ns > 1)
            for (int r = 1; r < R; ++r)
                for (int k = 0; k < Ns; ++k) {
                    const int m = r * k * (L / (Ns * R));
                    p32.push_back(t32[m]);
                    p64.push_back(t64[m]);
                }
        Ns *= R;
    }
    ntw = (int)p64.size();
    MM_REQUIRE(ntw < L || L == 1, "per-pass twiddle table larger than the line");
    const size_t nalloc = std::max<size_t>(1, p64.size());
    MM_HIP(hipMalloc(&twp32, sizeof(float2) * nalloc));
    MM_HIP(hipMalloc(&twp64, sizeof(double2) * nalloc));
    if (ntw > 0) {
        MM_HIP(hipMemcpy(twp32, p32.data(), sizeof(float2) * ntw, hipMemcpyHostToDevice));
        MM_HIP(hipMemcpy(twp64, p64.data(), sizeof(double2) * ntw, hipMemcpyHostToDevice));
    }
}

void FftPlanHost::release()
{
    if (tw32) (void)hipFree(tw32);
    if (tw64) (void)hipFree(tw64);
    if (twp32) (void)hipFree(twp32);
    if (twp64) (void)hipFree(twp64);
    tw32 = tw64 = twp32 = twp64 = nullptr;
}

bool mm_is_smooth(int n)
{
    if (n < 1) return false;
    for (int f : {2, 3, 5})
        while (n % f == 0) n /= f;
    return n == 1;
}

// Any padded size P >= 2n-1 gives the same linear convolution for open
// boundaries (the tensor is zero between the +/- offsets), so the given size
// is kept if it is radix-friendly and even, else the next such size is used.
// A periodic axis (given == n) is a circular convolution of period n and
// keeps its size, which must then be radix-friendly itself.
int mm_fft_size_for(int n, int given)
{
    if (n == 1) return 1;
    if (given < 2ll * n - 1) {
        MM_REQUIRE(given == n, "tensor size along an axis must be the mesh size (periodic) or >= 2n-1 (open)");
        MM_REQUIRE(mm_is_smooth(n), "a periodic axis needs a mesh size of the form 2^a 3^b 5^c");
        return n;
    }
    if (given % 2 == 0 && mm_is_smooth(given)) return given;
    int p = 2 * n - 1;  // fits: given is no smaller
    while (!(p % 2 == 0 && mm_is_smooth(p))) {
        MM_REQUIRE(p < INT_MAX, "no transform length for this mesh size");
        ++p;
    }
    return p;
}

static int g_max_lds = 0;
static std::once_flag g_lds_once;

int mm_max_lds_bytes()
{
    std::call_once(g_lds_once, []() {
        int dev = 0;
        (void)hipGetDevice(&dev);
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
            v = 65536;
        g_max_lds = v;
    });
    return g_max_lds;
}

int mm_num_cus()
{
    int dev = 0, n = 0;
    MM_HIP(hipGetDevice(&dev));
    MM_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    return n;
}

// ---------------------------------------------------------------------------
// launch-shape table ("wisdom")
// ---------------------------------------------------------------------------
static std::mutex g_wis_mu;
static std::map<std::string, MmShape> g_wisdom;
static thread_local MmShape g_candidate;
static thread_local bool g_have_candidate = false;

// "<arch>/<CUs>" of the current device, e.g. gfx950/256
static std::string device_tag()
{
    static std::mutex mu;
    static std::map<int, std::string> tags;
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(mu);
    auto it = tags.find(dev);
    if (it != tags.end()) return it->second;
    hipDeviceProp_t p;
    std::string tag = "unknown";
    if (hipGetDeviceProperties(&p, dev) == hipSuccess) {
        std::string arch = p.gcnArchName;
        tag = arch.substr(0, arch.find(':')) + "/" + std::to_string(p.multiProcessorCount);
    }
    tags[dev] = tag;
    return tag;
}

static std::string shape_key(int nx, int ny, int nz, size_t real_bytes)
{
    return std::to_string(nx) + "x" + std::to_string(ny) + "x" + std::to_string(nz) +
           (real_bytes == 4 ? " fp32 " : " fp64 ") + device_tag();
}

MmShape mm_shape_for(int nx, int ny, int nz, size_t real_bytes)
{
    if (g_have_candidate) return g_candidate;
    const std::string key = shape_key(nx, ny, nz, real_bytes);
    std::lock_guard<std::mutex> lk(g_wis_mu);
    auto it = g_wisdom.find(key);
    return it != g_wisdom.end() ? it->second : MmShape{0, 0, 0, 0, 0};
}

void mm_shape_set_candidate(const MmShape *s)
{
    g_have_candidate = s != nullptr;
    if (s) g_candidate = *s;
}

void mm_wisdom_put(int nx, int ny, int nz, size_t real_bytes, const MmShape &s)
{
    const std::string key = shape_key(nx, ny, nz, real_bytes);
    std::lock_guard<std::mutex> lk(g_wis_mu);
    g_wisdom[key] = s;
}

// File format: '#' comment lines, then one entry per line,
// "<nx>x<ny>x<nz> <fp32|fp64> <arch>/<CUs> lpw_x tk_y tk_z rpw stage_threads".
// An import reads the whole file first and takes nothing from an invalid one.
extern "C" int mm_wisdom_import(const char *path, int *n_entries)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(path, "null argument");
    std::ifstream f(path);
    MM_REQUIRE((bool)f, std::string("cannot open wisdom file ") + path);
    std::map<std::string, MmShape> got;
    std::string line;
    int lineno = 0;
    while (std::getline(f, line)) {
        ++lineno;
        const size_t b = line.find_first_not_of(" \t\r");
        if (b == std::string::npos || line[b] == '#') continue;
        std::istringstream ls(line);
        std::string mesh, prec, dev, extra;
        MmShape v;
        const bool ok = (bool)(ls >> mesh >> prec >> dev >> v.lpw_x >> v.tk_y >> v.tk_z >> v.rpw >> v.stage_threads) &&
                        !(ls >> extra);
        int nx = 0, ny = 0, nz = 0;
        char x1 = 0, x2 = 0;
        std::istringstream ms(mesh);
        const bool mesh_ok = (bool)(ms >> nx >> x1 >> ny >> x2 >> nz) && x1 == 'x' && x2 == 'x' && nx > 0 && ny > 0 &&
                             nz > 0 && !(ms >> extra);
        const bool vals_ok = v.lpw_x >= 0 && v.tk_y >= 0 && v.tk_z >= 0 && v.rpw >= 0 && v.stage_threads >= 0 &&
                             v.lpw_x <= 1024 && v.tk_y <= 1024 && v.tk_z <= 1024 && v.rpw <= 1024 &&
                             v.stage_threads <= 1024;
        MM_REQUIRE(ok && mesh_ok && vals_ok && (prec == "fp32" || prec == "fp64"),
                   std::string("invalid wisdom file ") + path + " at line " + std::to_string(lineno));
        got[mesh + " " + prec + " " + dev] = v;
    }
    {
        std::lock_guard<std::mutex> lk(g_wis_mu);
        for (const auto &kv : got) g_wisdom[kv.first] = kv.second;
    }
    if (n_entries) *n_entries = (int)got.size();
    MM_CAPI_END
}

extern "C" int mm_wisdom_export(const char *path)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(path, "null argument");
    std::ostringstream os;
    os << "# libmmhip launch-shape wisdom: mesh precision device lpw_x tk_y tk_z rpw stage_threads\n";
    {
        std::lock_guard<std::mutex> lk(g_wis_mu);
        for (const auto &kv : g_wisdom)
            os << kv.first << " " << kv.second.lpw_x << " " << kv.second.tk_y << " " << kv.second.tk_z << " "
               << kv.second.rpw << " " << kv.second.stage_threads << "\n";
    }
    std::ofstream f(path);
    MM_REQUIRE((bool)f, std::string("cannot write wisdom file ") + path);
    f << os.str();
    MM_REQUIRE((bool)f, std::string("cannot write wisdom file ") + path);
    MM_CAPI_END
}

extern "C" int mm_wisdom_forget(void)
{
    MM_CAPI_BEGIN
    std::lock_guard<std::mutex> lk(g_wis_mu);
    g_wisdom.clear();
    MM_CAPI_END
}

ConvLaunch mm_choose_launch(const ConvGeom &g, const FftPlanHost &px, const FftPlanHost &py,
                                const FftPlanHost &pz, size_t csize)
{
    const int lds = mm_max_lds_bytes();
    const MmShape w = mm_shape_for(g.nx, g.ny, g.nz, csize / 2);
    ConvLaunch ln;
    ln.lpw_x = env_int("MM_LPW_X", w.lpw_x > 0 ? w.lpw_x : std::max(1, 256 / px.tline));
    while (ln.lpw_x > 1 && (lines_lds<MM_SKEW_X>(ln.lpw_x, px.L, csize) > (size_t)lds || ln.lpw_x * px.tline > 1024)) --ln.lpw_x;
    const int nl_y = g.is2d ? 3 : 1;
    // default tile widths by line length, measured on MI355X (FP32 steps/s,
    // same-run A/B): y 8 columns, 2 for lines of 2048 or more (1024x1024x2
    // cells: +3 %; 256x256x16: 8 best; 512x512x64: 8 better than 4 by 4 %);
    // z 512 / Pz columns within [16, 64] (256x256x16: 16 best of 8..64;
    // 1024x1024x2, Pz 4: 64 +4 % against 16), halved while a workgroup
    // needs more than 64 KiB of LDS (512x512x64 FP64, Pz 128: 8 columns,
    // 56 KiB, +11 % against 16 at 111 KiB, one workgroup per CU; FP32 keeps
    // 16 at 55 KiB, 8 and 4 slower)
    const int tk_y0 = g.Py >= 2048 ? 2 : 8;
    int tk_z0 = std::max(16, std::min(64, 512 / std::max(1, g.Pz)));
    while (tk_z0 > 1 && lines_lds<MM_SKEW_Z>(3 * tk_z0, pz.L, csize) > 65536) tk_z0 /= 2;
    int tk = floor_pow2(env_int("MM_TK_Y", w.tk_y > 0 ? w.tk_y : tk_y0));
    while (tk > 1 && ((size_t)nl_y * tk * py.tline > 1024 || lines_lds<MM_SKEW_Y>(nl_y * tk, py.L, csize) > (size_t)lds)) tk /= 2;
    ln.tk_y = tk;
    MM_REQUIRE((size_t)nl_y * tk * py.tline <= 1024 && lines_lds<MM_SKEW_Y>(nl_y * tk, py.L, csize) <= (size_t)lds,
               "y transform length too large for one workgroup");
    int tz = floor_pow2(env_int("MM_TK_Z", w.tk_z > 0 ? w.tk_z : tk_z0));
    while (tz > 1 && ((size_t)3 * tz * pz.tline > 1024 || lines_lds<MM_SKEW_Z>(3 * tz, pz.L, csize) > (size_t)lds)) tz /= 2;
    ln.tk_z = tz;
    return ln;
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" int mm_conv_create(const double *N_host, int nx, int ny, int nz, int ex, int ey, int ez,
                              int precision, mm_conv_t **out)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(N_host && out, "null argument");
    MM_REQUIRE(precision == MM_FP64 || precision == MM_FP32, "precision must be MM_FP64 or MM_FP32");
    mm_conv *c = new mm_conv();
    c->precision = precision;
    try {
        if (precision == MM_FP64) {
            c->c64 = new ConvImpl<double>();
            c->c64->init(N_host, nx, ny, nz, ex, ey, ez);
        } else {
            c->c32 = new ConvImpl<float>();
            c->c32->init(N_host, nx, ny, nz, ex, ey, ez);
        }
    } catch (...) {
        if (c->c64) { c->c64->release(); delete c->c64; }
        if (c->c32) { c->c32->release(); delete c->c32; }
        delete c;
        throw;
    }
    *out = c;
    MM_CAPI_END
}

extern "C" int mm_conv_execute(mm_conv_t *conv, const double *M, double *H, void *stream)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(conv && M && H, "null argument");
    MM_REQUIRE(conv->precision == MM_FP64, "convolution was created for FP32; use mm_conv_execute_f32");
    conv->c64->execute(M, H, (hipStream_t)stream);
    MM_CAPI_END
}

extern "C" int mm_conv_execute_f32(mm_conv_t *conv, const float *M, float *H, void *stream)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(conv && M && H, "null argument");
    MM_REQUIRE(conv->precision == MM_FP32, "convolution was created for FP64; use mm_conv_execute");
    conv->c32->execute(M, H, (hipStream_t)stream);
    MM_CAPI_END
}

extern "C" int mm_conv_fft_size(const mm_conv_t *conv, int *fft_xyz)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(conv && fft_xyz, "null argument");
    const ConvGeom &g = conv->c64 ? conv->c64->g : conv->c32->g;
    fft_xyz[0] = g.Px;
    fft_xyz[1] = g.Py;
    fft_xyz[2] = g.Pz;
    MM_CAPI_END
}

extern "C" int mm_conv_destroy(mm_conv_t *conv)
{
    MM_CAPI_BEGIN
    if (!conv) return MM_OK;
    if (conv->c64) { conv->c64->release(); delete conv->c64; }
    if (conv->c32) { conv->c32->release(); delete conv->c32; }
    delete conv;
    MM_CAPI_END
}

// ---------------------------------------------------------------------------
// direct-sum convolution
// ---------------------------------------------------------------------------
// H(r) = sum_r' N((r - r') mod E) M(r') over the whole mesh, the tensor in the
// layout of GenerateDemagTensor (6 entries per point, x fastest).  One thread
// per target cell; the workgroup walks the source cells in tiles staged in
// LDS (M of 256 source cells, three components), the source order of every
// thread z, y, x as the reference's loop.
#define MM_SIMPLE_TILE 256
__global__ void __launch_bounds__(MM_SIMPLE_TILE) k_conv_simple(const double *__restrict__ N, int nx, int ny, int nz,
                                                               int ex, int ey, int ez, const double *__restrict__ M,
                                                               double *__restrict__ H)
{
    __shared__ double ms[3][MM_SIMPLE_TILE];
    const int n = nx * ny * nz;
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const bool act = i < n;
    const int x = act ? i % nx : 0, y = act ? (i / nx) % ny : 0, z = act ? i / (nx * ny) : 0;
    double hx = 0.0, hy = 0.0, hz = 0.0;
    for (int j0 = 0; j0 < n; j0 += MM_SIMPLE_TILE) {
        const int jl = j0 + (int)threadIdx.x;
        __syncthreads();
        for (int c = 0; c < 3; ++c) ms[c][threadIdx.x] = jl < n ? M[(size_t)c * n + jl] : 0.0;
        __syncthreads();
        if (!act) continue;
        const int cnt = min(MM_SIMPLE_TILE, n - j0);
        int m = j0 % nx, o = j0 / (nx * ny), nn = (j0 / nx) % ny;
        for (int t = 0; t < cnt; ++t) {
            const int X = (x - m + ex) % ex, Y = (y - nn + ey) % ey, Z = (z - o + ez) % ez;
            const double *Np = N + 6 * ((size_t)X + (size_t)ex * ((size_t)Y + (size_t)ey * Z));
            const double Mx = ms[0][t], My = ms[1][t], Mz = ms[2][t];
            hx += Np[0] * Mx + Np[1] * My + Np[2] * Mz;
            hy += Np[1] * Mx + Np[3] * My + Np[4] * Mz;
            hz += Np[2] * Mx + Np[4] * My + Np[5] * Mz;
            if (++m == nx) {
                m = 0;
                if (++nn == ny) {
                    nn = 0;
                    ++o;
                }
            }
        }
    }
    if (act) {
        H[i] = hx;
        H[(size_t)n + i] = hy;
        H[2 * (size_t)n + i] = hz;
    }
}

struct mm_conv_simple {
    double *N = nullptr;
    int nx = 0, ny = 0, nz = 0, ex = 0, ey = 0, ez = 0;
};

extern "C" int mm_conv_simple_create(const double *N_host, int nx, int ny, int nz, int ex, int ey, int ez,
                                     mm_conv_simple_t **out)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(N_host && out, "null argument");
    MM_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1 && ex >= nx && ey >= ny && ez >= nz, "bad sizes");
    MM_REQUIRE((size_t)nx * ny * nz < (1u << 30), "mesh too large for the direct sum");
    mm_conv_simple *c = new mm_conv_simple();
    c->nx = nx;
    c->ny = ny;
    c->nz = nz;
    c->ex = ex;
    c->ey = ey;
    c->ez = ez;
    const size_t bytes = sizeof(double) * 6 * (size_t)ex * ey * ez;
    if (hipMalloc(&c->N, bytes) != hipSuccess) {
        delete c;
        MM_REQUIRE(false, "device allocation failed");
    }
    const hipError_t e = hipMemcpy(c->N, N_host, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(c->N);
        delete c;
        MM_HIP(e);
    }
    *out = c;
    MM_CAPI_END
}

extern "C" int mm_conv_simple_execute(mm_conv_simple_t *c, const double *M, double *H, void *stream)
{
    MM_CAPI_BEGIN
    MM_REQUIRE(c && M && H, "null argument");
    const int n = c->nx * c->ny * c->nz;
    hipLaunchKernelGGL(k_conv_simple, dim3((n + MM_SIMPLE_TILE - 1) / MM_SIMPLE_TILE), dim3(MM_SIMPLE_TILE), 0,
                       (hipStream_t)stream, c->N, c->nx, c->ny, c->nz, c->ex, c->ey, c->ez, M, H);
    MM_HIP(hipGetLastError());
    MM_CAPI_END
}

extern "C" int mm_conv_simple_destroy(mm_conv_simple_t *c)
{
    MM_CAPI_BEGIN
    if (!c) return MM_OK;
    if (c->N) (void)hipFree(c->N);
    delete c;
    MM_CAPI_END
}
