// Pruned, deconvolving FFTs for fine grids of any 5-smooth size (2^a 3^b 5^c),
// the general counterpart of the power-of-two kernels in mn_fftp.hip.
//
// As there, one pass per axis transforms that axis's lines and keeps (type 1)
// or fills (type 2) only its N_d modes, with dec_d fused, so that a 3D type-1
// transform moves grid + 2 (n0 n1 N2) + 2 (n0 N1 N2) + fk instead of the four
// full-grid passes, transposes and crop pass of a library transform. What
// bounds it is memory traffic; a stage's LDS round trip comes second, hence
// radices up to 16 (three stages for most sizes up to 1000).
//
// A workgroup transforms TI lines of N values in LDS by Stockham stages of
// radix 2 to 16. N, and with it every radix, stride and division, is a
// compile-time constant (mn_fftg.h): one kernel with run-time radices did the
// same arithmetic, but its index work and spilled registers held it to 1.4 to
// 2.0 TB/s. The lengths of the table (all even 5-smooth ones up to 2048, and
// the odd ones that splitting needs) have three kernels each;
// the files mn_fftg_a.hip to mn_fftg_f.hip only divide the compile time. The
// first stage reads its inputs from global memory (all loads issued before
// any is used) and the last stage writes its outputs there. The transform in
// the kernel is the e^{+i} one; the other sign conjugates its inputs and
// outputs.
// Measured (type 1 / type 2, us; library transform with its crop or pad pass
// in brackets): 270 x 240 x 180 60 / 53 (210 / 229), 4.0 and 4.5 TB/s of the
// bytes above, 400^3 319 / 345 (1256 / 1436), 160^3 with 128^3 modes 35 / 35
// (75 / 80), 1250 x 900 17 / 17 (40 / 43), 1012500 points 23 / 23 (51 / 52),
// 8192 points 11.5 / 11.5 (18 / 18).
//
// Axes longer than 2048 (too long for LDS, or for useful runs of a strided
// axis) are split as n = n1 n2: a pass over the n1-point lines of stride n2, whose
// outputs are multiplied by exp(2 pi i k1 b / n), and one over the n2-point
// lines; mode pruning and deconvolution go to whichever pass touches the
// mode side.
//
// The grid may be stored with extents e_d >= n_d: type 1 then adds the cells
// at x + n_d < e_d (the overhang of footprints past the period) to cell x as
// the first pass loads it, and type 2 stores every cell to its image as well,
// so that owner-computes spreads and gathers, whose blocks need multiples of
// 8 cells, serve every grid size without a fold or copy pass.
//
// ref: nd.py:374-383 (_fft_grid), nd.py:416-435 (crop + deconvolution),
// nd.py:878-906 (type-2 pad + deconvolution).
#include <cmath>
#include <map>
#include <mutex>
#include <utility>

#include "mn_fftg.h"

namespace mn {
namespace {

// tw[m] = exp(2 pi i m / n), rounded from fp64
__global__ void k_fg_twiddles(float2 *tw, int n) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    double s, c;
    sincospi(2.0 * (double)m / (double)n, &s, &c);
    tw[m] = make_float2((float)c, (float)s);
}

// Device tables of the stage twiddles, one per (device, n): n is 5-smooth and
// at most 2048, so there are a few hundred at the very most (4 MB); they
// are released with the other transform caches (mn_fft_cache_clear).
std::mutex g_fg_mu;
std::map<std::pair<int, int>, float2 *> g_fg_tw;

int fg_twiddles(int n, hipStream_t s, const float2 **out) {
    int dev = 0;
    MN_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_fg_mu);
    const auto key = std::make_pair(dev, n);
    auto it = g_fg_tw.find(key);
    if (it == g_fg_tw.end()) {
        float2 *t = nullptr;
        MN_HIP_CHECK(hipMalloc(&t, sizeof(float2) * (size_t)n));
        k_fg_twiddles<<<(n + 255) / 256, 256, 0, s>>>(t, n);
        hipError_t e = hipGetLastError();
        // later calls may come on other streams: the table is complete first
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            (void)hipFree(t);
            set_error(std::string("fft twiddles: ") + hipGetErrorString(e));
            return MN_ERUNTIME;
        }
        it = g_fg_tw.emplace(key, t).first;
    }
    *out = it->second;
    return MN_OK;
}

constexpr int64_t FG_SPLIT = 2048;  // longer axes are split in two passes

const FgEntry *fg_find(int64_t n) {
    static const std::map<int64_t, FgEntry> table = [] {
        std::map<int64_t, FgEntry> t;
        for (auto get : {fg_entries_a, fg_entries_b, fg_entries_c, fg_entries_d, fg_entries_e,
                         fg_entries_f}) {
            int k = 0;
            const FgEntry *e = get(&k);
            for (int i = 0; i < k; ++i) t[e[i].n] = e[i];
        }
        return t;
    }();
    const auto it = table.find(n);
    return it == table.end() ? nullptr : &it->second;
}

// One pass over a.nlines lines of n values.
int fg_pass(int kind, int64_t n, const float2 *in, float2 *out, const FgArgs &a, hipStream_t s) {
    const FgEntry *e = fg_find(n);
    if (!e) {
        set_error("fft: unsupported length");
        return MN_EINVAL;
    }
    const int64_t ntile = (a.nlines + e->ti - 1) / e->ti;
    if (ntile > 0x7fffffff) {
        set_error("fft: too many lines");
        return MN_EINVAL;
    }
    const float2 *tw = nullptr;
    int rc = fg_twiddles((int)n, s, &tw);
    if (rc) return rc;
    if (e->lds > 60000)
        MN_HIP_CHECK(hipFuncSetAttribute((const void *)e->k[kind],
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)e->lds));
    e->k[kind]<<<(unsigned)ntile, e->threads, e->lds, s>>>(in, out, tw, a);
    MN_LAUNCH_CHECK("fft pass");
    return MN_OK;
}

// The split n = n1 n2 of a long axis into two table lengths as near each other
// as can be; false if there is none.
bool fg_split(int64_t n, int64_t *n1, int64_t *n2) {
    for (int64_t d = (int64_t)std::sqrt((double)n) + 1; d >= 16; --d) {
        if (n % d == 0 && fg_find(d) && fg_find(n / d)) {
            *n1 = d;
            *n2 = n / d;
            return true;
        }
    }
    return false;
}

bool fg_axis_ok(int64_t n) {
    int64_t a, b;
    return n >= 4 && n <= FG_SPLIT * FG_SPLIT &&
           (n <= FG_SPLIT ? fg_find(n) != nullptr : fg_split(n, &a, &b));
}

struct FgPlan {
    int dim;
    int64_t n[3], N[3], e[3], batch;
};

int fg_check(int dim, const int64_t n_up[3], const int64_t N[3], const int64_t ext[3],
             int64_t batch, FgPlan *p) {
    MN_REQUIRE(dim >= 1 && dim <= 3, "general fft: dim must be 1, 2 or 3");
    MN_REQUIRE(batch >= 1, "general fft: batch must be >= 1");
    p->dim = dim;
    p->batch = batch;
    for (int d = 0; d < dim; ++d) {
        MN_REQUIRE(fg_axis_ok(n_up[d]), "general fft: fine-grid sizes must be 2^a 3^b 5^c in range");
        MN_REQUIRE(N[d] >= 1 && N[d] <= n_up[d], "general fft: mode count out of range");
        p->n[d] = n_up[d];
        p->N[d] = N[d];
        p->e[d] = ext ? ext[d] : n_up[d];
        MN_REQUIRE(p->e[d] >= n_up[d] && p->e[d] <= 2 * n_up[d],
                   "general fft: grid extents must be in [n, 2 n]");
        if (p->e[d] != n_up[d])
            MN_REQUIRE(dim >= 2 && n_up[dim - 1] <= FG_SPLIT,
                       "general fft: extents need two dims and a last axis of at most 2048");
    }
    if (ext)
        for (int d = 0; d < dim; ++d)
            MN_REQUIRE(dim == 1 || n_up[dim - 1] <= FG_SPLIT || ext[d] == n_up[d],
                       "general fft: extents need a last axis of at most 2048");
    return MN_OK;
}

// Walks the passes of a transform. run(kind, line length, args, elems): elems
// is the size of the pass's output array.
template <typename F>
int fg_walk(const FgPlan &p, bool type1, int isign, const float *const *dec, F &&run) {
    const int dim = p.dim, last = dim - 1;
    bool ext = false;
    for (int d = 0; d < dim; ++d) ext = ext || p.e[d] != p.n[d];
    for (int step = 0; step < dim; ++step) {
        const int d = type1 ? last - step : step;
        // arrays (outer, n or N, inner); axes before d are full, after d modes
        int64_t outer = p.batch, inner = 1;
        for (int k = 0; k < d; ++k) outer *= p.n[k];
        for (int k = d + 1; k < dim; ++k) inner *= p.N[k];
        const int64_t n = p.n[d], M = p.N[d];
        FgArgs a{};
        a.M = (int)M;
        a.hM = (int)(M / 2);
        a.nfull = (int)n;
        a.dec = dec ? dec[d] : nullptr;
        a.sg = isign >= 0 ? 1.0f : -1.0f;
        a.oc = 1;
        int rc;
        if (n <= FG_SPLIT) {
            a.pstep = 1;
            a.nlines = outer * inner;
            a.ghost = ext && d == last;
            // base of line (o, q, r) on the grid side and on the mode side
            int64_t g1 = n * inner, g2 = 0, gq = 0, m1 = M * inner, m2 = 0, mq = 0;
            a.ni = a.inner = inner;
            if (a.ghost) {
                const int64_t e2 = p.e[last];
                if (dim == 3) {  // o = (batch, x), q = y
                    const int64_t e1 = p.e[1];
                    a.oc = p.n[0];
                    a.ni = p.n[1];
                    g1 = p.e[0] * e1 * e2;
                    g2 = e1 * e2;
                    gq = e2;
                    m1 = p.n[0] * p.n[1] * M;
                    m2 = p.n[1] * M;
                    a.gq = p.e[1] - p.n[1];
                    a.go = p.e[0] - p.n[0];
                    a.gqo = p.n[1] * gq;
                    a.goo = p.n[0] * g2;
                } else {  // o = batch, q = x
                    a.ni = p.n[0];
                    g1 = p.e[0] * e2;
                    gq = e2;
                    m1 = p.n[0] * M;
                    a.gq = p.e[0] - p.n[0];
                    a.gqo = p.n[0] * gq;
                }
                mq = M;
                a.inner = 1;
                a.ge = (int)(e2 - n);
            }
            a.ib1 = type1 ? g1 : m1;
            a.ib2 = type1 ? g2 : m2;
            a.ibq = type1 ? gq : mq;
            a.ob1 = type1 ? m1 : g1;
            a.ob2 = type1 ? m2 : g2;
            a.obq = type1 ? mq : gq;
            a.ies = a.oes = inner;
            a.icontig = a.ocontig = inner == 1;
            rc = run(type1 ? FG_CROP : FG_PAD, n, a, outer * inner * (type1 ? M : n));
            if (rc) return rc;
            continue;
        }
        int64_t n1, n2;
        if (!fg_split(n, &n1, &n2)) {
            set_error("general fft: axis too long");
            return MN_EINVAL;
        }
        // first pass: n1-point lines of stride n2, line q = b
        FgArgs A = a;
        A.useq = 1;
        A.pstep = (int)n2;
        A.ntw = (int)n;
        A.nlines = outer * n2 * inner;
        A.ni = n2 * inner;
        A.inner = inner;
        A.ib1 = type1 ? n * inner : M * inner;
        A.ibq = type1 ? inner : 0;
        A.ies = type1 ? n2 * inner : inner;
        A.ob1 = n * inner;
        A.obq = inner;
        A.oes = n2 * inner;
        rc = run(type1 ? FG_MID : FG_PAD, n1, A, outer * n * inner);
        if (rc) return rc;
        // second pass: n2-point lines, line q = k1, output k1 + n1 k2
        FgArgs B = a;
        B.useq = 1;
        B.pstep = (int)n1;
        B.nlines = outer * n1 * inner;
        B.ni = n1 * inner;
        B.inner = inner;
        B.ib1 = n * inner;
        B.ibq = n2 * inner;
        B.ies = inner;
        B.icontig = inner == 1;
        B.ob1 = type1 ? M * inner : n * inner;
        B.obq = type1 ? 0 : inner;
        B.oes = type1 ? inner : n1 * inner;
        rc = run(type1 ? FG_CROP : FG_MID, n2, B, outer * inner * (type1 ? M : n));
        if (rc) return rc;
    }
    return MN_OK;
}

// Bytes of the two buffers the intermediate arrays alternate between.
void fg_work(const FgPlan &p, bool type1, int64_t w[2]) {
    w[0] = w[1] = 0;
    int64_t prev = 0;
    int k = 0;
    // the last pass writes the result: count every pass but that one
    (void)fg_walk(p, type1, 1, nullptr, [&](int, int64_t, const FgArgs &, int64_t elems) {
        if (k > 0 && prev * 8 > w[(k - 1) & 1]) w[(k - 1) & 1] = prev * 8;
        prev = elems;
        ++k;
        return MN_OK;
    });
    for (int i = 0; i < 2; ++i) w[i] = (w[i] + 255) / 256 * 256;
}

int fg_run(const FgPlan &p, bool type1, int isign, const float2 *in, const float *const *dec,
           void *work, int64_t work_bytes, float2 *out, hipStream_t s) {
    int64_t w[2];
    fg_work(p, type1, w);
    MN_REQUIRE(work_bytes >= w[0] + w[1] && (w[0] + w[1] == 0 || work),
               "general fft: work buffer too small");
    int npass = 0;
    (void)fg_walk(p, type1, isign, nullptr, [&](int, int64_t, const FgArgs &, int64_t) {
        ++npass;
        return MN_OK;
    });
    char *wb = static_cast<char *>(work);
    float2 *bufs[2] = {reinterpret_cast<float2 *>(wb), reinterpret_cast<float2 *>(wb + w[0])};
    const float2 *src = in;
    int k = 0;
    return fg_walk(p, type1, isign, dec,
                   [&](int kind, int64_t n, const FgArgs &a, int64_t) {
                       float2 *dst = k + 1 == npass ? out : bufs[k & 1];
                       const int rc = fg_pass(kind, n, src, dst, a, s);
                       src = dst;
                       ++k;
                       return rc;
                   });
}

}  // namespace

void fftg_cache_clear() {
    std::lock_guard<std::mutex> lock(g_fg_mu);
    for (auto &kv : g_fg_tw) (void)hipFree(kv.second);
    g_fg_tw.clear();
}

}  // namespace mn

using namespace mn;

extern "C" {

int mn_fftg_supported(int dim, const int64_t n_up[3]) {
    if (dim < 1 || dim > 3) return 0;
    for (int d = 0; d < dim; ++d)
        if (!fg_axis_ok(n_up[d])) return 0;
    return 1;
}

int64_t mn_fftg_work_bytes(int dim, const int64_t n_up[3], const int64_t N[3], int64_t batch) {
    FgPlan p{};
    if (fg_check(dim, n_up, N, nullptr, batch, &p)) return -1;
    int64_t a[2], b[2];
    fg_work(p, true, a);
    fg_work(p, false, b);
    const int64_t t1 = a[0] + a[1], t2 = b[0] + b[1];
    return t1 > t2 ? t1 : t2;
}

int mn_fftg_crop_deconv(int dim, const int64_t n_up[3], const int64_t N[3], const int64_t ext[3],
                        int64_t batch, int isign, const void *grid, const float *const dec[3],
                        void *work, int64_t work_bytes, void *fk, mn_stream_t stream) {
    clear_error();
    FgPlan p{};
    int rc = fg_check(dim, n_up, N, ext, batch, &p);
    if (rc) return rc;
    MN_REQUIRE(grid && fk, "general fft: NULL pointer");
    for (int d = 0; d < dim; ++d) MN_REQUIRE(dec[d], "general fft: NULL deconvolution vector");
    return fg_run(p, true, isign, static_cast<const float2 *>(grid), dec, work, work_bytes,
                  static_cast<float2 *>(fk), as_stream(stream));
}

int mn_fftg_pad_deconv(int dim, const int64_t n_up[3], const int64_t N[3], const int64_t ext[3],
                       int64_t batch, int isign, const void *fk, const float *const dec[3],
                       void *work, int64_t work_bytes, void *grid, mn_stream_t stream) {
    clear_error();
    FgPlan p{};
    int rc = fg_check(dim, n_up, N, ext, batch, &p);
    if (rc) return rc;
    MN_REQUIRE(grid && fk, "general fft: NULL pointer");
    for (int d = 0; d < dim; ++d) MN_REQUIRE(dec[d], "general fft: NULL deconvolution vector");
    return fg_run(p, false, isign, static_cast<const float2 *>(fk), dec, work, work_bytes,
                  static_cast<float2 *>(grid), as_stream(stream));
}

}  // extern "C"
