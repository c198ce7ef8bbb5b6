// Kernels of the general pruned FFT (see mn_fftg.hip): one pass over lines of
// a compile-time length N.
#pragma once

#include "mn_common.h"

namespace mn {

struct FgArgs {
    int64_t nlines;
    // line = o ni + q inner + r; its base in either array is
    // (o / oc) b1 + (o % oc) b2 + q bq + r, its element stride es
    int64_t ni, inner, oc;
    int64_t ib1, ib2, ibq, ies;
    int64_t ob1, ob2, obq, oes;
    int icontig, ocontig;       // a line's elements are contiguous (es == 1)
    // modes kept of the pruned side: element l of a line is FFT position
    // l pstep + q of nfull (q taken as 0 unless useq)
    int nfull, pstep, useq, M, hM;
    const float *dec;
    int ntw;                    // twiddle modulus of a split axis's first pass, else 0
    // images of a grid stored with larger extents (ghost): line q (and
    // o % oc) below gq (go) also lives at base + gqo (+ goo), element p < ge
    // at p + N
    int ghost;
    int64_t gq, go, gqo, goo;
    int ge;
    float sg;                   // +1, or -1: conjugate inputs and outputs
};

// One line length's kernels: crop (full lines in, kept modes out), pad (modes
// in, full lines out) and mid (full in and out), their tile and workgroup.
typedef void (*FgKernel)(const float2 *, float2 *, const float2 *, FgArgs);
struct FgEntry {
    int n, ti, threads;
    size_t lds;
    FgKernel k[3];
};
enum { FG_CROP = 0, FG_PAD = 1, FG_MID = 2 };

// the entries of each instantiation file, ascending by length
const FgEntry *fg_entries_a(int *count);
const FgEntry *fg_entries_b(int *count);
const FgEntry *fg_entries_c(int *count);
const FgEntry *fg_entries_d(int *count);
const FgEntry *fg_entries_e(int *count);
const FgEntry *fg_entries_f(int *count);

namespace fg {

// Stage radices of n = 2^a 3^b 5^c (two stages at least) from {2, 3, 4, 5, 6,
// 8, 9, 10, 16}, few of them, larger ones first: the first stage's loads are
// the ones to overlap.
struct Radices {
    int k, r[8];
};
constexpr Radices radices(int n) {
    Radices p{};
    int c2 = 0, c3 = 0, c5 = 0;
    for (; n % 2 == 0; n /= 2) ++c2;
    for (; n % 3 == 0; n /= 3) ++c3;
    for (; n % 5 == 0; n /= 5) ++c5;
    if (n != 1) return p;
    for (; c3 >= 2; c3 -= 2) p.r[p.k++] = 9;
    for (; c5 > 0 && c2 > 0; --c5, --c2) p.r[p.k++] = 10;
    for (; c5 > 0; --c5) p.r[p.k++] = 5;
    if (c3) {
        if (c2 % 3 == 1) {
            p.r[p.k++] = 6;
            --c2;
        } else {
            p.r[p.k++] = 3;
        }
    }
    while (c2 > 0) {  // the twos evenly over the fewest stages
        const int st = (c2 + 3) / 4, e = (c2 + st - 1) / st;
        p.r[p.k++] = 1 << e;
        c2 -= e;
    }
    if (p.k == 1 && p.r[0] > 3 && p.r[0] != 5) {  // one radix: two stages of it
        const int v = p.r[0], x = v == 9 ? 3 : (v == 10 ? 5 : (v == 6 ? 3 : (v == 4 ? 2 : 4)));
        p.r[0] = x;
        p.r[1] = v / x;
        p.k = 2;
    }
    for (int i = 1; i < p.k; ++i)
        for (int j = i; j > 0 && p.r[j] > p.r[j - 1]; --j) {
            const int t = p.r[j];
            p.r[j] = p.r[j - 1];
            p.r[j - 1] = t;
        }
    return p;
}

// Tile of a line length: TI lines (16 give strided axes 128-byte runs; the
// longer lines take fewer, so that two or three workgroups share a CU), LDS
// rows of PI = TI + 1 values (one pad column keeps walks along a line and
// across lines off the same banks, and constant offsets between a
// butterfly's values), and one butterfly per thread of the large radices.
template <int N>
struct Cfg {
    static constexpr Radices R = radices(N);
    static constexpr int TI = N <= 320 ? 16 : (N <= 1024 ? 8 : 4);
    static constexpr int PI = TI + 1;
    static constexpr int bmax() {
        int m = 0;
        for (int i = 0; i < R.k; ++i)
            if (R.r[i] >= 8 || R.r[i] == R.r[0]) m = N / R.r[i] > m ? N / R.r[i] : m;
        return m * TI;
    }
    static constexpr int T = bmax() >= 1024 ? 1024 : (bmax() + 63) / 64 * 64;
    static constexpr size_t LDS = sizeof(float2) * ((size_t)N * PI + N);
    static constexpr int ns(int s) {
        int p = 1;
        for (int i = 0; i < s; ++i) p *= R.r[i];
        return p;
    }
};

__device__ __forceinline__ float2 gadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 gsub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 gmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 gscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 gmul_i(float2 a) { return make_float2(-a.y, a.x); }

// In-register DFTs X[k] = sum_m v[m] exp(2 pi i m k / R).
__device__ __forceinline__ void gdft2(float2 &a, float2 &b) {
    const float2 t = a;
    a = gadd(t, b);
    b = gsub(t, b);
}
__device__ __forceinline__ void gdft3(float2 &v0, float2 &v1, float2 &v2) {
    constexpr float H3 = 0.86602540378443864676f;
    const float2 t1 = gadd(v1, v2);
    const float2 t2 = make_float2(v0.x - 0.5f * t1.x, v0.y - 0.5f * t1.y);
    const float2 t3 = gscale(gmul_i(gsub(v1, v2)), H3);
    v0 = gadd(v0, t1);
    v1 = gadd(t2, t3);
    v2 = gsub(t2, t3);
}
__device__ __forceinline__ void gdft4(float2 &v0, float2 &v1, float2 &v2, float2 &v3) {
    const float2 a0 = gadd(v0, v2), a1 = gsub(v0, v2), a2 = gadd(v1, v3), a3 = gmul_i(gsub(v1, v3));
    v0 = gadd(a0, a2);
    v2 = gsub(a0, a2);
    v1 = gadd(a1, a3);
    v3 = gsub(a1, a3);
}
__device__ __forceinline__ void gdft5(float2 &v0, float2 &v1, float2 &v2, float2 &v3, float2 &v4) {
    constexpr float C1 = 0.30901699437494742410f, C2 = -0.80901699437494742410f;
    constexpr float S1 = 0.95105651629515357212f, S2 = 0.58778525229247312917f;
    const float2 a1 = gadd(v1, v4), b1 = gsub(v1, v4), a2 = gadd(v2, v3), b2 = gsub(v2, v3);
    const float2 p1 = make_float2(v0.x + C1 * a1.x + C2 * a2.x, v0.y + C1 * a1.y + C2 * a2.y);
    const float2 p2 = make_float2(v0.x + C2 * a1.x + C1 * a2.x, v0.y + C2 * a1.y + C1 * a2.y);
    const float2 q1 = gmul_i(make_float2(S1 * b1.x + S2 * b2.x, S1 * b1.y + S2 * b2.y));
    const float2 q2 = gmul_i(make_float2(S2 * b1.x - S1 * b2.x, S2 * b1.y - S1 * b2.y));
    v0 = gadd(v0, gadd(a1, a2));
    v1 = gadd(p1, q1);
    v4 = gsub(p1, q1);
    v2 = gadd(p2, q2);
    v3 = gsub(p2, q2);
}
// a * exp(2 pi i (c, s as cosine and sine))
__device__ __forceinline__ float2 grot(float2 a, float c, float s) {
    return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
}
__device__ __forceinline__ void gdft8(float2 *v) {
    constexpr float R2 = 0.70710678118654752440f;
    gdft4(v[0], v[2], v[4], v[6]);
    gdft4(v[1], v[3], v[5], v[7]);
    const float2 o1 = make_float2((v[3].x - v[3].y) * R2, (v[3].x + v[3].y) * R2);
    const float2 o2 = gmul_i(v[5]);
    const float2 o3 = make_float2((-v[7].x - v[7].y) * R2, (v[7].x - v[7].y) * R2);
    const float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
    v[0] = gadd(e0, o0);
    v[4] = gsub(e0, o0);
    v[1] = gadd(e1, o1);
    v[5] = gsub(e1, o1);
    v[2] = gadd(e2, o2);
    v[6] = gsub(e2, o2);
    v[3] = gadd(e3, o3);
    v[7] = gsub(e3, o3);
}
__device__ __forceinline__ void gdft6(float2 *v) {  // 2 x 3: even and odd inputs
    gdft3(v[0], v[2], v[4]);
    gdft3(v[1], v[3], v[5]);
    const float2 o1 = grot(v[3], 0.5f, 0.86602540378443864676f);
    const float2 o2 = grot(v[5], -0.5f, 0.86602540378443864676f);
    const float2 e0 = v[0], e1 = v[2], e2 = v[4], o0 = v[1];
    v[0] = gadd(e0, o0);
    v[3] = gsub(e0, o0);
    v[1] = gadd(e1, o1);
    v[4] = gsub(e1, o1);
    v[2] = gadd(e2, o2);
    v[5] = gsub(e2, o2);
}
__device__ __forceinline__ void gdft9(float2 *v) {  // 3 x 3
    gdft3(v[0], v[3], v[6]);
    gdft3(v[1], v[4], v[7]);
    gdft3(v[2], v[5], v[8]);
    // column m's output k times exp(2 pi i m k / 9)
    v[4] = grot(v[4], 0.76604444311897803520f, 0.64278760968653932632f);
    v[7] = grot(v[7], 0.17364817766693034885f, 0.98480775301220805937f);
    v[5] = grot(v[5], 0.17364817766693034885f, 0.98480775301220805937f);
    v[8] = grot(v[8], -0.93969262078590838405f, 0.34202014332566873304f);
    gdft3(v[0], v[1], v[2]);
    gdft3(v[3], v[4], v[5]);
    gdft3(v[6], v[7], v[8]);
    // output k + 3 m sits in v[3 k + m]
    const float2 a = v[1], b = v[2], c = v[5];
    v[1] = v[3];
    v[3] = a;
    v[2] = v[6];
    v[6] = b;
    v[5] = v[7];
    v[7] = c;
}
__device__ __forceinline__ void gdft10(float2 *v) {  // 2 x 5
    gdft5(v[0], v[2], v[4], v[6], v[8]);
    gdft5(v[1], v[3], v[5], v[7], v[9]);
    const float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], e4 = v[8], o0 = v[1];
    const float2 o1 = grot(v[3], 0.80901699437494742410f, 0.58778525229247312917f);
    const float2 o2 = grot(v[5], 0.30901699437494742410f, 0.95105651629515357212f);
    const float2 o3 = grot(v[7], -0.30901699437494742410f, 0.95105651629515357212f);
    const float2 o4 = grot(v[9], -0.80901699437494742410f, 0.58778525229247312917f);
    v[0] = gadd(e0, o0);
    v[5] = gsub(e0, o0);
    v[1] = gadd(e1, o1);
    v[6] = gsub(e1, o1);
    v[2] = gadd(e2, o2);
    v[7] = gsub(e2, o2);
    v[3] = gadd(e3, o3);
    v[8] = gsub(e3, o3);
    v[4] = gadd(e4, o4);
    v[9] = gsub(e4, o4);
}
__device__ __forceinline__ void gdft16(float2 *v) {  // 4 x 4
    constexpr float C1 = 0.92387953251128675613f, S1 = 0.38268343236508977173f;
    constexpr float R2 = 0.70710678118654752440f;
#pragma unroll
    for (int m = 0; m < 4; ++m) gdft4(v[m], v[m + 4], v[m + 8], v[m + 12]);
    // column m's output k (in v[m + 4 k]) times exp(2 pi i m k / 16)
    v[5] = grot(v[5], C1, S1);
    v[9] = grot(v[9], R2, R2);
    v[13] = grot(v[13], S1, C1);
    v[6] = grot(v[6], R2, R2);
    v[10] = gmul_i(v[10]);
    v[14] = grot(v[14], -R2, R2);
    v[7] = grot(v[7], S1, C1);
    v[11] = grot(v[11], -R2, R2);
    v[15] = grot(v[15], -C1, -S1);
#pragma unroll
    for (int k = 0; k < 4; ++k) gdft4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    // output k + 4 m sits in v[4 k + m]
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int m = 0; m < k; ++m) {
            const float2 t = v[4 * k + m];
            v[4 * k + m] = v[4 * m + k];
            v[4 * m + k] = t;
        }
}

template <int R>
__device__ __forceinline__ void gdft(float2 *v) {
    if constexpr (R == 2) gdft2(v[0], v[1]);
    else if constexpr (R == 3) gdft3(v[0], v[1], v[2]);
    else if constexpr (R == 4) gdft4(v[0], v[1], v[2], v[3]);
    else if constexpr (R == 5) gdft5(v[0], v[1], v[2], v[3], v[4]);
    else if constexpr (R == 6) gdft6(v);
    else if constexpr (R == 8) gdft8(v);
    else if constexpr (R == 9) gdft9(v);
    else if constexpr (R == 10) gdft10(v);
    else gdft16(v);
}

__device__ __forceinline__ int mode_at(int p, int n, int M, int hM) {
    return p < M - hM ? p + hM : (p >= n - hM ? p - (n - hM) : -1);
}

// Per-line state of a tile.
template <int TI>
struct Lines {
    int64_t ib[TI], ob[TI];  // bases; -1: past the last line
    int q[TI];
    int img[TI];             // bit 0: image at gqo, bit 1: at goo
};

template <int N, int NR>
__device__ __forceinline__ void bfly(int b, int contig, int &t, int &j) {
    constexpr int TI = Cfg<N>::TI;
    t = contig ? b / NR : b % TI;
    j = contig ? b % NR : b / TI;
}

template <int N, int KIND>
__device__ __forceinline__ void first_stage(const FgArgs &a, const Lines<Cfg<N>::TI> &ln,
                                            const float2 *__restrict__ in, float2 *buf) {
    using C = Cfg<N>;
    constexpr int R = C::R.r[0], NR = N / R, NB = NR * C::TI, T = C::T, F = (NB + T - 1) / T;
    float2 v[F][R];
    float d[F][R];
    uint32_t kept[F];  // bit r: value r is a kept mode
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const int b = threadIdx.x + f * T;
        int t, j;
        bfly<N, NR>(b < NB ? b : 0, a.icontig, t, j);
        const int64_t ib = b < NB ? ln.ib[t] : -1;
        if constexpr (KIND == FG_PAD) {
            const int q = ln.q[t];
            kept[f] = 0;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                // index 0 stands in where no mode is kept, so that every
                // load is issued at once; the value is dropped below
                const int m = mode_at((j + r * NR) * a.pstep + q, a.nfull, a.M, a.hM);
                const bool ok = ib >= 0 && m >= 0;
                v[f][r] = in[ok ? ib + (int64_t)m * a.ies : 0];
                d[f][r] = a.dec[ok ? m : 0];
                kept[f] |= (ok ? 1u : 0u) << r;
            }
        } else {
            // lines past the end read element 0, and are never stored
            const int64_t o = ib >= 0 ? ib + (int64_t)j * a.ies : 0, st = ib >= 0 ? NR * a.ies : 0;
#pragma unroll
            for (int r = 0; r < R; ++r) v[f][r] = in[o + r * st];
        }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const int b = threadIdx.x + f * T;
        if (b < NB) {
            int t, j;
            bfly<N, NR>(b, a.icontig, t, j);
            if constexpr (KIND == FG_CROP) {
                const int64_t ib = ln.ib[t];
                if (a.ghost && ib >= 0) {
                    const int im = ln.img[t];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int l = j + r * NR;
                        const bool gz = l < a.ge;
                        if (im | (int)gz) {
                            float2 x = v[f][r];
                            if (gz) x = gadd(x, in[ib + l + N]);
                            for (int k = 1; k < 4; ++k)
                                if ((im & k) == k) {
                                    const int64_t o = ib + l + ((k & 1) ? a.gqo : 0) +
                                                      ((k & 2) ? a.goo : 0);
                                    x = gadd(x, in[o]);
                                    if (gz) x = gadd(x, in[o + N]);
                                }
                            v[f][r] = x;
                        }
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (KIND == FG_PAD)
                    v[f][r] = (kept[f] >> r) & 1u ? gscale(v[f][r], d[f][r]) : make_float2(0.f, 0.f);
                v[f][r].y *= a.sg;
            }
            gdft<R>(v[f]);
            float2 *w = buf + j * R * C::PI + t;
#pragma unroll
            for (int r = 0; r < R; ++r) w[r * C::PI] = v[f][r];
        }
    }
    __syncthreads();
}

// Middle stage s (LDS to LDS, in place: every butterfly is read before the
// barrier and written after it); tw[m] = exp(2 pi i m / N).
template <int N, int S>
__device__ __forceinline__ void middle_stages(float2 *buf, const float2 *tw) {
    using C = Cfg<N>;
    if constexpr (S + 1 < C::R.k) {
        constexpr int R = C::R.r[S], NR = N / R, NB = NR * C::TI, T = C::T, F = (NB + T - 1) / T;
        constexpr int Ns = C::ns(S), TS = N / (Ns * R);
        float2 v[F][R];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int b = threadIdx.x + f * T;
            if (b < NB) {
                const int t = b % C::TI, j = b / C::TI, k = j % Ns;
                const float2 *p = buf + j * C::PI + t;
#pragma unroll
                for (int r = 0; r < R; ++r) v[f][r] = p[r * NR * C::PI];
#pragma unroll
                for (int r = 1; r < R; ++r) v[f][r] = gmul(v[f][r], tw[k * r * TS]);
                gdft<R>(v[f]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int b = threadIdx.x + f * T;
            if (b < NB) {
                const int t = b % C::TI, j = b / C::TI, k = j % Ns;
                float2 *p = buf + ((j - k) * R + k) * C::PI + t;
#pragma unroll
                for (int r = 0; r < R; ++r) p[r * Ns * C::PI] = v[f][r];
            }
        }
        __syncthreads();
        middle_stages<N, S + 1>(buf, tw);
    }
}

template <int N, int KIND>
__device__ __forceinline__ void last_stage(const FgArgs &a, const Lines<Cfg<N>::TI> &ln,
                                           const float2 *buf, const float2 *tw,
                                           float2 *__restrict__ out) {
    using C = Cfg<N>;
    constexpr int R = C::R.r[C::R.k - 1], NR = N / R, NB = NR * C::TI, T = C::T;
    constexpr int F = (NB + T - 1) / T;
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const int b = threadIdx.x + f * T;
        if (b >= NB) break;
        int t, j;
        bfly<N, NR>(b, a.ocontig, t, j);
        const int64_t ob = ln.ob[t];
        const int q = ln.q[t];
        int im[R];
        float dm[R];
        if constexpr (KIND == FG_CROP) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                im[r] = mode_at((j + r * NR) * a.pstep + q, a.nfull, a.M, a.hM);
                dm[r] = a.dec[im[r] >= 0 ? im[r] : 0];
            }
        }
        float2 v[R];
        const float2 *p = buf + j * C::PI + t;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = p[r * NR * C::PI];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = gmul(v[r], tw[j * r]);
        gdft<R>(v);
        if (KIND != FG_CROP && a.ntw) {
            // exp(2 pi i k q / ntw), k q < ntw, from fp64
#pragma unroll
            for (int r = 0; r < R; ++r) {
                double sn, cs;
                sincospi(2.0 * (double)((j + r * NR) * q) / (double)a.ntw, &sn, &cs);
                v[r] = grot(v[r], (float)cs, (float)sn);
            }
        }
        if (ob < 0) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r].y *= a.sg;
        if constexpr (KIND == FG_CROP) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (im[r] >= 0) out[ob + (int64_t)im[r] * a.oes] = gscale(v[r], dm[r]);
        } else {
            const int64_t o = ob + (int64_t)j * a.oes, st = NR * a.oes;
#pragma unroll
            for (int r = 0; r < R; ++r) out[o + r * st] = v[r];
            if (KIND == FG_PAD && a.ghost) {
                const int g = ln.img[t];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int l = j + r * NR;
                    const bool gz = l < a.ge;
                    if (g | (int)gz) {
                        if (gz) out[ob + l + N] = v[r];
                        for (int k = 1; k < 4; ++k)
                            if ((g & k) == k) {
                                const int64_t i = ob + l + ((k & 1) ? a.gqo : 0) +
                                                  ((k & 2) ? a.goo : 0);
                                out[i] = v[r];
                                if (gz) out[i + N] = v[r];
                            }
                    }
                }
            }
        }
    }
}

template <int N, int KIND>
__global__ __launch_bounds__(Cfg<N>::T) void k_fftg(const float2 *__restrict__ in,
                                                    float2 *__restrict__ out,
                                                    const float2 *__restrict__ twg, FgArgs a) {
    using C = Cfg<N>;
    extern __shared__ float2 fg_lds[];
    __shared__ Lines<C::TI> ln;
    float2 *tw = fg_lds + N * C::PI;
    const int tid = threadIdx.x;
    const int64_t ntile = (a.nlines + C::TI - 1) / C::TI;
    const int64_t line0 = xcd_remap(blockIdx.x, ntile) * C::TI;
    for (int m = tid; m < N; m += C::T) tw[m] = twg[m];
    if (tid < C::TI) {
        const int64_t line = line0 + tid;
        const int64_t o = line / a.ni, i = line - o * a.ni;
        const int64_t q = i / a.inner, r = i - q * a.inner;
        const int64_t oh = o / a.oc, ol = o - oh * a.oc;
        const bool ok = line < a.nlines;
        ln.ib[tid] = ok ? oh * a.ib1 + ol * a.ib2 + q * a.ibq + r : -1;
        ln.ob[tid] = ok ? oh * a.ob1 + ol * a.ob2 + q * a.obq + r : -1;
        ln.q[tid] = a.useq ? (int)q : 0;
        ln.img[tid] = a.ghost ? ((q < a.gq ? 1 : 0) | (ol < a.go ? 2 : 0)) : 0;
    }
    __syncthreads();
    first_stage<N, KIND>(a, ln, in, fg_lds);
    middle_stages<N, 1>(fg_lds, tw);
    last_stage<N, KIND>(a, ln, fg_lds, tw, out);
}

template <int N>
FgEntry entry() {
    using C = Cfg<N>;
    static_assert(C::R.k >= 2, "two stages at least");
    return FgEntry{N, C::TI, C::T, C::LDS, {k_fftg<N, FG_CROP>, k_fftg<N, FG_PAD>, k_fftg<N, FG_MID>}};
}

}  // namespace fg
}  // namespace mn
