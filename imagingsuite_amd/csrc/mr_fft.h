// LDS-resident Stockham FFT for one complex line of compile-time length P,
// shared by the parallel-beam and the FDK ramp filters.
//
// The line lives in LDS as float2, padded (lpad); every pass reads its butterfly
// inputs into registers, synchronises, and writes the outputs back in natural
// (Stockham autosort) order, so no bit reversal is needed.  Twiddles come from a
// P-entry table tw[k] = exp(-2 pi i k / P) computed in double on the host.
#pragma once

#include <hip/hip_runtime.h>

namespace mr {

constexpr int ilog2c(int v) { return v <= 1 ? 0 : 1 + ilog2c(v >> 1); }

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, -a.y * b.y), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// ---------------------------------------------------------------------------
// Radix-8 Stockham passes (one radix-2 or radix-4 pass first
// when log2 P is not a multiple of 3), so P = 8192 takes 5 passes instead of
// 7.  The line is stored with one pad entry every 16 (index lpad(i)), which
// spreads the strided writes of the early passes over all LDS banks.  The
// twiddles come from an LDS copy of the first P/8 entries of the table
// (w = exp(-+2 pi i base / P), base < P/8 in every radix-8 pass); the other
// six powers of a butterfly are products of w (at most three multiplications
// deep).  Length of the padded line: lds_len(P).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lpad(int i) { return i + (i >> 4); }
constexpr int lds_len(int P) { return P + P / 16; }

template <bool INV>
__device__ __forceinline__ void dft4(float2 &v0, float2 &v1, float2 &v2, float2 &v3)
{
    const float2 a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3), d = csub(v1, v3);
    const float2 a3 = INV ? make_float2(-d.y, d.x) : make_float2(d.y, -d.x);
    v0 = cadd(a0, a2);
    v2 = csub(a0, a2);
    v1 = cadd(a1, a3);
    v3 = csub(a1, a3);
}

template <int R, bool INV>
__device__ __forceinline__ void dft_r(float2 (&v)[R])
{
    if constexpr (R == 2) {
        const float2 t = v[0];
        v[0] = cadd(t, v[1]);
        v[1] = csub(t, v[1]);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else {
        constexpr float c = 0.70710678118654752440f;
        float2 a[4], b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            a[r] = cadd(v[r], v[r + 4]);
            b[r] = csub(v[r], v[r + 4]);
        }
        // b_r *= exp(-+2 pi i r / 8)
        b[1] = INV ? make_float2(c * (b[1].x - b[1].y), c * (b[1].x + b[1].y))
                   : make_float2(c * (b[1].x + b[1].y), c * (b[1].y - b[1].x));
        b[2] = INV ? make_float2(-b[2].y, b[2].x) : make_float2(b[2].y, -b[2].x);
        b[3] = INV ? make_float2(-c * (b[3].x + b[3].y), c * (b[3].x - b[3].y))
                   : make_float2(c * (b[3].y - b[3].x), -c * (b[3].x + b[3].y));
        dft4<INV>(a[0], a[1], a[2], a[3]);
        dft4<INV>(b[0], b[1], b[2], b[3]);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            v[2 * m] = a[m];
            v[2 * m + 1] = b[m];
        }
    }
}

// Filter of the line: forward transform, product with the spectrum hs, inverse
// transform.  load(j, v) gives butterfly j of the first pass its R inputs j + r
// P/R, store(q, j, v) takes the results j + r P/8 of butterfly j of the last
// pass, the thread's q-th: functors for all of a butterfly's points, so that
// their memory accesses are in flight together, and no LDS round trip (and its
// barriers) of their own.  The spectrum multiplies the last forward pass's
// outputs.  after_load() runs between the inputs' loads and the first exchange,
// before_store(q, j) ahead of the last pass.  STORE_LDS: store writes the LDS
// line.
template <int P, int NT, int R, int NS, bool INV, class Load, class AfterLoad, class Sync, class Put>
__device__ __forceinline__ void fft_pass_io(const float2 *__restrict__ twl, Load load, AfterLoad after_load, Sync sync,
                                            Put put)
{
    constexpr int B = P / R, PER = (B + NT - 1) / NT, LR = ilog2c(R), L = ilog2c(P), LNS = ilog2c(NS);
    const int t = threadIdx.x;
    float2 v[PER][R];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) load(j, v[q]);
    }
    after_load();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) {
            if (R == 8 && NS > 1) {
                const int k = j & (NS - 1);
                float2 w1 = twl[k << (L - 3 - LNS)];
                if (INV) w1.y = -w1.y;
                const float2 w2 = cmul(w1, w1), w3 = cmul(w1, w2), w4 = cmul(w2, w2);
                const float2 w5 = cmul(w1, w4), w6 = cmul(w3, w3), w7 = cmul(w3, w4);
                const float2 w[8] = {make_float2(1.f, 0.f), w1, w2, w3, w4, w5, w6, w7};
#pragma unroll
                for (int r = 1; r < R; ++r) v[q][r] = cmul(v[q][r], w[r]);
            }
            dft_r<R, INV>(v[q]);
        }
    }
    sync();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) put(q, j, ((j >> LNS) << (LNS + LR)) + (j & (NS - 1)), v[q]);
    }
}

// passes NS, 8 NS, ... up to but not including the last, LDS to LDS
template <int P, int NT, int NS, bool INV>
__device__ __forceinline__ void fft_mid_passes(float2 *a, const float2 *__restrict__ twl)
{
    if constexpr (NS * 8 < P) {
        auto load = [&](int j, float2 (&v)[8]) {
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = a[lpad(j + r * (P / 8))];
        };
        auto put = [&](int, int, int d0, float2 (&v)[8]) {
#pragma unroll
            for (int r = 0; r < 8; ++r) a[lpad(d0 + r * NS)] = v[r];
        };
        fft_pass_io<P, NT, 8, NS, INV>(twl, load, [] {}, [] { __syncthreads(); }, put);
        __syncthreads();
        fft_mid_passes<P, NT, NS * 8, INV>(a, twl);
    }
}

template <int P, int NT, bool STORE_LDS, class Load, class AfterLoad, class BeforeStore, class Store>
__device__ __forceinline__ void fft_filter(float2 *a, const float2 *__restrict__ tw, const float *__restrict__ hs,
                                           Load load, AfterLoad after_load, BeforeStore before_store, Store store)
{
    constexpr int L = ilog2c(P), FIRST = L % 3 == 1 ? 2 : (L % 3 == 2 ? 4 : 8), B = P / 8;   // FIRST: radix
    constexpr int PER = (B + NT - 1) / NT;
    static_assert(P > FIRST, "two passes or more");
    const int t = threadIdx.x;
    float2 *twl = a + lds_len(P);
    for (int i = t; i < P / 8; i += NT) twl[i] = tw[i];   // read behind the first pass's barrier
    auto nothing = [] {};
    auto barrier = [] { __syncthreads(); };
    auto from_lds = [&](int j, auto &v) {
        constexpr int R = sizeof(v) / sizeof(float2);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = a[lpad(j + r * (P / R))];
    };
    auto first_put = [&](int, int, int d0, auto &v) {
        constexpr int R = sizeof(v) / sizeof(float2);
#pragma unroll
        for (int r = 0; r < R; ++r) a[lpad(d0 + r)] = v[r];
    };
    fft_pass_io<P, NT, FIRST, 1, false>(twl, load, after_load, nothing, first_put);
    __syncthreads();
    fft_mid_passes<P, NT, FIRST, false>(a, twl);
    // ahead of its use where the registers allow
    constexpr bool AHEAD = P <= 4096;
    float h[PER][8];
    auto fetch = [&](int q, int j) {
#pragma unroll
        for (int r = 0; r < 8; ++r) h[q][r] = hs[j + r * B];
    };
#pragma unroll
    for (int q = 0; AHEAD && q < PER; ++q) fetch(q, min(t + q * NT, B - 1));
    auto spectrum = [&](int q, int j, int, float2 (&v)[8]) {
        if (!AHEAD) fetch(q, j);
#pragma unroll
        for (int r = 0; r < 8; ++r) a[lpad(j + r * B)] = make_float2(v[r].x * h[q][r], v[r].y * h[q][r]);
    };
    fft_pass_io<P, NT, 8, B, false>(twl, from_lds, nothing, barrier, spectrum);
    __syncthreads();
    fft_pass_io<P, NT, FIRST, 1, true>(twl, from_lds, nothing, barrier, first_put);
    __syncthreads();
    fft_mid_passes<P, NT, FIRST, true>(a, twl);
#pragma unroll
    for (int q = 0; AHEAD && q < PER; ++q) before_store(q, min(t + q * NT, B - 1));
    auto last = [&](int q, int j, int, float2 (&v)[8]) {
        if (!AHEAD) before_store(q, j);
        store(q, j, v);
    };
    if constexpr (STORE_LDS) {
        fft_pass_io<P, NT, 8, B, true>(twl, from_lds, nothing, barrier, last);
        __syncthreads();
    } else {
        fft_pass_io<P, NT, 8, B, true>(twl, from_lds, nothing, nothing, last);
    }
}

}  // namespace mr
