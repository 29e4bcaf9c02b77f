// LDS-resident FFT filter of one complex line of compile-time length P, shared
// by the parallel-beam and the FDK ramp filters: forward transform, product
// with a real spectrum, inverse transform.
//
// Radix-8 stages, each in place: a thread reads eight points of the line into
// registers and writes its results to the same eight places.  The forward
// stages decimate in frequency (span P, P/8, ...), the inverse ones in time
// (back up), so the spectrum is met in digit-reversed order, where its product
// and the stages on either side of it are one pass over registers: no
// reordering, and one exchange through LDS per stage boundary.  The line's
// remaining factor 2 or 4 is that middle stage.
//
// A stage of span N works on runs of N points by N / 8 consecutive threads, so
// from span 512 down a run stays within one wave and needs no block barrier:
// P = 4096 has two (after the first and before the last stage).
//
// Bank conflicts: point i lies at i ^ ((i >> 3) & 31).  In every stage the five
// index bits that vary over 32 consecutive lanes (bits 0 .. 4 for a stride of
// 32 or more, the low bits and those above the three stage bits for smaller
// ones, bits 3 .. 7 in the middle stage) then reach all 32 pairs of banks.
//
// Twiddles: powers 1, 2 and 4 of each stage are table entries (in double on the
// host, coalesced loads ahead of the stage's exchange), the others products of
// them.  A filtered row is small beside its input where a ramp meets smooth
// data, so the twiddles' errors count: with all powers made from the first the
// result is 1.6 to 2 times further from double than with these (rows of 2048:
// 2.1e-5 against 1.2e-5 of the result, all seven from a table 1.1e-5).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace mr {

constexpr int ilog2c(int v) { return v <= 1 ? 0 : 1 + ilog2c(v >> 1); }

// Stages of the P-point line: kFftStages(P) of radix 8 with a twiddle, then the
// middle stage of radix fft_mid(P).
constexpr int fft_mid(int P) { return ilog2c(P) % 3 == 0 ? 8 : 1 << (ilog2c(P) % 3); }
constexpr int fft_stages(int P) { return ilog2c(P / fft_mid(P)) / 3; }
// Table offset of stage s: spans P, P/8, ... with 3 x span / 8 entries each.
constexpr int fft_tw_offset(int P, int s) { return s == 0 ? 0 : fft_tw_offset(P, s - 1) + 3 * (P >> (3 * s)); }
// Frequency of point p of the digit-reversed line.
constexpr int fft_frequency(int P, int p)
{
    int f = 0, scale = 1, span = P;
    for (int s = 0; s < fft_stages(P); ++s, scale *= 8, span /= 8) f += scale * (p / (span / 8) % 8);
    return f + scale * (p % fft_mid(P));
}

__host__ __device__ constexpr int fft_swz(int i) { return i ^ ((i >> 3) & 31); }

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, -a.y * b.y), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

template <int N, class F> __device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

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

// a b, or a times the conjugate of b
template <bool CONJ> __device__ __forceinline__ float2 cmul_or_conj(float2 a, float2 b)
{
    if (!CONJ) return cmul(a, b);
    return make_float2(__builtin_fmaf(a.x, b.x, a.y * b.y), __builtin_fmaf(a.y, b.x, -a.x * b.y));
}

// v[m] w^m from the powers 1, 2 and 4 (CONJ: of the conjugate)
template <bool CONJ> __device__ __forceinline__ void twiddle8(float2 (&v)[8], const float2 (&w)[3])
{
    const float2 w3 = cmul(w[0], w[1]);
    v[1] = cmul_or_conj<CONJ>(v[1], w[0]);
    v[2] = cmul_or_conj<CONJ>(v[2], w[1]);
    v[3] = cmul_or_conj<CONJ>(v[3], w3);
    v[4] = cmul_or_conj<CONJ>(v[4], w[2]);
    v[5] = cmul_or_conj<CONJ>(v[5], cmul(w[0], w[2]));
    v[6] = cmul_or_conj<CONJ>(v[6], cmul(w[1], w[2]));
    v[7] = cmul_or_conj<CONJ>(v[7], cmul(w3, w[2]));
}

// the first stage's transform when points 4 .. 7 are zero
__device__ __forceinline__ void dft8_half(float2 (&v)[8])
{
    constexpr float c = 0.70710678118654752440f;
    float2 a[4] = {v[0], v[1], v[2], v[3]};
    float2 b[4] = {v[0], make_float2(c * (v[1].x + v[1].y), c * (v[1].y - v[1].x)), make_float2(v[2].y, -v[2].x),
                   make_float2(c * (v[3].y - v[3].x), -c * (v[3].x + v[3].y))};
    dft4<false>(a[0], a[1], a[2], a[3]);
    dft4<false>(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        v[2 * m] = a[m];
        v[2 * m + 1] = b[m];
    }
}

// Orders a stage's exchange among T consecutive threads.
template <int T> __device__ __forceinline__ void fft_sync()
{
    if constexpr (T > 64) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// The eight points of butterfly j in the stage of stride T (span 8 T).
template <int T> struct FftPoints {
    int base;
    __device__ __forceinline__ explicit FftPoints(int j) : base(fft_swz((j / T) * (8 * T) + (j & (T - 1)))) {}
    // index bits of base and r T are disjoint, and fft_swz is linear in them
    __device__ __forceinline__ int operator()(int r) const { return T >= 256 ? base + r * T : base ^ fft_swz(r * T); }
};

// Filter of the line.  load(j, v) gives inputs j + r P/8 in v[r], store(q, j, v)
// takes those results (HALF: r < 4; the other inputs are zero and the other
// results not wanted) of butterfly j, the thread's q-th; a functor for all of a
// thread's points can have its loads in flight together.  after_load() runs
// between the inputs' loads and the first exchange, before_store(q, j) ahead of
// the last one.  tw: the stages' tables; hs: the spectrum in the order of
// spectrum_order().
template <int P, int NT, bool HALF, class Load, class AfterLoad, class BeforeStore, class Store>
__device__ __forceinline__ void fft_filter(float2 *a, const float2 *__restrict__ tw, const float *__restrict__ hs,
                                           Load load, AfterLoad after_load, BeforeStore before_store, Store store)
{
    constexpr int B = P / 8, PER = (B + NT - 1) / NT, S = fft_stages(P), R = fft_mid(P);
    const int t = threadIdx.x;
    // the twiddles of the next stage, requested ahead of its exchange
    float2 w[PER][3];
    auto fetch = [&](auto sc) {
        constexpr int s = decltype(sc)::value, T = B >> (3 * s);
#pragma unroll
        for (int q = 0; q < PER; ++q)
#pragma unroll
            for (int m = 0; m < 3; ++m) w[q][m] = tw[fft_tw_offset(P, s) + m * T + ((t + q * NT) & (T - 1))];
    };
    fetch(std::integral_constant<int, 0>{});
    float2 v[8];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) {
            load(j, v);
            if constexpr (HALF) dft8_half(v);
            else dft_r<8, false>(v);
            twiddle8<false>(v, w[q]);
            const FftPoints<B> at(j);
#pragma unroll
            for (int r = 0; r < 8; ++r) a[at(r)] = v[r];
        }
    }
    after_load();
    float h[PER][8];
    auto next = [&](auto sc) {   // what follows forward stage s - 1
        constexpr int s = decltype(sc)::value;
        if constexpr (s < S) fetch(sc);
        else
#pragma unroll
            for (int q = 0; q < PER; ++q)
#pragma unroll
                for (int r = 0; r < 8; ++r) h[q][r] = hs[r * B + min(t + q * NT, B - 1)];
    };
    next(std::integral_constant<int, 1>{});
    fft_sync<B>();
    static_for<S - 1>([&](auto sc) {
        constexpr int s = decltype(sc)::value + 1, T = B >> (3 * s);
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int j = t + q * NT;
            if (j < B) {
                const FftPoints<T> at(j);
#pragma unroll
                for (int r = 0; r < 8; ++r) v[r] = a[at(r)];
                dft_r<8, false>(v);
                twiddle8<false>(v, w[q]);
#pragma unroll
                for (int r = 0; r < 8; ++r) a[at(r)] = v[r];
            }
        }
        next(std::integral_constant<int, s + 1>{});
        fft_sync<T>();
    });
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) {
            const FftPoints<1> at(j);
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = a[at(r)];
#pragma unroll
            for (int g = 0; g < 8; g += R) {
                float2 x[R];
#pragma unroll
                for (int r = 0; r < R; ++r) x[r] = v[g + r];
                dft_r<R, false>(x);
#pragma unroll
                for (int r = 0; r < R; ++r) x[r] = make_float2(x[r].x * h[q][g + r], x[r].y * h[q][g + r]);
                dft_r<R, true>(x);
#pragma unroll
                for (int r = 0; r < R; ++r) a[at(g + r)] = x[r];
            }
        }
    }
    static_for<S - 1>([&](auto sc) {
        constexpr int s = S - 1 - decltype(sc)::value, T = B >> (3 * s);
        fetch(std::integral_constant<int, s>{});
        fft_sync<T>();
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int j = t + q * NT;
            if (j < B) {
                const FftPoints<T> at(j);
#pragma unroll
                for (int r = 0; r < 8; ++r) v[r] = a[at(r)];
                twiddle8<true>(v, w[q]);
                dft_r<8, true>(v);
#pragma unroll
                for (int r = 0; r < 8; ++r) a[at(r)] = v[r];
            }
        }
    });
    fetch(std::integral_constant<int, 0>{});
#pragma unroll
    for (int q = 0; q < PER; ++q) before_store(q, min(t + q * NT, B - 1));
    fft_sync<B>();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int j = t + q * NT;
        if (j < B) {
            const FftPoints<B> at(j);
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = a[at(r)];
            twiddle8<true>(v, w[q]);
            dft_r<8, true>(v);
            store(q, j, v);
        }
    }
}

}  // namespace mr
