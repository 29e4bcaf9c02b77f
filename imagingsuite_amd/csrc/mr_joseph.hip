// Matched Joseph projector pair for parallel beam on gfx950: forward A and
// its exact adjoint A^T.  No reference counterpart exists (the reference's
// LinearForwardProjector, frameworks/tomography/Framework/ReconAlgorithms/
// ReconAlgorithms/linearforwardprojector.cpp:15-143, is 2-D only and is not
// the adjoint of any back-projector); the geometry is the one of the
// reference's parallel-beam back-projector (StdBackProjectorBase.cpp:73-80):
//   u(x, y) = center + cos(phi) (y + 1 - c) - sin(phi) (x + 1 - c),  c = nx / 2.
//
// With m = max(|sin phi|, |cos phi|) both operators use the same kernel
//   K(t) = max(0, 1 - |t| / m) / m,
// A[phi][n][z]  = sum_{x,y} K(u(x,y) - n) vol[y][x][z]   (ray-driven Joseph
//                 stepping along the axis the ray is closest to: linear
//                 interpolation between the two nearest voxels, step 1/m)
// AT[y][x][z]   = sum_{phi,n} K(u(x,y) - n) sino[phi][n][z]   (voxel-driven:
//                 the two detector bins around u with weights K)
// so A^T is the transpose of A in exact arithmetic.
//
// Layout: volume [nx(y)][nx(x)][nz] (MatrixZXY), sinogram [n_ang][n_det][nz]
// (slice fastest).  Each thread owns ZT slices held as float4 vectors.
#include "mr_common.h"
#include "mr_filter.h"
#include "mr_joseph.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

namespace mr {

struct JosephArgs {
    const float *src;
    float *dst;
    const float4 *tab;  // per angle: (su, cos, sin, 1/m)   su = c (sin - cos) + center
    int nx, nz, nd, na;
};

// Loads below are never predicated: out-of-volume neighbours read a clamped,
// valid address with weight zero, so the compiler can keep the loads of
// several unrolled steps in flight together.
template <int ZT>
__device__ __forceinline__ void lerp_accumulate(float (&acc)[ZT], const float *p0, const float *p1, float w0,
                                                float w1)
{
#pragma unroll
    for (int g = 0; g < ZT / 4; ++g) {
        const float4 v0 = *reinterpret_cast<const float4 *>(p0 + 4 * g);
        const float4 v1 = *reinterpret_cast<const float4 *>(p1 + 4 * g);
        acc[4 * g + 0] = __builtin_fmaf(w1, v1.x, __builtin_fmaf(w0, v0.x, acc[4 * g + 0]));
        acc[4 * g + 1] = __builtin_fmaf(w1, v1.y, __builtin_fmaf(w0, v0.y, acc[4 * g + 1]));
        acc[4 * g + 2] = __builtin_fmaf(w1, v1.z, __builtin_fmaf(w0, v0.z, acc[4 * g + 2]));
        acc[4 * g + 3] = __builtin_fmaf(w1, v1.w, __builtin_fmaf(w0, v0.w, acc[4 * g + 3]));
    }
}

// Range [lo, hi) of the step index t = 0..N-1 for which the crossing
// position q(t) = A + B t can fall in [-1, N) (where a voxel pair gets a
// nonzero weight), widened by two steps against rounding; the loop body
// still tests every step exactly.
__device__ __forceinline__ void step_range(float A, float B, int N, int &lo, int &hi)
{
    lo = 0;
    hi = N;
    if (fabsf(B) > 1e-20f) {
        float t1 = (-1.0f - A) / B, t2 = ((float)N - A) / B;
        if (t1 > t2) {
            const float tmp = t1;
            t1 = t2;
            t2 = tmp;
        }
        lo = max(0, (int)fmaxf(floorf(t1) - 2.0f, -1.0f));
        hi = min(N, (int)fminf(ceilf(t2) + 2.0f, (float)N));
    } else if (A < -1.0f || A >= (float)N) {
        hi = 0;
    }
}

// Forward: one thread per (angle, bin) and ZT slices.
template <int ZT>
__global__ __launch_bounds__(256) void joseph_forward_kernel(JosephArgs a)
{
    const int n = blockIdx.x * 64 + (threadIdx.x & 63);
    const int ang = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int z0 = blockIdx.z * ZT;
    if (n >= a.nd || ang >= a.na) return;
    const float4 t = a.tab[ang];
    const float su = t.x, c = t.y, s = t.z, inv_m = t.w;
    const int N = a.nx;
    float acc[ZT];
#pragma unroll
    for (int z = 0; z < ZT; ++z) acc[z] = 0.0f;
    const float fn = (float)n;
    if (fabsf(s) >= fabsf(c)) {
        // step over rows y: x(y) solves u(x, y) = n
        const float inv_s = 1.0f / s;
        int lo, hi;
        step_range((su + c - fn) * inv_s - 1.0f, c * inv_s, N, lo, hi);
#pragma unroll 2
        for (int y = lo; y < hi; ++y) {
            const float xf = (su + c * (float)(y + 1) - fn) * inv_s - 1.0f;
            const float fl = floorf(xf);
            const int x0 = (int)fl;
            const float f = xf - fl;
            const float w0 = (x0 >= 0 && x0 < N) ? 1.0f - f : 0.0f;
            const float w1 = (x0 + 1 >= 0 && x0 + 1 < N) ? f : 0.0f;
            const int xa = min(max(x0, 0), N - 1), xb = min(max(x0 + 1, 0), N - 1);
            const float *row = a.src + ((size_t)y * N) * a.nz + z0;
            lerp_accumulate<ZT>(acc, row + (size_t)xa * a.nz, row + (size_t)xb * a.nz, w0, w1);
        }
    } else {
        // step over columns x: y(x) solves u(x, y) = n
        const float inv_c = 1.0f / c;
        int lo, hi;
        step_range((fn - su + s) * inv_c - 1.0f, s * inv_c, N, lo, hi);
#pragma unroll 2
        for (int x = lo; x < hi; ++x) {
            const float yf = (fn - su + s * (float)(x + 1)) * inv_c - 1.0f;
            const float fl = floorf(yf);
            const int y0 = (int)fl;
            const float f = yf - fl;
            const float w0 = (y0 >= 0 && y0 < N) ? 1.0f - f : 0.0f;
            const float w1 = (y0 + 1 >= 0 && y0 + 1 < N) ? f : 0.0f;
            const int ya = min(max(y0, 0), N - 1), yb = min(max(y0 + 1, 0), N - 1);
            const float *col = a.src + (size_t)x * a.nz + z0;
            lerp_accumulate<ZT>(acc, col + (size_t)ya * N * a.nz, col + (size_t)yb * N * a.nz, w0, w1);
        }
    }
    float *out = a.dst + ((size_t)ang * a.nd + n) * a.nz + z0;
#pragma unroll
    for (int g = 0; g < ZT / 4; ++g)
        *reinterpret_cast<float4 *>(out + 4 * g) =
            make_float4(acc[4 * g] * inv_m, acc[4 * g + 1] * inv_m, acc[4 * g + 2] * inv_m, acc[4 * g + 3] * inv_m);
}

// LDS-staged forward over a chunk of angles that all step along the same
// axis (class 0: |sin| >= |cos|, rows y; class 1: columns x).  A block owns
// kFwdNB detector bins x (up to) kFwdKA angles x ZT slices, one ray per
// thread.  It walks the lines L = 0..N-1 of its class R at a time: for
// each line it stages the kFwdW voxels (x ZT slices) from the lowest crossing
// of any of its rays, then every ray interpolates its two voxels from LDS.
// Staged positions outside the volume are zeros and carry weight zero, so the
// sums are those of the direct kernel, accumulated over the same lines in
// the same order.  Neighbouring angles cross a line close together, so one
// staged segment serves all the chunk's rays: the volume is read once per
// chunk instead of once per angle.  The host builds the chunks so that every
// line's crossings of a block fit in kFwdW - 2 voxels.
constexpr int kFwdNB = 16, kFwdKA = 16, kFwdR = 1, kFwdW = 80;

template <int ZT, int R>
__global__ __launch_bounds__(256) void joseph_forward_lds_kernel(JosephArgs a, const int4 *__restrict__ chunks,
                                                                 const int *__restrict__ order, int n_chunks,
                                                                 int nbt, int nzs)
{
    constexpr int NB = kFwdNB, W = kFwdW, RS = ZT + 4, G = ZT / 4;
    __shared__ float seg[R][W][RS];
    __shared__ int lo_s[R], hi_s[R];
    const int total = n_chunks * nbt * nzs;
    const int per = (total + 7) >> 3;
    const int b = (int)blockIdx.x;
    const int wi = (b & 7) * per + (b >> 3);   // XCD b % 8 takes the (b % 8)-th eighth
    if (wi >= total) return;
    const int bt = wi % nbt;
    const int rest = wi / nbt;
    const int ci = rest % n_chunks;
    const int zs = rest / n_chunks;
    const int4 ch = chunks[ci];                // first, count, class
    const int ai = threadIdx.x / NB, bi = threadIdx.x % NB;
    const int n = bt * NB + bi;
    const bool active = ai < ch.y && n < a.nd;
    const bool edge = active && (bi == 0 || bi == NB - 1 || n == a.nd - 1);
    const int ang = order[ch.x + min(ai, ch.y - 1)];
    const float4 t = a.tab[ang];
    const float su = t.x, c = t.y, s = t.z, inv_m = t.w;
    const int N = a.nx;
    const int z0 = zs * ZT;
    const bool rows = ch.z == 0;
    // crossing of line L: ((a0 + b1 (L+1)) + cn) * inv - 1
    const float a0 = rows ? su : -su, b1 = rows ? c : s;
    const float fn = (float)n;
    const float cn = rows ? -fn : fn;
    const float inv = rows ? 1.0f / s : 1.0f / c;
    const size_t strideL = rows ? (size_t)N * a.nz : (size_t)a.nz;
    const size_t strideP = rows ? (size_t)a.nz : (size_t)N * a.nz;
    float acc[ZT];
#pragma unroll
    for (int z = 0; z < ZT; ++z) acc[z] = 0.0f;
    for (int L0 = 0; L0 < N; L0 += R) {
        if (threadIdx.x < R) {
            lo_s[threadIdx.x] = 0x7fffffff;
            hi_s[threadIdx.x] = -0x7fffffff;
        }
        __syncthreads();
        if (edge) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float pf = ((a0 + b1 * (float)(L0 + r + 1)) + cn) * inv - 1.0f;
                const int p0 = (int)floorf(pf);
                atomicMin(&lo_s[r], p0);
                atomicMax(&hi_s[r], p0);
            }
        }
        __syncthreads();
        // the group is skipped when no ray crosses the volume on its lines
        bool any = false;
#pragma unroll
        for (int r = 0; r < R; ++r)
            any = any || (L0 + r < N && hi_s[r] >= -1 && lo_s[r] < N);
        if (any) {
            // only the voxels a line's rays read: lo .. hi + 1
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int L = L0 + r, lo = lo_s[r], nj = min(hi_s[r] - lo + 2, W);
                const float *line = a.src + (size_t)min(L, N - 1) * strideL + z0;
                for (int e = threadIdx.x; e < nj * G; e += 256) {
                    const int j = e / G, g = e - j * G;
                    const int p = lo + j;
                    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    if (L < N && p >= 0 && p < N)
                        v = *reinterpret_cast<const float4 *>(line + (size_t)p * strideP + 4 * g);
                    *reinterpret_cast<float4 *>(&seg[r][j][4 * g]) = v;
                }
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (L0 + r < N) {
                    const float pf = ((a0 + b1 * (float)(L0 + r + 1)) + cn) * inv - 1.0f;
                    const float fl = floorf(pf);
                    const int p0 = (int)fl;
                    const float f = pf - fl;
                    const float w0 = (p0 >= 0 && p0 < N) ? 1.0f - f : 0.0f;
                    const float w1 = (p0 + 1 >= 0 && p0 + 1 < N) ? f : 0.0f;
                    const int j = min(max(p0 - lo_s[r], 0), W - 2);
                    const float *v0 = &seg[r][j][0];
                    const float *v1 = v0 + RS;
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const float4 x0 = *reinterpret_cast<const float4 *>(v0 + 4 * g);
                        const float4 x1 = *reinterpret_cast<const float4 *>(v1 + 4 * g);
                        acc[4 * g + 0] = __builtin_fmaf(w1, x1.x, __builtin_fmaf(w0, x0.x, acc[4 * g + 0]));
                        acc[4 * g + 1] = __builtin_fmaf(w1, x1.y, __builtin_fmaf(w0, x0.y, acc[4 * g + 1]));
                        acc[4 * g + 2] = __builtin_fmaf(w1, x1.z, __builtin_fmaf(w0, x0.z, acc[4 * g + 2]));
                        acc[4 * g + 3] = __builtin_fmaf(w1, x1.w, __builtin_fmaf(w0, x0.w, acc[4 * g + 3]));
                    }
                }
            }
        }
        __syncthreads();
    }
    if (!active) return;
    float *out = a.dst + ((size_t)ang * a.nd + n) * a.nz + z0;
#pragma unroll
    for (int g = 0; g < G; ++g)
        *reinterpret_cast<float4 *>(out + 4 * g) =
            make_float4(acc[4 * g] * inv_m, acc[4 * g + 1] * inv_m, acc[4 * g + 2] * inv_m, acc[4 * g + 3] * inv_m);
}

// The same forward with one barrier per R lines.  The block first computes,
// for every line, the span of its rays' crossings (the minimum and maximum
// floor(crossing) over the edge rays, the first and last valid bin of each of
// its angles, with the same float expression) into LDS; while its rays
// interpolate R lines from one buffer, direct loads stage the next R into the
// other.  A line is staged by 256 / R threads in 16-byte chunks, G of a
// position's slices and one unused (an offset past the range loads zeros
// there), so that positions lie ZT + 4 floats apart; the spans are read two
// steps ahead.  Slice counts are any multiple of 4: groups beyond the last are
// staged as zeros and not stored.  Values and order of the sums are those of
// joseph_forward_lds_kernel, or with direct set of joseph_forward_kernel, which
// adds the column class's terms in another order: bit-identical to either.
//
// What limits it is the latency of a line (position, LDS address, LDS read,
// barrier) at 3 to 5 waves per SIMD (512^2 x 16 x 360: LDS 43 % busy, 43 % of the
// wave cycles waiting), and for volumes that do not stay in the caches their
// fetch, once per chunk of angles (1024^2 x 64 x 900: 27 GB in 4.9 ms); the form
// before staged through registers and read its spans when it needed them.
// Projection in microseconds, before and now: 512^2 x 16 x 360 (R = 2) 430, 260;
// 512^2 x 32 x 360 (R = 1) 567, 378 (502 with R = 2); 1024^2 x 64 x 200 5302, 3847
// (4976 with R = 2); slice counts that took joseph_forward_kernel: 300^2 x 20 x 200
// 461, 136; 700^2 x 8 x 200 (8 slices, R = 4) 924, 333.
// Dynamic LDS: N + 3 R spans.
template <int ZT, int R>
__global__ __launch_bounds__(256, R == 4 ? 4 : 5) void joseph_forward_dma_kernel(
    JosephArgs a, const int4 *__restrict__ chunks, const int *__restrict__ order, int n_chunks, int nbt, int nzs,
    int direct)
{
    constexpr int NB = kFwdNB, KA = kFwdKA, W = kFwdW, G = ZT / 4, GP = G + 1, RS = 4 * GP;
    constexpr int TL = 256 / R, NE = (W * GP + TL - 1) / TL;
    __shared__ __align__(16) float seg[2][R][W * RS];
    __shared__ float4 ep[2 * KA];    // edge rays: (a0, b1, cn, inv)
    extern __shared__ int2 jspans[]; // [lo, hi] of line L; lines N .. N + 3 R - 1 are dead
    const int total = n_chunks * nbt * nzs;
    const int per = (total + 7) >> 3;
    const int b = (int)blockIdx.x;
    const int wi = (b & 7) * per + (b >> 3);   // XCD b % 8 takes the (b % 8)-th eighth
    if (wi >= total) return;
    const int bt = wi % nbt;
    const int rest = wi / nbt;
    const int ci = rest % n_chunks;
    const int zs = rest / n_chunks;
    const int4 ch = chunks[ci];                // first, count, class
    const int tid = (int)threadIdx.x;
    // lanes 16 q .. 16 q + 15 of a wave take 4 angles x 4 neighbouring bins,
    // whose crossings of a line lie within a few staged rows: one angle's 16
    // bins spread over about 20 rows, and rows 16 apart share LDS banks
    const int ai = ((tid >> 2) & 3) | ((tid >> 4) & 12), bi = (tid & 3) | ((tid >> 2) & 12);
    const int n = bt * NB + bi;
    const bool active = ai < ch.y && n < a.nd;
    const int ang = order[ch.x + min(ai, ch.y - 1)];
    const float4 t = a.tab[ang];
    const float su = t.x, c = t.y, s = t.z, inv_m = t.w;
    const int N = a.nx;
    const int z0 = zs * ZT;
    const bool rows = ch.z == 0;
    // crossing of line L: ((a0 + b1 (L+1)) + cn) * inv - 1
    const bool own = direct && !rows;
    const float b1 = rows ? c : s;
    const float fn = (float)n;
    const float a0 = own ? fn - su : (rows ? su : -su);
    const float cn = own ? 0.0f : (rows ? -fn : fn);
    const float inv = rows ? 1.0f / s : 1.0f / c;
    const size_t strideL = rows ? (size_t)N * a.nz : (size_t)a.nz;
    const size_t strideP = rows ? (size_t)a.nz : (size_t)N * a.nz;
    if (tid < 2 * KA) {
        // edge ray tid: angle tid / 2, the block's first (even) or last valid (odd) bin
        const int ea = tid >> 1;
        const int en = min(bt * NB + ((tid & 1) ? NB - 1 : 0), a.nd - 1);
        const float4 et = a.tab[order[ch.x + min(ea, ch.y - 1)]];
        const float efn = (float)en;
        ep[tid] = make_float4(own ? efn - et.x : (rows ? et.x : -et.x), rows ? et.y : et.z,
                              own ? 0.0f : (rows ? -efn : efn), rows ? 1.0f / et.z : 1.0f / et.y);
    }
    __syncthreads();
    const int ne = 2 * ch.y;
    for (int L = tid; L < N + 3 * R; L += 256) {
        int lo = 0x7fffffff, hi = -0x7fffffff;
        for (int e = 0; L < N && e < ne; ++e) {
            const float4 q = ep[e];
            const int p0 = (int)floorf(((q.x + q.y * (float)(L + 1)) + q.z) * q.w - 1.0f);
            lo = min(lo, p0);
            hi = max(hi, p0);
        }
        // a line is dead when no ray of the block crosses the volume on it
        jspans[L] = hi >= -1 && lo < N ? make_int2(lo, hi) : make_int2(0x7fffffff, 0x7fffffff);
    }
    __syncthreads();
    float acc[ZT];
#pragma unroll
    for (int z = 0; z < ZT; ++z) acc[z] = 0.0f;
    // chunks of this thread: position j and byte offset from the line's first position
    const int sr = __builtin_amdgcn_readfirstlane(tid / TL), le = tid - sr * TL;
    int st_j[NE];
    unsigned st_off[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = le + TL * i, j = e / GP, g = e - j * GP;
        const bool used = e < W * GP && g < G && z0 + 4 * g < a.nz;
        st_j[i] = j;
        st_off[i] = used ? (unsigned)j * (unsigned)(4 * strideP) + 16u * (unsigned)g : 0x80000000u;
    }
    auto stage = [&](int L, int2 sp, float *dst) {
        if (sp.x == 0x7fffffff) return;
        const int nj = min(sp.y - sp.x + 2, W);   // only the voxels a line's rays read: lo .. hi + 1
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.src + ((long)L * (long)strideL + (long)sp.x * (long)strideP + z0)), (short)0, 0x7FFFFFFF,
            0x00020000);
        const int w64 = __builtin_amdgcn_readfirstlane(le & ~63);
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            if (w64 + TL * i >= nj * GP) break;
            const unsigned off = (unsigned)(sp.x + st_j[i]) < (unsigned)N ? st_off[i] : 0x80000000u;
            if (le + TL * i < W * GP)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs, (__attribute__((address_space(3))) void *)(dst + 4 * (w64 + TL * i)), 16, off, 0, 0, 0);
        }
    };
    auto span = [&](int L) {
        const int2 v = jspans[L];
        return make_int2(__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y));
    };
    int2 cur[R], nxt[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        cur[r] = span(r);
        nxt[r] = span(R + r);
    }
    stage(sr, span(sr), seg[0][sr]);
    lds_loads_barrier();
    for (int L0 = 0, buf = 0; L0 < N; L0 += R, buf ^= 1) {
        int2 far[R];
#pragma unroll
        for (int r = 0; r < R; ++r) far[r] = jspans[L0 + 2 * R + r];
        int2 mine = nxt[0];
#pragma unroll
        for (int r = 1; r < R; ++r)
            if (sr == r) mine = nxt[r];
        stage(L0 + R + sr, mine, seg[buf ^ 1][sr]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (cur[r].x == 0x7fffffff) continue;
            const float pf = ((a0 + b1 * (float)(L0 + r + 1)) + cn) * inv - 1.0f;
            const float fl = floorf(pf);
            const int p0 = (int)fl;
            const float f = pf - fl;
            const float w0 = (p0 >= 0 && p0 < N) ? 1.0f - f : 0.0f;
            const float w1 = (p0 + 1 >= 0 && p0 + 1 < N) ? f : 0.0f;
            const int j = min(max(p0 - cur[r].x, 0), W - 2);
            const float *v0 = &seg[buf][r][j * RS];
            const float *v1 = v0 + RS;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float4 x0 = *reinterpret_cast<const float4 *>(v0 + 4 * g);
                const float4 x1 = *reinterpret_cast<const float4 *>(v1 + 4 * g);
                acc[4 * g + 0] = __builtin_fmaf(w1, x1.x, __builtin_fmaf(w0, x0.x, acc[4 * g + 0]));
                acc[4 * g + 1] = __builtin_fmaf(w1, x1.y, __builtin_fmaf(w0, x0.y, acc[4 * g + 1]));
                acc[4 * g + 2] = __builtin_fmaf(w1, x1.z, __builtin_fmaf(w0, x0.z, acc[4 * g + 2]));
                acc[4 * g + 3] = __builtin_fmaf(w1, x1.w, __builtin_fmaf(w0, x0.w, acc[4 * g + 3]));
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            cur[r] = nxt[r];
            nxt[r] = make_int2(__builtin_amdgcn_readfirstlane(far[r].x), __builtin_amdgcn_readfirstlane(far[r].y));
        }
        lds_loads_barrier();
    }
    if (!active) return;
    float *out = a.dst + ((size_t)ang * a.nd + n) * a.nz + z0;
#pragma unroll
    for (int g = 0; g < G; ++g)
        if (z0 + 4 * g < a.nz)
            *reinterpret_cast<float4 *>(out + 4 * g) = make_float4(acc[4 * g] * inv_m, acc[4 * g + 1] * inv_m,
                                                                   acc[4 * g + 2] * inv_m, acc[4 * g + 3] * inv_m);
}

// Adjoint: one thread per (x, y) voxel column and ZT slices.
template <int ZT>
__global__ __launch_bounds__(256) void joseph_adjoint_kernel(JosephArgs a)
{
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int z0 = blockIdx.z * ZT;
    const int N = a.nx;
    if (x >= N || y >= N) return;
    float acc[ZT];
#pragma unroll
    for (int z = 0; z < ZT; ++z) acc[z] = 0.0f;
    const float xf = (float)(x + 1), yf = (float)(y + 1);
#pragma unroll 2
    for (int ang = 0; ang < a.na; ++ang) {
        const float4 t = a.tab[ang];
        const float u = (t.x + t.y * yf) - t.z * xf;
        const float fl = floorf(u);
        const int n1 = (int)fl;
        const float f = u - fl;
        const float inv_m = t.w;
        const bool ok1 = n1 >= 0 && n1 < a.nd, ok2 = n1 + 1 >= 0 && n1 + 1 < a.nd;
        const float w1 = ok1 ? fmaxf(0.0f, 1.0f - f * inv_m) * inv_m : 0.0f;
        const float w2 = ok2 ? fmaxf(0.0f, 1.0f - (1.0f - f) * inv_m) * inv_m : 0.0f;
        const int na = min(max(n1, 0), a.nd - 1), nb = min(max(n1 + 1, 0), a.nd - 1);
        const float *base = a.src + (size_t)ang * a.nd * a.nz + z0;
        lerp_accumulate<ZT>(acc, base + (size_t)na * a.nz, base + (size_t)nb * a.nz, w1, w2);
    }
    float *out = a.dst + ((size_t)y * N + x) * a.nz + z0;
#pragma unroll
    for (int g = 0; g < ZT / 4; ++g)
        *reinterpret_cast<float4 *>(out + 4 * g) =
            make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
}

// LDS-staged adjoint: the structure of the parallel back-projector's tiled
// kernel (16 x 16 voxel tile, ZT slices, C angles staged per chunk by direct
// loads into the other of two buffers, the XCD-striped tile order) with the Joseph
// kernel K as weights.  For each angle the tile stages the SPAN detector bins from
// floor(u) of its lowest corner, one bin of rounding margin below; bins outside [0, n_det) are staged as zeros, which is where the
// direct kernel's clamped loads have weight zero, and so are slices past the
// last.  (Staged between two barriers per chunk: 512^2 x 16 x 360 207 against 166
// us, 512^2 x 32 x 360 358 against 272, 1024^2 x 64 x 200 1.32 against 1.16 ms.)  As
// there, the compiler waits for the loads ahead of a chunk's first read and the
// CU's other blocks cover them (without that wait 0.94 to 1.03 times as long), and
// no unit bounds it alone: 512^2 x 16 x 360 keeps the LDS busy for 53 % of the
// cycles, issues 0.23 vector instructions per cycle and SIMD and waits for 36 %
// of the wave cycles.
constexpr int kJSpan = 26;

template <int ZT, int C>
__global__ __launch_bounds__(256) void joseph_adjoint_lds_kernel(JosephArgs a, int ntx, int nty, int ntz)
{
    constexpr int T = 16, SPAN = kJSpan, G = ZT / 4, GP = G + 1, NE = (SPAN * GP + 63) / 64;
    static_assert(64 % C == 0, "a chunk lies in one group of 64 angles");
    __shared__ __align__(16) float sm[2][C][SPAN][4 * GP];
    // block -> tile: XCD c (= block % 8) takes the c-th eighth of the tiles in
    // slice-chunk, 4-column stripe, row order
    const int n = ntx * nty * ntz;
    const int per = (n + 7) >> 3;
    const int b = (int)blockIdx.x;
    const int tidx = (b & 7) * per + (b >> 3);
    if (tidx >= n) return;
    const int plane = ntx * nty;
    const int bz = tidx / plane;
    const int r = tidx - bz * plane;
    const int sw = 4;
    const int s = r / (sw * nty);
    const int q = r - s * sw * nty;
    const int w = min(sw, ntx - sw * s);
    const int by = q / w, bx = sw * s + (q - by * w);

    const int N = a.nx;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int x0 = bx * T, y0 = by * T;
    const int x = x0 + tx, y = y0 + ty;
    const int z0 = bz * ZT;
    const bool in_vol = x < N && y < N;
    float acc[ZT];
#pragma unroll
    for (int z = 0; z < ZT; ++z) acc[z] = 0.0f;
    const float xf = (float)(x + 1), yf = (float)(y + 1);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // wave w stages angles w, w + 4, ... of a chunk in 16-byte chunks: G of a
    // bin's slices and one lane whose offset lies past the buffer
    int st_b[NE];
    unsigned st_off[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int b = (lane + 64 * i) / GP, g = (lane + 64 * i) - b * GP;
        st_b[i] = b;
        st_off[i] = g < G && z0 + 4 * g < a.nz ? 4u * (unsigned)b * (unsigned)a.nz + 16u * (unsigned)g : 0x80000000u;
    }
    // lowest bin of angle 64 j + lane
    auto lowest = [&](int kb) {
        const float4 t = a.tab[min(kb + lane, a.na - 1)];
        const float ya = (float)(y0 + 1), yb = (float)(y0 + T);
        const float xa = (float)(x0 + 1), xb = (float)(x0 + T);
        const float la = t.x + t.y * ya, lb = t.x + t.y * yb;
        const float umin = fminf(fminf(la - t.z * xa, la - t.z * xb), fminf(lb - t.z * xa, lb - t.z * xb));
        return (int)floorf(umin) - 1;
    };
    auto stage = [&](int kb, int low, float (&dst)[C][SPAN][4 * GP]) {
#pragma unroll
        for (int kk = wv; kk < C; kk += 4) {
            if (kb + kk >= a.na) break;
            const int n0 = __builtin_amdgcn_readlane(low, (kb + kk) & 63);
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(a.src + (((long)(kb + kk) * a.nd + n0) * a.nz + z0)), (short)0, 0x7FFFFFFF, 0x00020000);
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const unsigned off = (unsigned)(n0 + st_b[i]) < (unsigned)a.nd ? st_off[i] : 0x80000000u;
                if (lane + 64 * i < SPAN * GP)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rs, (__attribute__((address_space(3))) void *)(&dst[kk][0][0] + 256 * i), 16, off, 0, 0, 0);
            }
        }
    };
    int low = lowest(0), low_next = low;
    stage(0, low, sm[0]);
    lds_loads_barrier();
    for (int kb = 0, buf = 0; kb < a.na; kb += C, buf ^= 1) {
        if (kb + C < a.na) {
            if (((kb + C) & 63) == 0) low_next = lowest(kb + C);
            stage(kb + C, low_next, sm[buf ^ 1]);
        }
        if (in_vol) {
#pragma unroll
            for (int kk = 0; kk < C; ++kk) {
                if (kb + kk >= a.na) break;
                const float4 t = tab_entry(a.tab, kb + kk);
                const float u = (t.x + t.y * yf) - t.z * xf;
                const float fl = floorf(u);
                const int n1 = (int)fl;
                const float f = u - fl;
                const float inv_m = t.w;
                const float w1 = fmaxf(0.0f, 1.0f - f * inv_m) * inv_m;
                const float w2 = fmaxf(0.0f, 1.0f - (1.0f - f) * inv_m) * inv_m;
                const int loc = min(max(n1 - __builtin_amdgcn_readlane(low, (kb + kk) & 63), 0), SPAN - 2);
                const float *A = &sm[buf][kk][loc][0];
                const float *B = A + (ZT + 4);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float4 va = *reinterpret_cast<const float4 *>(A + 4 * g);
                    const float4 vb = *reinterpret_cast<const float4 *>(B + 4 * g);
                    acc[4 * g + 0] = __builtin_fmaf(w2, vb.x, __builtin_fmaf(w1, va.x, acc[4 * g + 0]));
                    acc[4 * g + 1] = __builtin_fmaf(w2, vb.y, __builtin_fmaf(w1, va.y, acc[4 * g + 1]));
                    acc[4 * g + 2] = __builtin_fmaf(w2, vb.z, __builtin_fmaf(w1, va.z, acc[4 * g + 2]));
                    acc[4 * g + 3] = __builtin_fmaf(w2, vb.w, __builtin_fmaf(w1, va.w, acc[4 * g + 3]));
                }
            }
        }
        low = low_next;
        lds_loads_barrier();
    }
    if (!in_vol) return;
    float *out = a.dst + ((size_t)y * N + x) * a.nz + z0;
#pragma unroll
    for (int g = 0; g < G; ++g)
        if (z0 + 4 * g < a.nz)
            *reinterpret_cast<float4 *>(out + 4 * g) =
                make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
}

std::vector<float> joseph_tables(const mr_joseph_geom &g, const float *angles, size_t n_ang)
{
    std::vector<float> tab(4 * n_ang);
    const double dirw = g.direction == 0 ? -1.0 : 1.0;
    const double cx = (double)(g.nx / 2);
    for (size_t i = 0; i < n_ang; ++i) {
        const double phi = dirw * (double)angles[i] * 3.14159265358979323846 / 180.0;
        const double s = std::sin(phi), c = std::cos(phi);
        tab[4 * i + 0] = (float)(cx * (s - c) + (double)g.center);
        tab[4 * i + 1] = (float)c;
        tab[4 * i + 2] = (float)s;
        tab[4 * i + 3] = (float)(1.0 / std::max(std::fabs(s), std::fabs(c)));
    }
    return tab;
}

// Angle chunks of the LDS forward: angles of one stepping class in order of
// direction, cut so that on every line the crossings of any block's rays
// (kFwdNB bins x the chunk's angles) span at most kFwdW - 3 voxels (one voxel
// of margin for float rounding; the interpolation needs p0 and p0 + 1).  The
// span of affine functions of the line index is largest at the first or
// last line, so those two are checked.
JosephPacked joseph_pack(const mr_joseph_geom &g, const float *angles, size_t n_ang)
{
    JosephPacked pk;
    pk.tab = joseph_tables(g, angles, n_ang);
    const int N = (int)g.nx, nd = (int)g.n_det;
    const int nbt = (nd + kFwdNB - 1) / kFwdNB;
    for (int cls = 0; cls < 2; ++cls) {
        std::vector<std::pair<double, int>> idx;
        for (size_t i = 0; i < n_ang; ++i) {
            const float c = pk.tab[4 * i + 1], s = pk.tab[4 * i + 2];
            const int k = std::fabs(s) >= std::fabs(c) ? 0 : 1;
            if (k != cls) continue;
            double dir = std::atan2((double)s, (double)c);
            if (dir < 0) dir += 2.0 * 3.14159265358979323846;
            idx.push_back({dir, (int)i});
        }
        std::sort(idx.begin(), idx.end());
        // per bin tile and end line: min / max crossing over the chunk
        std::vector<double> mn(2 * nbt), mx(2 * nbt), tmn(2 * nbt), tmx(2 * nbt);
        int first = (int)pk.order.size(), count = 0;
        auto flush = [&]() {
            if (count > 0) pk.chunks.push_back(make_int4(first, count, cls, 0));
            first = (int)pk.order.size();
            count = 0;
        };
        for (const auto &e : idx) {
            const int i = e.second;
            const double su = pk.tab[4 * i], c = pk.tab[4 * i + 1], s = pk.tab[4 * i + 2];
            const double a0 = cls == 0 ? su : -su, b1 = cls == 0 ? c : s, inv = cls == 0 ? 1.0 / s : 1.0 / c;
            double worst = 0.0;
            for (int bt = 0; bt < nbt; ++bt) {
                const int na = bt * kFwdNB, nb = std::min(na + kFwdNB - 1, nd - 1);
                for (int end = 0; end < 2; ++end) {
                    const double L1 = end == 0 ? 1.0 : (double)N;
                    double lo = 1e300, hi = -1e300;
                    for (int nn : {na, nb}) {
                        const double cn = cls == 0 ? -(double)nn : (double)nn;
                        const double pf = ((a0 + b1 * L1) + cn) * inv - 1.0;
                        lo = std::min(lo, pf);
                        hi = std::max(hi, pf);
                    }
                    const int k = 2 * bt + end;
                    tmn[k] = count ? std::min(mn[k], lo) : lo;
                    tmx[k] = count ? std::max(mx[k], hi) : hi;
                    worst = std::max(worst, tmx[k] - tmn[k]);
                }
            }
            if (count > 0 && (count == kFwdKA || std::ceil(worst) + 1.0 > (double)(kFwdW - 2))) {
                flush();
                // restart the extents with this angle alone
                for (int bt = 0; bt < nbt; ++bt) {
                    const int na = bt * kFwdNB, nb = std::min(na + kFwdNB - 1, nd - 1);
                    for (int end = 0; end < 2; ++end) {
                        const double L1 = end == 0 ? 1.0 : (double)N;
                        double lo = 1e300, hi = -1e300;
                        for (int nn : {na, nb}) {
                            const double cn = cls == 0 ? -(double)nn : (double)nn;
                            const double pf = ((a0 + b1 * L1) + cn) * inv - 1.0;
                            lo = std::min(lo, pf);
                            hi = std::max(hi, pf);
                        }
                        tmn[2 * bt + end] = lo;
                        tmx[2 * bt + end] = hi;
                    }
                }
            }
            mn = tmn;
            mx = tmx;
            pk.order.push_back(i);
            ++count;
        }
        flush();
    }
    return pk;
}

size_t JosephPacked::bytes() const
{
    return sizeof(float) * tab.size() + sizeof(int4) * chunks.size() + sizeof(int) * order.size();
}

// One buffer: tables, then chunks, then the angle order.
int joseph_upload(const JosephPacked &pk, void *d_base, hipStream_t s, JosephDevTables &dt)
{
    char *b = static_cast<char *>(d_base);
    const size_t o1 = sizeof(float) * pk.tab.size(), o2 = o1 + sizeof(int4) * pk.chunks.size();
    MR_HIP(hipMemcpyAsync(b, pk.tab.data(), o1, hipMemcpyHostToDevice, s));
    if (!pk.chunks.empty())
        MR_HIP(hipMemcpyAsync(b + o1, pk.chunks.data(), o2 - o1, hipMemcpyHostToDevice, s));
    if (!pk.order.empty())
        MR_HIP(hipMemcpyAsync(b + o2, pk.order.data(), sizeof(int) * pk.order.size(), hipMemcpyHostToDevice, s));
    dt.tab = reinterpret_cast<const float4 *>(b);
    dt.chunks = reinterpret_cast<const int4 *>(b + o1);
    dt.order = reinterpret_cast<const int *>(b + o2);
    dt.n_chunks = (int)pk.chunks.size();
    return MR_OK;
}

int joseph_check(const mr_joseph_geom *g, size_t n_ang)
{
    MR_REQUIRE(g != nullptr, "geometry is NULL");
    MR_REQUIRE(g->nx >= 2 && g->n_det >= 2 && g->nz >= 4, "sizes too small");
    MR_REQUIRE(g->nz % 4 == 0, "nz must be a multiple of 4");
    MR_REQUIRE(n_ang >= 1 && n_ang <= 65535 * 4, "angle count out of range");
    MR_REQUIRE(g->direction == 0 || g->direction == 1, "direction must be 0 (CW) or 1 (CCW)");
    return MR_OK;
}

// Whether a slice count that is no multiple of 16 takes the staged forward (total
// blocks of slice tiles zt) or joseph_forward_kernel (one wave per 64 rays and 4
// slices), from what one line of the volume takes with either, in microseconds.
// A staged block serves 16 bins of the angles of its chunk - 16 where they lie
// close, one where a wide volume and few angles let no two share a chunk - in
// the same time, so the number of blocks counts.  The direct kernel's waves all
// run at once up to one per SIMD (1024), then one after the other, each with the
// cache misses of its slices.  Fitted to 500 sizes (64^2 to 2048^2, 4 to 60 slices, 8
// to 360 angles); whole calls, staged / direct, the faster one is taken: 2048^2 x 4 x
// 60 3.86 / 1.18 ms, 1024^2 x 12 x 20 0.72 / 0.34, 128^2 x 20 x 60 0.082 / 0.061; 300^2 x
// 20 x 200 0.14 / 0.46, 1024^2 x 12 x 90 1.18 / 1.85, 400^2 x 4 x 180 0.14 / 0.22.
static bool forward_staged(const mr_joseph_geom &g, size_t n_ang, int zt, long total)
{
    if (total < 128) return false;
    const double blocks = (double)total / 1024.0;
    const double waves = (double)g.n_det * (double)n_ang * (double)g.nz / (64.0 * 4.0 * 1024.0);
    const double staged = zt == 8 ? std::max(0.22, 0.32 * blocks) : std::max(0.42, 0.40 * blocks);
    const double direct =
        waves <= 1.0 ? 0.28 : std::max(0.45, (0.08 + 0.03 * (double)std::min<size_t>(g.nz, 24)) * waves);
    return 1.08 * staged < direct;
}

// Enqueues A (forward) or A^T on s with a resident angle table; no host sync.
int joseph_launch(const mr_joseph_geom *g, const float *src, float *dst, const JosephDevTables &dt, size_t n_ang,
                  bool forward, hipStream_t s)
{
    mr::JosephArgs a{src, dst, dt.tab, (int)g->nx, (int)g->nz, (int)g->n_det, (int)n_ang};
    constexpr int ZT = 4;
    if (forward) {
        mr::ProfScope prof("joseph_forward", s);
        // The staged form with direct loads: 32 slices and a line per barrier
        // where the slice count is a multiple of 32, 8 slices and 4 lines up to
        // 8 slices, else 16 slices and 2 lines; while its spans fit in LDS
        // beside the lines (64 KB) and a staged line's offsets in 32 bits.
        const int zt = g->nz % 32 == 0 ? 32 : (g->nz > 8 ? 16 : 8), R = zt == 32 ? 1 : (zt == 16 ? 2 : 4);
        const int nbt = (int)((g->n_det + kFwdNB - 1) / kFwdNB), nzs = (int)((g->nz + zt - 1) / zt);
        const long total = (long)dt.n_chunks * nbt * nzs;
        const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
        const size_t dyn = sizeof(int2) * (g->nx + 3 * R);
        const size_t fixed = sizeof(float) * 2 * R * kFwdW * (zt + 4) + sizeof(float4) * 2 * kFwdKA;
        const int direct = g->nz % 16 == 0 ? 0 : 1;
        if (dt.n_chunks > 0 && total < (1L << 31) - 8 && dyn + fixed <= 65536 && g->nx * g->nz < 6500000 &&
            (!direct || forward_staged(*g, n_ang, zt, total))) {
            if (zt == 32)
                hipLaunchKernelGGL((mr::joseph_forward_dma_kernel<32, 1>), grid, dim3(256), dyn, s, a, dt.chunks,
                                   dt.order, dt.n_chunks, nbt, nzs, direct);
            else if (zt == 16)
                hipLaunchKernelGGL((mr::joseph_forward_dma_kernel<16, 2>), grid, dim3(256), dyn, s, a, dt.chunks,
                                   dt.order, dt.n_chunks, nbt, nzs, direct);
            else
                hipLaunchKernelGGL((mr::joseph_forward_dma_kernel<8, 4>), grid, dim3(256), dyn, s, a, dt.chunks,
                                   dt.order, dt.n_chunks, nbt, nzs, direct);
        } else if (g->nz % 16 == 0 && dt.n_chunks > 0) {
            MR_REQUIRE(total < (1L << 31) - 8, "Joseph forward grid too large");
            // larger volumes: the per-line form gives the same bits
            if (zt == 32)
                hipLaunchKernelGGL((mr::joseph_forward_lds_kernel<32, kFwdR>), grid, dim3(256), 0, s, a, dt.chunks,
                                   dt.order, dt.n_chunks, nbt, nzs);
            else
                hipLaunchKernelGGL((mr::joseph_forward_lds_kernel<16, kFwdR>), grid, dim3(256), 0, s, a, dt.chunks,
                                   dt.order, dt.n_chunks, nbt, nzs);
        } else {
            // other slice counts, few blocks or a large volume: direct ray-driven gathers
            mr::ProfScope gathers("joseph_forward_direct", s);
            dim3 grid((unsigned)((g->n_det + 63) / 64), (unsigned)((n_ang + 3) / 4), (unsigned)(g->nz / ZT));
            hipLaunchKernelGGL(mr::joseph_forward_kernel<ZT>, grid, dim3(256), 0, s, a);
        }
    } else {
        mr::ProfScope prof("joseph_adjoint", s);
        // slice tiles of 32 where the count is a multiple of it, 8 up to 8
        // slices, else 16 (a rest is staged as zeros).  Slice counts that are not
        // a multiple of 16 take the voxel-driven kernel, which gives the same
        // bits, below 512 tiles: 128^2 x 24 x 60 (128 tiles) 18 against 28 us,
        // 300^2 x 20 x 200 (722) 125 against 80, 700^2 x 8 x 200 220 against 103.
        const int zt = g->nz % 32 == 0 ? 32 : (g->nz > 8 ? 16 : 8);
        const int ntx = (int)((g->nx + 15) / 16), ntz = (int)((g->nz + zt - 1) / zt);
        const long nt = (long)ntx * ntx * ntz;
        const dim3 grid((unsigned)(8 * ((nt + 7) / 8)));
        if (nt >= (1L << 30) || (g->nz % 16 != 0 && nt < 512)) {
            // (also more tiles than the tile numbers hold)
            dim3 g3((unsigned)ntx, (unsigned)ntx, (unsigned)(g->nz / ZT));
            hipLaunchKernelGGL(mr::joseph_adjoint_kernel<ZT>, g3, dim3(256), 0, s, a);
        } else if (zt == 32) {
            hipLaunchKernelGGL((mr::joseph_adjoint_lds_kernel<32, 4>), grid, dim3(256), 0, s, a, ntx, ntx, ntz);
        } else if (zt == 16) {
            hipLaunchKernelGGL((mr::joseph_adjoint_lds_kernel<16, 4>), grid, dim3(256), 0, s, a, ntx, ntx, ntz);
        } else {
            hipLaunchKernelGGL((mr::joseph_adjoint_lds_kernel<8, 8>), grid, dim3(256), 0, s, a, ntx, ntx, ntz);
        }
    }
    MR_HIP(hipGetLastError());
    return MR_OK;
}

}  // namespace mr

namespace {

int joseph_common(const mr_joseph_geom *g, const float *src, const float *angles, size_t n_ang, float *dst,
                  void *stream, bool forward)
{
    mr::clear_error();
    int rc = mr::joseph_check(g, n_ang);
    if (rc != MR_OK) return rc;
    MR_REQUIRE(src != nullptr && dst != nullptr && angles != nullptr, "NULL pointer");
    hipStream_t s = (hipStream_t)stream;
    const mr::JosephPacked pk = mr::joseph_pack(*g, angles, n_ang);
    void *d_buf = nullptr;
    MR_HIP(hipMallocAsync(&d_buf, pk.bytes(), s));
    mr::JosephDevTables dt;
    rc = mr::joseph_upload(pk, d_buf, s, dt);
    if (rc == MR_OK) rc = mr::joseph_launch(g, src, dst, dt, n_ang, forward, s);
    hipError_t e2 = hipFreeAsync(d_buf, s);
    if (rc != MR_OK) return rc;
    if (e2 != hipSuccess) return mr::hip_fail(e2, "hipFreeAsync", __FILE__, __LINE__);
    // the host table must outlive the asynchronous copy
    MR_HIP(hipStreamSynchronize(s));
    return MR_OK;
}

}  // namespace

extern "C" int mr_joseph_forward(const mr_joseph_geom *geom, const float *d_volume, const float *angles,
                                 size_t n_ang, float *d_sino, void *stream)
{
    MR_GUARD_BEGIN
    return joseph_common(geom, d_volume, angles, n_ang, d_sino, stream, true);
    MR_GUARD_END
}

extern "C" int mr_joseph_adjoint(const mr_joseph_geom *geom, const float *d_sino, const float *angles,
                                 size_t n_ang, float *d_volume, void *stream)
{
    MR_GUARD_BEGIN
    return joseph_common(geom, d_sino, angles, n_ang, d_volume, stream, false);
    MR_GUARD_END
}
