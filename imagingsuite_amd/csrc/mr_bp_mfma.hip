// Parallel-beam back-projection on the matrix cores (fused mode of
// MultiProjBPparallel / MultiProjBP, linear interpolation).
//
// For one projection, the voxels of a 4 x 4 patch reach detector positions u
// within 3 (|cos| + |sin|) <= 4.25 columns of the patch's lowest corner, so a
// window of 8 columns starting at an even column holds every column they
// interpolate.  The update of a patch by 4 projections and 16 slices is then
// a 16 x 32 by 32 x 16 product,
//   vol[voxel][slice] += sum_{g < 4, i < 8} W[voxel][8 g + i] S_g[c0_g + i][slice],
// with W the two interpolation weights of the voxel in projection g's window
// (a hat function of the position, zeros elsewhere): one
// v_mfma_f32_16x16x32_f16 per operand pair, lane (16 g + m) building the
// weights of voxel m and reading the window of projection g.
//
// Operands.  A float weight or sample a is the sum of two halves, ah =
// half(a) and al = half(a - ah), 22 significant bits; a product is ah bh + al
// bh + ah bl in float (al bl, below 2^-22 of the product, is dropped).  The
// samples are first scaled per slice by a power of two that brings the
// slice's largest magnitude to [2^14, 2^15): a sample keeps 22 bits down to
// 2^-17 of the largest of its slice and an absolute 2^-40 of it below; the
// volume is scaled back on the way out (exact).  Positions are the
// reference's float operations, as everywhere.  A group of 4 projections is
// summed from zero in the matrix unit and added to the voxel's running sum
// once, against eight fused multiply-adds, so the sum's rounding is smaller
// than the float kernel's by more than the split adds, as long as the samples
// of a slice are of similar size: error against 64-bit sums of the same samples
// (relative rms, MFMA / FMA kernel) 1.55e-6 / 1.62e-6 at 512^2 x 400 projections,
// 4.90e-6 / 5.00e-6 at 1024^2 x 1800, equal to three digits where the float
// positions dominate.
//
// One sample far above the others (a sentinel for a dead pixel, one projection's
// weight) takes bits from the rest of its slice: at 1e7 times them the sums' error
// would be 9 times the float kernel's, at 1e9 600 times.  So a slice of which more
// than a sixteenth of the samples (those that are not zero; counted on an eighth of
// them) lie below 2^-17 of the largest does not fit, nor do samples that are not
// finite or slices whose largest magnitude is outside [2^-63, 2^74):
// bp_scale_kernel raises a flag on the device, the kernel here leaves without
// writing and the VALU kernel (gated by the same flag) does the work.  A voxel that
// only meets such small samples, in a slice that holds few enough of them to
// fit, has an error of about 2^-40 of the slice's largest per projection.
//
// What bounds it (2048^2 x 256 x 1500): the LDS reads of the windows (2 KB per
// patch, 16 slices and group) keep the LDS busy for 67 % of the cycles, the matrix
// unit (3 products of 16 cycles per wave) is busy for 45 %, the VALU (weights:
// about 40 instructions per patch) issues 0.16 instructions per cycle and SIMD,
// and 40 % of the wave cycles wait for one of them.  bp_lds_kernel takes 107 ms
// for it, this one 60-64 (the clock falls with the samples' toggling); whole FBP
// of that stack 110 against 65 ms, 701^2 x 37 x 603 1.54 against 0.89.
// The batch's form below keeps 45 registers in memory (all four widths of the
// tile in one kernel of 128 registers), 64-slice tiles of 16 x 16 voxels three.
#include "mr_bp.h"
#include "mr_common.h"

#include <algorithm>
#include <cstdint>
#include <string>

namespace mr {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// scales and split samples
// ---------------------------------------------------------------------------

// Largest value and sums over a wave.
__device__ __forceinline__ unsigned wave_max(unsigned m)
{
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
    return m;
}
__device__ __forceinline__ unsigned wave_sum(unsigned n)
{
    for (int o = 32; o > 0; o >>= 1) n += (unsigned)__shfl_xor((int)n, o);
    return n;
}

// part[v][chunk] = largest |proj[idx[k]][v][u] * w[idx[k]]| (its float bits;
// infinities and NaN compare above every finite value) over one of at most
// kScaleChunks runs of kc used projections; a wave takes every fourth.
constexpr int kScaleChunks = 64;
__global__ __launch_bounds__(256) void bp_absmax_kernel(const float *__restrict__ proj, const int *__restrict__ idx,
                                                        const float *__restrict__ wts, int nu, int nv, int nk, int kc,
                                                        unsigned *__restrict__ part)
{
    __shared__ unsigned red[4];
    const int v = blockIdx.x, k0 = blockIdx.y * kc, k1 = min(nk, k0 + kc);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned m = 0;
    for (int k = k0 + wv; k < k1; k += 4) {
        const int p = idx[k];
        const float w = wts[p];
        const float *row = proj + ((size_t)p * nv + v) * nu;
        if ((nu & 3) == 0) {
            for (int u = lane; u < nu / 4; u += 64) {
                const float4 x = reinterpret_cast<const float4 *>(row)[u];
                m = max(max(m, __float_as_uint(x.x * w) & 0x7fffffffu), __float_as_uint(x.y * w) & 0x7fffffffu);
                m = max(max(m, __float_as_uint(x.z * w) & 0x7fffffffu), __float_as_uint(x.w * w) & 0x7fffffffu);
            }
        } else {
            for (int u = lane; u < nu; u += 64) m = max(m, __float_as_uint(row[u] * w) & 0x7fffffffu);
        }
    }
    m = wave_max(m);
    if (lane == 0) red[wv] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[(size_t)v * gridDim.y + blockIdx.y] = max(max(red[0], red[1]), max(red[2], red[3]));
}

// How wide a slice's range is: behind the maxima of bp_absmax_kernel, part holds
// per [v][four chunks] how many samples are below 2^-17 of the slice's largest, and
// how many are not zero, among every eighth run of 64 columns (shifted by a run
// from one projection to the next, so that all columns take part).
constexpr unsigned kSmall = 17u << 23;   // 2^-17 in the bits of a float
__global__ __launch_bounds__(256) void bp_range_kernel(const float *__restrict__ proj, const int *__restrict__ idx,
                                                       const float *__restrict__ wts, int nu, int nv, int nk, int kc,
                                                       int nchunk, unsigned *__restrict__ part)
{
    __shared__ unsigned red[4][2];
    const int v = blockIdx.x, k0 = blockIdx.y * 4 * kc, k1 = min(nk, k0 + 4 * kc);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const unsigned m = wave_max(lane < nchunk ? part[(size_t)v * nchunk + lane] : 0u);
    const unsigned least = m > kSmall ? m - kSmall : 0u;
    unsigned small = 0, nonzero = 0;
    for (int k = k0 + wv; k < k1; k += 4) {
        const int p = idx[k];
        const float w = wts[p];
        const float *row = proj + ((size_t)p * nv + v) * nu;
        for (int u = 64 * (k & 7) + lane; u < nu; u += 512) {
            const unsigned x = __float_as_uint(row[u] * w) & 0x7fffffffu;
            small += x != 0 && x < least ? 1u : 0u;
            nonzero += x != 0 ? 1u : 0u;
        }
    }
    small = wave_sum(small);
    nonzero = wave_sum(nonzero);
    if (lane == 0) {
        red[wv][0] = small;
        red[wv][1] = nonzero;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[(size_t)nv * nchunk + ((size_t)threadIdx.x * nv + v) * gridDim.y + blockIdx.y] =
            red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

// scale[v] = (factor on the samples of slice v, its inverse); *flag = 1 when
// some slice does not fit the split: not finite, outside the exponent range, or
// more than a sixteenth of its samples below 2^-17 of its largest.  One block, 16
// lanes per slice (one lane: 22 us at 256 slices, against 6).
__global__ __launch_bounds__(1024) void bp_scale_kernel(const unsigned *__restrict__ part, int nv, int nchunk,
                                                        float2 *__restrict__ scale, int *__restrict__ flag)
{
    const int lane = threadIdx.x & 15;
    const int nrange = (nchunk + 3) / 4;   // at most 16
    int bad = 0;
    for (int v0 = 0; v0 < nv; v0 += 64) {
        const int v = v0 + (threadIdx.x >> 4);
        unsigned m = 0, small = 0, nonzero = 0;
#pragma unroll
        for (int i = 0; i < kScaleChunks / 16; ++i) {
            const int c = lane + 16 * i;
            if (v >= nv || c >= nchunk) continue;
            m = max(m, part[(size_t)v * nchunk + c]);
        }
        if (v < nv && lane < nrange) {
            const unsigned *counts = part + (size_t)nv * nchunk + (size_t)v * nrange + lane;
            small = counts[0];
            nonzero = counts[(size_t)nv * nrange];
        }
        for (int o = 8; o > 0; o >>= 1) {
            m = max(m, (unsigned)__shfl_xor((int)m, o));
            small += (unsigned)__shfl_xor((int)small, o);
            nonzero += (unsigned)__shfl_xor((int)nonzero, o);
        }
        const int e = (int)(m >> 23);   // biased exponent of the largest magnitude
        float2 s = make_float2(1.0f, 1.0f);
        if (m != 0) {
            if (e < 64 || e > 200 || small > nonzero / 16) bad = 1;
            else s = make_float2(__uint_as_float((unsigned)(268 - e) << 23), __uint_as_float((unsigned)(e - 14) << 23));
        }
        if (lane == 0 && v < nv) scale[v] = s;
    }
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) *flag = bad;
}

// a - (float)low half of h, b - (float)high half of h (exact), one instruction each
__device__ __forceinline__ float2v residual2(half2v h, float a, float b)
{
    float2v r = {a, b};
#if defined(__HIP_DEVICE_COMPILE__)
    const unsigned x = __builtin_bit_cast(unsigned, h);
    float lo, hi;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(lo) : "v"(x), "v"(a));
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(hi) : "v"(x), "v"(b));
    r = (float2v){lo, hi};
#endif
    return r;
}

// (a, b) ~ hi + lo, each a pair of halves.
__device__ __forceinline__ void split_pair(float a, float b, unsigned &hi, unsigned &lo)
{
    const half2v h = __builtin_convertvector((float2v){a, b}, half2v);
    const half2v l = __builtin_convertvector(residual2(h, a, b), half2v);
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, l);
}

// split[k][pair][zt][plane][16]: dword (sample of column 2 pair, of column 2
// pair + 1) of slice 16 zt + i, as halves: the high (plane 0) and low (plane
// 1) part of proj[idx[k]][z][u] * w[idx[k]] * scale[z].  Zero for u >= nu and
// for slices >= nz4, which the back-projectors do not update.  A block
// transposes 64 columns x 64 slices.  With *flag set the buffer becomes the
// float sinogram [k][u][vpad] of launch_bp_prep instead, for the kernel that
// then runs.
__global__ __launch_bounds__(256) void bp_split_prep_kernel(const float *__restrict__ proj,
                                                            unsigned *__restrict__ split,
                                                            const int *__restrict__ idx,
                                                            const float *__restrict__ wts,
                                                            const float2 *__restrict__ scale,
                                                            const int *__restrict__ flag, int nu, int nv, int nvs,
                                                            int nz4, int vpad, int vp, int npair)
{
    __shared__ float tile[64][65];
    const int k = blockIdx.z, p = idx[k];
    const float w = wts[p];
    const int u0 = blockIdx.x * 64, v0 = blockIdx.y * 64;
    const float *src = proj + (size_t)p * nu * nvs;
    if ((nu & 3) == 0) {
        const int c4 = threadIdx.x & 15, rr = threadIdx.x >> 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = rr + 16 * i, v = v0 + r, u = u0 + 4 * c4;
            float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (v < nv && u < nu) x = *reinterpret_cast<const float4 *>(src + (size_t)v * nu + u);
            tile[r][4 * c4 + 0] = x.x * w;
            tile[r][4 * c4 + 1] = x.y * w;
            tile[r][4 * c4 + 2] = x.z * w;
            tile[r][4 * c4 + 3] = x.w * w;
        }
    } else {
        const int c = threadIdx.x & 63, rr = threadIdx.x >> 6;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = rr + 4 * i, v = v0 + r, u = u0 + c;
            tile[r][c] = (v < nv && u < nu) ? src[(size_t)v * nu + u] * w : 0.0f;
        }
    }
    __syncthreads();
    if (*flag) {
        float *dst = reinterpret_cast<float *>(split) + (size_t)k * nu * vpad;
        const int r = threadIdx.x & 63, c0 = threadIdx.x >> 6;
        if (v0 + r < vpad)
            for (int c = c0; c < 64; c += 4)
                if (u0 + c < nu) dst[(size_t)(u0 + c) * vpad + v0 + r] = tile[r][c];
        return;
    }
    const int r = threadIdx.x & 63, v = v0 + r;
    if (v >= vp) return;
    const float sc = v < nz4 ? scale[v].x : 0.0f;
    unsigned *dst = split + (size_t)k * npair * 2 * vp + (size_t)(v >> 4) * 32 + (v & 15);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int c = (threadIdx.x >> 6) + 4 * i, pair = (u0 >> 1) + c;   // 32 pairs of the tile
        if (pair >= npair) break;
        unsigned hi, lo;
        split_pair(tile[r][2 * c] * sc, tile[r][2 * c + 1] * sc, hi, lo);
        dst[(size_t)pair * 2 * vp] = hi;
        dst[(size_t)pair * 2 * vp + 16] = lo;
    }
}

// ---------------------------------------------------------------------------
// back-projection
// ---------------------------------------------------------------------------

// A block of NW waves owns TX x TY voxels and 16 NT slices; a wave owns a row
// of 4 patches, all slices, in 4 NT accumulators per patch.  For each chunk of
// 4 projections the block stages the NP column pairs its voxels' windows lie
// in, into one of NB buffers (2: the loads of the next chunk are in flight
// while this one is used, one barrier per chunk; 1: two barriers, several
// blocks per CU).
constexpr int bpm_pairs(int tx, int ty)
{
    // window starts lie within floor(sqrt((tx - 4)^2 + (ty - 4)^2) / 2 + slack) + 1 pairs of the tile's first
    // one and are 4 pairs long
    return tx == 32 && ty == 32 ? 24 : 13;
}
template <int NT, int TX, int TY, int NB>
struct BpmShape {
    static constexpr int PW = 4;
    static constexpr int NW = (TX / 16) * (TY / 4);
    static constexpr int NTHR = 64 * NW;
    static constexpr int ROW = 32 * NT;            // dwords of a staged pair: [zt][plane][16]
    static constexpr int PPL = 64 / (8 * NT);      // pairs per wave load (16 bytes per lane)
    static constexpr int LANES = PPL * 8 * NT;     // lanes of a wave load
    static constexpr int WPP = NW / 4;             // waves staging one projection
    static constexpr int NL = (bpm_pairs(TX, TY) + PPL * WPP - 1) / (PPL * WPP);   // loads per wave and chunk
    static constexpr int NP = NL * PPL * WPP;
    static constexpr int GS = NP * ROW + 16;       // projection stride in dwords: 16 banks apart, so that lanes
                                                   // of two projections that read together use different banks
    static constexpr int BUF = 4 * GS;
    static constexpr int LDS = NB * BUF * 4 + 256; // bytes: the buffers, two slots of 4 table entries, selectors
};

__device__ __forceinline__ bool bpm_tile_of_block(const BpmArgs &a, int &bx, int &by, int &bz)
{
    const int n = a.ntx * a.nty * a.ntz;
    const int per = (n + 7) >> 3;
    const int b = (int)blockIdx.x;
    const int t = (b & 7) * per + (b >> 3);
    if (t >= n) return false;
    const int plane = a.ntx * a.nty;
    bz = t / plane;
    const int r = t - bz * plane;
    const int s = r / (a.sw * a.nty);
    const int q = r - s * a.sw * a.nty;
    const int w = min(a.sw, a.ntx - a.sw * s);
    by = q / w;
    bx = a.sw * s + (q - by * w);
    return true;
}

// LDS by byte offset: a window's address is one shift and addition away from
// the bits of its rounded position.
__device__ __forceinline__ unsigned lds_offset(const unsigned *p)
{
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned *)p;
}
template <class T>
__device__ __forceinline__ T lds_read(unsigned at)
{
    return *(const __attribute__((address_space(3))) T *)(uintptr_t)at;
}

template <int NT, int TX, int TY, int NB, int WV>
__device__ __forceinline__ void bpm_tile(const BpmArgs &a, int bx, int by, int bz, unsigned *lds)
{
    using S = BpmShape<NT, TX, TY, NB>;
    constexpr int PW = S::PW;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, m = lane & 15;        // projection of the group / voxel (A) or slice (B, C)
    const int xl = m & 3, yl = m >> 2;
    const int tx0 = bx * TX, ty0 = by * TY;
    const int wx0 = tx0 + (wv % (TX / 16)) * 16, wy0 = ty0 + (wv / (TX / 16)) * 4;
    const int z0 = a.zt0 * 16 + bz * 16 * NT;

    bool inside = false;
    for (int i = tid; i < TY; i += S::NTHR) {
        if (ty0 + i < a.nu) {
            const int2 mk = a.mask[ty0 + i];
            inside = inside || (max(mk.x, tx0) < min(mk.y, tx0 + TX));
        }
    }
    const bool live = __syncthreads_or(inside ? 1 : 0) != 0 && z0 < a.nz4;

    // accumulators: acc[patch][zt][i] = voxel 4 g + i (row g of the patch, column i), slice z0 + 16 zt + m
    float4v acc[PW][NT];
#pragma unroll
    for (int q = 0; q < PW; ++q)
#pragma unroll
        for (int zt = 0; zt < NT; ++zt) acc[q][zt] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
    if (a.chain && live) {
        // continue the sums of earlier projections (exact: a power of two)
#pragma unroll
        for (int q = 0; q < PW; ++q)
#pragma unroll
            for (int zt = 0; zt < NT; ++zt) {
                const int z = z0 + 16 * zt + m, y = wy0 + g, x = wx0 + 4 * q;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (y < a.nu && x + i < a.nu && z < a.nv)
                        acc[q][zt][i] = a.vol[((size_t)y * a.nu + x + i) * a.nvs + z] * a.scale[z].x;
            }
    }

    if (live && a.nk > 0) {
        const unsigned pairb = 8u * (unsigned)a.vp, projb = (unsigned)a.npair * pairb;
        // Table entries of the next chunk travel through two LDS slots as the
        // samples do: a vector load here would stall every wave of the block
        // once per chunk.  No voxel's position is valid in a projection past
        // the last one.
        float4 *ltab = reinterpret_cast<float4 *>(lds + NB * S::BUF);
        const __amdgpu_buffer_rsrc_t trs =
            __builtin_amdgcn_make_buffer_rsrc((void *)a.tab, (short)0, a.nk * 16, 0x00020000);
        auto stage_table = [&](int kb, int slot) {
            if (tid < 4)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    trs, (__attribute__((address_space(3))) void *)(ltab + 4 * slot), 16, 16 * (kb + tid), 0, 0, 0);
        };
        auto valid = [&](float4 t, int kb) { return kb + g < a.nk ? t : make_float4(-1.0e6f, 0.0f, 0.0f, 0.0f); };
        const float fnu1 = (float)(a.nu - 1);
        // Lower bounds of positions come from tile and patch centres, kSlack
        // below the real ones, so float rounding never puts a voxel under
        // its window: a voxel lies at most 2 + 3 (|cos| + |sin|) + 4 kSlack
        // < 7 columns above its window's first column.  Halved (pairs) and
        // rounded to an integer by adding kMagic.
        constexpr float kSlack = 0.0625f, kMagic = 12582912.0f;   // 1.5 2^23
        const float tcx = (float)tx0 + 0.5f * (TX + 1), tcy = (float)ty0 + 0.5f * (TY + 1);
        auto reach = [&](const float4 &t, float &lo, float &hi) {
            const float ext = __builtin_fmaf(fabsf(t.y), 0.5f * (TY - 1), fabsf(t.z) * (0.5f * (TX - 1))) + 2.0f * kSlack;
            const float cen = __builtin_fmaf(t.y, tcy, __builtin_fmaf(-t.z, tcx, t.x));
            lo = cen - ext;
            hi = cen + ext;
        };
        // first staged pair of the lane's projection, as the bits of kMagic + pair
        auto first_pair = [&](float lo) -> unsigned { return __float_as_uint((lo * 0.5f - 0.5f) + kMagic); };
        // Staging: loads straight into LDS, PPL pairs per wave load, WPP
        // waves per projection.  Offsets before the buffer or past its end
        // give zeros; pairs outside the detector and slices at or beyond vp
        // read finite neighbours, which meet zero weights or slices that are
        // not stored.
        const int skk = wv / S::WPP, sr0 = (wv % S::WPP) * S::NL;
        const unsigned st_lane = (unsigned)(lane / (8 * NT)) * pairb + 16u * (unsigned)(lane % (8 * NT)) +
                                 8u * (unsigned)z0 + (unsigned)skk * projb;
        auto stage = [&](int kb, unsigned s0, unsigned *buf) {
            const char *cb = reinterpret_cast<const char *>(a.split) + (size_t)kb * projb;
            const long rem = (long)(a.nk - kb) * projb;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void *)cb, (short)0, (int)min(rem, 0x7FFFFFF0L), 0x00020000);
            const int sp = (int)((unsigned)__builtin_amdgcn_readlane((int)s0, 16 * skk) - __float_as_uint(kMagic));
            unsigned soff = (unsigned)(sp + sr0 * S::PPL) * pairb;
            unsigned *dst = buf + skk * S::GS + sr0 * S::PPL * S::ROW;
            if (S::LANES == 64 || lane < S::LANES) {
#pragma unroll
                for (int j = 0; j < S::NL; ++j) {
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)dst, 16,
                                                             st_lane + soff, 0, 0, 0);
                    soff += S::PPL * pairb;
                    dst += S::PPL * S::ROW;
                }
            }
        };
        const float yf = (float)(wy0 + 1 + yl), xf = (float)(wx0 + 1 + xl);
        const float pcx = (float)wx0 + 2.5f, pcy = (float)wy0 + 2.5f;   // centre of the wave's first patch
        // Byte selectors that put the weights of columns n and n + 1 (a dword
        // of two halves) into the four dwords of a window's eight columns;
        // entry 7 selects zeros.
        unsigned *sel = lds + NB * S::BUF + 32;
        if (tid < 32) {
            const int d = (tid >> 2) - 2 * (tid & 3);   // n - 2 j
            const unsigned v = d == 0 ? 0x03020100u : (d == -1 ? 0x0c0c0302u : (d == 1 ? 0x01000c0cu : 0x0c0c0c0cu));
            sel[tid] = tid < 28 ? v : 0x0c0c0c0cu;
        }
        const unsigned kBits = __float_as_uint(kMagic);
        const unsigned sel_at = lds_offset(sel) - (kBits << 4);
        auto update = [&](const unsigned *buf, const float4 &t, unsigned s0, bool edge) {
            const float lsu = t.x + t.y * yf;
            // the first patch's lower bound in pairs, less the half that rounds it down
            float v = __builtin_fmaf(t.y, pcy, __builtin_fmaf(-t.z, pcx, t.x));
            v = __builtin_fmaf(__builtin_fmaf(fabsf(t.y) + fabsf(t.z), -1.5f, v), 0.5f, -0.5f - 0.5f * kSlack);
            const float s2 = t.z + t.z;
            const unsigned win_at = lds_offset(buf + g * S::GS + m) - s0 * (4 * S::ROW);
            // window of patch q: the voxel's two weights (high and low
            // halves), their selectors and the window's LDS address
            auto window = [&](int q, unsigned &wh, unsigned &wl, uint4v &sl) -> unsigned {
                const float u = lsu - t.z * (xf + (float)(4 * q));
                const float jm = v + kMagic;
                v -= s2;
                const float j2 = jm - kMagic;
                unsigned at = __float_as_uint(jm) * (4 * S::ROW) + win_at;
                float p = __builtin_fmaf(j2, -2.0f, u);   // position in the window
                if (edge) {
                    asm volatile("");   // a branch, not selects: most chunks skip it
                    // (int)u truncates: u in (-1, 0) counts as column 0 with weight |u| on column 1
                    p = u > -1.0f && u < fnu1 ? __builtin_fmaf(j2, -2.0f, fabsf(u)) : 7.25f;
                    at = (unsigned)min(max((int)(__float_as_uint(jm) - s0), 0), S::NP - 4) * (4 * S::ROW) +
                         lds_offset(buf + g * S::GS + m);
                }
                // column below the position (the one before it for a whole
                // number, which gives the same weights); 7: no weight
                const float nm = (p - 0.5f) + kMagic;
                sl = lds_read<uint4v>((__float_as_uint(nm) << 4) + sel_at);
                const float f = p - (nm - kMagic);
                split_pair(1.0f - f, f, wh, wl);
                return at;
            };
            // the four dwords of the lane's window per operand.  The empty
            // asm keeps the compiler from pairing dwords of different
            // operands into one read and moving them apart again.
            auto operands = [&](unsigned w, int zt, half8 &bh, half8 &bl) {
                const unsigned at = w + 128 * zt;
                bh = __builtin_bit_cast(half8, (uint4v){lds_read<unsigned>(at), lds_read<unsigned>(at + 4 * S::ROW),
                                                        lds_read<unsigned>(at + 8 * S::ROW),
                                                        lds_read<unsigned>(at + 12 * S::ROW)});
                asm volatile("" ::: "memory");
                bl = __builtin_bit_cast(
                    half8, (uint4v){lds_read<unsigned>(at + 64), lds_read<unsigned>(at + 4 * S::ROW + 64),
                                    lds_read<unsigned>(at + 8 * S::ROW + 64), lds_read<unsigned>(at + 12 * S::ROW + 64)});
                asm volatile("" ::: "memory");
            };
            half8 bh[2], bl[2];
            unsigned wh, wl;
            uint4v sl;
            unsigned w = window(0, wh, wl, sl);
            operands(w, 0, bh[0], bl[0]);
#pragma unroll
            for (int q = 0; q < PW; ++q) {
                uint4v ah, al;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ah[j] = __builtin_amdgcn_perm(0u, wh, sl[j]);
                    al[j] = __builtin_amdgcn_perm(0u, wl, sl[j]);
                }
                const half8 Ah = __builtin_bit_cast(half8, ah), Al = __builtin_bit_cast(half8, al);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int zt = 0; zt < NT; ++zt) {
                    // the next slice tile's (or patch's) LDS reads are under
                    // way while this one multiplies
                    const int c = (q * NT + zt) & 1;
                    if (zt + 1 < NT) operands(w, zt + 1, bh[c ^ 1], bl[c ^ 1]);
                    else if (q + 1 < PW) {
                        w = window(q + 1, wh, wl, sl);
                        operands(w, 0, bh[c ^ 1], bl[c ^ 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // the group's sum starts from zero and joins the running
                    // sum by a float addition: the matrix unit aligns its
                    // addends to the largest and drops what falls below,
                    // which against a running sum would leave a bias
                    float4v d = {0.0f, 0.0f, 0.0f, 0.0f};
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, bl[c], d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(Al, bh[c], d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, bh[c], d, 0, 0, 0);
                    acc[q][zt] += d;
                    asm volatile("" : "+v"(acc[q][zt]));   // here: sunk to the loop's end, every d would stay live
                }
            }
        };
        float4 t = valid(a.tab[min(g, a.nk - 1)], 0);
        float lo, hi;
        reach(t, lo, hi);
        unsigned s0 = first_pair(lo);
        bool edge = !__all(lo >= 0.0f && hi < fnu1);
        stage(0, s0, lds);
        stage_table(4, 1);
        lds_loads_barrier();
        int buf = 0;
        for (int kb = 0; kb < a.nk; kb += 4) {
            const int slot = (kb >> 2) & 1;
            reach(valid(ltab[4 * (slot ^ 1) + g], kb + 4), lo, hi);
            stage_table(kb + 8, slot);
            const unsigned s1 = first_pair(lo);
            const bool edge1 = !__all(lo >= 0.0f && hi < fnu1);
            unsigned *cur = lds + buf;
            if (NB == 2) {
                buf = S::BUF - buf;
                if (kb + 4 < a.nk) stage(kb + 4, s1, lds + buf);
            }
            update(cur, t, s0, edge);
            if (NB == 1) {
                lds_loads_barrier();
                if (kb + 4 < a.nk) stage(kb + 4, s1, lds);
            }
            t = valid(ltab[4 * (slot ^ 1) + g], kb + 4);   // read again: registers are short in update
            s0 = s1;
            edge = edge1;
            lds_loads_barrier();
        }
    }
    float inv[NT];
#pragma unroll
    for (int zt = 0; zt < NT; ++zt) inv[zt] = z0 + 16 * zt + m < a.nv ? a.scale[z0 + 16 * zt + m].y : 1.0f;
    // store: slices of one voxel are contiguous, 16 lanes write 64 bytes
#pragma unroll
    for (int q = 0; q < PW; ++q) {
        const int y = wy0 + g, x = wx0 + 4 * q;
        if (y >= a.nu) continue;
        const int2 mk = a.mask[y];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (x + i >= a.nu) continue;
            const bool in = x + i >= mk.x && x + i < mk.y;
            float *out = a.vol + ((size_t)y * a.nu + x + i) * a.nvs + z0 + m;
#pragma unroll
            for (int zt = 0; zt < NT; ++zt)
                if (z0 + 16 * zt + m < a.nv) out[16 * zt] = in ? acc[q][zt][i] * inv[zt] : 0.0f;
            // up to three slices past the last group of four, where that ends a tile
            if (z0 + 16 * NT == a.nz4 && a.nz4 + m < a.nv) out[16 * NT] = 0.0f;
        }
    }
}

template <int NT, int TX, int TY, int NB, int WV>
__global__ __launch_bounds__((BpmShape<NT, TX, TY, NB>::NTHR), WV) void bp_mfma_kernel(BpmArgs a)
{
    extern __shared__ __align__(16) unsigned bpm_lds[];
    if (*a.flag) return;
    int bx, by, bz;
    if (!bpm_tile_of_block(a, bx, by, bz)) return;
    bpm_tile<NT, TX, TY, NB, WV>(a, bx, by, bz, bpm_lds);
}

// Slice tiles [zt0, zt0 + ntz NT) of the volume.
template <int NT, int TX, int TY, int NB, int WV>
static int launch_bpm(BpmArgs a, int zt0, int ntz, hipStream_t s)
{
    using S = BpmShape<NT, TX, TY, NB>;
    a.ntx = (a.nu + TX - 1) / TX;
    a.nty = (a.nu + TY - 1) / TY;
    a.ntz = ntz;
    a.zt0 = zt0;
    a.sw = 4;
    const long n = (long)a.ntx * a.nty * a.ntz;
    if (S::LDS > 65536)
        MR_HIP(hipFuncSetAttribute((const void *)bp_mfma_kernel<NT, TX, TY, NB, WV>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS));
    ProfScope prof("bp_parallel", s);
    hipLaunchKernelGGL((bp_mfma_kernel<NT, TX, TY, NB, WV>), dim3((unsigned)(8 * ((n + 7) / 8))), dim3(S::NTHR),
                       S::LDS, s, a);
    MR_HIP(hipGetLastError());
    return MR_OK;
}

template <int NT>
static int launch_bpm_tile(const BpmArgs &a, int tile, int zt0, int ntz, hipStream_t s)
{
    return tile == 32 ? launch_bpm<NT, 32, 32, 2, 4>(a, zt0, ntz, s) : launch_bpm<NT, 16, 16, 1, 4>(a, zt0, ntz, s);
}

static int scale_chunks(size_t nk, int &kc)
{
    kc = (int)std::max<size_t>(8, (nk + kScaleChunks - 1) / kScaleChunks);
    return (int)((nk + kc - 1) / kc);
}

size_t bpm_part_words(size_t nv, size_t nk)
{
    int kc;
    return 3 * nv * (size_t)scale_chunks(nk, kc);
}

int launch_bp_scale(const float *proj, const int *idx, const float *wts, int nu, int nv, int nk, unsigned *part,
                    float2 *scale, int *flag, hipStream_t s)
{
    ProfScope prof("bp_scale", s);
    int kc;
    const int nchunk = scale_chunks((size_t)nk, kc);
    hipLaunchKernelGGL(bp_absmax_kernel, dim3((unsigned)nv, (unsigned)nchunk), dim3(256), 0, s, proj, idx, wts, nu, nv,
                       nk, kc, part);
    hipLaunchKernelGGL(bp_range_kernel, dim3((unsigned)nv, (unsigned)((nchunk + 3) / 4)), dim3(256), 0, s, proj, idx,
                       wts, nu, nv, nk, kc, nchunk, part);
    hipLaunchKernelGGL(bp_scale_kernel, dim3(1), dim3(1024), 0, s, part, nv, nchunk, scale, flag);
    MR_HIP(hipGetLastError());
    return MR_OK;
}

int launch_bp_split_prep(const BpmArgs &a, const float *proj, const int *idx, const float *wts, int vpad,
                         hipStream_t s)
{
    ProfScope prof("bp_prep", s);
    // (vpad, the float sinogram's slices, exceeds vp where nv % 16 is 1, 2 or 3)
    dim3 g((unsigned)((2 * a.npair + 63) / 64), (unsigned)((std::max(a.vp, vpad) + 63) / 64), (unsigned)a.nk);
    hipLaunchKernelGGL(bp_split_prep_kernel, g, dim3(256), 0, s, proj, const_cast<unsigned *>(a.split), idx, wts,
                       a.scale, a.flag, a.nu, a.nv, a.nvs, a.nz4, vpad, a.vp, a.npair);
    MR_HIP(hipGetLastError());
    return MR_OK;
}

// Where the matrix-core form is the faster one (whole calls, fused, against
// bp_lds_kernel): from 17 slices (1024^2 x 32 x 625: 1.40 against 1.71 ms, 2048^2 x
// 256 x 300: 13.3 against 20.0; a single tile of 16 leaves the weights' cost to 16
// slices: equal from 400^2) and from 1.5e9 voxel-projection updates, below which
// its extra launches cost what it saves (300^2 x 40 x 450, 1.6e9: 0.25 against 0.24
// ms; 400^2 x 40 x 300, 1.9e9: 0.20 against 0.26; 512^2 x 32 x 360: 0.23 against
// 0.27).  Each of its one or two launches (run_bpm: chunks of four slice tiles, then
// a chunk of the rest) must have about two blocks per CU, as a block's own latency
// is long: with 484 blocks 350^2 x 64 x 511 0.32 against 0.40 ms, 350^2 x 80 x 409
// 0.39 against 0.50; with 361 300^2 x 64 x 382 0.24 either way, 300^2 x 100 x 445
// equal; with 256 256^2 x 80 x 763 0.62 against 0.40 and with 64 128^2 x 100 x 916
// 0.84 against 0.35.  One or two slice tiles need as much work per column of
// blocks (350^2 x 32 x 1021: 0.41 against 0.50, 400^2 x 20 x 1250 0.55 against 0.57,
// but 350^2 x 24 x 511 0.22 against 0.20, 300^2 x 32 x 1046 even).  Four
// projections must fit the 60 MiB chunk of the no-allocation entry point, which
// gives the same bits by adding whole groups of four.
// Tile: 32 x 32 voxels (half the staging per voxel, one block of 16 waves per
// CU) for long scans over many tiles (2048^2 x 256 x 1500: 62.9 against 68.0 ms,
// 1024^2 x 64 x 900: 3.01 against 3.11), else 16 x 16 (four blocks per CU overlap
// each other's ends; 774^2 x 170 x 126: 0.82 against 0.88 ms, 329^2 x 51 x 1408:
// 0.83 against 1.06; 1024^2 x 64 x 300: 1.04 either way).
bool bpm_shape(int nu, int nv, int nk, int &tile)
{
    const size_t proj_bytes = 8 * (size_t)bpm_npair(nu) * (size_t)bpm_vp(nv);
    if (nv <= 16 || nk < 32 || 4 * proj_bytes > ((size_t)60 << 20)) return false;
    if ((double)nu * nu * nv * nk < 1.5e9) return false;
    const int nzt = bpm_vp(nv) / 16;
    const long n16 = (long)((nu + 15) / 16) * ((nu + 15) / 16), chunks = nzt % 4 ? 1 : nzt / 4;   // of the smaller launch
    if (nzt <= 2 ? n16 * nv < 12000 : n16 * chunks < 480) return false;
    const long n32 = (long)((nu + 31) / 32) * ((nu + 31) / 32) * ((nzt + 3) / 4);
    tile = nk >= 800 && n32 >= 512 ? 32 : 16;
    return true;
}

int run_bpm(const BpmArgs &a, int tile, hipStream_t s)
{
    // slices in chunks of four tiles of 16, what is left in one chunk of its own
    const int nzt = a.vp / 16, full = nzt / 4, rest = nzt % 4;
    int rc = MR_OK;
    if (full > 0) rc = launch_bpm_tile<4>(a, tile, 0, full, s);
    if (rc == MR_OK && rest == 1) rc = launch_bpm_tile<1>(a, tile, 4 * full, 1, s);
    if (rc == MR_OK && rest == 2) rc = launch_bpm_tile<2>(a, tile, 4 * full, 1, s);
    if (rc == MR_OK && rest == 3) rc = launch_bpm_tile<3>(a, tile, 4 * full, 1, s);
    return rc;
}

// Persistent form over the work items of a batch: items[i] = (stack, tile x,
// tile y, first slice tile | slice tiles << 16), eight partitions as in
// bp_batch_kernel.  Stacks whose samples do not fit the split are left to
// the VALU kernel.
__global__ __launch_bounds__(256, 4) void bp_mfma_batch_kernel(const BpmArgs *__restrict__ stacks,
                                                               const int4 *__restrict__ items,
                                                               const int *__restrict__ part_begin, int *counters)
{
    extern __shared__ __align__(16) unsigned bpm_lds[];
    __shared__ int item;
    int part = (int)(blockIdx.x & 7);
    for (;;) {
        if (threadIdx.x == 0) {
            int it = -1;
            for (int tries = 0; tries < 8; ++tries) {
                const int k = atomicAdd(&counters[part], 1);
                const int idx = part_begin[part] + k;
                if (idx < part_begin[part + 1]) {
                    it = idx;
                    break;
                }
                part = (part + 1) & 7;
            }
            item = it;
        }
        __syncthreads();
        // uniform: the item's and the stack's fields stay in scalar registers
        const int it = __builtin_amdgcn_readfirstlane(item);
        __syncthreads();
        if (it < 0) break;
        const int4 w = items[it];
        BpmArgs a = stacks[w.x];
        if (*a.flag) continue;
        a.zt0 = w.w & 0xffff;
        switch (w.w >> 16) {
        case 1: bpm_tile<1, 16, 16, 1, 4>(a, w.y, w.z, 0, bpm_lds); break;
        case 2: bpm_tile<2, 16, 16, 1, 4>(a, w.y, w.z, 0, bpm_lds); break;
        case 3: bpm_tile<3, 16, 16, 1, 4>(a, w.y, w.z, 0, bpm_lds); break;
        default: bpm_tile<4, 16, 16, 1, 4>(a, w.y, w.z, 0, bpm_lds); break;
        }
        __syncthreads();
    }
}

int bpm_batch_grid(int &grid)
{
    constexpr int lds = BpmShape<4, 16, 16, 1>::LDS;
    int dev = 0, ncu = 0, nb = 0;
    MR_HIP(hipGetDevice(&dev));
    MR_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    MR_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, bp_mfma_batch_kernel, 256, lds));
    grid = std::max(1, nb) * std::max(1, ncu);
    return MR_OK;
}

int launch_bpm_batch(const BpmArgs *d_stacks, const int4 *d_items, const int *d_parts, int *d_counters, int grid,
                     hipStream_t s)
{
    hipLaunchKernelGGL(bp_mfma_batch_kernel, dim3((unsigned)grid), dim3(256), (BpmShape<4, 16, 16, 1>::LDS), s,
                       d_stacks, d_items, d_parts, d_counters);
    MR_HIP(hipGetLastError());
    return MR_OK;
}

}  // namespace mr
