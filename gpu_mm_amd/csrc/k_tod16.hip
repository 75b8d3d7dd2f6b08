// 16-bit TOD encoding on gfx950: one FP32 scale per TOD row, values stored as FP16 or BF16.
//
// scale[r] = max(max_s |tod[r][s]| / (0.5 * M), FLT_MIN), M = largest finite value of the type
// (65504 for FP16, 0x1.fep127 for BF16), so every encoded value lies in [-M/2, M/2]; the FLT_MIN
// floor keeps the scale a normal float (an all-zero row gets scale FLT_MIN and zeros).
//
// Optional error feedback (order 1 or 2): each thread encodes a contiguous run of its row in
// sample order and adds the previous samples' rounding errors e to the next value before rounding
// (v_k = u_k + e_{k-1}, order 1; v_k = u_k + 2 e_{k-1} - e_{k-2}, order 2; e_k = v_k - round(v_k)).
// The decoded TOD then carries the first (second) difference of the rounding errors instead of
// the errors themselves; tod2map sums samples with slowly varying bilinear weights, so in the map
// the differences largely cancel (FP16, 2048x262144 raster: map error 2.1e-4 -> 9.9e-5 / 8.3e-5
// of the map RMS, while the per-sample TOD error grows by ~1.5x / 2.7x). The chain restarts at
// each thread's run (row_len / 256 samples); a non-finite error is dropped.
// This has no counterpart in the reference, which stores TODs as float32 only.
//
// Bound: the row is read twice (its scale comes before its values) and written once, 671 MB at 512 rows
// of 131072 samples, which take 128 us with error feedback (5.2 TB/s; 109 us without). With a lane
// walking its run straight through HBM, 2 KiB from its neighbour's, the same call took 1515 us. With
// few rows the chain of feedbacks is the bound: 330 us for one row of 2^21 samples (8192 steps).

#include "gmm_internal.hpp"

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace gmm {

namespace {

constexpr int ENC_CHAINS = 256;                    // error-feedback runs per row
constexpr int ENC_THREADS = 256;
constexpr int ENC_TILE = 32;                       // samples of each run staged at a time
constexpr int ENC_STRIDE = ENC_TILE + 4;           // floats per staged run: 16-byte slots, 16 lanes on distinct banks

// fmaxf ignores NaN, so NaN values leave the scale alone and are encoded as NaN. A row that holds an
// infinity gets an infinite scale (its finite values encode as 0, infinities as NaN).
template<typename TT>
__device__ inline float row_scale(float m)
{
    constexpr float half_max = std::is_same<TT, _Float16>::value ? 32752.0f : 0x1.fep126f;
    return fmaxf(m / half_max, FLT_MIN);
}

// Largest m of the block's NT threads, the same in every thread.
template<int NT>
__device__ inline float block_reduce_max(float m, float *s_max)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0)
        s_max[threadIdx.x >> 6] = m;
    __syncthreads();
    m = s_max[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++)
        m = fmaxf(m, s_max[w]);
    return m;
}

// Largest magnitude of src[0..n) over the block's NT threads, the same in every thread.
template<int NT, bool Vec>
__device__ inline float block_max(const float *__restrict__ src, int64_t n, float *s_max)
{
    float m = 0.0f;
    if (Vec) {
        const float4 *s4 = reinterpret_cast<const float4 *>(src);
        constexpr int U = 8;                       // loads in flight per thread
        int64_t i = threadIdx.x;
        for (; i + (U - 1) * NT < n / 4; i += U * NT) {
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                v[u] = s4[i + u * NT];
#pragma unroll
            for (int u = 0; u < U; u++)
                m = fmaxf(fmaxf(m, fmaxf(fabsf(v[u].x), fabsf(v[u].y))), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
        }
        for (; i < n / 4; i += NT) {
            const float4 v = s4[i];
            m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
        }
    }
    else {
        for (int64_t i = threadIdx.x; i < n; i += NT)
            m = fmaxf(m, fabsf(src[i]));
    }
    return block_reduce_max<NT>(m, s_max);
}

// Correctly rounded x / sc from the rounded reciprocal of sc: a product and two corrections by FMA
// (P. W. Markstein, IBM J. Res. Dev. 34, 1990: a quotient within an ulp becomes the rounded one),
// 5 instructions where a division takes 10. It needs remainders that are exact: no underflow of
// |x| 2^-48, no overflow of 1 / sc.
struct RowQuotient
{
    float sc, r;
    bool fast;

    __device__ explicit RowQuotient(float s) : sc(s), r(1.0f / s), fast(s >= 0x1p-126f && s <= 0x1p+100f) { }
    // Least and largest magnitude of a set of values (zeros are exact and left out), and whether they
    // are in range.
    __device__ static void range(float x, uint32_t &lo, uint32_t &hi)
    {
        const uint32_t b = __float_as_uint(x) & 0x7fffffffu;
        lo = min(lo, b - 1);
        hi = max(hi, b);
    }
    __device__ bool covers(uint32_t lo, uint32_t hi) const
    {
        return fast && lo >= __float_as_uint(0x1p-90f) - 1 && hi < 0x7f800000u;
    }
    __device__ float operator()(float x) const
    {
        float q = x * r;
        q = fmaf(fmaf(-q, sc, x), r, q);
        return fmaf(fmaf(-q, sc, x), r, q);
    }
};

__device__ inline void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A lane's ENC_TILE samples in LDS (own) become their encoded values, each four in the first half of
// the slot of theirs. fast: the quotients come from the reciprocal, ahead of the chain of feedbacks, and
// no value or rounding error is infinite or NaN.
template<typename TT, int Order>
__device__ inline void feedback_tile(float *__restrict__ own, const RowQuotient &div, bool fast, float &e1, float &e2)
{
    typedef TT tv4 __attribute__((ext_vector_type(4)));
    if (fast) {
        auto step = [&](float x) {
            const float u = x + ((Order == 1) ? e1 : 2.0f * e1 - e2);
            const TT q = TT(u);
            e2 = e1;
            e1 = u - float(q);
            return q;
        };
        float4 next = *reinterpret_cast<const float4 *>(own);
#pragma unroll 4
        for (int j = 0; j < ENC_TILE; j += 4) {
            const float x0 = div(next.x), x1 = div(next.y), x2 = div(next.z), x3 = div(next.w);
            next = *reinterpret_cast<const float4 *>(own + ((j + 4 < ENC_TILE) ? j + 4 : 0));
            tv4 o;
            o.x = step(x0);
            o.y = step(x1);
            o.z = step(x2);
            o.w = step(x3);
            *reinterpret_cast<tv4 *>(own + j) = o;
        }
    }
    else {
#pragma unroll 1
        for (int j = 0; j < ENC_TILE; j += 4) {
            const float4 x4 = *reinterpret_cast<const float4 *>(own + j);
            const float x[4] = { x4.x, x4.y, x4.z, x4.w };
            tv4 o;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float u = x[k] / div.sc + ((Order == 1) ? e1 : 2.0f * e1 - e2);
                const TT q = TT(u);
                float e = u - float(q);
                e = (fabsf(e) <= FLT_MAX) ? e : 0.0f;
                e2 = e1;
                e1 = e;
                o[k] = q;
            }
            *reinterpret_cast<tv4 *>(own + j) = o;
        }
    }
}

// Error feedback over 64 of a row's runs (chains 64 * group ...), one per lane of the calling wave. The
// runs are read and written a tile of ENC_TILE samples of each at a time, consecutive lanes taking
// consecutive samples of a run, and LDS turns the tile between that order and a lane per run. 's' holds
// 64 * ENC_STRIDE floats of the wave's own. A wave of few on its SIMD waits for its loads: whole tiles
// (Vec: a multiple of 4 samples per row and run, 16-byte aligned) are loaded one ahead, without branches
// around an access, which would make the compiler wait for every access in flight.
template<typename TT, int Order, bool Vec>
__device__ inline void encode_chains(TT *__restrict__ dst, const float *__restrict__ src, int64_t row_len, float sc,
                                     int group, float *__restrict__ s)
{
    typedef TT tv4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const int64_t run = (row_len + ENC_CHAINS - 1) / ENC_CHAINS;
    const int64_t first = int64_t(group) * 64 * run;
    if (first >= row_len)
        return;
    const RowQuotient div(sc);
    float e1 = 0.0f, e2 = 0.0f;
    int64_t t0 = 0;

    if constexpr (Vec) {
        constexpr int LPR = ENC_TILE / 4, RPA = 64 / LPR, NACC = 64 / RPA;   // lanes per run, runs per access, accesses
        const int64_t nwhole = (first + 64 * run <= row_len) ? run / ENC_TILE * ENC_TILE : 0;
        // Access i: run i * RPA + lane / LPR, samples 4 * (lane % LPR) ...: a uniform base and a lane offset.
        const uint32_t ofs = uint32_t(lane / LPR) * uint32_t(run) + 4 * uint32_t(lane % LPR);
        float *place = s + (lane / LPR) * ENC_STRIDE + 4 * (lane % LPR);
        float4 v[NACC];
        auto load = [&](int64_t t) {
#pragma unroll
            for (int i = 0; i < NACC; i++)
                v[i] = *reinterpret_cast<const float4 *>(src + (first + t + i * RPA * run) + ofs);
        };
        if (nwhole > 0)
            load(0);
        for (; t0 < nwhole; t0 += ENC_TILE) {
            uint32_t lo = 0xffffffffu, hi = 0;
#pragma unroll
            for (int i = 0; i < NACC; i++) {
                *reinterpret_cast<float4 *>(place + i * RPA * ENC_STRIDE) = v[i];
                div.range(v[i].x, lo, hi);
                div.range(v[i].y, lo, hi);
                div.range(v[i].z, lo, hi);
                div.range(v[i].w, lo, hi);
            }
            load((t0 + ENC_TILE < nwhole) ? t0 + ENC_TILE : 0);
            const bool fast = !__any(!div.covers(lo, hi));
            wave_sync_lds();
            feedback_tile<TT, Order>(s + lane * ENC_STRIDE, div, fast, e1, e2);
            wave_sync_lds();
#pragma unroll
            for (int i = 0; i < NACC; i++)
                *reinterpret_cast<tv4 *>(dst + (first + t0 + i * RPA * run) + ofs) =
                    *reinterpret_cast<const tv4 *>(place + i * RPA * ENC_STRIDE);
            wave_sync_lds();
        }
    }

    // The rest, sample by sample: the runs' last tile, the row's last group, or everything.
    constexpr int RPA = 64 / ENC_TILE;
    const int col = lane % ENC_TILE;
    for (; t0 < run; t0 += ENC_TILE) {
        uint32_t lo = 0xffffffffu, hi = 0;
        const bool in = t0 + col < run;
        const int64_t p0 = first + int64_t(lane / ENC_TILE) * run + t0 + col;
#pragma unroll 8
        for (int i = 0; i < 64 / RPA; i++) {
            const int64_t p = p0 + i * RPA * run;
            const float x = (in && p < row_len) ? src[p] : 0.0f;
            s[(i * RPA + lane / ENC_TILE) * ENC_STRIDE + col] = x;
            div.range(x, lo, hi);
        }
        const bool fast = !__any(!div.covers(lo, hi));
        wave_sync_lds();
        feedback_tile<TT, Order>(s + lane * ENC_STRIDE, div, fast, e1, e2);
        wave_sync_lds();
#pragma unroll 8
        for (int i = 0; i < 64 / RPA; i++) {
            const int64_t p = p0 + i * RPA * run;
            const float *slot = s + (i * RPA + lane / ENC_TILE) * ENC_STRIDE + (col & ~3);
            if (in && p < row_len)
                dst[p] = reinterpret_cast<const TT *>(slot)[col & 3];
        }
        wave_sync_lds();
    }
}

// Samples [i0, i1) rounded independently by the block's threads.
template<typename TT, bool Vec, int NT>
__device__ inline void encode_plain(TT *__restrict__ dst, const float *__restrict__ src, int64_t i0, int64_t i1, float sc)
{
    typedef TT tv4 __attribute__((ext_vector_type(4)));
    if (Vec) {
#pragma unroll 4
        for (int64_t i = i0 / 4 + threadIdx.x; i < i1 / 4; i += NT) {
            const float4 x = reinterpret_cast<const float4 *>(src)[i];
            const tv4 o = { TT(x.x / sc), TT(x.y / sc), TT(x.z / sc), TT(x.w / sc) };
            reinterpret_cast<tv4 *>(dst)[i] = o;
        }
    }
    else {
        for (int64_t i = i0 + threadIdx.x; i < i1; i += NT)
            dst[i] = TT(src[i] / sc);
    }
}

// Short rows, one block of NT threads each (64 or 128 when the row has no more samples: the waves without
// any take their time too): a lane keeps its run, of at most ENC_WALK samples, in registers, so that the
// row is read once. Staged, a whole tile moves for the few samples of such a run: 100000 rows of 64 samples
// with feedback 648 us staged, 49 here, 8000 of 1024 88 and 35, 4000 of 2048 59 and 34. Vec: rows and runs
// of whole groups of four, as for encode_chains.
constexpr int ENC_WALK = 8;

template<typename TT, int Order, bool Vec, int NT>
__global__ void __launch_bounds__(NT)
tod16_walk_kernel(TT *__restrict__ out, float *__restrict__ scale, const float *__restrict__ tod, int64_t row_len, int run)
{
    // u is rounded before it is rounded to 16 bits: no x + 2 e as an FMA with a 16-bit result.
#pragma clang fp contract(off)
    typedef TT tv4 __attribute__((ext_vector_type(4)));
    __shared__ float s_max[NT / 64];
    const float *src = tod + int64_t(blockIdx.x) * row_len;
    TT *dst = out + int64_t(blockIdx.x) * row_len;
    const int first = int(threadIdx.x) * run, n = min(run, int(row_len) - first);      // n <= 0 past the end
    float v[ENC_WALK], m = 0.0f;
#pragma unroll
    for (int k = 0; k < ENC_WALK; k += 4)
        if (Vec && k < run) {
            const float4 x = (k < n) ? *reinterpret_cast<const float4 *>(src + first + k) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            v[k] = x.x;
            v[k + 1] = x.y;
            v[k + 2] = x.z;
            v[k + 3] = x.w;
        }
#pragma unroll
    for (int k = 0; k < ENC_WALK; k++)
        if (k < run) {
            if (!Vec)
                v[k] = (k < n) ? src[first + k] : 0.0f;
            m = fmaxf(m, fabsf(v[k]));
        }
    const float sc = row_scale<TT>(block_reduce_max<NT>(m, s_max));
    if (threadIdx.x == 0)
        scale[blockIdx.x] = sc;
    float e1 = 0.0f, e2 = 0.0f;
    tv4 o;
#pragma unroll
    for (int k = 0; k < ENC_WALK; k++)
        if (k < run) {
            float u = v[k] / sc;
            if (Order)
                u += (Order == 1) ? e1 : 2.0f * e1 - e2;      // also of zeros: -0 + 0 is 0
            const TT q = TT(u);
            const float e = u - float(q);
            e2 = e1;
            e1 = (fabsf(e) <= FLT_MAX) ? e : 0.0f;
            if (Vec) {
                o[k & 3] = q;
                if ((k & 3) == 3 && k < n)
                    *reinterpret_cast<tv4 *>(dst + first + k - 3) = o;
            }
            else if (k < n)
                dst[first + k] = q;
        }
}

// One block per row: its scale, by all of the block's waves, then its values (with error feedback by four
// of them, 64 runs each).
template<typename TT, int Order, bool Vec, int NT>
__global__ void __launch_bounds__(NT)
tod16_row_kernel(TT *__restrict__ out, float *__restrict__ scale, const float *__restrict__ tod, int64_t row_len)
{
    __shared__ float s_max[NT / 64];
    __shared__ __align__(16) float s_tile[Order ? ENC_CHAINS / 64 : 1][Order ? 64 * ENC_STRIDE : 1];
    const float *src = tod + int64_t(blockIdx.x) * row_len;
    TT *dst = out + int64_t(blockIdx.x) * row_len;
    const float sc = row_scale<TT>(block_max<NT, Vec>(src, row_len, s_max));
    if (threadIdx.x == 0)
        scale[blockIdx.x] = sc;
    if constexpr (Order == 0)
        encode_plain<TT, Vec, NT>(dst, src, 0, row_len, sc);
    else if (threadIdx.x < ENC_CHAINS)
        encode_chains<TT, Order, Vec>(dst, src, row_len, sc, int(threadIdx.x >> 6), s_tile[threadIdx.x >> 6]);
}

// Few long rows: 'nsplit' blocks per row find its largest magnitude, one value each in 'part' (the
// start of the output, which the encoding overwrites) ...
template<bool Vec>
__global__ void __launch_bounds__(ENC_THREADS)
tod16_split_max_kernel(float *__restrict__ part, const float *__restrict__ tod, int64_t row_len, int nsplit)
{
    __shared__ float s_max[ENC_THREADS / 64];
    const int64_t row = blockIdx.x / nsplit;
    const int i = int(blockIdx.x % nsplit);
    const int64_t per = ((row_len + nsplit - 1) / nsplit + 3) & ~int64_t(3);
    const int64_t i0 = min(row_len, i * per), i1 = min(row_len, i0 + per);
    const float m = block_max<ENC_THREADS, Vec>(tod + row * row_len + i0, i1 - i0, s_max);
    if (threadIdx.x == 0)
        part[blockIdx.x] = m;
}

// ... a wave per row takes the largest of them ...
template<typename TT>
__global__ void __launch_bounds__(64)
tod16_split_scale_kernel(const float *__restrict__ part, float *__restrict__ scale, int nsplit)
{
    float m = 0.0f;
    for (int i = threadIdx.x; i < nsplit; i += 64)
        m = fmaxf(m, part[int64_t(blockIdx.x) * nsplit + i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        m = fmaxf(m, __shfl_xor(m, off, 64));
    if (threadIdx.x == 0)
        scale[blockIdx.x] = row_scale<TT>(m);
}

// ... and the row is encoded by one block per 64 runs, or (independent rounding) by 'nsplit' blocks.
template<typename TT, int Order, bool Vec>
__global__ void __launch_bounds__(Order ? 64 : ENC_THREADS)
tod16_split_encode_kernel(TT *__restrict__ out, const float *__restrict__ scale, const float *__restrict__ tod,
                          int64_t row_len, int nsplit)
{
    __shared__ __align__(16) float s_tile[Order ? 64 * ENC_STRIDE : 1];
    const int64_t row = blockIdx.x / nsplit;
    const int i = int(blockIdx.x % nsplit);
    const float sc = scale[row];
    const float *src = tod + row * row_len;
    TT *dst = out + row * row_len;
    if constexpr (Order == 0) {
        const int64_t per = ((row_len + nsplit - 1) / nsplit + 3) & ~int64_t(3);
        const int64_t i0 = min(row_len, i * per);
        encode_plain<TT, Vec, ENC_THREADS>(dst, src, i0, min(row_len, i0 + per), sc);
    }
    else
        encode_chains<TT, Order, Vec>(dst, src, row_len, sc, i, s_tile);
}

// A block per row when the rows fill the GPU, or when a row is so short that two more launches cost
// more than one block takes to read it (65536 samples: 20 us in one block, 8 + 13 us in three launches);
// else several blocks per row.
constexpr int64_t ENC_ROWS = 256;
constexpr int64_t ENC_SHORT = 16384;
constexpr int64_t ENC_SPLIT_MIN = 4096;            // samples per block of a split row, at least

template<typename TT, int Order, bool Vec>
void encode_order(TT *out, float *scale, const float *tod, int64_t nrows, int64_t row_len, hipStream_t stream)
{
    // Independent rounding has no runs: from 256 samples on, groups of four are as fast or faster.
    if (row_len <= (Order ? ENC_WALK * ENC_CHAINS : ENC_CHAINS)) {
        const int run = int((row_len + ENC_CHAINS - 1) / ENC_CHAINS);
        if (row_len <= 64)
            tod16_walk_kernel<TT, Order, false, 64><<<unsigned(nrows), 64, 0, stream>>>(out, scale, tod, row_len, run);
        else if (row_len <= 128)
            tod16_walk_kernel<TT, Order, false, 128><<<unsigned(nrows), 128, 0, stream>>>(out, scale, tod, row_len, run);
        else
            tod16_walk_kernel<TT, Order, Vec && Order != 0, ENC_CHAINS><<<unsigned(nrows), ENC_CHAINS, 0, stream>>>(
                out, scale, tod, row_len, run);
        return;
    }
    if (nrows >= ENC_ROWS || row_len <= ENC_SHORT) {
        // 16 waves keep enough loads in flight for the scale of a long row (512 x 131072: 127 us against
        // 133 with 4); a short one has no use for them.
        if (row_len <= ENC_SHORT)
            tod16_row_kernel<TT, Order, Vec, 256><<<unsigned(nrows), 256, 0, stream>>>(out, scale, tod, row_len);
        else
            tod16_row_kernel<TT, Order, Vec, 1024><<<unsigned(nrows), 1024, 0, stream>>>(out, scale, tod, row_len);
        return;
    }
    const int nsplit = int(std::min<int64_t>((1024 + nrows - 1) / nrows, row_len / ENC_SPLIT_MIN));
    // 4 bytes per block at the start of the output, which holds at least 2 * ENC_SPLIT_MIN per block.
    float *part = reinterpret_cast<float *>((reinterpret_cast<uintptr_t>(out) + 3) & ~uintptr_t(3));
    tod16_split_max_kernel<Vec><<<unsigned(nrows * nsplit), ENC_THREADS, 0, stream>>>(part, tod, row_len, nsplit);
    tod16_split_scale_kernel<TT><<<unsigned(nrows), 64, 0, stream>>>(part, scale, nsplit);
    const int ngroup = Order ? ENC_CHAINS / 64 : nsplit;
    tod16_split_encode_kernel<TT, Order, Vec><<<unsigned(nrows * ngroup), Order ? 64 : ENC_THREADS, 0, stream>>>(
        out, scale, tod, row_len, ngroup);
}

template<typename TT>
void encode_typed(TT *out, float *scale, const float *tod, int64_t nrows, int64_t row_len, int order, hipStream_t stream)
{
    // Whole groups of 4 samples per row and per run, 16-byte aligned input and 8-byte aligned output.
    const int64_t run = (row_len + ENC_CHAINS - 1) / ENC_CHAINS;
    const bool vec = (row_len % 4 == 0) && (order == 0 || run % 4 == 0)
                     && (reinterpret_cast<uintptr_t>(tod) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
    auto go = [&](auto o) {
        constexpr int Order = decltype(o)::value;
        if (vec)
            encode_order<TT, Order, true>(out, scale, tod, nrows, row_len, stream);
        else
            encode_order<TT, Order, false>(out, scale, tod, nrows, row_len, stream);
    };
    if (order == 2)
        go(std::integral_constant<int, 2>());
    else if (order == 1)
        go(std::integral_constant<int, 1>());
    else
        go(std::integral_constant<int, 0>());
}

}  // namespace

void launch_tod16_encode(void *out, int tod_type, float *scale, const float *tod, int64_t nrows,
                         int64_t row_len, int error_feedback, hipStream_t stream)
{
    if (tod_type == TOD_F16)
        encode_typed(static_cast<_Float16 *>(out), scale, tod, nrows, row_len, error_feedback, stream);
    else
        encode_typed(static_cast<__bf16 *>(out), scale, tod, nrows, row_len, error_feedback, stream);
    GMM_HIP(hipGetLastError());
}

}  // namespace gmm
