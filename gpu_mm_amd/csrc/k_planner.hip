// Plan construction on gfx950: preplan count, deterministic emit, device scan, stable LSD
// radix sort in LDS, and the operators' work lists. All kernels assume 64-lane waves.

#include "gmm_internal.hpp"
#include "gmm_locate.hpp"
#include "gmm_wave.hpp"

namespace gmm {

namespace {

constexpr int WAVE = 64;

__device__ inline int lane_id() { return threadIdx.x & 63; }

__device__ inline uint64_t lanemask_lt() { return (1ull << lane_id()) - 1ull; }

__device__ inline uint32_t wave_reduce_or(uint32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v |= __shfl_xor(v, off, WAVE);
    return v;
}

__device__ inline uint32_t wave_reduce_add(uint32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, WAVE);
    return v;
}

// One extraction round over the remaining candidate cells of the two half-waves.
// 'k' holds up to four distinct candidate keys per lane (NO_CELL = none). Returns false when
// both halves are exhausted; otherwise removes one cell per non-empty half from every lane of
// that half and returns it in 'c' (NO_CELL for an exhausted half).
__device__ inline bool extract_one(uint32_t k[4], uint32_t &c, bool &lo_hit, bool &hi_hit)
{
    uint32_t first = (k[0] != NO_CELL) ? k[0] : ((k[1] != NO_CELL) ? k[1] : ((k[2] != NO_CELL) ? k[2] : k[3]));
    uint64_t m = __ballot(first != NO_CELL);
    if (m == 0)
        return false;
    uint32_t mlo = uint32_t(m), mhi = uint32_t(m >> 32);
    uint32_t clo = NO_CELL, chi = NO_CELL;
    if (mlo)
        clo = __builtin_amdgcn_readlane(first, __builtin_ctz(mlo));
    if (mhi)
        chi = __builtin_amdgcn_readlane(first, 32 + __builtin_ctz(mhi));
    lo_hit = (mlo != 0);
    hi_hit = (mhi != 0);
    c = (lane_id() < 32) ? clo : chi;
#pragma unroll
    for (int j = 0; j < 4; j++)
        k[j] = (k[j] == c) ? NO_CELL : k[j];
    return true;
}

// The four corner indices of a sample's bilinear footprint (locate_pixel's,
// include/gpu_mm_internals.hpp:124-164), located by locate_op with its range checks deferred to
// 'chk'.
template<bool Periodic>
__device__ inline void sample_corners(float y, float x, const Geom &g, Checks &chk, Pixel<float> &p)
{
    float dy, dx;
    locate_op<Periodic>(y, x, g, chk, p.iy0, p.ix0, dy, dx);
    p.iy1 = p.iy0 + 1;
    p.ix1 = Periodic ? ((p.ix0 + 1 < g.nx) ? p.ix0 + 1 : 0) : p.ix0 + 1;
}

// Footprint cells of one sample. An inactive lane holds NO_CELL everywhere; its y = x = 0 lie in
// range and leave the checks unchanged.
template<bool Periodic>
__device__ inline void sample_cells(float y, float x, const Geom &g, Checks &chk, bool active, uint32_t k[4])
{
    Pixel<float> p;
    sample_corners<Periodic>(y, x, g, chk, p);
    footprint_cells(p, k);
    if (!active)
        k[0] = k[1] = k[2] = k[3] = NO_CELL;
}

// ------------------------------------------------------------------------------------------
// Both passes over the pointing (count and emit) read a 32-sample line with eight lanes, four samples
// each, a wave eight lines at a time. The cells of a line come from the range of its coordinates: trunc
// and the shift to cells are monotonic, so the lowest corner's cell and the highest one's bound the
// line, and when they are the same or neighbours along one axis, the line's cells are exactly these
// (the lowest sample touches the one, the highest the other). A line that spans two cells along both
// axes takes the union of its samples' corners in these 2 x 2 cells. Anything else (longer lines, the
// wrap of periodic x) is found sample by sample, by repeated extraction, two such lines at a time: 4.2e6
// scattered samples take 154 us to count and 597 us in all to plan (one line at a time, loaded again for
// the count and the emit's two passes, 202 and 760; sample by sample throughout 159 and 629); 6.7e7 at 3
// pixels per sample 223 and 840 us (266 and 1010; 321 and 1024).
// Working through every sample's four corners, with ballots over them, took 68 and 101 instructions
// per sample, 0.93 and 1.38 ms of VALU issue in the 1.01 and 1.62 ms of the passes on 2048x262144
// samples. By ranges the count takes 0.65 ms (6.7 TB/s: the 4.3 GB it reads) and the emit 0.89 ms (41
// instructions per sample, 0.56 ms; loading a step ahead spills and takes 0.98).

constexpr int SCAN_LINES = 8;                 // lines per wave and load

// One lane's four samples: the range of their coordinates as bit patterns of c + 0 (as in Checks: those
// of valid coordinates are in the order of the numbers).
struct QuadRange
{
    uint32_t ylo, yhi, xlo, xhi;
};

// y and x of the lane's samples: n (0..4) of them from p = the first one's y on (the first one's values
// beyond n, zeros when n == 0). Non-temporal: each pass reads its pointing once (count 757 -> 635 us).
template<bool Vec>
__device__ inline void load_quad(const float *__restrict__ p, int64_t nsamp, int n, float (&y)[4], float (&x)[4])
{
    if (Vec) {
        typedef float f4v __attribute__((ext_vector_type(4)));
        f4v a = { 0.0f, 0.0f, 0.0f, 0.0f }, b = a;
        if (n > 0) {
            a = __builtin_nontemporal_load(reinterpret_cast<const f4v *>(p));
            b = __builtin_nontemporal_load(reinterpret_cast<const f4v *>(p + nsamp));
        }
        y[0] = a.x; y[1] = a.y; y[2] = a.z; y[3] = a.w;
        x[0] = b.x; x[1] = b.y; x[2] = b.z; x[3] = b.w;
    }
    else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int j = (k < n) ? k : 0;
            y[k] = (n > 0) ? p[j] : 0.0f;
            x[k] = (n > 0) ? p[nsamp + j] : 0.0f;
        }
    }
}

// Samples of lines [line, l1) that exist (the last line may be partial), at most 'cap': wave-uniform, so
// that a lane's count is one clamp of the difference to its place.
__device__ inline int samples_left(int64_t line, int64_t l1, int64_t nsamp, int cap)
{
    return int(max<int64_t>(0, min<int64_t>(cap, min(nsamp, l1 * LINE) - line * LINE)));
}

// Lines a wave takes at a time: eight, or fewer where the blocks don't fill the GPU and have not as many for
// each wave, for the sake of slow ones, which a wave does in pairs (preplan of 32768 scattered samples 59 us,
// 45 so; with the GPU full it costs the count of ordinary lines 1.6 us).
__device__ inline int lines_per_wave(int64_t nlines, int nwaves)
{
    return (gridDim.x < 256) ? int(min<int64_t>(SCAN_LINES, (nlines + nwaves - 1) / nwaves)) : SCAN_LINES;
}

// x after the wrap of locate_op: in [0, nx] for every valid x.
template<bool Periodic>
__device__ inline float wrap_x(float x, const Geom &g)
{
    if (Periodic) {
        x = (x >= 0.0f) ? x : (x + g.fnx);
        x = (x <= g.fnx) ? x : (x - g.fnx);
    }
    return x;
}

__device__ inline void range4(const float (&v)[4], uint32_t &lo, uint32_t &hi)
{
    uint32_t b[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        b[k] = __float_as_uint(v[k] + 0.0f);
    lo = min(min(b[0], b[1]), min(b[2], b[3]));
    hi = max(max(b[0], b[1]), max(b[2], b[3]));
}

// Range of a lane's samples, the checks of locate_op added to chk. x is left wrapped.
template<bool Periodic>
__device__ inline QuadRange quad_range(const float (&y)[4], float (&x)[4], bool on, const Geom &g, Checks &chk)
{
    if (Periodic) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            chk.px = fmaxf(chk.px, fmaxf(g.xlo - x[k], x[k] - g.xhi));
            chk.pn += x[k];
            x[k] = wrap_x<true>(x[k], g);
        }
    }
    QuadRange r;
    range4(y, r.ylo, r.yhi);
    range4(x, r.xlo, r.xhi);
    chk.uy = max(chk.uy, r.yhi);
    if (!Periodic)
        chk.ux = max(chk.ux, r.xhi);
    if (!on) {
        r.ylo = r.xlo = 0xffffffffu;
        r.yhi = r.xhi = 0;
    }
    return r;
}

template<bool Periodic>
__device__ inline int pixel_x(float x, const Geom &g) { return int(clamp0(x, Periodic ? g.fnx : g.fnx2)); }
template<bool Periodic>
__device__ inline int pixel_x(uint32_t bits, const Geom &g) { return pixel_x<Periodic>(__uint_as_float(bits), g); }
__device__ inline int pixel_y(float y, const Geom &g) { return int(clamp0(y, g.fny2)); }
__device__ inline int pixel_y(uint32_t bits, const Geom &g) { return pixel_y(__uint_as_float(bits), g); }

// Cells of one line, the same in its eight lanes: bit 2 * r + c of 'at' stands for cell (cy + r,
// cx + c). slow: found sample by sample instead (at = 0).
struct LineCells
{
    int cy, cx;
    int xhi;               // largest ix0 of the line
    uint32_t at;
    bool slow;
};

template<bool Periodic>
__device__ inline LineCells line_cells(const QuadRange &q, const float (&y)[4], const float (&x)[4], bool on,
                                       const Geom &g)
{
    auto umin = [](uint32_t a, uint32_t b) { return min(a, b); };
    auto umax = [](uint32_t a, uint32_t b) { return max(a, b); };
    const uint32_t ylo = group8_reduce(q.ylo, umin), yhi = group8_reduce(q.yhi, umax);
    const uint32_t xlo = group8_reduce(q.xlo, umin), xhi = group8_reduce(q.xhi, umax);
    LineCells l;
    l.xhi = pixel_x<Periodic>(xhi, g);
    l.cy = pixel_y(ylo, g) >> 6;
    l.cx = pixel_x<Periodic>(xlo, g) >> 6;
    const int dy = ((pixel_y(yhi, g) + 1) >> 6) - l.cy, dx = ((l.xhi + 1) >> 6) - l.cx;
    // Periodic x: ix0 = nx - 1 (and x = nx, which is pixel 0) have a corner at ix = 0.
    l.slow = (unsigned(dy) > 1u) || (unsigned(dx) > 1u) || (Periodic && l.xhi + 1 >= g.nx);
    l.at = l.slow ? 0u : 1u | (uint32_t(dx) << 1) | (uint32_t(dy) << 2);
    const bool both = !l.slow && dx + dy == 2;
    if (__any(both)) {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int iy = pixel_y(y[k], g), ix = pixel_x<Periodic>(x[k], g);
            const int r0 = (iy >> 6) - l.cy, r1 = ((iy + 1) >> 6) - l.cy, c0 = (ix >> 6) - l.cx, c1 = ((ix + 1) >> 6) - l.cx;
            const uint32_t cols = (1u << (c0 & 1)) | (1u << (c1 & 1));
            m |= (cols << (2 * (r0 & 1))) | (cols << (2 * (r1 & 1)));
        }
        m = group8_reduce(on ? m : 0u, [](uint32_t a, uint32_t b) { return a | b; });
        l.at = both ? m : l.at;
    }
    return l;
}

// The samples of a wave's eight lines in LDS, for those of its lines that are slow.
struct __align__(16) WaveSamples
{
    float y[SCAN_LINES * LINE], x[SCAN_LINES * LINE];

    __device__ void put(const float (&yq)[4], const float (&xq)[4])
    {
        const int lane = lane_id();
        *reinterpret_cast<float4 *>(y + 4 * lane) = make_float4(yq[0], yq[1], yq[2], yq[3]);
        *reinterpret_cast<float4 *>(x + 4 * lane) = make_float4(xq[0], xq[1], xq[2], xq[3]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// Two slow lines at a time, la in lanes 0..31 and lb in 32..63 (lb = la: one line only), a sample per lane:
// their footprint cells go to k for extract_one(). s0: first sample of the wave's lines.
template<bool Periodic>
__device__ inline void slow_pair(const WaveSamples &w, int la, int lb, int64_t s0, int64_t nsamp, const Geom &g, uint32_t k[4])
{
    const int lane = lane_id(), i = LINE * ((lane < 32) ? la : lb) + (lane & 31);
    Checks unchecked;                          // the line's ranges were checked already
    const bool act = (lane < 32 || lb != la) && s0 + i < nsamp;
    sample_cells<Periodic>(w.y[i], w.x[i], g, unchecked, act, k);
}

// The next pair of the slow lines in m, a bit for the first lane of each.
__device__ inline void next_pair(uint64_t &m, int &la, int &lb)
{
    la = __builtin_ctzll(m) >> 3;
    m &= m - 1;
    lb = m ? __builtin_ctzll(m) >> 3 : la;
    m &= m - 1;
}

// ------------------------------------------------------------------------------------------
// Preplan: number of distinct (line, cell) pairs per planner block
// (src_lib/PointingPrePlan.cu:37-108 computes the same per-block counts).

constexpr int PP_THREADS = 512;
constexpr int PP_UNROLL = 2;

template<bool Periodic, bool Vec>
__global__ void __launch_bounds__(PP_THREADS) __attribute__((amdgpu_waves_per_eu(8)))
preplan_count_kernel(const float *__restrict__ xp, int64_t nsamp, int64_t ncl, int64_t ncl_per_block,
                     int ny, int nx, uint32_t *__restrict__ nmt_out, uint32_t *__restrict__ err_out)
{
    __shared__ uint32_t s_cnt[PP_THREADS / WAVE], s_err[PP_THREADS / WAVE];
    __shared__ WaveSamples s_samples[PP_THREADS / WAVE];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    constexpr int NW = PP_THREADS / WAVE;
    const int q = lane & 7;

    const int64_t l0 = int64_t(blockIdx.x) * ncl_per_block;
    const int64_t l1 = min(ncl, l0 + ncl_per_block);
    uint32_t cnt = 0;                          // lanes q == 0: cells of the lane's lines
    uint32_t slow_cnt = 0;                     // wave-uniform
    const Geom g = make_geom(ny, nx, Periodic);
    Checks chk;

    const int lpw = lines_per_wave(l1 - l0, NW);
    for (int64_t lb = l0 + lpw * wave; lb < l1; lb += lpw * NW * PP_UNROLL) {
        float y[PP_UNROLL][4], x[PP_UNROLL][4];
        int n[PP_UNROLL];
#pragma unroll
        for (int u = 0; u < PP_UNROLL; u++) {
            const int64_t line = lb + lpw * NW * u;                // the wave's first line of the group
            n[u] = min(max(samples_left(line, l1, nsamp, lpw * LINE) - 4 * lane, 0), 4);
            load_quad<Vec>(xp + line * LINE + 4 * lane, nsamp, n[u], y[u], x[u]);
        }
#pragma unroll
        for (int u = 0; u < PP_UNROLL; u++) {
            const QuadRange r = quad_range<Periodic>(y[u], x[u], n[u] > 0, g, chk);
            const LineCells l = line_cells<Periodic>(r, y[u], x[u], n[u] > 0, g);
            const bool lead = (q == 0) && n[u] > 0;
            cnt += lead ? uint32_t(__popc(l.at)) : 0u;
            uint64_t m = __ballot(lead && l.slow);
            if (m)
                s_samples[wave].put(y[u], x[u]);
            while (m) {
                int la, lb2;
                next_pair(m, la, lb2);
                uint32_t k[4], c;
                slow_pair<Periodic>(s_samples[wave], la, lb2, (lb + lpw * NW * u) * LINE, nsamp, g, k);
                bool lo, hi;
                while (extract_one(k, c, lo, hi))
                    slow_cnt += uint32_t(lo) + uint32_t(hi);
            }
        }
    }

    const uint32_t err = wave_reduce_or(chk.bits(g));
    cnt = wave_reduce_add(cnt) + slow_cnt;
    if (lane == 0) {
        s_cnt[wave] = cnt;
        s_err[wave] = err;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t c = 0, e = 0;
        for (int w = 0; w < NW; w++) {
            c += s_cnt[w];
            e |= s_err[w];
        }
        nmt_out[blockIdx.x] = c;
        err_out[blockIdx.x] = e;
    }
}

// Inclusive scan of the per-block counts (padded to PREPLAN_SIZE with the total) and OR of the
// error words into err[0]; the 64-bit total goes to err[1] (low) and err[2] (high).
// One block of PREPLAN_SIZE threads. Replaces the host round trip of PointingPrePlan.cu:195-216.
__global__ void __launch_bounds__(PREPLAN_SIZE)
preplan_finish_kernel(uint32_t *nmt, uint32_t *err, int nblocks)
{
    constexpr int NW = PREPLAN_SIZE / WAVE;
    __shared__ uint32_t s_wave[NW], s_lo[NW], s_hi[NW], s_err[NW];
    const int t = threadIdx.x;
    uint32_t v = (t < nblocks) ? nmt[t] : 0u;
    // The total in 64 bits from sums of 16-bit halves (all lanes adding to one word take 6 us).
    const uint32_t lo = wave_reduce_add(v & 0xffffu), hi = wave_reduce_add(v >> 16);
    const uint32_t e = wave_reduce_or((t < nblocks) ? err[t] : 0u);
    if (lane_id() == 0) {
        s_lo[t / WAVE] = lo;
        s_hi[t / WAVE] = hi;
        s_err[t / WAVE] = e;
    }
    uint32_t total;
    uint32_t excl = block_exclusive_scan<PREPLAN_SIZE>(v, s_wave, total);   // synchronizes
    nmt[t] = (t < nblocks) ? (excl + v) : total;
    if (t == 0) {
        uint64_t sum = 0;
        uint32_t flags = 0;
        for (int w = 0; w < NW; w++) {
            sum += uint64_t(s_lo[w]) + (uint64_t(s_hi[w]) << 16);
            flags |= s_err[w];
        }
        err[0] = flags;
        err[1] = uint32_t(sum);
        err[2] = uint32_t(sum >> 32);
    }
}

// ------------------------------------------------------------------------------------------
// Emit: writes the plan entries of each planner block into its window
// [nmt_cumsum[b-1], nmt_cumsum[b]) in line order; inside a line in an order that the sort by cell
// replaces. The entry layout and the consistency check against the preplan count follow
// src_lib/PointingPlan.cu:75-89, 116, 227. Bits 48..63 carry the entry's owned-quad mask through the
// sort (its last pass stores it apart): the ranges give it for lines of one or two cells, others are
// marked QM_PENDING and done by qmask_kernel afterwards.

constexpr int EM_THREADS = 512;
constexpr int EM_NW = EM_THREADS / WAVE;               // 64 lines per block step (128 measure the same)
constexpr uint16_t QM_PENDING = 0x8000;
constexpr int QM_SHIFT = 48;
constexpr int NML_SHIFT = 8;

// At most 64 VGPRs (8 waves per SIMD, 4 blocks per CU): the planner grid (1024 blocks at most)
// is then resident at once on 256 CUs instead of leaving a tail.
template<bool Periodic, bool Vec>
__global__ void __launch_bounds__(EM_THREADS) __attribute__((amdgpu_waves_per_eu(8)))
plan_emit_kernel(const float *__restrict__ xp, int64_t nsamp, int64_t ncl, int64_t ncl_per_block,
                 int ny, int nx, const uint32_t *__restrict__ nmt_cumsum,
                 uint64_t *__restrict__ out, uint32_t *__restrict__ err_out)
{
    __shared__ uint32_t s_total[2][EM_NW];
    __shared__ uint32_t s_err[EM_NW], s_nml[EM_NW];
    __shared__ WaveSamples s_samples[EM_NW];
    __shared__ uint32_t s_cells[EM_NW][SCAN_LINES][LINE];      // cells of the wave's slow lines
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int li = lane >> 3, q = lane & 7;
    const int b = blockIdx.x;

    const int64_t l0 = int64_t(b) * ncl_per_block;
    const int64_t l1 = min(ncl, l0 + ncl_per_block);
    const uint32_t base = (b > 0) ? nmt_cumsum[b - 1] : 0u;
    const uint32_t limit = nmt_cumsum[b] - base;
    out += base;

    uint32_t err = 0;
    uint32_t running = 0;   // entries written by earlier steps (block-uniform)
    uint32_t nml = 0;       // multi-cell lines (wave-uniform)
    const Geom g = make_geom(ny, nx, Periodic);
    Checks chk;
    int parity = 0;

    const int lpw = lines_per_wave(l1 - l0, EM_NW);
    for (int64_t ls = l0; ls < l1; ls += lpw * EM_NW) {
        const int64_t lw = ls + lpw * wave;                // the wave's first line
        const int n = min(max(samples_left(lw, l1, nsamp, lpw * LINE) - 4 * lane, 0), 4);
        float y[4], x[4];
        load_quad<Vec>(xp + lw * LINE + 4 * lane, nsamp, n, y, x);

        const bool on = n > 0, lead = (q == 0) && on;
        const QuadRange r = quad_range<Periodic>(y, x, on, g, chk);
        const LineCells l = line_cells<Periodic>(r, y, x, on, g);
        const uint64_t slow = __ballot(lead && l.slow);
        const uint64_t present = __ballot(on);
        const int shift = lane & ~7;
        const uint32_t quads = uint32_t(present >> shift) & 0xffu;
        // Lanes q < 4 write the line's cell number q, if it is one; its first sample's cell carries the
        // zflag.
        const uint32_t at = (quads & 1u) ? l.at : 0u;
        uint32_t cnt = lead ? uint32_t(__popc(at)) : 0u;
        uint32_t m = quads, z = 0;                          // owned quads of the lane's entry, its flags
        if (__any(at > 1u)) {
            // Two cells side by side: the left one evaluates all when the right one's samples (if it
            // owns any) lie in its halo; else, and for two cells in a column, each its own (the rule of
            // qmask_kernel).
            const bool xpair = at == 3u, ypair = at == 5u;
            const bool owns = (l.xhi >> 6) == l.cx + 1, takes = xpair && owns && (l.xhi & 63) <= HALO_X - 2;
            const bool each = ypair || (xpair && owns && !takes);
            if (at > 1u)
                m = (xpair && q == 0) ? (quads | (takes ? QM_TAKES_RIGHT : 0u)) : (xpair ? 0u : QM_PENDING);
            if (__any(each)) {
                const int ixlo = pixel_x<Periodic>(r.xlo, g), ixhi = pixel_x<Periodic>(r.xhi, g);
                const int iylo = pixel_y(r.ylo, g), iyhi = pixel_y(r.yhi, g);
                const bool first = on && (xpair ? (ixlo >> 6) == l.cx : (iylo >> 6) == l.cy);
                const bool second = on && (xpair ? (ixhi >> 6) == l.cx + 1 : (iyhi >> 6) == l.cy + 1);
                const uint32_t qa = uint32_t(__ballot(first) >> shift) & 0xffu, qb = uint32_t(__ballot(second) >> shift) & 0xffu;
                m = each ? ((q == 0) ? qa : qb) : m;
            }
            const uint32_t zc = uint32_t(2 * ((pixel_y(y[0], g) >> 6) - l.cy) + ((pixel_x<Periodic>(x[0], g) >> 6) - l.cx));
            const bool zf = dpp<DPP_QUAD0>(zc) == uint32_t(q);
            z = (at > 1u) ? (uint32_t(MFLAG >> 32) | (zf ? uint32_t(ZFLAG >> 32) : 0u)) : 0u;
            nml += uint32_t(__popcll(__ballot(lead && at > 1u)));
        }
        if (slow)
            s_samples[wave].put(y, x);
        for (uint64_t sm = slow; sm;) {
            int la, lb;
            next_pair(sm, la, lb);
            uint32_t k[4], c, nlo = 0, nhi = 0, mine = NO_CELL;
            slow_pair<Periodic>(s_samples[wave], la, lb, lw * LINE, nsamp, g, k);
            bool lo, hi;
            while (extract_one(k, c, lo, hi)) {
                mine = (uint32_t(lane & 31) == ((lane < 32) ? nlo : nhi)) ? c : mine;
                nlo += lo;
                nhi += hi;
            }
            if (mine != NO_CELL)
                s_cells[wave][(lane < 32) ? la : lb][lane & 31] = mine;
            cnt = (lane == 8 * la) ? nlo : ((lane == 8 * lb) ? nhi : cnt);
            nml += uint32_t(nlo > 1) + uint32_t(nhi > 1);
        }

        // Offsets of the wave's lines, then of the step's waves, in line order.
        const uint32_t inc = wave_inclusive_sum(cnt);
        if (lane == WAVE - 1)
            s_total[parity][wave] = inc;
        __syncthreads();
        uint32_t before = running, step_total = 0;
#pragma unroll
        for (int w = 0; w < EM_NW; w++) {
            const uint32_t t = s_total[parity][w];
            before += (w < wave) ? t : 0u;
            step_total += t;
        }
        // The line's offset: the sum up to its first lane less its own count.
        const uint32_t off = before + __shfl(inc - cnt, lane & ~7, WAVE);

        if (q < 4 && ((at >> q) & 1u)) {
            const uint32_t pos = off + uint32_t(__popc(at & ((1u << q) - 1u)));
            const uint64_t mt = (uint64_t((m << (QM_SHIFT - 32)) | z) << 32) | (uint64_t(lw + li) << ICL_SHIFT)
                              | cell_key(l.cy + (q >> 1), l.cx + (q & 1));
            if (pos < limit)
                out[pos] = mt;
            else
                err |= ERR_INCONSISTENT_NMT;
        }
        for (uint64_t sm = slow; sm;) {
            int la, lb;
            next_pair(sm, la, lb);
            const int ln = (lane < 32) ? la : lb, sub = lane & 31;
            const uint32_t soff = __shfl(off, 8 * ln, WAVE), c = __shfl(cnt, 8 * ln, WAVE);
            const bool mine = lane < 32 || lb != la;
            // The first cell extracted is the first sample's.
            auto store = [&](uint32_t i, uint32_t key) {
                const uint64_t mt = uint64_t(key) | (uint64_t(lw + ln) << ICL_SHIFT) | (uint64_t(QM_PENDING) << QM_SHIFT)
                                  | ((c > 1) ? MFLAG : 0ull) | ((c > 1 && i == 0) ? ZFLAG : 0ull);
                if (soff + i < limit)
                    out[soff + i] = mt;
                else
                    err |= ERR_INCONSISTENT_NMT;
            };
            if (mine && uint32_t(sub) < c)
                store(uint32_t(sub), s_cells[wave][ln][sub]);
            // Cells beyond 32 of a line (not reachable by ordinary scans) are extracted again.
            if (__any(mine && c > 32)) {
                uint32_t k[4], key, i = 0;
                slow_pair<Periodic>(s_samples[wave], la, lb, lw * LINE, nsamp, g, k);
                bool lo, hi;
                while (extract_one(k, key, lo, hi)) {
                    if (sub == 0 && i >= 32 && key != NO_CELL)
                        store(i, key);
                    i += ((lane < 32) ? lo : hi) ? 1u : 0u;
                }
            }
        }

        running += step_total;
        parity ^= 1;
    }

    if (running != limit)
        err |= ERR_INCONSISTENT_NMT;

    err = wave_reduce_or(err | chk.bits(g));
    if (lane == 0) {
        s_err[wave] = err;
        s_nml[wave] = nml;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t e = 0, m = 0;
        for (int w = 0; w < EM_NW; w++) {
            e |= s_err[w];
            m += s_nml[w];
        }
        // The block's multi-cell lines above its error bits (at most 2^16 lines per block; a count that all
        // blocks add to takes 10 us).
        err_out[b] = e | (m << NML_SHIFT);
    }
}

// ------------------------------------------------------------------------------------------
// Device-wide exclusive scan of uint32 (reduce-then-scan, recursive over tile sums).

constexpr int SC_THREADS = 256;
constexpr int SC_ITEMS = 16;
constexpr int SC_TILE = SC_THREADS * SC_ITEMS;

__global__ void __launch_bounds__(SC_THREADS)
scan_tile_sums_kernel(const uint32_t *__restrict__ in, int64_t n, uint32_t *__restrict__ sums)
{
    __shared__ uint32_t s_wave[SC_THREADS / WAVE];
    const int64_t t0 = int64_t(blockIdx.x) * SC_TILE;
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < SC_ITEMS; i++) {
        int64_t j = t0 + int64_t(i) * SC_THREADS + threadIdx.x;
        v += (j < n) ? in[j] : 0u;
    }
    v = wave_reduce_add(v);
    if (lane_id() == 0)
        s_wave[threadIdx.x / WAVE] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int w = 0; w < SC_THREADS / WAVE; w++)
            s += s_wave[w];
        sums[blockIdx.x] = s;
    }
}

__global__ void __launch_bounds__(SC_THREADS)
scan_tiles_kernel(uint32_t *__restrict__ data, int64_t n, const uint32_t *__restrict__ offsets)
{
    __shared__ uint32_t s_wave[SC_THREADS / WAVE];
    const int64_t t0 = int64_t(blockIdx.x) * SC_TILE + int64_t(threadIdx.x) * SC_ITEMS;
    uint32_t v[SC_ITEMS];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < SC_ITEMS; i++) {
        int64_t j = t0 + i;
        v[i] = (j < n) ? data[j] : 0u;
        sum += v[i];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan<SC_THREADS>(sum, s_wave, total);
    if (offsets)
        run += offsets[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SC_ITEMS; i++) {
        int64_t j = t0 + i;
        if (j < n)
            data[j] = run;
        run += v[i];
    }
}

// ------------------------------------------------------------------------------------------
// Stable LSD radix sort of plan entries by dense cell key (iycell * kx + ixcell).
// Per pass: per-tile digit histograms -> device scan (digit-major) -> stable scatter.
// Stability inside a tile: wave w owns items [w*1024, (w+1)*1024) of the tile, processed in
// rounds of 64; equal digits inside a round are ranked by lane via ballot matching.

constexpr int RS_THREADS = 256;
constexpr int RS_NW = RS_THREADS / WAVE;
constexpr int RS_ROUNDS = 16;
constexpr int RS_TILE = RS_THREADS * RS_ROUNDS;   // 4096
constexpr int RS_MAXBITS = 8;
constexpr int RS_RADIX = 1 << RS_MAXBITS;

__device__ inline uint32_t dense_key(uint64_t mt, uint32_t kx)
{
    uint32_t c = uint32_t(mt) & CELL_MASK;
    return (c >> 10) * kx + (c & 1023u);
}

__device__ inline void store_item(uint64_t *__restrict__ out, uint16_t *__restrict__ qmask, int64_t i, uint64_t item)
{
    if (qmask) {
        out[i] = item & ((1ull << QM_SHIFT) - 1ull);
        qmask[i] = uint16_t(item >> QM_SHIFT);
    }
    else
        out[i] = item;
}

__global__ void __launch_bounds__(RS_THREADS)
radix_hist_kernel(const uint64_t *__restrict__ in, int64_t n, uint32_t kx, int shift, uint32_t dmask,
                  uint32_t *__restrict__ hist, int64_t ntiles)
{
    __shared__ uint32_t s_hist[RS_RADIX];
    s_hist[threadIdx.x] = 0;
    __syncthreads();
    const int64_t t0 = int64_t(blockIdx.x) * RS_TILE;
#pragma unroll 4
    for (int r = 0; r < RS_ROUNDS; r++) {
        int64_t j = t0 + int64_t(r) * RS_THREADS + threadIdx.x;
        if (j < n) {
            uint32_t d = (dense_key(in[j], kx) >> shift) & dmask;
            atomicAdd(&s_hist[d], 1u);
        }
    }
    __syncthreads();
    hist[int64_t(threadIdx.x) * ntiles + blockIdx.x] = s_hist[threadIdx.x];
}

// With 'qmask' (the plan's last pass) the items are stored apart: the entry and its mask (bits 48..63).
__global__ void __launch_bounds__(RS_THREADS)
radix_scatter_kernel(const uint64_t *__restrict__ in, uint64_t *__restrict__ out, uint16_t *__restrict__ qmask, int64_t n,
                     uint32_t kx, int shift, int nbits, const uint32_t *__restrict__ hist_scanned,
                     int64_t ntiles)
{
    __shared__ uint32_t s_cnt[RS_NW][RS_RADIX];
    const int lane = lane_id(), wave = threadIdx.x / WAVE;
    const uint32_t dmask = (1u << nbits) - 1u;

    for (int i = threadIdx.x; i < RS_NW * RS_RADIX; i += RS_THREADS)
        (&s_cnt[0][0])[i] = 0;
    __syncthreads();

    const int64_t w0 = int64_t(blockIdx.x) * RS_TILE + int64_t(wave) * (RS_TILE / RS_NW);
    uint64_t item[RS_ROUNDS];
    uint32_t dig[RS_ROUNDS], rank[RS_ROUNDS];

#pragma unroll
    for (int r = 0; r < RS_ROUNDS; r++) {
        int64_t j = w0 + int64_t(r) * WAVE + lane;
        bool valid = (j < n);
        item[r] = valid ? in[j] : 0ull;
        uint32_t d = valid ? ((dense_key(item[r], kx) >> shift) & dmask) : 0u;
        dig[r] = d;

        uint64_t peers = __ballot(valid);
        for (int bit = 0; bit < nbits; bit++) {
            uint64_t bb = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? bb : ~bb;
        }
        uint32_t below = __popcll(peers & lanemask_lt());
        uint32_t old = valid ? s_cnt[wave][d] : 0u;
        if (valid && below == 0)
            s_cnt[wave][d] = old + uint32_t(__popcll(peers));
        rank[r] = old + below;
    }
    __syncthreads();

    // Digit-major prefix over waves, plus this tile's global offset for the digit.
    if (threadIdx.x < (1 << nbits)) {
        uint32_t d = threadIdx.x;
        uint32_t acc = hist_scanned[int64_t(d) * ntiles + blockIdx.x];
        for (int w = 0; w < RS_NW; w++) {
            uint32_t c = s_cnt[w][d];
            s_cnt[w][d] = acc;
            acc += c;
        }
    }
    __syncthreads();

#pragma unroll
    for (int r = 0; r < RS_ROUNDS; r++) {
        int64_t j = w0 + int64_t(r) * WAVE + lane;
        if (j < n)
            store_item(out, qmask, s_cnt[wave][dig[r]] + rank[r], item[r]);
    }
}

// One cell only: nothing to sort.
__global__ void split_items_kernel(const uint64_t *__restrict__ in, uint64_t *__restrict__ out,
                                   uint16_t *__restrict__ qmask, int64_t n)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        store_item(out, qmask, i, in[i]);
}

// ------------------------------------------------------------------------------------------
// Work lists: per-cell [begin, end) in the sorted plan, cut into chunks of <= cap entries, one list per
// operator, in plan order; rank_chunks_kernel or a stable sort by size then puts them in theirs.

__global__ void fill_u32_kernel(uint32_t *p, int64_t n, uint32_t v)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// First entry of the sorted plan whose cell key is at least k.
__device__ inline uint32_t key_lower_bound(const uint64_t *__restrict__ mt, int64_t n, uint32_t kx, uint32_t k)
{
    uint32_t lo = 0, hi = uint32_t(n);
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (dense_key(mt[mid], kx) < k)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

__device__ inline uint32_t nchunks_for(uint32_t cnt, uint32_t cap) { return (cnt + cap - 1) / cap; }

// Chunks of a cell's entries [b, b + cnt), stored from position 'at' of the list on.
__device__ inline void store_chunks(uint32_t icell, uint32_t b, uint32_t cnt, uint32_t cap, uint32_t at,
                                    Chunk *__restrict__ list, int64_t max_chunks)
{
    const uint32_t nc = nchunks_for(cnt, cap);
    for (uint32_t j = 0; j < nc; j++) {
        Chunk c;
        c.icell = icell;
        c.begin = b + uint32_t((uint64_t(cnt) * j) / nc);
        c.end = b + uint32_t((uint64_t(cnt) * (j + 1)) / nc);
        c.flags = (nc > 1) ? CHUNK_SHARED : 0u;
        if (int64_t(at) + j < max_chunks)
            list[at + j] = c;
    }
}

// One list as the kernels see it: the sizes to choose from, how many chunks each of them makes (in all,
// and [size][block of cell_runs_kernel]), and the number of chunks of the list.
struct WorkListOut
{
    Chunk *list;
    int64_t max_chunks;
    ChunkCaps caps;
    uint32_t *cap_counts;
    uint32_t *block_counts;
    uint32_t *count;
};

constexpr int WL_THREADS = 256;

// First entry of each cell of the global map, one cell a thread, by binary search (25 dependent loads,
// 10 us; marking the ends of the runs in a pass over the plan took 59 us on the 2048x262144 raster); and
// the number of chunks that each size of the two lists would make.
__global__ void __launch_bounds__(WL_THREADS)
cell_runs_kernel(const uint64_t *__restrict__ mt, int64_t n, uint32_t kx, int64_t nkeys, uint32_t *__restrict__ begin,
                 WorkListOut a, WorkListOut b)
{
    __shared__ uint32_t s_begin[WL_THREADS + 1], s_counts[2 * NCAPS];
    const int64_t k0 = int64_t(blockIdx.x) * WL_THREADS, k = k0 + threadIdx.x;
    const uint32_t b0 = key_lower_bound(mt, n, kx, uint32_t(min(k, nkeys)));
    s_begin[threadIdx.x] = b0;
    if (threadIdx.x == 0)
        s_begin[WL_THREADS] = key_lower_bound(mt, n, kx, uint32_t(min(k0 + WL_THREADS, nkeys)));
    if (threadIdx.x < 2 * NCAPS)
        s_counts[threadIdx.x] = 0;
    if (k <= nkeys)
        begin[k] = b0;
    __syncthreads();
    const uint32_t cnt = max(s_begin[threadIdx.x + 1], b0) - b0;
    if (__any(cnt)) {
        for (uint32_t j = 0; j < a.caps.n + b.caps.n; j++) {
            const bool ina = j < a.caps.n;
            const uint32_t sum = wave_reduce_add(nchunks_for(cnt, ina ? a.caps.cap[j] : b.caps.cap[j - a.caps.n]));
            if (lane_id() == 0)
                atomicAdd(&s_counts[ina ? j : NCAPS + j - a.caps.n], sum);
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * NCAPS) {
        const bool ina = threadIdx.x < NCAPS;
        const uint32_t j = threadIdx.x % NCAPS, c = s_counts[threadIdx.x];
        (ina ? a.block_counts : b.block_counts)[j * gridDim.x + blockIdx.x] = c;
        if (c)
            atomicAdd((ina ? a.cap_counts : b.cap_counts) + j, c);
    }
}

__device__ inline uint32_t chosen_cap(const WorkListOut &l)
{
    for (uint32_t j = 0; j + 1 < l.caps.n; j++)
        if (l.cap_counts[j] <= l.caps.limit[j])
            return j;
    return l.caps.n - 1;
}

__global__ void __launch_bounds__(WL_THREADS)
work_list_kernel(const uint32_t *__restrict__ begin, uint32_t kx, int64_t nkeys, WorkListOut a, WorkListOut b)
{
    // The grid is cell_runs_kernel's. Each block adds up the chunks of the blocks before it (at most 4096
    // words a list), so that the lists come in plan order, the same in every run.
    __shared__ uint32_t s_wave[WL_THREADS / WAVE], s_before[2][WL_THREADS / WAVE];
    const int64_t k = int64_t(blockIdx.x) * WL_THREADS + threadIdx.x;
    const uint32_t b0 = (k < nkeys) ? begin[k] : 0u, cnt = (k < nkeys) ? max(begin[k + 1], b0) - b0 : 0u;
    const uint32_t ja = chosen_cap(a), jb = chosen_cap(b), cap_a = a.caps.cap[ja], cap_b = b.caps.cap[jb];
    uint32_t xa = 0, xb = 0;
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += WL_THREADS) {
        xa += a.block_counts[ja * gridDim.x + i];
        xb += b.block_counts[jb * gridDim.x + i];
    }
    xa = wave_reduce_add(xa);
    xb = wave_reduce_add(xb);
    if (lane_id() == 0) {
        s_before[0][threadIdx.x / WAVE] = xa;
        s_before[1][threadIdx.x / WAVE] = xb;
    }
    uint32_t ta, tb;
    xa = block_exclusive_scan<WL_THREADS>(nchunks_for(cnt, cap_a), s_wave, ta);     // synchronizes
    xb = block_exclusive_scan<WL_THREADS>(nchunks_for(cnt, cap_b), s_wave, tb);
#pragma unroll
    for (int w = 0; w < WL_THREADS / WAVE; w++) {
        xa += s_before[0][w];
        xb += s_before[1][w];
    }
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) {
        *a.count = xa + ta;
        *b.count = xb + tb;
    }
    if (cnt > 0) {
        const uint32_t icell = cell_key(int(k / kx), int(k % kx));
        store_chunks(icell, b0, cnt, cap_a, xa, a.list, a.max_chunks);
        store_chunks(icell, b0, cnt, cap_b, xb, b.list, b.max_chunks);
    }
}

// Largest-first order of a list (entries equal in size in plan order), so that the operators' last
// blocks are short ones (tod2map 1.4% faster on the 2048x262144 raster): each wave counts the chunks
// that go before its four. blockIdx.y tells the list. Lists of more than RANK_MAX chunks are left to the
// radix sort: n^2 comparisons cross its time near 9000 chunks (plans of as many cells with 30 entries each,
// ranked / sorted, in us: 4096 chunks 150 / 197, 8192 203 / 216, 11264 256 / 223, 15872 334 / 233).
constexpr uint32_t RANK_MAX = 9000;
constexpr int RK_PER_WAVE = 4;
constexpr int RK_LOADS = 8;                              // in flight (4947 chunks: 42 us one by one, 30 so)
constexpr int RK_PER_BLOCK = RK_PER_WAVE * (WL_THREADS / WAVE);

struct RankList
{
    const Chunk *src;
    Chunk *dst;
    const uint32_t *count;
    int64_t max_chunks;
};

__global__ void __launch_bounds__(WL_THREADS)
rank_chunks_kernel(RankList a, RankList b, uint32_t least)
{
    const RankList l = blockIdx.y ? b : a;
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t n = *l.count;
    const uint32_t i0 = blockIdx.x * RK_PER_BLOCK + wave * RK_PER_WAVE;
    if (i0 >= n || n <= least || n > min<int64_t>(RANK_MAX, l.max_chunks))
        return;
    Chunk own[RK_PER_WAVE];
    uint32_t rank[RK_PER_WAVE] = {};
#pragma unroll
    for (int i = 0; i < RK_PER_WAVE; i++)
        own[i] = l.src[min(i0 + i, n - 1)];
    for (uint32_t j0 = 0; j0 < n; j0 += RK_LOADS * WAVE) {
        Chunk c[RK_LOADS];
#pragma unroll
        for (int k = 0; k < RK_LOADS; k++)
            c[k] = l.src[min(j0 + k * WAVE + lane, n - 1)];
#pragma unroll
        for (int k = 0; k < RK_LOADS; k++) {
            const bool in = j0 + k * WAVE + lane < n;
            const uint32_t len = c[k].end - c[k].begin;
#pragma unroll
            for (int i = 0; i < RK_PER_WAVE; i++) {
                const uint32_t mine = own[i].end - own[i].begin;
                rank[i] += uint32_t(__popcll(__ballot(in && (len > mine || (len == mine && c[k].begin < own[i].begin)))));
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RK_PER_WAVE; i++)
        if (lane == 0 && i0 + i < n)
            l.dst[rank[i]] = own[i];
}

// Owned-quad masks for the operators (ownership rule at HALO_X in gmm_common.hpp). For entry e
// of cell Y = (cy, cx) and line l, with has(X) = "l has a sample whose (iy0, ix0) corner is in
// X", fit(X) = "every such sample has ix0 % 64 <= HALO_X - 2 and ix0 + 1 < nx" and touches(X) =
// "a bilinear corner of some sample of l is in X" (exactly: the plan has an entry (l, X)):
//   eligible(X) = has(X) && fit(X) && touches(X - 1)        (X - 1: the cell to the left)
//   R(l, X)     = has(X + 1) && fit(X + 1) && !eligible(X)  (X's entry evaluates X + 1's samples)
// A sample of cell X is evaluated by X - 1 iff R(l, X - 1), else by X. R(l, X) excludes that
// X's own samples go left, so no block both gives and takes, and each sample has exactly one
// evaluator; every entry of l computes these from the same 32 samples, so they agree. Bit q of
// qmask[e] is set iff quad q (samples 4q..4q+3) holds a sample that Y evaluates; QM_TAKES_RIGHT
// is R(l, Y). A line that lies in one cell gives all quads that hold a sample to it. Works on the
// entries that plan_emit_kernel marked QM_PENDING (97 us on the 2048x262144 raster; 461 when it did all
// of them, from 1.65 GB of pointing read again).
template<bool Periodic>
__global__ void __launch_bounds__(256)
qmask_kernel(const uint64_t *__restrict__ mt, int64_t n, const float *__restrict__ xp, int64_t nsamp, int ny,
             int nx, uint16_t *__restrict__ qmask)
{
    // Each wave takes 64 entries at a time, one per lane. An entry of a single-cell line owns
    // every quad of its line that holds a sample: written directly. The entries of multi-cell
    // lines are listed in LDS and handled eight at a time, eight lanes each (one quad per lane).
    __shared__ uint32_t s_list[256 / WAVE][WAVE];
    const int lane = lane_id(), wave = threadIdx.x / WAVE;
    const int g = lane >> 3, q = lane & 7;
    // The planner's passes have checked the pointing's range already.
    const Geom geo = make_geom(ny, nx, Periodic);
    Checks unchecked;
    uint32_t *list = s_list[wave];
    // Line summary bits, OR-reduced over the entry's 32 samples.
    constexpr uint32_t HAS_L = 1, BAD_L = 2, HAS_Y = 4, BAD_Y = 8, HAS_R = 16, BAD_R = 32, TOUCH_L = 64,
                       TOUCH_LL = 128;
    const int64_t nwaves = int64_t(gridDim.x) * (256 / WAVE);
    for (int64_t base = (int64_t(blockIdx.x) * (256 / WAVE) + wave) * WAVE; base < n; base += nwaves * WAVE) {
        const int64_t e = base + lane;
        const bool pending = (e < n) && (qmask[e] & QM_PENDING);
        if (!__any(pending))
            continue;
        const uint64_t m = pending ? mt[e] : 0ull;
        const bool multi = pending && (m & MFLAG);
        if (pending && !multi) {
            // Samples past the end of a partial last line do not exist.
            const int64_t s0 = int64_t(uint32_t(m >> ICL_SHIFT) & ICL_MASK) * LINE;
            const int64_t nv = max<int64_t>(0, min<int64_t>(LINE, nsamp - s0));
            qmask[e] = uint16_t((1u << uint32_t((nv + 3) / 4)) - 1u);
        }
        const uint64_t mb = __ballot(multi);
        if (mb == 0)
            continue;
        if (multi)
            list[__builtin_amdgcn_mbcnt_hi(uint32_t(mb >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mb), 0u))] = uint32_t(lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int nm = __popcll(mb);
        for (int r0 = 0; r0 < nm; r0 += 8) {
            const bool on = r0 + g < nm;
            const int src = on ? int(list[r0 + g]) : 0;
            const uint64_t em = __shfl(m, src, WAVE);
            const int64_t ee = base + src;
            uint32_t sum = 0, own_y = 0, own_r = 0;     // own_*: per sample k, bit k
            const uint32_t icell = uint32_t(em) & CELL_MASK;
            const int cy = int(icell >> 10), cx = int(icell & 1023u);
            const int64_t s0 = int64_t(uint32_t(em >> ICL_SHIFT) & ICL_MASK) * LINE + 4 * q;
            const uint32_t nv = on ? uint32_t(max<int64_t>(0, min<int64_t>(4, nsamp - s0))) : 0u;
            float yv[4], xv[4];
            if (nv > 0) {
                // All loads first (indices clamped to the last sample), so that they overlap.
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int64_t sk = s0 + min<int64_t>(k, nv - 1);
                    yv[k] = xp[sk];
                    xv[k] = xp[nsamp + sk];
                }
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (uint32_t(k) >= nv)
                    continue;
                Pixel<float> p;
                sample_corners<Periodic>(yv[k], xv[k], geo, unchecked, p);
                // Cells of the footprint relative to Y: the owner (p.iy0, p.ix0) is in Y's cell
                // row iff iy0 >> 6 == cy; its column offset is d, that of the ix1 corner d1.
                const bool inrow = (p.iy0 >> 6) == cy;
                const bool rowhit = inrow || ((p.iy1 >> 6) == cy);
                const int d = (p.ix0 >> 6) - cx, d1 = (p.ix1 >> 6) - cx;
                const bool fit = ((p.ix0 & 63) <= HALO_X - 2) && (p.ix0 + 1 < nx);
                // HAS/BAD bit pairs of the cells Y - 1, Y, Y + 1 sit at bit 2 * (d + 1).
                if (inrow && d >= -1 && d <= 1)
                    sum |= (fit ? 1u : 3u) << (2 * (d + 1));
                own_y |= (inrow && d == 0) ? (1u << k) : 0u;
                own_r |= (inrow && d == 1) ? (1u << k) : 0u;
                if (rowhit) {
                    sum |= (d == -1 || d1 == -1) ? TOUCH_L : 0u;
                    sum |= (d == -2 || d1 == -2) ? TOUCH_LL : 0u;
                }
            }
            // OR over the 8 lanes of the entry (aligned groups of 8 within the wave).
            sum |= __shfl_xor(sum, 1, WAVE);
            sum |= __shfl_xor(sum, 2, WAVE);
            sum |= __shfl_xor(sum, 4, WAVE);
            const bool elig_l = (sum & HAS_L) && !(sum & BAD_L) && (sum & TOUCH_LL);
            const bool elig_y = (sum & HAS_Y) && !(sum & BAD_Y) && (sum & TOUCH_L);
            const bool taken_y = elig_y && !elig_l;                  // R(l, Y - 1)
            const bool takes_r = (sum & HAS_R) && !(sum & BAD_R) && !elig_y;   // R(l, Y)
            const bool bit = (own_y != 0 && !taken_y) || (own_r != 0 && takes_r);
            const uint64_t b = __ballot(bit);
            if (on && q == 0)
                qmask[ee] = uint16_t(((b >> (lane & ~7)) & 0xffu) | (takes_r ? QM_TAKES_RIGHT : 0u));
        }
        // The list is read before the next batch writes it (LDS operations of a wave complete
        // in issue order; the fence keeps the compiler from reordering them).
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// Error bits and multi-cell lines of the emit pass's blocks, by a block of PREPLAN_SIZE threads: the bits go
// to *err_word and counts[PC_ERROR], the number of lines to counts[PC_NMLINES].
__device__ inline void gather_plan_errors(const uint32_t *__restrict__ in, int n, uint32_t *__restrict__ err_word,
                                          uint32_t *__restrict__ counts)
{
    __shared__ uint32_t s_err[PREPLAN_SIZE / WAVE], s_nml[PREPLAN_SIZE / WAVE];
    const uint32_t v = (int(threadIdx.x) < n) ? in[threadIdx.x] : 0u;
    const uint32_t e = wave_reduce_or(v & ((1u << NML_SHIFT) - 1u)), m = wave_reduce_add(v >> NML_SHIFT);
    if (lane_id() == 0) {
        s_err[threadIdx.x / WAVE] = e;
        s_nml[threadIdx.x / WAVE] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t err = 0, nml = 0;
        for (int w = 0; w < PREPLAN_SIZE / WAVE; w++) {
            err |= s_err[w];
            nml += s_nml[w];
        }
        *err_word = err;
        counts[PC_NMLINES] = nml;
        counts[PC_ERROR] = err;
    }
}

__global__ void __launch_bounds__(PREPLAN_SIZE)
plan_errors_kernel(const uint32_t *__restrict__ in, int n, uint32_t *__restrict__ err_word, uint32_t *__restrict__ counts)
{
    gather_plan_errors(in, n, err_word, counts);
    if (threadIdx.x < PC_TOTAL && threadIdx.x != PC_NMLINES && threadIdx.x != PC_ERROR)
        counts[threadIdx.x] = 0;
}

// ------------------------------------------------------------------------------------------
// Small plans, up to SP_MAX entries: what follows the emit pass (error words, sort, work lists) in one
// launch of one block, the entries in LDS. Such a plan's time is launches: with one each for the error
// words, the digit histograms, their scan, the scatter (per pass), the lists and their order, preplan and
// plan of 1000 entries took 93 us, now 75; of 7900, where the one block takes 23 us, 100 and 91.

constexpr int SP_THREADS = PREPLAN_SIZE;
constexpr int SP_NW = SP_THREADS / WAVE;
constexpr int SP_ROUNDS = 8;
constexpr int SP_RANK = SP_THREADS;                      // longest list that is ordered here
constexpr int SP_BEGIN_BITS = 13, SP_LEN_BITS = 11;      // a chunk has at most 1024 entries
static_assert(SP_THREADS * SP_ROUNDS == SP_MAX && SP_MAX == 1 << SP_BEGIN_BITS, "one item per thread and round");

// A list's chunks as words: ~length, begin, shared, so that they are in the list's order.
__device__ inline uint32_t sp_pack(uint32_t begin, uint32_t end, bool shared)
{
    const uint32_t inv = (1u << SP_LEN_BITS) - 1u - (end - begin);
    return (inv << (SP_BEGIN_BITS + 1)) | (begin << 1) | (shared ? CHUNK_SHARED : 0u);
}

__device__ inline Chunk sp_unpack(uint32_t v, const uint64_t *items)
{
    Chunk c;
    c.begin = (v >> 1) & (SP_MAX - 1);
    c.end = c.begin + (1u << SP_LEN_BITS) - 1u - (v >> (SP_BEGIN_BITS + 1));
    c.flags = v & CHUNK_SHARED;
    c.icell = uint32_t(items[c.begin]) & CELL_MASK;
    return c;
}

// The list of chunks of the cells that start at start[0 .. ncells). In 'dst' in order when there are at most SP_RANK, else in 'tmp' in any (the host then orders it).
__device__ inline void sp_work_list(const uint64_t *items, const uint16_t *start, uint32_t ncells, const WorkListOut &l,
                                    Chunk *__restrict__ dst, uint32_t *s_key, uint32_t *s_wave)
{
    const uint32_t t = threadIdx.x;
    uint32_t at, total, cap;
    for (uint32_t j = 0;; j++) {
        cap = l.caps.cap[j];
        uint32_t mine = 0;
        for (uint32_t c = t; c < ncells; c += SP_THREADS)
            mine += nchunks_for(uint32_t(start[c + 1]) - start[c], cap);
        at = block_exclusive_scan<SP_THREADS>(mine, s_wave, total);
        if (j + 1 >= l.caps.n || total <= l.caps.limit[j])
            break;
    }
    if (t == 0)
        *l.count = total;
    const bool ordered = total <= SP_RANK;
    for (uint32_t c = t; c < ncells; c += SP_THREADS) {
        const uint32_t b = start[c], cnt = uint32_t(start[c + 1]) - b, nc = nchunks_for(cnt, cap);
        for (uint32_t j = 0; j < nc; j++, at++) {
            const uint32_t v = sp_pack(b + cnt * j / nc, b + cnt * (j + 1) / nc, nc > 1);
            if (ordered)
                s_key[at] = v;
            else if (int64_t(at) < l.max_chunks)
                l.list[at] = sp_unpack(v, items);
        }
    }
    __syncthreads();
    if (ordered && t < total) {
        const uint32_t v = s_key[t];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < total; j++)
            rank += (s_key[j] < v) ? 1u : 0u;
        if (int64_t(rank) < l.max_chunks)
            dst[rank] = sp_unpack(v, items);
    }
    __syncthreads();
}

__global__ void __launch_bounds__(SP_THREADS)
small_plan_kernel(const uint64_t *__restrict__ in, uint32_t n, uint32_t kx, int bits, uint64_t *__restrict__ out,
                  uint16_t *__restrict__ qmask, WorkListOut a, WorkListOut b, Chunk *__restrict__ dst_a,
                  Chunk *__restrict__ dst_b, const uint32_t *__restrict__ err_in, int nblocks,
                  uint32_t *__restrict__ err_word, uint32_t *__restrict__ counts)
{
    __shared__ uint64_t s_item[SP_MAX];
    __shared__ uint32_t s_cnt[SP_NW][RS_RADIX];
    __shared__ uint16_t s_start[SP_MAX + 1];
    __shared__ uint32_t s_key[SP_RANK], s_wave[SP_NW];
    const int t = threadIdx.x, lane = lane_id(), wave = t / WAVE;

    gather_plan_errors(err_in, nblocks, err_word, counts);

    // The stable radix sort of the tiles above, on one tile: wave w owns items [w * 64 * rounds, ...).
    const int rounds = int((n + SP_THREADS - 1) / SP_THREADS);
    const uint32_t w0 = uint32_t(wave * rounds * WAVE + lane);
    for (int r = 0; r < rounds; r++) {
        const uint32_t i = w0 + r * WAVE;
        if (i < n)
            s_item[i] = in[i];
    }
    const int npasses = (bits + RS_MAXBITS - 1) / RS_MAXBITS;
    const int per = npasses ? (bits + npasses - 1) / npasses : 0;
    for (int pass = 0, shift = 0; pass < npasses; pass++, shift += per) {
        const int nb = min(bits - shift, per);
        const uint32_t dmask = (1u << nb) - 1u;
        for (int i = t; i < SP_NW * RS_RADIX; i += SP_THREADS)
            (&s_cnt[0][0])[i] = 0;
        __syncthreads();
        uint64_t item[SP_ROUNDS];
        uint32_t dig[SP_ROUNDS], rank[SP_ROUNDS];
#pragma unroll
        for (int r = 0; r < SP_ROUNDS; r++) {
            if (r >= rounds)
                break;
            const uint32_t i = w0 + r * WAVE;
            const bool valid = i < n;
            item[r] = valid ? s_item[i] : 0ull;
            const uint32_t d = valid ? ((dense_key(item[r], kx) >> shift) & dmask) : 0u;
            dig[r] = d;
            uint64_t peers = __ballot(valid);
            for (int bit = 0; bit < nb; bit++) {
                const uint64_t bb = __ballot((d >> bit) & 1u);
                peers &= ((d >> bit) & 1u) ? bb : ~bb;
            }
            const uint32_t below = uint32_t(__popcll(peers & lanemask_lt()));
            const uint32_t old = valid ? s_cnt[wave][d] : 0u;
            if (valid && below == 0)
                s_cnt[wave][d] = old + uint32_t(__popcll(peers));
            rank[r] = old + below;
        }
        __syncthreads();
        uint32_t sum = 0, total;
        if (t < RS_RADIX)
            for (int w = 0; w < SP_NW; w++)
                sum += s_cnt[w][t];
        uint32_t at = block_exclusive_scan<SP_THREADS>(sum, s_wave, total);
        if (t < RS_RADIX)
            for (int w = 0; w < SP_NW; w++) {
                const uint32_t c = s_cnt[w][t];
                s_cnt[w][t] = at;
                at += c;
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SP_ROUNDS; r++) {
            if (r >= rounds)
                break;
            if (w0 + r * WAVE < n)
                s_item[s_cnt[wave][dig[r]] + rank[r]] = item[r];
        }
        __syncthreads();
    }
    __syncthreads();
    for (uint32_t i = t; i < n; i += SP_THREADS)
        store_item(out, qmask, i, s_item[i]);

    // First entries of the cells, in order: thread t looks at entries [t * rounds, ...).
    auto starts = [&](uint32_t i) {
        return i < n && (i == 0 || ((uint32_t(s_item[i]) ^ uint32_t(s_item[i - 1])) & CELL_MASK));
    };
    uint32_t mine = 0, ncells;
    for (int r = 0; r < rounds; r++)
        mine += starts(uint32_t(t * rounds + r)) ? 1u : 0u;
    uint32_t at = block_exclusive_scan<SP_THREADS>(mine, s_wave, ncells);
    for (int r = 0; r < rounds; r++)
        if (starts(uint32_t(t * rounds + r)))
            s_start[at++] = uint16_t(t * rounds + r);
    if (t == 0)
        s_start[ncells] = uint16_t(n);
    __syncthreads();
    sp_work_list(s_item, s_start, ncells, a, dst_a, s_key, s_wave);
    sp_work_list(s_item, s_start, ncells, b, dst_b, s_key, s_wave);
}

// ------------------------------------------------------------------------------------------
// Test aids.

template<bool Periodic>
__global__ void quantize_kernel(const float *__restrict__ xp, int64_t nsamp, int ny, int nx,
                                int32_t *__restrict__ iypix, int32_t *__restrict__ ixpix,
                                uint32_t *__restrict__ err_word)
{
    uint32_t err = 0;
    for (int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; s < nsamp; s += int64_t(gridDim.x) * blockDim.x) {
        Pixel<float> p;
        err |= locate_pixel(xp[s], xp[s + nsamp], ny, nx, Periodic, p);
        iypix[s] = p.iy0;
        ixpix[s] = p.ix0;
    }
    err = wave_reduce_or(err);
    if (lane_id() == 0 && err)
        atomicOr(err_word, err);
}

// Walks the work list exactly as the planned operators do: each wave takes its wave_slice() of
// the chunk, in batches of 64 entries (one per lane, one load) and steps of 8 entries (lane
// 8*li + q on entry li of the step, with the entry broadcast from the batch by a shuffle), and
// counts the visits of each entry (lane q == 0); a visit to an entry of another cell sets bit 0
// of the error word, an entry reached twice within one wave bit 1.
__global__ void iterator_test_kernel(const uint64_t *__restrict__ plan_mt, const Chunk *__restrict__ chunks,
                                     uint32_t *__restrict__ visits, uint32_t *__restrict__ err_word)
{
    const int lane = lane_id(), wave = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    const int li = lane >> 3, q = lane & 7;
    const Chunk ch = chunks[blockIdx.x];
    uint32_t wb, we;
    wave_slice(ch, wave, nw, wb, we);
    uint32_t err = 0, last = 0xffffffffu;
    for (uint32_t base = wb; base < we; base += 64) {
        const uint32_t cnt = min(64u, we - base);
        const uint32_t key = (uint32_t(lane) < cnt) ? (uint32_t(plan_mt[base + lane]) & CELL_MASK) : 0u;
        for (uint32_t j = 0; j < cnt; j += 8) {
            const uint32_t idx = j + li;
            const uint32_t k = __shfl(key, int(min(idx, 63u)), WAVE);
            if (idx >= cnt)
                continue;
            const uint32_t e = base + idx;
            if (k != ch.icell)
                err |= 1u;
            if (last != 0xffffffffu && e <= last)
                err |= 2u;
            last = e;
            if (q == 0)
                atomicAdd(visits + e, 1u);
        }
    }
    err = wave_reduce_or(err);
    if (lane == 0 && err)
        atomicOr(err_word, err);
}

// Long lists are put largest first by the radix sort: items (index << 20 | key) with key = 8192 -
// entries, then the chunks gathered in item order.
__global__ void chunk_key_kernel(const Chunk *__restrict__ chunks, int64_t n, uint64_t *__restrict__ items)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        const uint32_t len = chunks[i].end - chunks[i].begin;
        const uint32_t key = 8192u - min(len, 8192u);
        items[i] = (uint64_t(i) << 20) | key;
    }
}

__global__ void chunk_gather_kernel(const uint64_t *__restrict__ items, const Chunk *__restrict__ src, int64_t n,
                                    Chunk *__restrict__ dst)
{
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        dst[i] = src[items[i] >> 20];
}

inline int grid_for(int64_t n, int threads, int64_t cap = 65536)
{
    int64_t g = (n + threads - 1) / threads;
    g = (g < 1) ? 1 : g;
    return int((g < cap) ? g : cap);
}

}  // namespace

// ==========================================================================================
// Host launchers.

// float4 access to every line's groups of four samples.
static bool vec_pointing(const float *xp, int64_t nsamp)
{
    return (reinterpret_cast<uintptr_t>(xp) & 15) == 0 && nsamp % 4 == 0;
}

void launch_preplan_count(const float *xp, int64_t nsamp, const gmm_preplan &pp,
                          uint32_t *nmt_out, uint32_t *err_out, hipStream_t stream)
{
    const auto &p = pp.pparams;
    const bool vec = vec_pointing(xp, nsamp);
    auto k = pp.periodic_xcoord ? (vec ? preplan_count_kernel<true, true> : preplan_count_kernel<true, false>)
                                : (vec ? preplan_count_kernel<false, true> : preplan_count_kernel<false, false>);
    k<<<unsigned(p.planner_nblocks), PP_THREADS, 0, stream>>>(xp, nsamp, p.ncl, p.ncl_per_threadblock,
        int(pp.nypix_global), int(pp.nxpix_global), nmt_out, err_out);
    GMM_HIP(hipGetLastError());
}

void launch_preplan_finish(uint32_t *nmt, const uint32_t *err, int64_t nblocks,
                           uint32_t * /*summary_gpu*/, hipStream_t stream)
{
    preplan_finish_kernel<<<1, PREPLAN_SIZE, 0, stream>>>(nmt, const_cast<uint32_t *>(err), int(nblocks));
    GMM_HIP(hipGetLastError());
}

void launch_plan_emit(const float *xp, const gmm_preplan &pp, uint64_t *out_mt,
                      uint32_t *err_out, hipStream_t stream)
{
    const auto &p = pp.pparams;
    const bool vec = vec_pointing(xp, pp.nsamp);
    auto k = pp.periodic_xcoord ? (vec ? plan_emit_kernel<true, true> : plan_emit_kernel<true, false>)
                                : (vec ? plan_emit_kernel<false, true> : plan_emit_kernel<false, false>);
    k<<<unsigned(p.planner_nblocks), EM_THREADS, 0, stream>>>(xp, pp.nsamp, p.ncl, p.ncl_per_threadblock,
        int(pp.nypix_global), int(pp.nxpix_global), pp.nmt_cumsum_gpu, out_mt, err_out);
    GMM_HIP(hipGetLastError());
}

int64_t scan_scratch_nbytes(int64_t n)
{
    if (n <= SC_TILE)
        return 0;
    int64_t nt = (n + SC_TILE - 1) / SC_TILE;
    return align128(4 * nt) + scan_scratch_nbytes(nt);
}

void exclusive_scan_u32(uint32_t *data, int64_t n, void *scratch, hipStream_t stream)
{
    if (n <= 0)
        return;
    if (n <= SC_TILE) {
        scan_tiles_kernel<<<1, SC_THREADS, 0, stream>>>(data, n, nullptr);
        GMM_HIP(hipGetLastError());
        return;
    }
    int64_t nt = (n + SC_TILE - 1) / SC_TILE;
    uint32_t *sums = reinterpret_cast<uint32_t *>(scratch);
    scan_tile_sums_kernel<<<unsigned(nt), SC_THREADS, 0, stream>>>(data, n, sums);
    GMM_HIP(hipGetLastError());
    exclusive_scan_u32(sums, nt, reinterpret_cast<uint8_t *>(scratch) + align128(4 * nt), stream);
    scan_tiles_kernel<<<unsigned(nt), SC_THREADS, 0, stream>>>(data, n, sums);
    GMM_HIP(hipGetLastError());
}

namespace {

struct SortLayout
{
    int64_t ntiles;
    int64_t hist_off, hist_scan_off;   // histogram, scan scratch
    int64_t total;
};

SortLayout sort_layout(int64_t nmt)
{
    SortLayout L;
    L.ntiles = (nmt + RS_TILE - 1) / RS_TILE;
    int64_t o = 0;
    L.hist_off = o;      o += align128(4 * RS_RADIX * L.ntiles);
    L.hist_scan_off = o; o += align128(scan_scratch_nbytes(RS_RADIX * L.ntiles));
    L.total = o;
    return L;
}

constexpr int64_t CAP_MAX = 8192;                        // entries per work unit

// Blocks of the work list kernels, and the words that cell_runs_kernel leaves for each list.
int64_t work_list_blocks(int64_t nkeys) { return nkeys / WL_THREADS + 1; }            // begin[nkeys] too
int64_t block_count_words(int64_t nkeys) { return NCAPS * work_list_blocks(nkeys); }

WorkListOut m2t_out(const gmm_preplan &pp, const PlanLists &l, uint32_t *counts)
{
    return WorkListOut{l.tmp_m2t, l.max_m2t, pp.caps_m2t, counts + PC_CAPS_M2T, l.block_counts, counts + PC_CHUNKS_M2T};
}

WorkListOut t2m_out(const gmm_preplan &pp, const PlanLists &l, uint32_t *counts)
{
    return WorkListOut{l.tmp_t2m, l.max_t2m, pp.caps_t2m, counts + PC_CAPS_T2M,
                       l.block_counts + block_count_words(pp.nycells_g * pp.nxcells_g), counts + PC_CHUNKS_T2M};
}

// Sizes for a plan of nmt entries on 'slots' blocks that run at once: lists of at most k * slots chunks (k
// full rounds) with chunks up to 5, 15, 30 and 50% above an even share, ordered by the time that the
// rounds take when a block costs as much as 'fixed' entries; no chunk is smaller than 'least' for the sake
// of a round. Three rounds 50% above, the costliest of the twelve, are not tried (NCAPS). Last comes
// 'general', which any list may take.
ChunkCaps make_caps(int64_t nmt, int64_t slots, int64_t fixed, int kmax, int64_t least, int64_t general)
{
    struct Option { int64_t cap, limit, cost; };
    std::vector<Option> opt;
    for (int k = 1; k <= kmax; k++)
        for (int percent : {105, 115, 130, 150}) {
            const int64_t share = k * slots * 100;
            const int64_t cap = std::max<int64_t>(least, (nmt * percent + share - 1) / share);
            if (cap <= CAP_MAX && int(opt.size()) < NCAPS - 1)
                opt.push_back(Option{cap, k * slots, k * (fixed + cap)});
        }
    std::stable_sort(opt.begin(), opt.end(), [](const Option &a, const Option &b) { return a.cost < b.cost; });
    ChunkCaps c = {};
    for (const Option &o : opt) {
        c.cap[c.n] = uint32_t(o.cap);
        c.limit[c.n++] = uint32_t(o.limit);
    }
    c.cap[c.n] = uint32_t(general);
    c.limit[c.n++] = 0xffffffffu;
    return c;
}

int64_t max_chunks(const ChunkCaps &c, int64_t nmt, int64_t nkeys)
{
    int64_t n = (nmt + c.cap[c.n - 1] - 1) / c.cap[c.n - 1] + std::min(nmt, nkeys);
    for (uint32_t j = 0; j + 1 < c.n; j++)
        n = std::max(n, std::min<int64_t>(c.limit[j], nmt));
    return n;
}

void launch_work_lists(const uint64_t *mt, int64_t n, uint32_t kx, int64_t nkeys, uint32_t *begin, const WorkListOut &a,
                       const WorkListOut &b, hipStream_t stream)
{
    const unsigned grid = unsigned(work_list_blocks(nkeys));
    cell_runs_kernel<<<grid, WL_THREADS, 0, stream>>>(mt, n, kx, nkeys, begin, a, b);
    GMM_HIP(hipGetLastError());
    work_list_kernel<<<grid, WL_THREADS, 0, stream>>>(begin, kx, nkeys, a, b);
    GMM_HIP(hipGetLastError());
}

// Orders the lists of more than 'least' and up to RANK_MAX chunks, which have at most nmax.
void launch_rank(const PlanLists &l, const uint32_t *counts, int64_t nmax, uint32_t least, hipStream_t stream)
{
    const RankList a{l.tmp_m2t, l.m2t, counts + PC_CHUNKS_M2T, l.max_m2t}, b{l.tmp_t2m, l.t2m, counts + PC_CHUNKS_T2M, l.max_t2m};
    const int64_t n = std::min<int64_t>(nmax, RANK_MAX);
    rank_chunks_kernel<<<dim3(unsigned((n + RK_PER_BLOCK - 1) / RK_PER_BLOCK), 2), WL_THREADS, 0, stream>>>(a, b, least);
    GMM_HIP(hipGetLastError());
}

}  // namespace

// Entries per work unit of the operators. A tod2map block clears and flushes a 116 KiB tile, atomically
// when its cell is split, and has its CU to itself: lists are cut for one to three full rounds of the 256
// CUs where their cells allow it (tod2map with chunks of half a CU's share against this, in us: 145 000
// entries of 64 x 65536 samples 36 / 32; rotated scans of 256 and 1024 x 65536 131 / 92 and 388 / 323; the
// fast one of 768 x 50004 311 / 275; with one round as the only choice the last two gain nothing; rasters
// over more cells than that the same). map2tod, two blocks a CU and bound by memory, balances best in many
// small chunks (263 us on the 768 x 50004; 285 with tod2map's), except when they would not fill a round
// (64 x 65536 samples 25.8 us in chunks of 512, 22.7 in one round; 8 x 4096 10.9 and 9.5). Each chunk of a
// split cell adds to the map with a rounding of its own, so that tod2map's stay at 512 entries or more.
constexpr int64_t TILE_COST = 700, STAGE_COST = 100;     // a block's fixed work, in entries

void plan_chunk_caps(gmm_preplan &pp)
{
    const int64_t nmt = pp.plan_nmt, nkeys = pp.nycells_g * pp.nxcells_g, cus = 256;
    const int64_t m2t = std::min(CAP_MAX, std::max<int64_t>(512, (nmt + 12 * cus - 1) / (12 * cus)));
    const int64_t t2m = std::min(CAP_MAX, std::max<int64_t>(1024, (nmt + 2 * cus - 1) / (2 * cus)));
    pp.caps_m2t = make_caps(nmt, 2 * cus, STAGE_COST, (nmt <= 512 * 2 * cus) ? 1 : 0, 128, m2t);
    pp.caps_t2m = make_caps(nmt, cus, TILE_COST, 3, 512, t2m);
    pp.max_nchunks = max_chunks(pp.caps_m2t, nmt, nkeys);
    pp.max_nchunks_t2m = max_chunks(pp.caps_t2m, nmt, nkeys);
}

int64_t plan_scratch_nbytes(const gmm_preplan &pp)
{
    const int64_t nkeys = pp.nycells_g * pp.nxcells_g;
    return sort_layout(pp.plan_nmt).total + align128(int64_t(sizeof(Chunk)) * (pp.max_nchunks + pp.max_nchunks_t2m))
         + align128(8 * block_count_words(nkeys)) + align128(4 * (nkeys + 1));
}

PlanLists plan_lists(const gmm_preplan &pp, Chunk *m2t, Chunk *t2m, void *scratch)
{
    PlanLists l;
    l.m2t = m2t;
    l.t2m = t2m;
    l.max_m2t = pp.max_nchunks;
    l.max_t2m = pp.max_nchunks_t2m;
    l.tmp_m2t = reinterpret_cast<Chunk *>(static_cast<uint8_t *>(scratch) + sort_layout(pp.plan_nmt).total);
    l.tmp_t2m = l.tmp_m2t + pp.max_nchunks;
    const int64_t nkeys = pp.nycells_g * pp.nxcells_g;
    uint8_t *begin = static_cast<uint8_t *>(scratch) + plan_scratch_nbytes(pp) - align128(4 * (nkeys + 1));
    l.begin = reinterpret_cast<uint32_t *>(begin);
    l.block_counts = reinterpret_cast<uint32_t *>(begin - align128(8 * block_count_words(nkeys)));
    return l;
}

void plan_sort(const gmm_preplan &pp, uint64_t *a, uint64_t *b, uint64_t *out, uint16_t *qmask,
               void *scratch, int64_t scratch_nbytes, hipStream_t stream)
{
    const int64_t n = pp.plan_nmt;
    const uint32_t kx = uint32_t(pp.nxcells_g);
    SortLayout L = sort_layout(n);
    GMM_REQUIRE(scratch_nbytes >= L.total, "plan_sort: scratch too small");
    uint8_t *sc = reinterpret_cast<uint8_t *>(scratch);
    uint32_t *hist = reinterpret_cast<uint32_t *>(sc + L.hist_off);

    const int bits = pp.key_bits;
    if (bits == 0) {
        split_items_kernel<<<grid_for(n, 256, 4096), 256, 0, stream>>>(a, out, qmask, n);
        GMM_HIP(hipGetLastError());
        return;
    }
    const int npasses = (bits + RS_MAXBITS - 1) / RS_MAXBITS;
    const int per = (bits + npasses - 1) / npasses;

    const uint64_t *src = a;
    for (int pass = 0, shift = 0; pass < npasses; pass++, shift += per) {
        int nb = (bits - shift < per) ? (bits - shift) : per;
        uint64_t *dst = (pass == npasses - 1) ? out : ((src == a) ? b : a);
        radix_hist_kernel<<<unsigned(L.ntiles), RS_THREADS, 0, stream>>>(src, n, kx, shift, (1u << nb) - 1u, hist, L.ntiles);
        GMM_HIP(hipGetLastError());
        exclusive_scan_u32(hist, int64_t(1 << nb) * L.ntiles, sc + L.hist_scan_off, stream);
        radix_scatter_kernel<<<unsigned(L.ntiles), RS_THREADS, 0, stream>>>(src, dst, (dst == out) ? qmask : nullptr, n,
                                                                             kx, shift, nb, hist, L.ntiles);
        GMM_HIP(hipGetLastError());
        src = dst;
    }
}

void plan_schedule(const gmm_preplan &pp, const uint64_t *sorted_mt, const PlanLists &l, uint32_t *counts_gpu,
                   hipStream_t stream)
{
    const int64_t n = pp.plan_nmt;
    const int64_t nkeys = pp.nycells_g * pp.nxcells_g;
    launch_work_lists(sorted_mt, n, uint32_t(pp.nxcells_g), nkeys, l.begin, m2t_out(pp, l, counts_gpu),
                      t2m_out(pp, l, counts_gpu), stream);
    launch_rank(l, counts_gpu, std::max(l.max_m2t, l.max_t2m), 0, stream);
}

void plan_small(const gmm_preplan &pp, const uint64_t *items, uint64_t *out, uint16_t *qmask, const PlanLists &l,
                const uint32_t *err_in, uint32_t *err_word, uint32_t *counts_gpu, hipStream_t stream)
{
    uint32_t cap = 0;
    for (const ChunkCaps *c : {&pp.caps_m2t, &pp.caps_t2m})
        cap = std::max(cap, *std::max_element(c->cap, c->cap + c->n));
    GMM_REQUIRE(pp.plan_nmt <= SP_MAX && cap < (1u << SP_LEN_BITS), "plan_small: plan too large");
    small_plan_kernel<<<1, SP_THREADS, 0, stream>>>(items, uint32_t(pp.plan_nmt), uint32_t(pp.nxcells_g), pp.key_bits, out,
                                                    qmask, m2t_out(pp, l, counts_gpu), t2m_out(pp, l, counts_gpu), l.m2t,
                                                    l.t2m, err_in, int(pp.pparams.planner_nblocks), err_word, counts_gpu);
    GMM_HIP(hipGetLastError());
}

void plan_masks(const gmm_preplan &pp, const uint64_t *sorted_mt, const float *xp, uint16_t *qmask, hipStream_t stream)
{
    const int64_t n = pp.plan_nmt;
    const int grid = int(std::min<int64_t>((n + 255) / 256, 8192));
    if (pp.periodic_xcoord)
        qmask_kernel<true><<<grid, 256, 0, stream>>>(sorted_mt, n, xp, pp.nsamp, int(pp.nypix_global),
                                                     int(pp.nxpix_global), qmask);
    else
        qmask_kernel<false><<<grid, 256, 0, stream>>>(sorted_mt, n, xp, pp.nsamp, int(pp.nypix_global),
                                                      int(pp.nxpix_global), qmask);
    GMM_HIP(hipGetLastError());
}

bool order_long_lists(const gmm_preplan &pp, const PlanLists &l, int64_t n_m2t, int64_t n_t2m, const uint32_t *counts_gpu,
                      uint64_t *a, uint64_t *b, void *scratch, hipStream_t stream)
{
    if (pp.plan_nmt <= SP_MAX) {                                     // plan_small() did the short ones
        static_assert(SP_MAX <= RANK_MAX, "small plans' lists are ranked");
        if (n_m2t <= SP_RANK && n_t2m <= SP_RANK)
            return false;
        launch_rank(l, counts_gpu, std::max(n_m2t, n_t2m), SP_RANK, stream);
        return true;
    }
    // plan_schedule() did lists of up to RANK_MAX.
    // a and b hold plan_nmt items each, a list at most as many. 13-bit keys: kx = 1024 makes the sort's
    // key the item's low 20 bits.
    uint8_t *sc = reinterpret_cast<uint8_t *>(scratch);
    auto order = [&](const Chunk *src, Chunk *dst, int64_t nch) {
        if (nch <= RANK_MAX)
            return;
        SortLayout L = sort_layout(nch);
        uint32_t *hist = reinterpret_cast<uint32_t *>(sc + L.hist_off);
        chunk_key_kernel<<<grid_for(nch, 256), 256, 0, stream>>>(src, nch, a);
        GMM_HIP(hipGetLastError());
        const int bits = 13, npasses = 2, per = 7;
        uint64_t *from = a, *to = b;
        for (int pass = 0, shift = 0; pass < npasses; pass++, shift += per) {
            const int nb = (bits - shift < per) ? (bits - shift) : per;
            radix_hist_kernel<<<unsigned(L.ntiles), RS_THREADS, 0, stream>>>(from, nch, 1024u, shift, (1u << nb) - 1u, hist,
                                                                              L.ntiles);
            GMM_HIP(hipGetLastError());
            exclusive_scan_u32(hist, int64_t(1 << nb) * L.ntiles, sc + L.hist_scan_off, stream);
            radix_scatter_kernel<<<unsigned(L.ntiles), RS_THREADS, 0, stream>>>(from, to, nullptr, nch, 1024u, shift, nb,
                                                                                 hist, L.ntiles);
            GMM_HIP(hipGetLastError());
            std::swap(from, to);
        }
        chunk_gather_kernel<<<grid_for(nch, 256), 256, 0, stream>>>(from, src, nch, dst);
        GMM_HIP(hipGetLastError());
    };
    order(l.tmp_m2t, l.m2t, n_m2t);
    order(l.tmp_t2m, l.t2m, n_t2m);
    return std::max(n_m2t, n_t2m) > RANK_MAX;
}

constexpr int64_t GENERIC_KEYS = int64_t(1) << 20;

int64_t build_chunks_generic_scratch_nbytes()
{
    return align128(4 * (GENERIC_KEYS + 1)) + PC_NBYTES + 8 * block_count_words(GENERIC_KEYS);
}

int64_t build_chunks_generic(const uint64_t *plan_mt_gpu, int64_t nmt, int64_t chunk_cap,
                             Chunk *chunks_gpu, int64_t max_chunks, void *scratch, hipStream_t stream)
{
    uint32_t *begin = static_cast<uint32_t *>(scratch);
    uint32_t *counts = begin + align128(4 * (GENERIC_KEYS + 1)) / 4;
    uint32_t *block_counts = counts + PC_NBYTES / 4;
    fill_u32_kernel<<<1, 64, 0, stream>>>(counts, PC_TOTAL, 0u);
    GMM_HIP(hipGetLastError());
    ChunkCaps cap = {}, none = {};
    cap.n = none.n = 1;
    cap.cap[0] = uint32_t(chunk_cap);
    none.cap[0] = 1u << 30;
    const WorkListOut a{chunks_gpu, max_chunks, cap, counts + PC_CAPS_M2T, block_counts, counts + PC_CHUNKS_M2T};
    const WorkListOut b{chunks_gpu, 0, none, counts + PC_CAPS_T2M, block_counts + block_count_words(GENERIC_KEYS),
                        counts + PC_CHUNKS_T2M};
    launch_work_lists(plan_mt_gpu, nmt, 1024u, GENERIC_KEYS, begin, a, b, stream);
    return int64_t(read_word(counts + PC_CHUNKS_M2T, stream));
}

void launch_fill_u32(uint32_t *p, int64_t n, uint32_t v, hipStream_t stream)
{
    if (n <= 0)
        return;
    fill_u32_kernel<<<grid_for(n, 256, 4096), 256, 0, stream>>>(p, n, v);
    GMM_HIP(hipGetLastError());
}

void launch_plan_errors(const uint32_t *in, int64_t nblocks, uint32_t *err_word, uint32_t *counts, hipStream_t stream)
{
    plan_errors_kernel<<<1, PREPLAN_SIZE, 0, stream>>>(in, int(nblocks), err_word, counts);
    GMM_HIP(hipGetLastError());
}

void launch_quantize(const float *xp, int64_t nsamp, int ny, int nx, bool periodic,
                     int32_t *iypix, int32_t *ixpix, uint32_t *err_word, hipStream_t stream)
{
    fill_u32_kernel<<<1, 64, 0, stream>>>(err_word, 1, 0u);
    int g = grid_for(nsamp, 256, 16384);
    if (periodic)
        quantize_kernel<true><<<g, 256, 0, stream>>>(xp, nsamp, ny, nx, iypix, ixpix, err_word);
    else
        quantize_kernel<false><<<g, 256, 0, stream>>>(xp, nsamp, ny, nx, iypix, ixpix, err_word);
    GMM_HIP(hipGetLastError());
}

void launch_iterator_test(const uint64_t *plan_mt, const Chunk *chunks, int64_t nchunks,
                          int waves_per_block, uint32_t *visit_counts, uint32_t *err_word,
                          hipStream_t stream)
{
    fill_u32_kernel<<<1, 64, 0, stream>>>(err_word, 1, 0u);
    if (nchunks > 0)
        iterator_test_kernel<<<unsigned(nchunks), unsigned(64 * waves_per_block), 0, stream>>>(plan_mt, chunks, visit_counts, err_word);
    GMM_HIP(hipGetLastError());
}

}  // namespace gmm
