// Plan-free map2tod / tod2map on gfx950: bilinear gather straight from the local map in HBM (through
// L2), one lane per sample, or scatter through a window of sums in LDS, four samples per lane.
// Reference: src_lib/map2tod_unplanned.cu:17-127, src_lib/tod2map_unplanned.cu:17-121.

#include "gmm_internal.hpp"
#include "gmm_locate.hpp"
#include "gmm_wave.hpp"

namespace gmm {

namespace {

constexpr int UP_THREADS = 256;

__device__ inline uint32_t wave_or_u(uint32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v |= __shfl_xor(v, off, 64);
    return v;
}

struct LocalMapView
{
    const int64_t *__restrict__ cell_offsets;
    int nycells, nxcells;
    int64_t ystride, polstride;

    // Offset of the cell of pixel (iy, ix), negative if it is not in the local map; of the pixel in it.
    __device__ inline int64_t cell(int iy, int ix) const
    {
        const int cy = iy >> 6, cx = ix >> 6;
        if (unsigned(cy) >= unsigned(nycells) || unsigned(cx) >= unsigned(nxcells))
            return -1;
        return cell_offsets[int64_t(cy) * nxcells + cx];
    }
    __device__ inline int64_t inside(int iy, int ix) const { return int64_t(iy & 63) * ystride + (ix & 63); }

    // Offset of the T value of pixel (iy, ix), or -1 if its cell is not in the local map.
    __device__ inline int64_t offset(int iy, int ix) const
    {
        const int64_t o = cell(iy, ix);
        return (o < 0) ? int64_t(-1) : o + inside(iy, ix);
    }
};

// The first n (up to 4) of 4 consecutive samples, zeros after (a float4 with Vec, where n and the
// address are multiples of 4 samples).
template<bool Vec>
__device__ inline void load_quad(const float *__restrict__ p, int n, float (&v)[4])
{
    if (Vec) {
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (n > 0)
            q = *reinterpret_cast<const float4 *>(p);
        v[0] = q.x;
        v[1] = q.y;
        v[2] = q.z;
        v[3] = q.w;
    }
    else {
#pragma unroll
        for (int j = 0; j < 4; j++)
            v[j] = (j < n) ? p[j] : 0.0f;
    }
}

// Plan-free map2tod. The map lies in the caches, and what counts is how many addresses a wave sends there
// (a gather takes 16 clocks for its 64 lanes). When the corners of each of a wave's samples lie in one
// cell, as most do, one offset is looked up a sample, and the two corners of a row are read together: 7
// gathers a sample in place of 16: 4.2e6 samples at 0.1 pixel per sample 31.5 -> 26.4 us, at 45 degrees
// 55 -> 34; at 0.7 pixel per sample, where most waves cross a cell's edge, 32 both (lane by lane 36).
// (Two or four samples a lane at once: 34 and 40 us.)
struct __attribute__((packed, aligned(4))) Pair
{
    float a, b;
};

// Value at the pixel whose T, Q and U are given.
__device__ inline float stokes(float t, float q, float u, float cs, float sn) { return t + cs * q + sn * u; }

template<bool Periodic>
__global__ void __launch_bounds__(UP_THREADS)
unplanned_map2tod_kernel(float *__restrict__ tod, const float *__restrict__ lmap, const float *__restrict__ xp,
                         LocalMapView mv, uint32_t *__restrict__ errflags, int64_t nsamp,
                         int64_t nsamp_per_block, int ny, int nx, bool partial, bool accum)
{
    __shared__ uint32_t s_err;
    if (threadIdx.x == 0)
        s_err = 0;
    __syncthreads();

    const int64_t s0 = int64_t(blockIdx.x) * nsamp_per_block;
    const int64_t s1 = min(nsamp, s0 + nsamp_per_block);
    uint32_t err = 0;

    for (int64_t s = s0 + threadIdx.x; s < s1; s += UP_THREADS) {
        const float y = xp[s], x = xp[s + nsamp], alpha = xp[s + 2 * nsamp];
        Pixel<float> p;
        err |= locate_pixel(y, x, ny, nx, Periodic, p);
        const int64_t o = mv.offset(p.iy0, p.ix0);
        float sn, cs;
        sincos_angle(2.0f * alpha, sn, cs);
        const float wy0 = 1.0f - p.dy, wx0 = 1.0f - p.dx;
        float val;
        const bool one_cell = o >= 0 && (p.iy0 & 63) != 63 && (p.ix0 & 63) != 63 && p.iy1 == p.iy0 + 1
                           && p.ix1 == p.ix0 + 1;
        if (__all(one_cell)) {
            Pair m[2][3];
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int pl = 0; pl < 3; pl++)
                    m[r][pl] = *reinterpret_cast<const Pair *>(lmap + o + r * mv.ystride + pl * mv.polstride);
            val = (wy0 * wx0) * stokes(m[0][0].a, m[0][1].a, m[0][2].a, cs, sn);
            val += (wy0 * p.dx) * stokes(m[0][0].b, m[0][1].b, m[0][2].b, cs, sn);
            val += (p.dy * wx0) * stokes(m[1][0].a, m[1][1].a, m[1][2].a, cs, sn);
            val += (p.dy * p.dx) * stokes(m[1][0].b, m[1][1].b, m[1][2].b, cs, sn);
        }
        else {
            val = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int64_t oc = mv.offset((c & 2) ? p.iy1 : p.iy0, (c & 1) ? p.ix1 : p.ix0);
                const float w = ((c & 2) ? p.dy : wy0) * ((c & 1) ? p.dx : wx0);
                float v = 0.0f;
                if (oc >= 0)
                    v = stokes(lmap[oc], lmap[oc + mv.polstride], lmap[oc + 2 * mv.polstride], cs, sn);
                else if (!partial)
                    err |= ERR_NOT_IN_PIXELIZATION;
                val += w * v;
            }
        }
        tod[s] = accum ? (tod[s] + val) : val;
    }

    err = wave_or_u(err);
    if ((threadIdx.x & 63) == 0 && err)
        atomicOr(&s_err, err);
    __syncthreads();
    if (threadIdx.x == 0)
        errflags[blockIdx.x] = s_err;
}

// ------------------------------------------------------------------------------------------
// Plan-free tod2map. One float atomic to the map per sample, corner and plane takes 2318 us for 4.2e6
// samples at 0.1 pixel per sample: neighbouring samples hit the same pixels and wait for each other.
// Here a block takes 1024 consecutive samples at a time, 4 a lane, and sums their deposits in LDS
// before they go to the map (34 us; VALU issue is 25 of them), in a window along the straight line that
// the samples follow: at each place j of the window's major axis it holds the few pixels around the
// line, so that a scan in any direction fits (45 degrees: 69 us, the map rows it crosses are that many
// more atomic requests; 0.73 pixel per sample: 105 us). What falls outside goes to the map: samples that
// lie together summed in registers first (16 samples a detector at 0.1 pixel per sample 2370 -> 505 us of
// the call), others with consecutive samples in consecutive lanes, as without windows (with a lane's four
// one after the other, and their blocks' waves in turn, 3 pixels per sample along x took 1590 us, 667
// without windows, 600 now; random pointing 2460 us).
// The sums are float64: ds_add_f64 takes 9 clocks a wave, ds_add_f32 194 (measured). An element that
// was never added to holds -0.0 in its T plane, which no sum of values other than -0.0 gives.

constexpr int WIN_THREADS = 256, WIN_WAVES = WIN_THREADS / 64;
constexpr int WIN_SAMPLES = 4 * WIN_THREADS;
constexpr int WIN_N = 1024;                // pixels of the window (24 KiB of sums: 6 blocks per CU)
// Least number of a wave's 256 samples that are worth a round of their own (from a few detectors' turns to
// 5 pixels per sample 16, 32 and 64 are the same; 128 takes 2400 us for 4.2e6 samples at 1 pixel per
// sample along y, 32 takes 1610). Calls of a few blocks could do without rounds (1000 samples 54 us, 49
// straight to the map), but their sums would carry more float32 roundings.
constexpr int WIN_SHARE = 32;
// Lanes of a wave: with so many whose four samples step by a pixel or so, what its window does not hold is
// left for deposit_far(), where consecutive lanes then meet in cache lines. In slower waves they would meet
// in pixels and wait for each other (one detector's 2^21 samples at 0.58 pixel per sample, back and forth
// over the same rows, 250 us; 178 when the lanes' samples follow one after the other): there all but those
// for deposit_near(), if they are WIN_NEAR lanes or more, take the round together, and a few held ones are
// enough for it when most are not near. Calls without a block for each CU wait for each pass: their slow
// waves make one only (8 x 16384 samples 66 us, 70 with deposit_near()).
constexpr int WIN_SOME = 32, WIN_NEAR = 24, WIN_BLOCKS = 256;
constexpr int WIN_LEAD = 4;                // places before the least one seen (lanes show one of their 4 samples)
typedef double WindowSums[3][WIN_N];

// The window's major axis is x for lines that rise by at most a third: 8 pixels of y at each of 128
// places (room for a scan that turns inside the block and comes back a few pixels beside its way out),
// or 4 at 256 places for samples that go further. Else it is y: 8 pixels of x at each of 113 places, a
// stride of 9 against bank conflicts.
struct Window
{
    bool xmajor;
    int length, width;     // places along the major axis, pixels at each
    int jstride, kstride;
    int major0, minor0;    // (major0, minor0) is the first pixel of place WIN_LEAD
    int slope;             // 65536 * minor pixels per major pixel, at most 3 * 65536 in magnitude

    __device__ int place(int major) const { return major - major0 + WIN_LEAD; }
    // First minor pixel held at place j. (Far outside the window, on maps of more than 10922 pixels, the
    // product wraps, and the place is refused for its j.)
    __device__ int line(int j) const { return minor0 + (int(uint32_t(slope) * uint32_t(j - WIN_LEAD)) >> 16); }

    // Element of a pixel, or -1.
    __device__ int find(int iy, int ix) const
    {
        const int j = place(xmajor ? ix : iy), k = (xmajor ? iy : ix) - line(j);
        return (unsigned(j) < unsigned(length) && unsigned(k) < unsigned(width)) ? j * jstride + k * kstride : -1;
    }
};

// Positions packed with one axis on top, so that the extremes of that axis come with their place on
// the other: y << 16 | x of the least and the largest y, x << 16 | y of the least and the largest x.
struct Extremes
{
    uint32_t ylo, yhi, xlo, xhi;

    __device__ void merge(const Extremes &o)
    {
        ylo = min(ylo, o.ylo);
        yhi = max(yhi, o.yhi);
        xlo = min(xlo, o.xlo);
        xhi = max(xhi, o.xhi);
    }
    __device__ int dy() const { return int(yhi >> 16) - int(ylo >> 16); }
    __device__ int dx() const { return int(xhi >> 16) - int(xlo >> 16); }
};

__device__ inline Extremes wave_extremes(bool on, int iy, int ix)
{
    const uint32_t py = (uint32_t(iy) << 16) | (uint32_t(ix) & 0xffffu), px = (uint32_t(ix) << 16) | (uint32_t(iy) & 0xffffu);
    Extremes e;
    e.ylo = wave_min_u32(on ? py : 0xffffffffu);
    e.yhi = wave_max_u32(on ? py : 0u);
    e.xlo = wave_min_u32(on ? px : 0xffffffffu);
    e.xhi = wave_max_u32(on ? px : 0u);
    return e;
}

__device__ inline Window make_window(const Extremes &e)
{
    const int dy = e.dy(), dx = e.dx();
    Window w;
    w.xmajor = dx >= 3 * dy;
    w.length = w.xmajor ? ((dx <= 128 - 2 * WIN_LEAD) ? 128 : 256) : 113;
    w.width = w.xmajor ? WIN_N / w.length : 8;
    w.jstride = w.xmajor ? 1 : 9;
    w.kstride = w.xmajor ? w.length : 1;
    const uint32_t lo = w.xmajor ? e.xlo : e.ylo, hi = w.xmajor ? e.xhi : e.yhi;
    const int d = w.xmajor ? dx : dy;
    w.major0 = int(lo >> 16);
    w.slope = (d > 0) ? int(float(int(hi & 0xffffu) - int(lo & 0xffffu)) * (65536.0f / float(d))) : 0;
    w.slope = min(max(w.slope, -3 * 65536), 3 * 65536);
    // The line and the samples' pixels differ by up to a pixel, and a footprint is two pixels wide.
    w.minor0 = int(lo & 0xffffu) - (w.width / 2 - 1);
    return w;
}

__device__ inline void window_clear(WindowSums &acc)
{
    double2 *a2 = reinterpret_cast<double2 *>(&acc[0][0]);
    for (int i = threadIdx.x; i < 3 * WIN_N / 2; i += WIN_THREADS) {
        const double z = (i < WIN_N / 2) ? -0.0 : 0.0;
        a2[i] = make_double2(z, z);
    }
}

// Adds the window to the map and clears it. Consecutive lanes take consecutive pixels of a map row (256
// or 8 of them): the L2 takes about 35e9 atomic requests per second, whether a request carries one
// float or the 16 of a 64-byte line.
__device__ inline void window_flush(const Window &win, WindowSums &acc, float *__restrict__ lmap,
                                    const LocalMapView &mv, bool partial, uint32_t &err)
{
    constexpr int NE = WIN_N / WIN_THREADS;
    int e[NE];
    int64_t o[NE];
    double t[NE];
    // All of a thread's elements and their cells first, so that the loads overlap.
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int l = threadIdx.x + i * WIN_THREADS;
        const int k = win.xmajor ? l >> ((win.length == 128) ? 7 : 8) : (l & 7);
        const int j = win.xmajor ? (l & (win.length - 1)) : (l >> 3);
        const bool in = j < win.length;
        e[i] = in ? j * win.jstride + k * win.kstride : 0;
        t[i] = in ? acc[0][e[i]] : -0.0;
        const int major = win.major0 + j - WIN_LEAD, minor = win.line(j) + k;
        const int iy = win.xmajor ? minor : major, ix = win.xmajor ? major : minor;
        o[i] = mv.offset(iy, ix);
    }
#pragma unroll
    for (int i = 0; i < NE; i++) {
        if (__double_as_longlong(t[i]) == (long long)(1ull << 63))
            continue;
        const double q = acc[1][e[i]], u = acc[2][e[i]];
        acc[0][e[i]] = -0.0;
        acc[1][e[i]] = 0.0;
        acc[2][e[i]] = 0.0;
        if (o[i] >= 0) {
            unsafeAtomicAdd(lmap + o[i], float(t[i]));
            unsafeAtomicAdd(lmap + o[i] + mv.polstride, float(q));
            unsafeAtomicAdd(lmap + o[i] + 2 * mv.polstride, float(u));
        }
        else if (!partial)
            err |= ERR_NOT_IN_PIXELIZATION;
    }
}

__device__ inline void window_add(WindowSums &acc, int e, float t, float q, float u)
{
    unsafeAtomicAdd(&acc[0][e], double(t + 0.0f));        // + 0: a value of -0.0 counts as added
    unsafeAtomicAdd(&acc[1][e], double(q));
    unsafeAtomicAdd(&acc[2][e], double(u));
}

// A sample's place: the (iy0, ix0) corner of its footprint and the offsets from it.
struct Place
{
    int iy0, ix0;
    float dy, dx;
};

// The four corners of one sample: to the window or, outside it, to the map.
template<bool Periodic>
__device__ inline void deposit_sample(const Place &p, float t, float q, float u, const Window &win, WindowSums &acc,
                                      float *__restrict__ lmap, const LocalMapView &mv, int nx, bool partial, uint32_t &err)
{
#pragma unroll 1
    for (int i = 0; i < 4; i++) {
        const int iy = p.iy0 + (i >> 1);
        int ix = p.ix0 + (i & 1);
        if (Periodic)
            ix = (ix < nx) ? ix : 0;
        const float w = ((i & 2) ? p.dy : 1.0f - p.dy) * ((i & 1) ? p.dx : 1.0f - p.dx);
        const int e = win.find(iy, ix);
        if (e >= 0)
            window_add(acc, e, w * t, w * q, w * u);
        else {
            const int64_t o = mv.offset(iy, ix);
            if (o >= 0) {
                unsafeAtomicAdd(lmap + o, w * t);
                unsafeAtomicAdd(lmap + o + mv.polstride, w * q);
                unsafeAtomicAdd(lmap + o + 2 * mv.polstride, w * u);
            }
            else if (!partial)
                err |= ERR_NOT_IN_PIXELIZATION;
        }
    }
}

// Samples that no window holds go straight to the map. Four of a lane whose footprints are within 3 x 3
// pixels are summed in registers before ...
__device__ inline void deposit_near(const Place (&p)[4], const float (&t)[4], const float (&q)[4], const float (&u)[4],
                                    float *__restrict__ lmap, const LocalMapView &mv, bool partial, uint32_t &err)
{
    const int iy = min(min(p[0].iy0, p[1].iy0), min(p[2].iy0, p[3].iy0));
    const int ix = min(min(p[0].ix0, p[1].ix0), min(p[2].ix0, p[3].ix0));
    // The pixels' cells are those of the first and the last row and column: four lookups at once. (They do not
    // wrap: the three columns of nx - 2, nx - 1 and 0 can lie in three cells.)
    const int64_t o00 = mv.cell(iy, ix), o01 = mv.cell(iy, ix + 2), o10 = mv.cell(iy + 2, ix), o11 = mv.cell(iy + 2, ix + 2);
#pragma unroll 1
    for (int i = 0; i < 9; i++) {
        const int y = iy + i / 3, x = ix + i % 3;
        float a = 0.0f, b = 0.0f, c = 0.0f;
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int r = y - p[k].iy0, l = x - p[k].ix0;
            if (unsigned(r) <= 1u && unsigned(l) <= 1u) {
                const float w = (r ? p[k].dy : 1.0f - p[k].dy) * (l ? p[k].dx : 1.0f - p[k].dx);
                a = fmaf(w, t[k], a);
                b = fmaf(w, q[k], b);
                c = fmaf(w, u[k], c);
                any = true;
            }
        }
        if (any) {
            const bool row = (y ^ iy) >> 6, col = (x ^ ix) >> 6;
            int64_t o = row ? (col ? o11 : o10) : (col ? o01 : o00);
            if (o >= 0) {
                o += mv.inside(y, x);
                unsafeAtomicAdd(lmap + o, a);
                unsafeAtomicAdd(lmap + o + mv.polstride, b);
                unsafeAtomicAdd(lmap + o + 2 * mv.polstride, c);
            }
            else if (!partial)
                err |= ERR_NOT_IN_PIXELIZATION;
        }
    }
}

// ... and others, those of a wave's 256 samples from s on that are not done (sample i: bit i / 4 of
// 'done' in lanes i % 4, i % 4 + 4 ...), one per lane and consecutive lanes consecutive samples: their atomics share cache lines
// where the scan runs along a map row.
template<bool Periodic>
__device__ inline void deposit_far(float *__restrict__ lmap, const float *__restrict__ tod, const float *__restrict__ xp,
                                   int64_t nsamp, int64_t s, int64_t s1, uint64_t done, const Geom &g,
                                   const LocalMapView &mv, bool partial, uint32_t &err)
{
    Checks checked;                            // with the tile's samples
    const int lane = threadIdx.x & 63;
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        const int64_t i = s + 64 * r + lane;
        if (i >= s1 || ((done >> (16 * r + (lane >> 2))) & 1u))
            continue;
        const float y = xp[i], x = xp[nsamp + i], alpha = xp[2 * nsamp + i], t = tod[i];
        Place p;
        locate_op<Periodic>(y, x, g, checked, p.iy0, p.ix0, p.dy, p.dx);
        // The corners' cells are looked up at once.
        const int iy1 = p.iy0 + 1, ix1 = (Periodic && p.ix0 + 1 >= g.nx) ? 0 : p.ix0 + 1;
        const int64_t o00 = mv.cell(p.iy0, p.ix0), o01 = mv.cell(p.iy0, ix1), o10 = mv.cell(iy1, p.ix0), o11 = mv.cell(iy1, ix1);
        float sn, cs;
        sincos_angle(2.0f * alpha, sn, cs);
        const float q = t * cs, u = t * sn;
#pragma unroll 1
        for (int c = 0; c < 4; c++) {
            const bool row = c & 2, col = c & 1;
            int64_t o = row ? (col ? o11 : o10) : (col ? o01 : o00);
            const float w = (row ? p.dy : 1.0f - p.dy) * (col ? p.dx : 1.0f - p.dx);
            if (o >= 0) {
                o += mv.inside(row ? iy1 : p.iy0, col ? ix1 : p.ix0);
                unsafeAtomicAdd(lmap + o, w * t);
                unsafeAtomicAdd(lmap + o + mv.polstride, w * q);
                unsafeAtomicAdd(lmap + o + 2 * mv.polstride, w * u);
            }
            else if (!partial)
                err |= ERR_NOT_IN_PIXELIZATION;
        }
    }
}

// Where the four samples of a lane lie in a window, if they span at most two pixels along each axis:
// their footprints are then within 3 x 3 pixels.
struct QuadPlace
{
    int mj, mn;            // smallest corner on the major and minor axis
    uint32_t at;           // bit 2 * a + b: some sample's corner is at (mj + a, mn + b)
    int base[3];           // elements of (mj + m, mn)
    bool fast;             // the samples span more than three pixels along an axis
    bool near;             // the footprints are within 3 x 3 pixels and don't wrap,
    bool fits;             // which the window holds
};

template<bool Periodic>
__device__ inline QuadPlace place_quad(const Place (&p)[4], const Window &win, int nx)
{
    int pj[4], pn[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        pj[k] = win.xmajor ? p[k].ix0 : p[k].iy0;
        pn[k] = win.xmajor ? p[k].iy0 : p[k].ix0;
    }
    QuadPlace z;
    z.mj = min(min(pj[0], pj[1]), min(pj[2], pj[3]));
    z.mn = min(min(pn[0], pn[1]), min(pn[2], pn[3]));
    const int ej = max(max(pj[0], pj[1]), max(pj[2], pj[3])), en = max(max(pn[0], pn[1]), max(pn[2], pn[3]));
    z.at = 0;
#pragma unroll
    for (int k = 0; k < 4; k++)
        z.at |= (pj[k] != z.mj ? 4u : 1u) << (pn[k] != z.mn ? 1 : 0);
    const bool j2 = ej > z.mj, n2 = en > z.mn;
    const int j = win.place(z.mj);
    int lo = 0, hi = 0;                                   // minor places of (mj + m, mn)
#pragma unroll
    for (int m = 0; m < 3; m++) {
        const int k = z.mn - win.line(j + m);
        z.base[m] = (j + m) * win.jstride + k * win.kstride;
        if (m < 2 || j2) {
            lo = min(lo, k);
            hi = max(hi, k);
        }
    }
    z.fast = max(ej - z.mj, en - z.mn) > 2;
    // x0 = nx - 1 of periodic x has its second column at x = 0.
    z.near = ej - z.mj <= 1 && en - z.mn <= 1 && !(Periodic && (win.xmajor ? ej : en) + 1 >= nx);
    z.fits = z.near && j >= 0 && j + (j2 ? 2 : 1) < win.length && lo >= 0 && hi + (n2 ? 2 : 1) < win.width;
    return z;
}

// The four samples of a lane whose place fits: the pixels of their footprints are summed in registers
// and added to the window once each (at most 27 LDS atomics instead of 48).
__device__ inline void deposit_quad(const Place (&p)[4], const float (&t)[4], const float (&q)[4],
                                    const float (&u)[4], const QuadPlace &z, const Window &win, WindowSums &acc)
{
    float wj[4][3], wn[4][3];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float dj = win.xmajor ? p[k].dx : p[k].dy, dn = win.xmajor ? p[k].dy : p[k].dx;
        const bool sj = (win.xmajor ? p[k].ix0 : p[k].iy0) != z.mj, sn = (win.xmajor ? p[k].iy0 : p[k].ix0) != z.mn;
        wj[k][0] = sj ? 0.0f : 1.0f - dj;
        wj[k][1] = sj ? 1.0f - dj : dj;
        wj[k][2] = sj ? dj : 0.0f;
        wn[k][0] = sn ? 0.0f : 1.0f - dn;
        wn[k][1] = sn ? 1.0f - dn : dn;
        wn[k][2] = sn ? dn : 0.0f;
    }
    auto pix = [&](int m, int n) {
        float a = 0.0f, b = 0.0f, c = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float w = wj[k][m] * wn[k][n];
            a = fmaf(w, t[k], a);
            b = fmaf(w, q[k], b);
            c = fmaf(w, u[k], c);
        }
        window_add(acc, z.base[m] + n * win.kstride, a, b, c);
    };
    // Only pixels of some sample's footprint (a pixel next to them may be in an absent cell).
    const bool j2 = z.at & 0xcu, n2 = z.at & 0xau;
    if (z.at & 1u)
        pix(0, 0);
    pix(0, 1);
    pix(1, 0);
    pix(1, 1);
    if (n2)
        pix(1, 2);
    if (z.at & 2u)
        pix(0, 2);
    if (j2)
        pix(2, 1);
    if (z.at & 4u)
        pix(2, 0);
    if (z.at & 8u)
        pix(2, 2);
}

template<bool Periodic, bool Vec>
__global__ void __launch_bounds__(WIN_THREADS, 4)
unplanned_tod2map_kernel(float *__restrict__ lmap, const float *__restrict__ tod, const float *__restrict__ xp,
                         LocalMapView mv, uint32_t *__restrict__ errflags, int64_t nsamp,
                         int64_t nsamp_per_block, int ny, int nx, bool partial)
{
    __shared__ __align__(16) WindowSums acc;
    __shared__ Extremes s_ext[WIN_WAVES];
    __shared__ uint32_t s_err, s_split, s_use;
    if (threadIdx.x == 0)
        s_err = s_split = 0;
    window_clear(acc);

    const int wave = threadIdx.x >> 6;
    const int64_t s0 = int64_t(blockIdx.x) * nsamp_per_block;
    const int64_t s1 = min(nsamp, s0 + nsamp_per_block);
    const Geom g = make_geom(ny, nx, Periodic);
    Checks chk;
    uint32_t err = 0;

    for (int64_t base = s0; base < s1; base += WIN_SAMPLES) {
        const int64_t s = base + 4 * int64_t(threadIdx.x);
        const int n = int(max<int64_t>(0, min<int64_t>(4, s1 - s)));
        float y[4], x[4], alpha[4], t[4];
        load_quad<Vec>(xp + s, n, y);
        load_quad<Vec>(xp + nsamp + s, n, x);
        load_quad<Vec>(xp + 2 * nsamp + s, n, alpha);
        load_quad<Vec>(tod + s, n, t);
        // Samples past the end repeat the first one's place with a zero value.
        Place p[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            locate_op<Periodic>((k < n) ? y[k] : y[0], (k < n) ? x[k] : x[0], g, chk, p[k].iy0, p[k].ix0, p[k].dy, p[k].dx);
        const Extremes we = wave_extremes(n > 0, p[0].iy0, p[0].ix0);
        if ((threadIdx.x & 63) == 0)
            s_ext[wave] = we;
        __syncthreads();
        // sin and cos of 2 alpha: of sample 0, and by angle addition of the others where every lane's
        // steps are small enough for it (consecutive samples of one detector).
        float q[4], u[4], s0a, c0a;
        const float a0 = 2.0f * alpha[0];
        sincos_angle(a0, s0a, c0a);
        const float dmax = fmaxf(fmaxf(fabsf(2.0f * alpha[1] - a0), fabsf(2.0f * alpha[2] - a0)), fabsf(2.0f * alpha[3] - a0));
        const bool near = !__any(!(dmax <= 0.0185f));
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float sn = s0a, cs = c0a;
            if (k > 0) {
                if (near)
                    angle_step(s0a, c0a, 2.0f * alpha[k] - a0, sn, cs);
                else
                    sincos_angle(2.0f * alpha[k], sn, cs);
            }
            q[k] = t[k] * cs;
            u[k] = t[k] * sn;
        }
        // One window for the block or, where some wave does not fit it (a turn of the scan, a fast
        // one), one after the other for its waves.
        Extremes all = s_ext[0];
#pragma unroll
        for (int w = 1; w < WIN_WAVES; w++)
            all.merge(s_ext[w]);
        Window win = make_window(all);
        QuadPlace z = place_quad<Periodic>(p, win, nx);
        // 3 x 3 sums give every sample a (zero) weight in all nine pixels: a sample that is not finite
        // would reach pixels that it does not touch.
        const bool finite = fmaf(q[0], 0.0f, fmaf(q[1], 0.0f, fmaf(q[2], 0.0f, q[3] * 0.0f))) == 0.0f;
        bool fits = !__any(n > 0 && !(z.fits && finite));
        if (!fits && (threadIdx.x & 63) == 0)
            s_split = 1;
        if (threadIdx.x == 0)
            s_use = 0;
        __syncthreads();
        // A wave whose lanes' samples do not fit (faster than half a pixel per sample, a few of many
        // detectors, scattered) adds those that its window holds one by one, if they are enough to be worth
        // a round; the rest go to the map.
        const bool split = s_split;
        uint32_t held = 0, rounds = 1;
        bool use = __any(n > 0);
        if (split) {
            win = make_window(s_ext[wave]);
            z = place_quad<Periodic>(p, win, nx);
            fits = !__any(n > 0 && !(z.fits && finite));
            if (!fits) {
                int nheld = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    // (Of its four corners two opposite ones are looked at.)
                    const bool in = k < n && max(win.find(p[k].iy0, p[k].ix0), win.find(p[k].iy0 + 1, p[k].ix0 + 1)) >= 0;
                    held |= in ? 1u << k : 0u;
                    nheld += __popcll(__ballot(in));
                }
                const bool slow = __popcll(__ballot(n > 0 && z.fast)) < WIN_SOME, small = gridDim.x < WIN_BLOCKS;
                const int nmid = __popcll(__ballot(n > 0 && !z.fast && !z.near));
                const int napart = __popcll(__ballot(n > 0 && held == 0 && z.near));
                use = (slow && small) || nheld >= ((nmid >= WIN_SOME) ? 1 : WIN_SHARE);
                const bool apart = held == 0 && z.near && napart >= WIN_NEAR && !small;
                if (!use)
                    held = 0;
                else if (slow && !apart)
                    held = (1u << n) - 1u;
            }
            if (use && (threadIdx.x & 63) == 0)
                atomicOr(&s_use, 1u << wave);
            __syncthreads();
            rounds = s_use;
            if (threadIdx.x == 0)
                s_split = 0;                              // every wave has read it
        }
#pragma unroll 1
        for (; rounds; rounds &= rounds - 1) {
            const int w0 = __builtin_ctz(rounds);
            if (split)
                win = make_window(s_ext[w0]);
            if (n > 0 && (!split || wave == w0)) {
                if (fits)
                    deposit_quad(p, t, q, u, z, win, acc);
                else {
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        if ((held >> k) & 1u)
                            deposit_sample<Periodic>(p[k], t[k], q[k], u[k], win, acc, lmap, mv, nx, partial, err);
                }
            }
            __syncthreads();
            window_flush(win, acc, lmap, mv, partial, err);
            __syncthreads();
        }
        if (!fits) {
            const bool near = held == 0 && z.near;
            uint64_t done = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t b = __ballot(near || ((held >> k) & 1u));
                done = ((threadIdx.x & 3) == k) ? b : done;
            }
            if (near && n > 0)
                deposit_near(p, t, q, u, lmap, mv, partial, err);
            deposit_far<Periodic>(lmap, tod, xp, nsamp, base + 256 * wave, s1, done, g, mv, partial, err);
        }
    }

    err = wave_or_u(err | chk.bits(g));
    if ((threadIdx.x & 63) == 0 && err)
        atomicOr(&s_err, err);
    __syncthreads();
    if (threadIdx.x == 0)
        errflags[blockIdx.x] = s_err;
}

// Whole rounds of the block's threads, as few as max_blocks allow: a round is a chain of dependent loads, and
// small calls take as long as their blocks (8 x 4096 samples 10.6 us in 8 rounds a block, 4.2 in one).
int64_t samples_per_block(int64_t nsamp, int64_t max_blocks)
{
    const int64_t spb = (nsamp + max_blocks - 1) / max_blocks;
    return (spb + UP_THREADS - 1) / UP_THREADS * UP_THREADS;
}

// tod2map: whole windows of samples.
int64_t tod2map_samples_per_block(int64_t nsamp, int64_t max_blocks)
{
    const int64_t spb = (nsamp + max_blocks - 1) / max_blocks;
    return (spb + WIN_SAMPLES - 1) / WIN_SAMPLES * WIN_SAMPLES;
}

}  // namespace

int64_t unplanned_nblocks(int64_t nsamp, int64_t max_blocks)
{
    int64_t spb = samples_per_block(nsamp, max_blocks);
    return (nsamp + spb - 1) / spb;
}

void launch_unplanned_map2tod(float *tod, const float *lmap, const float *xp, const OpArgs &a,
                              uint32_t *errflags, int64_t max_blocks, bool accum, hipStream_t stream)
{
    const gmm_lpix &lp = *a.lpix;
    const int64_t spb = samples_per_block(a.nsamp, max_blocks);
    const int64_t nb = (a.nsamp + spb - 1) / spb;
    LocalMapView mv{lp.offsets_gpu, int(lp.nycells), int(lp.nxcells), lp.ystride, lp.polstride};
    auto k = lp.periodic_xcoord ? unplanned_map2tod_kernel<true> : unplanned_map2tod_kernel<false>;
    k<<<unsigned(nb), UP_THREADS, 0, stream>>>(tod, lmap, xp, mv, errflags, a.nsamp, spb,
                                               int(lp.nypix_global), int(lp.nxpix_global), a.partial, accum);
    GMM_HIP(hipGetLastError());
}

int64_t unplanned_tod2map_nblocks(int64_t nsamp, int64_t max_blocks)
{
    const int64_t spb = tod2map_samples_per_block(nsamp, max_blocks);
    return (nsamp + spb - 1) / spb;
}

void launch_unplanned_tod2map(float *lmap, const float *tod, const float *xp, const OpArgs &a,
                              uint32_t *errflags, int64_t max_blocks, hipStream_t stream)
{
    const gmm_lpix &lp = *a.lpix;
    const int64_t spb = tod2map_samples_per_block(a.nsamp, max_blocks);
    const int64_t nb = (a.nsamp + spb - 1) / spb;
    LocalMapView mv{lp.offsets_gpu, int(lp.nycells), int(lp.nxcells), lp.ystride, lp.polstride};
    const bool vec = ((reinterpret_cast<uintptr_t>(tod) | reinterpret_cast<uintptr_t>(xp)) & 15) == 0 && a.nsamp % 4 == 0;
    auto k = lp.periodic_xcoord ? (vec ? unplanned_tod2map_kernel<true, true> : unplanned_tod2map_kernel<true, false>)
                                : (vec ? unplanned_tod2map_kernel<false, true> : unplanned_tod2map_kernel<false, false>);
    k<<<unsigned(nb), WIN_THREADS, 0, stream>>>(lmap, tod, xp, mv, errflags, a.nsamp, spb,
                                                int(lp.nypix_global), int(lp.nxpix_global), a.partial);
    GMM_HIP(hipGetLastError());
}

}  // namespace gmm
