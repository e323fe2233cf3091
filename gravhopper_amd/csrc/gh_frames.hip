// Spatial order and local frames of the FP32 pair kernels.
//
// An FP32 pair force needs the separation x_j - x_i.  Casting absolute FP64 positions to
// FP32 first and subtracting afterwards loses 2^-24 |x| per coordinate, which for a
// star cluster 8 kpc from the coordinate origin is a relative error of order 1e-4 on
// its internal forces (the reference forms every difference in FP64,
// gravhopper/_jbgrav.c:155-168).  The FP32 kernels therefore never cast an absolute
// position.  Points are sorted along a Morton curve (about 11 levels in their root box) and
// cut into groups of consecutive sorted points (the kernels' blocks); each group g has
// an FP64 origin o_g, one of its own points, and the kernels work in the frame of one
// group: a point of group h enters as fl(x - o_h) + fl(o_h - o_g), both formed from FP64
// values.  The rounding error of a separation is then bounded by 2^-24 times the extents
// of the groups involved plus the separation itself, independent of where the system
// sits.
//
// A sorted group is compact unless the curve jumps between two clusters inside it (two
// galaxies far apart, or the rare large jump of the curve itself).  k_frames measures
// this per group: R = max |x - o| against the geometric mean s of the gaps between
// consecutive sorted points of the group; R > 2^kFrameLog2 s flags the group, and pairs
// involving a flagged group are computed in double-single form (hi + lo FP32 pairs of
// FP64 differences), whose separations are exact to 2^-24 |x_j - x_i| whatever the
// group's shape.
#include <algorithm>

#include "gh_box.h"
#include "gh_runsort.h"
#include "gh_internal.h"

namespace gh {

// 21-bit integer spread to every third bit (bit k of v goes to bit 3k).
__device__ __forceinline__ u64 spread3(u64 v)
{
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

// The sort uses key bits [kKeyShift, 63) of the 63-bit Morton key.
constexpr int kKeyShift = 31;

__device__ __forceinline__ u32 quantize(double x, double lo, double scale)
{
    double q = (x - lo) * scale;
    q = q > 0.0 ? q : 0.0;  // also maps NaN to 0
    return q < 2097151.0 ? (u32)q : 2097151u;
}

// Morton key of 21 levels (bit 3k + a: level 20 - k, axis a) of point i in the box
// box[0..2] = centre, box[3] = size.
__device__ __forceinline__ u64 morton_key(const double* __restrict__ pos, int64_t i,
                                          const double* box)
{
    const double size = box[3];
    const double scale = size > 0.0 ? 2097152.0 / size : 0.0;
    u64 k = 0;
    for (int a = 0; a < 3; a++)
        k |= spread3(quantize(pos[3 * i + a], box[a] - 0.5 * size, scale)) << a;
    return k;
}

// Morton keys of the points; idx = identity.
__global__ __launch_bounds__(kBlock) void k_morton(const double* __restrict__ pos, int64_t n,
                                                   const double* __restrict__ box,
                                                   u64* __restrict__ keys,
                                                   u32* __restrict__ idx,
                                                   int* __restrict__ nflag)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i == 0) *nflag = 0;
    if (i >= n) return;
    double b[4];
    for (int k = 0; k < 4; k++) b[k] = box[k];
    keys[i] = morton_key(pos, i, b);
    idx[i] = (u32)i;
}

// Small sorts, in runs of up to 1024 points (gh_runsort.h).  The sort of one call, radix passes
// of one launch each before: 43 us at N = 3000, now 19; 50 us at 16384, now 18.
// Bits kKeyShift .. 62 of the Morton key: from bit 0 on y and z of level 10, then x, y, z of
// levels 11 .. 20 (bit 3 k + a of the key is bit k of axis a).
static_assert(kKeyShift == 31, "the axes' shares of the 32 key bits");
__device__ __forceinline__ u32 spread3_11(u32 v)
{
    v = (v | (v << 16)) & 0x070000ffu;
    v = (v | (v << 8)) & 0x0700f00fu;
    v = (v | (v << 4)) & 0x430c30c3u;
    return (v | (v << 2)) & 0x49249249u;
}

// Root box (as k_bbox_final with eps = 0) of the n points from pos on, in every thread of the
// workgroup; minima and maxima are exact in any order.
__device__ __forceinline__ void points_box(const double* __restrict__ pos, int n, double box[4])
{
    double mn[3], mx[3];
    for (int a = 0; a < 3; a++) mn[a] = mx[a] = pos[a];  // the first point seeds
#pragma unroll 4
    for (int i = threadIdx.x; i < n; i += kRunThreads)
        for (int a = 0; a < 3; a++) {
            const double q = pos[3 * i + a];
            if (q < mn[a]) mn[a] = q;
            if (q > mx[a]) mx[a] = q;
        }
    run_extents(mn, mx);
    box_of_extents(mn, mx, 0.0, box);
}

// Run b of RUN points (RUN of the kRunThreads threads hold one each; all of them form the box
// of the run's segment): the keys in order, with the points they belong to.  Places behind the
// segment's points are filled with the largest key.  single: no segment has more than one run,
// whose order is then the segment's and goes to perm at once.
template <int RUN>
__global__ __launch_bounds__(kRunThreads) void k_rank_runs(
    const double* __restrict__ pos, int64_t n_all, const int* __restrict__ seg,
    const int64_t* __restrict__ seg_start, const int64_t* __restrict__ seg_count,
    u32* __restrict__ keys, u32* __restrict__ from, u32* __restrict__ perm,
    int* __restrict__ nflag, bool single)
{
    const int t = threadIdx.x;
    const int g = seg ? seg[blockIdx.x] : 0;
    const int64_t first = seg ? seg_start[g] : 0;
    const int n = (int)(seg ? seg_count[g] : n_all);
    if (blockIdx.x == 0 && t == 0) *nflag = 0;
    const double* p = pos + 3 * first;
    double box[4];
    points_box(p, n, box);
    const bool act = t < RUN;  // whole wavefronts
    const int64_t base = (int64_t)blockIdx.x * RUN;
    const int i = (int)(base - first) + t;
    u32 key = 0xffffffffu, idx = (u32)(base + t);
    if (act && i < n) {
        const double size = box[3], scale = size > 0.0 ? 2097152.0 / size : 0.0;
        u32 q[3];
        for (int a = 0; a < 3; a++) q[a] = quantize(p[3 * i + a], box[a] - 0.5 * size, scale);
        key = spread3_11(q[1] >> 10) | spread3_11(q[2] >> 10) << 1 | spread3_11(q[0] >> 11) << 2;
    } else if (act && seg) {
        perm[base + t] = idx;
    }
    const int at = sort_run<RUN>(key, idx, act);
    if (act && single) {
        if ((int64_t)idx - first < n) perm[base + at] = idx;
    } else if (act) {
        keys[base + at] = key;
        from[base + at] = idx;
    }
}

// The order of n points, or of segments of at most `most` points each (runs of `run` places,
// seg[b] the segment of run b), as o.perm().  keys[0] and keys[1] hold n_pad 32-bit words.  The
// merge has as many wavefronts as there are parts of 1024 keys to search, up to 16: more would
// hold places that other workgroups wait for (4 steps of 2000 simulations of 500 with runs of 256,
// us: radix passes 1525, 16 wavefronts 1589, one 1189).
static int rank_order(gh_ctx* c, OrderBufs& o, const double* d_pos, int64_t n, int64_t n_pad,
                      int run, const int* seg, const int64_t* start, const int64_t* count,
                      int64_t most, hipStream_t s)
{
    const dim3 runs((unsigned)(n_pad / run)), blocks((unsigned)(n_pad / 64));
    u32 *keys = o.keys[0].as<u32>(), *from = o.keys[1].as<u32>();
    u32* const perm = o.kept ? o.kept : o.idx[0].as<u32>();
    const bool single = most <= run;
#define GH_MERGE(RUN, WAVES)                                                                   \
    hipLaunchKernelGGL((k_run_merge<RUN, WAVES, 1, u32>), blocks, dim3(64 * WAVES), 0, s, keys, \
                       from, n, seg, start, count, (u32*)nullptr, perm)
#define GH_RANK(RUN)                                                                           \
    case RUN:                                                                                  \
        hipLaunchKernelGGL(k_rank_runs<RUN>, runs, dim3(kRunThreads), 0, s, d_pos, n, seg,     \
                           start, count, keys, from, perm, o.nflag.as<int>(), single);         \
        GH_TRY(check_launch(c, "k_rank_runs"));                                                \
        if (single)                                                                            \
            break;                                                                             \
        else if (most <= 1024)                                                                 \
            GH_MERGE(RUN, 1);                                                                  \
        else if (most <= 4096)                                                                 \
            GH_MERGE(RUN, 4);                                                                  \
        else                                                                                   \
            GH_MERGE(RUN, 16);                                                                 \
        break;
    switch (run) {
        GH_RANK(256)
        GH_RANK(512)
        GH_RANK(1024)
    default: return fail(c, GH_EARG, "internal: runs of %d keys", run);
    }
#undef GH_RANK
#undef GH_MERGE
    o.sel = 0;
    return check_launch(c, "k_run_merge");
}

__global__ __launch_bounds__(kBlock) void k_copy_order(const u32* __restrict__ a,
                                                       u32* __restrict__ b, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = a[i];
}

// Every run forms the box of all its segment's points, and every 64 points search all its runs,
// so the work grows as n^2.  Where this is the faster form, of n places in segments of at most
// `most` points: a force of 65536 particles took 1058 us with it and 1080 with the radix passes,
// of 98304 2083 and 2089, of 131072 3158 and 3135; a step of 4 simulations of 32768 1.11 ms and
// 1.22, of 32 of 16384 2.19 and 2.20, of 128 of 16384 7.84 and 7.75.  With the passes and with it,
// four steps of many small ones: 20000 of 20 4.07 and 2.08 ms, 4096 of 250 1.23 and 0.86, 1000
// of 1024 2.07 and 1.70, 300 of 2500 2.92 and 2.47.
static bool rank_form(const gh_ctx* c, int64_t n, int64_t most)
{
    return c->tune[GH_TUNE_SORT_DIRECT] >= 0 && n * most <= (int64_t)1 << 33;
}

int spatial_order(gh_ctx* c, OrderBufs& o, const double* d_pos, int64_t n, hipStream_t s)
{
    o.sorted = nullptr;
    if (n <= 0) return 0;
    for (int k = 0; k < 2; k++) {
        // (512: rank_order pads its 32-bit keys to whole runs)
        GH_TRY(ensure(c, o.keys[k], sizeof(u64) * (size_t)std::max(n, (int64_t)kRunThreads / 2)));
        GH_TRY(ensure(c, o.idx[k], sizeof(u32) * (size_t)n));
    }
    GH_TRY(ensure(c, o.box, sizeof(double) * 8));
    GH_TRY(ensure(c, o.nflag, 256));
    if (rank_form(c, n, n)) {
        const int64_t n_pad = (int64_t)blocks_for(n, kRunThreads) * kRunThreads;
        GH_TRY(rank_order(c, o, d_pos, n, n_pad, kRunThreads, nullptr, nullptr, nullptr, n, s));
        o.sorted = d_pos;
        o.sorted_n = n;
        return 0;
    }
    GH_TRY(bbox_dev(c, d_pos, n, 0.0, o.boxpart, o.box.as<double>(), s));
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, d_pos, n,
                       o.box.as<double>(), o.keys[0].as<u64>(), o.idx[0].as<u32>(),
                       o.nflag.as<int>());
    GH_TRY(check_launch(c, "k_morton"));
    // bits 31..62 (the top 10 2/3 levels): four 8-bit passes.  Deeper keys change the
    // blocks' compactness, and so the forces' rounding, by little (Plummer sphere,
    // 65536 particles, 1024-particle blocks: median relative error 3.0e-8 with 10 levels,
    // 3.4e-8 with 16) and cost two more passes.
    GH_TRY(radix_sort(c, o.keys, o.idx, o.hist, n, 1, kKeyShift, s, &o.sel, 63));
    if (o.kept) {
        hipLaunchKernelGGL(k_copy_order, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s,
                           o.idx[o.sel].as<u32>(), o.kept, n);
        GH_TRY(check_launch(c, "k_copy_order"));
    }
    o.sorted = d_pos;
    o.sorted_n = n;
    return 0;
}

// Root box (as k_bbox_final with eps = 0) of each segment's real points, one workgroup
// per segment: box[4 g ..] = centre, size.
__global__ __launch_bounds__(kBlock) void k_seg_box(const double* __restrict__ pos,
                                                    const int64_t* __restrict__ start,
                                                    const int64_t* __restrict__ count,
                                                    double* __restrict__ box)
{
    __shared__ double smin[3][kBlock], smax[3][kBlock];
    const int64_t a = start[blockIdx.x], n = count[blockIdx.x];
    double mn[3], mx[3];
    for (int k = 0; k < 3; k++) mn[k] = mx[k] = pos[3 * a + k];
    for (int64_t i = threadIdx.x; i < n; i += kBlock)
        for (int k = 0; k < 3; k++) {
            const double q = pos[3 * (a + i) + k];
            mn[k] = q < mn[k] ? q : mn[k];
            mx[k] = q > mx[k] ? q : mx[k];
        }
    for (int k = 0; k < 3; k++) {
        smin[k][threadIdx.x] = mn[k];
        smax[k][threadIdx.x] = mx[k];
    }
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int k = 0; k < 3; k++) {
                if (smin[k][threadIdx.x + w] < smin[k][threadIdx.x])
                    smin[k][threadIdx.x] = smin[k][threadIdx.x + w];
                if (smax[k][threadIdx.x + w] > smax[k][threadIdx.x])
                    smax[k][threadIdx.x] = smax[k][threadIdx.x + w];
            }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    double bs = smax[0][0] - smin[0][0];
    for (int k = 1; k < 3; k++)
        if ((smax[k][0] - smin[k][0]) > bs) bs = smax[k][0] - smin[k][0];
    for (int k = 0; k < 3; k++) box[4 * blockIdx.x + k] = 0.5 * (smin[k][0] + smax[k][0]);
    box[4 * blockIdx.x + 3] = bs;
}

// Keys of the padded, segmented layout: position p of block b belongs to segment
// seg[b]; its key is (segment << 32) | the key bits spatial_order sorts by (in the
// segment's box), and padding positions take their segment's largest key, so that a
// stable sort keeps every segment in place, in the order a single sort of it gives,
// with its padding last.
__global__ __launch_bounds__(kBlock) void k_morton_seg(const double* __restrict__ pos,
                                                       int64_t n_pad, int blk,
                                                       const int* __restrict__ seg,
                                                       const int64_t* __restrict__ start,
                                                       const int64_t* __restrict__ count,
                                                       const double* __restrict__ box,
                                                       u64* __restrict__ keys,
                                                       u32* __restrict__ idx,
                                                       int* __restrict__ nflag)
{
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p == 0) *nflag = 0;
    if (p >= n_pad) return;
    const int g = seg[p / blk];
    u64 k = ((u64)1 << (63 - kKeyShift)) - 1;
    if (p - start[g] < count[g]) {
        const double* bx = box + 4 * g;
        const double size = bx[3];
        const double scale = size > 0.0 ? 2097152.0 / size : 0.0;
        u64 m = 0;
        for (int a = 0; a < 3; a++)
            m |= spread3(quantize(pos[3 * p + a], bx[a] - 0.5 * size, scale)) << a;
        k = m >> kKeyShift;
    }
    keys[p] = ((u64)g << (63 - kKeyShift)) | k;
    idx[p] = (u32)p;
}

int spatial_order_seg(gh_ctx* c, OrderBufs& o, const double* d_pos, int64_t n_pad, int blk,
                      int nseg, const int* seg, const int64_t* start, const int64_t* count,
                      int64_t most, hipStream_t s)
{
    o.sorted = nullptr;
    if (n_pad <= 0) return 0;
    for (int k = 0; k < 2; k++) {
        GH_TRY(ensure(c, o.keys[k], sizeof(u64) * (size_t)n_pad));
        GH_TRY(ensure(c, o.idx[k], sizeof(u32) * (size_t)n_pad));
    }
    GH_TRY(ensure(c, o.box, sizeof(double) * 4 * (size_t)nseg));
    GH_TRY(ensure(c, o.nflag, 256));
    GH_TRY(ensure(c, o.hist, sizeof(u32) * 256 * (size_t)(blocks_for(n_pad, kRsChunk) + 1)));
    if (rank_form(c, n_pad, most))
        return rank_order(c, o, d_pos, 0, n_pad, blk, seg, start, count, most, s);
    hipLaunchKernelGGL(k_seg_box, dim3((unsigned)nseg), dim3(kBlock), 0, s, d_pos, start, count,
                       o.box.as<double>());
    GH_TRY(check_launch(c, "k_seg_box"));
    hipLaunchKernelGGL(k_morton_seg, dim3(blocks_for(n_pad, kBlock)), dim3(kBlock), 0, s, d_pos,
                       n_pad, blk, seg, start, count, o.box.as<double>(), o.keys[0].as<u64>(),
                       o.idx[0].as<u32>(), o.nflag.as<int>());
    GH_TRY(check_launch(c, "k_morton_seg"));
    int bits = 63 - kKeyShift;
    while (bits < 64 && ((int64_t)1 << (bits - (63 - kKeyShift))) < nseg) bits++;
    return radix_sort(c, o.keys, o.idx, o.hist, n_pad, 1, 0, s, &o.sel, bits);
}

__device__ __forceinline__ int exponent_of(double x)
{
    // binary exponent of |x| (x = 0 and subnormals give -1023)
    return (int)((__double_as_longlong(x) >> 52) & 0x7ff) - 1023;
}

__device__ __forceinline__ double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ long long wave_sum(long long v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// One workgroup per group of G consecutive sorted points.  Origin: the group's point at
// offset min(G/2, count-1) (a point of the group's majority part, so that a group with a
// few strays keeps a useful frame).  Writes loc / s64 for the group's G slots (padding:
// massless at the origin), frame = (origin, R), the compactness flag, and the FP32 mass all
// points of the group share (NaN where they do not, or where the group is padded).
template <int G>
__global__ __launch_bounds__(kBlock) void k_frames(const double* __restrict__ pos,
                                                   const double* __restrict__ mass,
                                                   const u32* __restrict__ perm, int64_t n,
                                                   const int* __restrict__ valid,
                                                   float4* __restrict__ loc,
                                                   double4* __restrict__ s64,
                                                   double4* __restrict__ frame,
                                                   int* __restrict__ flag,
                                                   int* __restrict__ nflag,
                                                   float* __restrict__ umass,
                                                   int* __restrict__ used)
{
    __shared__ float sLo[kBlock / 64], sHi[kBlock / 64];
    __shared__ double sR[kBlock / 64];
    __shared__ long long sE[kBlock / 64], sC[kBlock / 64];
    const int64_t p0 = (int64_t)blockIdx.x * G;
    int cnt = valid ? valid[blockIdx.x] : (int)(n - p0 < G ? n - p0 : G);
    if (cnt < 0) cnt = 0;
    double ox = 0.0, oy = 0.0, oz = 0.0;
    if (cnt > 0) {
        const int64_t pm = p0 + (G / 2 < cnt - 1 ? G / 2 : cnt - 1);
        const int64_t jm = perm ? (int64_t)perm[pm] : pm;
        ox = pos[3 * jm];
        oy = pos[3 * jm + 1];
        oz = pos[3 * jm + 2];
    }
    double R = 0.0;
    long long esum = 0, gcnt = 0;
    float mlo = HUGE_VALF, mhi = -HUGE_VALF;
    bool same = cnt == G;  // no padding, and no mass that is not a number
    for (int k = threadIdx.x; k < G; k += kBlock) {
        const int64_t p = p0 + k;
        if (k < cnt) {
            const int64_t j = perm ? (int64_t)perm[p] : p;
            const double x = pos[3 * j], y = pos[3 * j + 1], z = pos[3 * j + 2];
            const double m = mass ? mass[j] : 0.0;
            const double dx = x - ox, dy = y - oy, dz = z - oz;
            R = fmax(R, fmax(fabs(dx), fmax(fabs(dy), fabs(dz))));
            loc[p] = make_float4((float)dx, (float)dy, (float)dz, (float)m);
            mlo = fminf(mlo, (float)m);
            mhi = fmaxf(mhi, (float)m);
            same = same && m == m;
            if (s64) s64[p] = make_double4(x, y, z, m);
            if (k + 1 < cnt) {
                const int64_t j2 = perm ? (int64_t)perm[p + 1] : p + 1;
                const double g = fmax(fabs(pos[3 * j2] - x),
                                      fmax(fabs(pos[3 * j2 + 1] - y), fabs(pos[3 * j2 + 2] - z)));
                esum += exponent_of(g);
                gcnt += 1;
            }
        } else {
            loc[p] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (s64) s64[p] = make_double4(ox, oy, oz, 0.0);
        }
    }
    R = wave_max(R);
    esum = wave_sum(esum);
    gcnt = wave_sum(gcnt);
    for (int o = 32; o > 0; o >>= 1) {
        mlo = fminf(mlo, __shfl_xor(mlo, o));
        mhi = fmaxf(mhi, __shfl_xor(mhi, o));
    }
    if (__ballot(!same) != 0) mlo = -HUGE_VALF;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        sR[wave] = R;
        sE[wave] = esum;
        sC[wave] = gcnt;
        sLo[wave] = mlo;
        sHi[wave] = mhi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; w++) {
            R = fmax(R, sR[w]);
            esum += sE[w];
            gcnt += sC[w];
            mlo = fminf(mlo, sLo[w]);
            mhi = fmaxf(mhi, sHi[w]);
        }
        used[blockIdx.x] = cnt;
        umass[blockIdx.x] = mlo == mhi ? mlo : __builtin_nanf("");
        // log2 R - mean log2 gap > kFrameLog2, in integer exponents
        const long long eR = exponent_of(R);
        const bool loose = gcnt > 0 && eR * gcnt - esum > (long long)kFrameLog2 * gcnt;
        frame[blockIdx.x] = make_double4(ox, oy, oz, R);
        flag[blockIdx.x] = loose ? 1 : 0;
        if (loose) atomicAdd(nflag, 1);
    }
}

int gather_frames(gh_ctx* c, OrderBufs& o, const double* d_pos, const double* d_mass,
                  const u32* perm, int64_t n, int64_t n_pad, int group, const int* valid,
                  bool want_s64, hipStream_t s)
{
    if (n_pad <= 0) return 0;
    if (n_pad % group != 0) return fail(c, GH_EARG, "internal: group padding");
    const int64_t ng = n_pad / group;
    GH_TRY(ensure(c, o.loc, sizeof(float4) * (size_t)n_pad));
    if (want_s64) GH_TRY(ensure(c, o.s64, sizeof(double4) * (size_t)n_pad));
    GH_TRY(ensure(c, o.frame, sizeof(double4) * (size_t)ng));
    GH_TRY(ensure(c, o.flag, sizeof(int) * (size_t)ng));
    GH_TRY(ensure(c, o.nflag, 256));
    GH_TRY(ensure(c, o.umass, sizeof(float) * (size_t)ng));
    GH_TRY(ensure(c, o.used, sizeof(int) * (size_t)ng));
    double4* s64 = want_s64 ? o.s64.as<double4>() : nullptr;
#define GH_FRAMES(GG)                                                                       \
    hipLaunchKernelGGL(k_frames<GG>, dim3((unsigned)ng), dim3(kBlock), 0, s, d_pos, d_mass,  \
                       perm, n, valid, o.loc.as<float4>(), s64, o.frame.as<double4>(),       \
                       o.flag.as<int>(), o.nflag.as<int>(), o.umass.as<float>(),              \
                       o.used.as<int>())
    switch (group) {
        case 256: GH_FRAMES(256); break;
        case 512: GH_FRAMES(512); break;
        case 1024: GH_FRAMES(1024); break;
        default: return fail(c, GH_EARG, "internal: group size %d", group);
    }
#undef GH_FRAMES
    return check_launch(c, "k_frames");
}

}  // namespace gh
