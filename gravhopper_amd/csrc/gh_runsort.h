// Sorts of few keys in two launches, shared by the spatial order (gh_frames.hip) and the tree
// build (gh_tree.hip).  A workgroup forms the keys of a run of up to 1024 points and sorts them
// (sort_run); then a point's place in the order is its place in its run plus what a binary
// search finds in every other run (k_run_merge).  A radix sort of so few keys is bound by the
// latency of its passes; this is a chain of some 60 dependent LDS reads.  Ties go by index, as
// in a stable sort.
#pragma once

#include "gh_internal.h"

namespace gh {

constexpr int kRunThreads = 1024;

// x of another lane, by DPP control CTRL in the rows of ROWS; other rows keep their own.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_f64(double x)
{
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false));
}

// Extents over a workgroup of kRunThreads threads, from each thread's own, in every thread.
// Minima and maxima are exact in any order.
__device__ __forceinline__ void run_extents(double (&mn)[3], double (&mx)[3])
{
    constexpr int kWaves = kRunThreads / 64;
    static_assert(kWaves == 16, "one value per lane of a row");
    __shared__ double ext[6][kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto fold = [&](auto moved) {
        for (int a = 0; a < 3; a++) {
            const double lo = moved(mn[a]), hi = moved(mx[a]);
            if (lo < mn[a]) mn[a] = lo;
            if (hi > mx[a]) mx[a] = hi;
        }
    };
    auto over_row = [&] {  // every lane of a row of 16 ends with the row's extremes
        fold([](double x) { return dpp_f64<0x128>(x); });
        fold([](double x) { return dpp_f64<0x124>(x); });
        fold([](double x) { return dpp_f64<0x122>(x); });
        fold([](double x) { return dpp_f64<0x121>(x); });
    };
    over_row();
    fold([](double x) { return dpp_f64<0x142, 0xa>(x); });  // rows 0 and 2 into 1 and 3
    fold([](double x) { return dpp_f64<0x143, 0xc>(x); });  // row 1 into 2 and 3
    if (lane == 63)
        for (int a = 0; a < 3; a++) {
            ext[a][wave] = mn[a];
            ext[3 + a][wave] = mx[a];
        }
    __syncthreads();
    for (int a = 0; a < 3; a++) {
        mn[a] = ext[a][lane % kWaves];
        mx[a] = ext[3 + a][lane % kWaves];
    }
    over_row();
}

// How many of the N sorted keys from k on come before key: those smaller, and with `ties` those
// equal.
template <int N, class K>
__device__ __forceinline__ int count_before(const K* k, K key, bool ties)
{
    int at = 0;
#pragma unroll
    for (int h = N / 2; h > 0; h /= 2) {
        const K q = k[at + h - 1];
        at += q < key || (ties && q == key) ? h : 0;
    }
    const K q = k[at];
    return at + (q < key || (ties && q == key) ? 1 : 0);
}

// A point's place in the merger of its run of N keys, its place there `at`, with the other
// three of its group of four (run r of the group; ties: earlier runs first).
template <int N, class K>
__device__ __forceinline__ int place_in_four(const K* group, int r, int at, K key)
{
    int place = at;
#pragma unroll
    for (int o = 1; o < 4; o++) {
        const int other = r ^ o;
        place += count_before<N>(group + other * N, key, other < r);
    }
    return place;
}

__device__ __forceinline__ u32 lane_value(u32 x, int lane)
{
    return (u32)__builtin_amdgcn_readlane((int)x, lane);
}
__device__ __forceinline__ u64 lane_value(u64 x, int lane)
{
    return (u64)lane_value((u32)(x >> 32), lane) << 32 | lane_value((u32)x, lane);
}

// Sorts the run held by threads 0 .. RUN - 1 of the workgroup (act), one (key, idx) each in
// order of idx; on return thread t holds another entry of it and the entry's place.  All
// threads of the workgroup call.  A wavefront sorts 64 by counting, then four sorted lists
// become one, twice.
template <int RUN, class K>
__device__ __forceinline__ int sort_run(K& key, u32& idx, bool act)
{
    static_assert(RUN == 256 || RUN == 512 || RUN == 1024, "lists merged");
    __shared__ K sk[2][RUN];
    __shared__ u32 si[2][RUN];
    const int t = threadIdx.x, lane = t & 63;
    int at = 0;
    if (act) {
#pragma unroll
        for (int q = 0; q < 64; q++) {
            const K k = lane_value(key, q);
            at += k < key || (k == key && q < lane) ? 1 : 0;
        }
        sk[0][t - lane + at] = key;
        si[0][t - lane + at] = idx;
    }
    __syncthreads();
    if (act) {
        key = sk[0][t];
        idx = si[0][t];
        at = place_in_four<64>(&sk[0][t & ~255], (t >> 6) & 3, lane, key);
    }
    if constexpr (RUN > 256) {
        if (act) {
            sk[1][(t & ~255) + at] = key;
            si[1][(t & ~255) + at] = idx;
        }
        __syncthreads();
        if (act) {
            key = sk[1][t];
            idx = si[1][t];
            if constexpr (RUN == 512)
                at = (t & 255) + count_before<256>(&sk[1][t < 256 ? 256 : 0], key, t >= 256);
            else
                at = place_in_four<256>(sk[1], t >> 8, t & 255, key);
        }
    }
    return at;
}

// The order from the sorted runs of RUN keys: 64 E places of one run per workgroup, E to a
// lane.  A wavefront takes 1024 keys at a time into its part of LDS and searches each run of
// them.  Segments: with seg_start / seg_count, segment g of a padded layout is sorted on its
// own (run b belongs to segment seg[b]), its padding left in place behind its points; without,
// there are n_all points.  Runs are filled up with keys that no point's exceeds.  keys_out may
// be null.
template <int RUN, int WAVES, int E, class K>
__global__ __launch_bounds__(WAVES * 64) void k_run_merge(
    const K* __restrict__ keys, const u32* __restrict__ from, int64_t n_all,
    const int* __restrict__ seg, const int64_t* __restrict__ seg_start,
    const int64_t* __restrict__ seg_count, K* __restrict__ keys_out, u32* __restrict__ perm)
{
    constexpr int kPart = 1024, kRuns = kPart / RUN, kVec = 16 / sizeof(K);
    static_assert(RUN % (64 * E) == 0, "a workgroup's places are of one run");
    __shared__ alignas(16) K part[WAVES][kPart];
    __shared__ int below[WAVES][E][64];
    typedef K vec __attribute__((ext_vector_type(kVec)));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t base = (int64_t)blockIdx.x * 64 * E;
    const int g = seg ? seg[base / RUN] : 0;
    const int64_t first = seg ? seg_start[g] : 0;
    const int64_t n = seg ? seg_count[g] : n_all;
    const int64_t end = (n + RUN - 1) / RUN * RUN;   // keys of the segment's runs
    const int64_t own = (base - first) / RUN;        // this run in its segment
    K key[E];
    int count[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        key[e] = keys[base + 64 * e + lane];
        count[e] = 0;
    }
    for (int64_t k0 = (int64_t)wave * kPart; k0 < end; k0 += (int64_t)WAVES * kPart) {
        vec* mine = (vec*)part[wave];
#pragma unroll
        for (int q = 0; q < kPart / 64 / kVec; q++) {
            const int64_t k = k0 + kVec * (64 * q + lane);
            mine[64 * q + lane] = k < end ? *(const vec*)(keys + first + k) : (vec)(~(K)0);
        }
        __builtin_amdgcn_wave_barrier();  // LDS serves a wavefront in order
#pragma unroll 4
        for (int r = 0; r < kRuns; r++) {
            const int64_t run = k0 / RUN + r;
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int c = count_before<RUN>(&part[wave][r * RUN], key[e], run < own);
                count[e] += run == own ? 0 : c;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int e = 0; e < E; e++) below[wave][e][lane] = count[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) {
        if (wave != e) continue;
        const int64_t place = base + 64 * e + lane;
        const u32 idx = from[place];
        int64_t at = place - own * RUN;  // first + the place in the run
        for (int w = 0; w < WAVES; w++) at += below[w][e][lane];
        if ((int64_t)idx - first < n) {
            perm[at] = idx;
            if (keys_out) keys_out[at] = key[e];
        }
    }
}

}  // namespace gh
