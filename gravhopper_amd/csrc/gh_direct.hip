// Direct-summation kernels for gfx950.
//
//  k_direct_f64_relay, k_direct_f64_ring  IEEE FP64, the operation order of
//                 gravhopper/_jbgrav.c:140-193 (self) and :299-353 (targets) with every
//                 sum formed in ascending source order, so the result is bit-identical to
//                 the reference.  Built with -ffp-contract=off; the pair factor comes from
//                 gh_pairf64.h, correctly rounded like the compiler's division and square
//                 root.  The terms are computed by many wavefronts and added in order by
//                 one: a wavefront of its own (relay, few targets) or each in its turn
//                 (ring).  k_direct_f64_few, the fields of few sources: the same sums, one
//                 target per lane.
//  k_direct_f32   FP32 pair forces with v_rsq_f32, IPT targets per lane, 256-source
//                 tiles staged in LDS as float4 (x, y, z, m) and read as wave-wide
//                 broadcasts, FP32 sums per tile and an FP32 two-sum (hi, lo) across
//                 tiles; FP64 out.  Sources may be split over grid.y when there are too
//                 few targets to fill 256 CUs; the splits are added in split order.
//  k_direct_sym_f32  the self field with each unordered pair computed once.
//  Both FP32 kernels form coordinates only relative to FP64 origins of groups of
//  spatially sorted particles (gh_frames.hip), so their accuracy does not depend on
//  where the system sits; non-compact groups take double-single forms.
#include <cmath>
#include <type_traits>

#include "gh_internal.h"
#include "gh_pairf64.h"
#include "gh_turn.h"

namespace gh {

int64_t pad_to(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

// ------------------------------------------------------------------------------
// FP64, reference operation order
// ------------------------------------------------------------------------------
// inv[u] = 1/d[u]/sqrt(d[u]) as the reference rounds it (:167; :327-331 with 0 for d = 0
// when !SELF).  One range check covers the U values: a lane with any value outside
// pair_factor's range takes the plain expressions for all of its own.
template <bool SELF, int U>
__device__ __forceinline__ void pair_factors(const double (&d)[U], double (&inv)[U])
{
    u32 hi = 0u, lo = 0u;
#pragma unroll
    for (int u = 0; u < U; u++) {
        hi = max(hi, (u32)__double2hiint(d[u]) - kPairLoHi);
        lo = max(lo, (u32)__double2loint(d[u]));
        inv[u] = pair_factor(d[u], __builtin_amdgcn_rsq(d[u]));
    }
    if (__builtin_expect(hi >= kPairSpan || lo == kPairLowOnes, 0)) {
#pragma unroll
        for (int u = 0; u < U; u++)
            inv[u] = (!SELF && d[u] == 0.0) ? 0.0 : 1.0 / d[u] / sqrt(d[u]);
    }
}

// A workgroup barrier that orders LDS accesses only: loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The same sums with the terms and the additions on different wavefronts.  A workgroup
// takes T = P K targets: wavefronts 0 .. P - 1 compute the terms of chunks of 128 sources
// (lane l sources 2l and 2l + 1 of the chunk, K targets each) into LDS, and wavefront P adds
// them, lane L < 3 T holding one sum (a target's x, y or z) and adding its 128 terms in
// source order.  While a chunk is added the next one's terms are computed (two LDS buffers,
// one barrier per chunk), so a chunk costs the longer of the two, not both: the ordered
// chain of additions (dependent FP64 adds, 9.8 cycles each) is the floor at few targets,
// the FP64 issue rate of the terms at many.  The adding wavefront gets priority on its
// SIMD, since the others wait for it.
template <bool SELF, int P, int K>
__global__ __launch_bounds__((P + 1) * 64) void k_direct_f64_relay(
    const double* __restrict__ pos, const double* __restrict__ mass, int64_t np,
    const double* __restrict__ tgt, int64_t from, int64_t nt, double eps2,
    double* __restrict__ acc, StepUpdate up)
{
    constexpr int T = P * K, NS = 3 * T, CH = 128;
    static_assert(NS <= 64, "one lane per sum");
    // terms[b][l][L]: terms 2l and 2l + 1 of sum L in chunk buffer b; an odd row length
    // spreads the rows over the LDS banks
    constexpr int ROW = NS | 1;
    __shared__ double2 terms[2][CH / 2][ROW];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t i0 = from + (int64_t)blockIdx.x * T;
    // chunks are taken in pairs; one past the last adds zeros
    const int64_t chunks = (np + 2 * CH - 1) / (2 * CH) * 2;
    if (wave == P) {
        __builtin_amdgcn_s_setprio(3);
        const int L = lane < NS ? lane : NS - 1;
        // a chunk's terms are read Q rows at a time into one of two sets of registers while
        // the rows before are added from the other
        constexpr int Q = 8;
        double2 v[2][Q];
        double f = 0.0;
#pragma unroll
        for (int k = 0; k < Q; k++) v[1][k] = make_double2(0.0, 0.0);
        for (int64_t c = 0; c < chunks; c++) {
            lds_barrier();  // chunk c is in buffer c & 1
            const double2* t = &terms[c & 1][0][L];
#pragma unroll
            for (int q = 0; q < CH / 2 / Q; q++) {
#pragma unroll
                for (int k = 0; k < Q; k++) v[q & 1][k] = t[(q * Q + k) * ROW];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < Q; k++) {
                    f = f + v[(q + 1) & 1][k].x;
                    f = f + v[(q + 1) & 1][k].y;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int k = 0; k < Q; k++) {
            f = f + v[1][k].x;
            f = f + v[1][k].y;
        }
        if (lane < NS && i0 + lane / 3 < nt) {
            if (SELF && up.v)
                update_one(up, 3 * i0 + lane, f);
            else
                acc[3 * i0 + lane] = f;
        }
        return;
    }
    double xt[K], yt[K], zt[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        // a target past nt takes the last target's position; its sums are not stored
        const int64_t i = i0 + wave * K + k < nt ? i0 + wave * K + k : nt - 1;
        xt[k] = tgt[3 * i];
        yt[k] = tgt[3 * i + 1];
        zt[k] = tgt[3 * i + 2];
    }
    // sources are read in place from the (n,3) positions and the masses, one chunk ahead
    // (in two sets of registers, so that no copy waits for the loads)
    struct Source {
        double x[2], y[2], z[2], w[2];
    };
    auto load = [&](int64_t base) {
        const int64_t at = min(base, np - 1);
        const int last = (int)min(np - 1 - at, (int64_t)(CH - 1));
        const double* p = pos + 3 * at;
        Source s;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int l = min(2 * lane + h, last);
            s.x[h] = p[3 * l];
            s.y[h] = p[3 * l + 1];
            s.z[h] = p[3 * l + 2];
            s.w[h] = mass[at + l];
        }
        return s;
    };
    auto chunk = [&](int64_t base, const Source& s, int buf) {
        double dx[2 * K], dy[2 * K], dz[2 * K], d[2 * K], inv[2 * K];
#pragma unroll
        for (int k = 0; k < 2 * K; k++) {
            dx[k] = s.x[k & 1] - xt[k >> 1];
            dy[k] = s.y[k & 1] - yt[k >> 1];
            dz[k] = s.z[k & 1] - zt[k >> 1];
            double d2 = dx[k] * dx[k];
            d2 = d2 + dy[k] * dy[k];
            d2 = d2 + dz[k] * dz[k];
            d[k] = d2 + eps2;
        }
        pair_factors<SELF, 2 * K>(d, inv);
        double2* o = &terms[buf][lane][3 * K * wave];
        // the chunk holding the workgroup's own particles, and chunks past np
        const bool masked = base + CH > np || (SELF && base < i0 + T && base + CH > i0);
#pragma unroll
        for (int k = 0; k < K; k++) {
            double c[3][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                c[0][h] = s.w[h] * dx[2 * k + h] * inv[2 * k + h];
                c[1][h] = s.w[h] * dy[2 * k + h] * inv[2 * k + h];
                c[2][h] = s.w[h] * dz[2 * k + h] * inv[2 * k + h];
            }
            if (masked) {
                // +0.0 for the target itself and for sources past np: adding it leaves a
                // sum that starts at +0.0 unchanged
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int64_t j = base + 2 * lane + h;
                    const bool use = j < np && !(SELF && j == i0 + wave * K + k);
#pragma unroll
                    for (int a = 0; a < 3; a++) c[a][h] = use ? c[a][h] : 0.0;
                }
            }
#pragma unroll
            for (int a = 0; a < 3; a++) o[3 * k + a] = make_double2(c[a][0], c[a][1]);
        }
        lds_barrier();
    };
    Source a = load(0);
    for (int64_t c = 0; c < chunks; c += 2) {
        const Source b = load(CH * (c + 1));
        chunk(CH * c, a, 0);
        a = load(CH * (c + 2));
        chunk(CH * (c + 1), b, 1);
    }
}

// The value of lane l - 32 in lanes 32 .. 63 (lanes 0 .. 31 keep theirs).
__device__ __forceinline__ double from_lower_half(double v)
{
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double(hi[0], lo[0]);
}

// The sources of each target spread over the wavefronts of a workgroup in turns.  A
// workgroup takes 64 / H targets (H = 1 or 2 lanes per target); per turn a wavefront takes
// the next H C sources, C per lane, computes their terms in registers, waits until the
// sources before are added, adds its own in source order to the sums in LDS and passes the
// turn on.  So every sum is formed in the reference's order while W wavefronts share its
// arithmetic: W times as many wavefronts as one lane per target gives, which fills the
// chip and evens out its last round.  The sources of a wavefront's next 64 / (H C) turns
// are staged in LDS, loaded that many turns ahead.
template <bool SELF, int W, int C, int H>
__global__ __launch_bounds__(W * 64) void k_direct_f64_ring(const double* __restrict__ pos,
                                                            const double* __restrict__ mass,
                                                            int64_t np,
                                                            const double* __restrict__ tgt,
                                                            int64_t from, int64_t nt,
                                                            double eps2,
                                                            double* __restrict__ acc)
{
    constexpr int T = 64 / H, G = H * C, TURNS = 64 / G;
    __shared__ double sums[3][T];
    __shared__ int turn;
    __shared__ double4 stage[W][2][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int t = lane % T, h = lane / T;
    const int64_t i0 = from + (int64_t)blockIdx.x * T;
    const int64_t i = i0 + t < nt ? i0 + t : nt - 1;  // past nt: computed, not stored
    const double xi = tgt[3 * i], yi = tgt[3 * i + 1], zi = tgt[3 * i + 2];
    if (threadIdx.x < T) sums[0][t] = sums[1][t] = sums[2][t] = 0.0;
    if (threadIdx.x == 0) turn = 0;
    __syncthreads();
    // group g (G sources from g G on) is wavefront (g mod W)'s; its turns come in blocks of
    // TURNS, lane l loading source l % G of turn l / G
    const int groups = (int)((np + G - 1) / G);
    auto load = [&](int g) {
        const int64_t at = ((int64_t)g + (int64_t)(lane / G) * W) * G + lane % G;
        const int64_t j = at < np ? at : np - 1;
        return make_double4(pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], mass[j]);
    };
    double4 next = load(wave);
    int buf = 0;
    for (int g0 = wave; g0 < groups; g0 += W * TURNS, buf ^= 1) {
        stage[wave][buf][lane] = next;
        next = load(g0 + W * TURNS);
        __builtin_amdgcn_wave_barrier();
        for (int k = 0; k < TURNS; k++) {
            const int g = g0 + k * W;
            if (g >= groups) break;
            const int64_t base = (int64_t)g * G;
            const double4* s = &stage[wave][buf][k * G + h * C];
            double dx[C], dy[C], dz[C];
            // four sources at a time keep the FP64 pipe full; more only cost registers
#pragma unroll
            for (int u0 = 0; u0 < C; u0 += 4) {
                double w[4], d[4], inv[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const double4 q = s[u0 + u];
                    dx[u0 + u] = q.x - xi;
                    dy[u0 + u] = q.y - yi;
                    dz[u0 + u] = q.z - zi;
                    w[u] = q.w;
                    double d2 = dx[u0 + u] * dx[u0 + u];
                    d2 = d2 + dy[u0 + u] * dy[u0 + u];
                    d2 = d2 + dz[u0 + u] * dz[u0 + u];
                    d[u] = d2 + eps2;
                }
                pair_factors<SELF, 4>(d, inv);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    dx[u0 + u] = w[u] * dx[u0 + u] * inv[u];
                    dy[u0 + u] = w[u] * dy[u0 + u] * inv[u];
                    dz[u0 + u] = w[u] * dz[u0 + u] * inv[u];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (base + G > np || (SELF && base < i0 + T && base + G > i0)) {
                // +0.0 for the target itself and for sources past np: adding it leaves a
                // sum that starts at +0.0 unchanged
#pragma unroll
                for (int u = 0; u < C; u++) {
                    const int64_t j = base + h * C + u;
                    const bool use = j < np && !(SELF && j == i0 + t);
                    dx[u] = use ? dx[u] : 0.0;
                    dy[u] = use ? dy[u] : 0.0;
                    dz[u] = use ? dz[u] : 0.0;
                }
            }
            // every wavefront of the workgroup is resident and passes each of its turns on,
            // so this ends
            while (!turn_is(&turn, g)) __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_s_setprio(3);
            double f0 = sums[0][t], f1 = sums[1][t], f2 = sums[2][t];
#pragma unroll
            for (int p = 0; p < H; p++) {
                if (p > 0) {
                    f0 = from_lower_half(f0);
                    f1 = from_lower_half(f1);
                    f2 = from_lower_half(f2);
                }
#pragma unroll
                for (int u = 0; u < C; u++) {
                    f0 = f0 + dx[u];
                    f1 = f1 + dy[u];
                    f2 = f2 + dz[u];
                }
            }
            if (h == H - 1) {
                sums[0][t] = f0;
                sums[1][t] = f1;
                sums[2][t] = f2;
            }
            turn_pass(&turn, g + 1);
            __builtin_amdgcn_s_setprio(0);
        }
    }
    __syncthreads();
    if (threadIdx.x < T && i0 + t < nt) {
        acc[3 * i] = sums[0][t];
        acc[3 * i + 1] = sums[1][t];
        acc[3 * i + 2] = sums[2][t];
    }
}

// The field of few sources: one target per lane, the sources one after the other, whose records
// are the same for all and arrive through scalar loads, and four factors at a time.  Nothing is
// shared, so a workgroup is as long as its sums: bound by HBM for up to 4 sources (10^6 targets in
// 12 us, 48 MB), by the FP64 issue rate beyond (50 sources 71 us).
__global__ __launch_bounds__(kBlock) void k_direct_f64_few(const double* __restrict__ pos,
                                                           const double* __restrict__ mass, int np,
                                                           const double* __restrict__ tgt,
                                                           int64_t nt, double eps2,
                                                           double* __restrict__ acc)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= nt) return;
    const double xi = tgt[3 * i], yi = tgt[3 * i + 1], zi = tgt[3 * i + 2];
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;
    auto add = [&](auto count, int j) {
        constexpr int U = decltype(count)::value;
        double dx[U], dy[U], dz[U], d[U], inv[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            dx[u] = pos[3 * (j + u)] - xi;
            dy[u] = pos[3 * (j + u) + 1] - yi;
            dz[u] = pos[3 * (j + u) + 2] - zi;
            double d2 = dx[u] * dx[u];
            d2 = d2 + dy[u] * dy[u];
            d2 = d2 + dz[u] * dz[u];
            d[u] = d2 + eps2;
        }
        pair_factors<false, U>(d, inv);
#pragma unroll
        for (int u = 0; u < U; u++) {
            f0 = f0 + mass[j + u] * dx[u] * inv[u];
            f1 = f1 + mass[j + u] * dy[u] * inv[u];
            f2 = f2 + mass[j + u] * dz[u] * inv[u];
        }
    };
    int j = 0;
    for (; j + 4 <= np; j += 4) add(std::integral_constant<int, 4>(), j);
    for (; j < np; j++) add(std::integral_constant<int, 1>(), j);
    acc[3 * i] = f0;
    acc[3 * i + 1] = f1;
    acc[3 * i + 2] = f2;
}

// Kernel shape for the FP64 sums.  Up to kF64RelayMax targets k_direct_f64_relay: the chain of
// ordered additions is what bounds it, so the fewest wavefronts that keep up with it, and as many
// targets per workgroup as give each CU one workgroup, or two of 6 or 9 where that is as many as
// fit (us for 2100, 3001, 5000 targets of 65536 sources with 12 in six wavefronts 469, 472, 767,
// with 9 418, 636, 968, with 6 445, 455, 767, with 20 696, 699, 704).  Beyond, k_direct_f64_ring:
// the issue rate of the terms bounds it, and the shape decides how evenly the wavefronts fill the
// CUs: two lanes per target (32 targets per workgroup) until 64 targets per workgroup give half of
// the CUs one, eight wavefronts per workgroup until there are two workgroups per CU, and whole
// rounds apart (f64_whole_rounds).  Measured on Plummer spheres, us per evaluation (the best of the
// other family beside it; "before" is one or few targets per wavefront, with the compiler's
// division and square root):
//   N        500  1000  2000  4000  6000 | 8000  12000  16384  20000  32768  65536  100003  262144
//   relay    7.3  10.0  17.9  41.2  80.7 |  141    289    529    817   2063
//   ring                      60.6  86.0 |  110    287    389    656   1518   6000   14460   91900
//   before   9.2  14.7  29.7  78.5   169 |  241    483   1017   1399   3589  13545   30155  142460
// 3001 targets of 65536 sources: 455 (before 1300); 200 of 100000: 393 (1062).
// Few sources are a chunk of the relay at most, whose many small workgroups then cost more than
// the ring's: 50 sources at 3000 and 6500 targets 7.5 and 9.9 us, with the ring 7.1 and 7.1; 100
// at 3000 7.5 and 7.8.
constexpr int64_t kF64FewSources = 64;
enum class F64Ring { none, w8_h2, w8_h1, w4_h2, w4_h1 };
struct F64Shape {
    int targets;  // relay: per workgroup
    F64Ring ring;
};
static F64Shape f64_shape(const gh_ctx* c, int64_t np, int64_t nt)
{
    const int tune = c->tune[GH_TUNE_DIRECT_F64_TPW];
    const bool relay = tune < 0 || (tune == 0 && nt <= (np <= kF64FewSources ? 2048 : kF64RelayMax));
    if (relay) {
        int64_t t = tune < 0 ? -(int64_t)tune : 0;
        if (tune == 0)
            t = nt <= 256 ? 1 : nt <= 768 ? 3 : nt <= 1024 ? 4 : nt <= 2048 ? 8 : nt <= 2304 ? 9
                : nt <= 3072 ? 6 : nt <= 4096 ? 16 : nt <= 4608 ? 9 : nt <= 5120 ? 20 : 6;
        for (int has : {1, 3, 4, 6, 8, 9, 16})
            if (t <= has) return {has, F64Ring::none};
        return {20, F64Ring::none};
    }
    const bool one_lane = tune ? tune >= 64 : nt > 8192;
    if (nt <= 16384) return {0, one_lane ? F64Ring::w8_h1 : F64Ring::w8_h2};
    return {0, one_lane ? F64Ring::w4_h1 : F64Ring::w4_h2};
}

// Targets 0 .. whole - 1 that take a launch of their own, 0 for none.  A workgroup of 64 targets
// on each of the 256 CUs is a round of 16384.  The few workgroups beyond whole rounds run last on
// a CU each that they do not fill (N = 100003: 27 after 1536 held the launch for 1.2 rounds), so
// they go to the shape for as many targets, which spreads them over the chip.  Up to half a round
// that always gains; beyond, a launch of them costs more than it takes off the other.  Us with
// one launch and with two: N = 16500 684 and 538, 24000 928 and 916, 34000 2331 and 1787, 40768
// 2778 and 2429, 50000 4650 and 3629, 73536 8479 and 7605, 100003 16483 and 14040, 200000 57417
// and 54251; not taken: 24884 1228 and 1263, 41768 2903 and 2897, 74536 8491 and 8663.  One round
// is taken by eight wavefronts per workgroup, more by four (16500 538 and 602; 100003 14444 and
// 14040).
constexpr int64_t kF64Round = 256 * 64;
static int64_t f64_whole_rounds(const gh_ctx* c, int64_t nt)
{
    const int64_t rest = nt % kF64Round;
    return c->tune[GH_TUNE_DIRECT_F64_TPW] == 0 && nt > kF64Round && rest <= kF64Round / 2
               ? nt - rest
               : 0;
}

// The field of few sources at many targets, which k_direct_f64_few takes: there a workgroup of the
// ring has hardly a turn for each of its wavefronts, and starting and ending it is what counts.
// Us with the ring and with it: 1 source at 100000 targets 16.5 and 7.6, at 10^6 97 and 12; 16
// at 20000 11.8 and 7.6; 64 at 50000 14.1 and 13.7; 200 at 200000 70.5 and 71.5, at 10^6 308 and
// 263; 1000 at 10^6 1369 and 1311; not taken: 32 at 30000 8.4 and 9.3, 500 at 200000 153 and 175.
static bool f64_few(const gh_ctx* c, int64_t np, int64_t nt)
{
    return c->tune[GH_TUNE_DIRECT_F64_TPW] == 0 && nt > kF64Round && np <= nt / 1000;
}

// ------------------------------------------------------------------------------
// FP32 pairs, compensated accumulation
// ------------------------------------------------------------------------------
// Every FP32 kernel works in local frames (gh_frames.hip): the particles are sorted
// along a Morton curve, each block of consecutive sorted particles has an FP64 origin,
// and a kernel forms its FP32 coordinates relative to one block's origin from FP64
// values.  Blocks whose flag is set (not compact) are handled by the double-single
// (DS) forms, which carry every coordinate as hi + lo FP32 words of an FP64
// difference and form separations as (hi_j - hi_i) + (lo_j - lo_i).
__device__ __forceinline__ void two_sum_into(float& hi, float& lo, float t)
{
    // Knuth's branch-free two-sum: hi + lo + t == s + (lo + e) exactly before the
    // final rounding of the low word.
    const float s = hi + t;
    const float bp = s - hi;
    const float e = (hi - (s - bp)) + (t - bp);
    hi = s;
    lo = lo + e;
}

// hi + lo split of an FP64 value: hi = fl32(d), lo = fl32(d - hi) (d - hi is exact).
__device__ __forceinline__ void split_ds(double d, float& hi, float& lo)
{
    hi = (float)d;
    lo = (float)(d - (double)hi);
}

// One-sided kernel: IPT targets per lane, 256-source tiles staged in LDS and read as
// wave-wide broadcasts, FP32 sums per tile and an FP32 two-sum (hi, lo) across tiles;
// FP64 out.  Workgroup b holds the sorted targets of group b (256 IPT of them), whose
// frame is tframe[b]; every source tile is re-based into that frame from the FP64
// sources (src64, any order, massless padding).  DS: the group is flagged, and its
// separations are double-single.  (A launch of its own for the flagged groups, which are
// few or none, cost 4 us.)  Sources may
// be split over grid.y when there are too few targets to fill 256 CUs; the splits are
// added in split order.  perm (sorted target -> caller's index) places the results;
// with splits the per-split fields go to out in sorted order instead.
template <int IPT, bool GUARD, bool DS>
__device__ __forceinline__ void one_sided_group(
    float4 (&tile)[kBlock], float4 (&tile_lo)[kBlock], const double4* __restrict__ src64,
    int64_t np_pad, int64_t j_per_split, const float4* __restrict__ tloc,
    const double4* __restrict__ t64, const double4* __restrict__ tframe,
    const u32* __restrict__ perm, int64_t nt, float eps2, double* __restrict__ out)
{
    const double4 o = tframe[blockIdx.x];
    const int64_t i0 = (int64_t)blockIdx.x * (kBlock * IPT) + threadIdx.x;
    const int64_t j_begin = (int64_t)blockIdx.y * j_per_split;
    const int64_t j_end = min(np_pad, j_begin + j_per_split);

    eps2 = in_vgpr(eps2);
    float xi[IPT], yi[IPT], zi[IPT], xl[IPT], yl[IPT], zl[IPT];
    float hx[IPT], hy[IPT], hz[IPT], lx[IPT], ly[IPT], lz[IPT];
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        const int64_t i = i0 + (int64_t)k * kBlock;
        xi[k] = yi[k] = zi[k] = xl[k] = yl[k] = zl[k] = 0.f;
        if (i < nt) {
            if (DS) {
                const double4 q = t64[i];
                split_ds(q.x - o.x, xi[k], xl[k]);
                split_ds(q.y - o.y, yi[k], yl[k]);
                split_ds(q.z - o.z, zi[k], zl[k]);
            } else {
                const float4 t = tloc[i];
                xi[k] = t.x;
                yi[k] = t.y;
                zi[k] = t.z;
            }
        }
        hx[k] = hy[k] = hz[k] = lx[k] = ly[k] = lz[k] = 0.f;
    }

    for (int64_t base = j_begin; base < j_end; base += kBlock) {
        __syncthreads();
        {
            const double4 q = src64[base + threadIdx.x];
            if (DS) {
                float4 h, l;
                split_ds(q.x - o.x, h.x, l.x);
                split_ds(q.y - o.y, h.y, l.y);
                split_ds(q.z - o.z, h.z, l.z);
                h.w = (float)q.w;
                l.w = 0.f;
                tile[threadIdx.x] = h;
                tile_lo[threadIdx.x] = l;
            } else {
                tile[threadIdx.x] = make_float4((float)(q.x - o.x), (float)(q.y - o.y),
                                                (float)(q.z - o.z), (float)q.w);
            }
        }
        __syncthreads();
        float ax[IPT], ay[IPT], az[IPT];
#pragma unroll
        for (int k = 0; k < IPT; k++) ax[k] = ay[k] = az[k] = 0.f;
#pragma unroll 8
        for (int jj = 0; jj < kBlock; jj++) {
            const float4 s = tile[jj];
            float4 sl = make_float4(0.f, 0.f, 0.f, 0.f);
            if (DS) sl = tile_lo[jj];
#pragma unroll
            for (int k = 0; k < IPT; k++) {
                float dx = s.x - xi[k];
                float dy = s.y - yi[k];
                float dz = s.z - zi[k];
                if (DS) {
                    dx = dx + (sl.x - xl[k]);
                    dy = dy + (sl.y - yl[k]);
                    dz = dz + (sl.z - zl[k]);
                }
                float r2 = __builtin_fmaf(dx, dx, eps2);
                r2 = __builtin_fmaf(dy, dy, r2);
                r2 = __builtin_fmaf(dz, dz, r2);
                const float ri = __builtin_amdgcn_rsqf(r2);
                const float ri2 = ri * ri;
                float sc = (s.w * ri) * ri2;
                if (GUARD) sc = clamp_finite(sc);
                ax[k] = __builtin_fmaf(dx, sc, ax[k]);
                ay[k] = __builtin_fmaf(dy, sc, ay[k]);
                az[k] = __builtin_fmaf(dz, sc, az[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < IPT; k++) {
            two_sum_into(hx[k], lx[k], ax[k]);
            two_sum_into(hy[k], ly[k], ay[k]);
            two_sum_into(hz[k], lz[k], az[k]);
        }
    }

    const bool split = gridDim.y > 1;
    double* o_split = out + (int64_t)blockIdx.y * nt * 3;
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        const int64_t i = i0 + (int64_t)k * kBlock;
        if (i < nt) {
            double* d = split ? o_split + 3 * i : out + 3 * (int64_t)perm[i];
            d[0] = (double)hx[k] + (double)lx[k];
            d[1] = (double)hy[k] + (double)ly[k];
            d[2] = (double)hz[k] + (double)lz[k];
        }
    }
}

template <int IPT, bool GUARD>
__global__ __launch_bounds__(kBlock) void k_direct_f32(const double4* __restrict__ src64,
                                                       int64_t np_pad, int64_t j_per_split,
                                                       const float4* __restrict__ tloc,
                                                       const double4* __restrict__ t64,
                                                       const double4* __restrict__ tframe,
                                                       const int* __restrict__ tflag,
                                                       const u32* __restrict__ perm,
                                                       int64_t nt, float eps2,
                                                       double* __restrict__ out)
{
    __shared__ float4 tile[kBlock], tile_lo[kBlock];
    if (tflag[blockIdx.x] == 0)
        one_sided_group<IPT, GUARD, false>(tile, tile_lo, src64, np_pad, j_per_split, tloc, t64,
                                           tframe, perm, nt, eps2, out);
    else
        one_sided_group<IPT, GUARD, true>(tile, tile_lo, src64, np_pad, j_per_split, tloc, t64,
                                          tframe, perm, nt, eps2, out);
}

// ------------------------------------------------------------------------------
// FP32 pairs, each unordered pair computed once (self field only)
// ------------------------------------------------------------------------------
// Particles (in sorted order) are cut into blocks of BLK = 256*IPT.  A workgroup takes
// one block pair (I, J), I <= J.  Its 4 wavefronts hold the 256*IPT i-particles of
// block I in registers (IPT per lane); block J is staged in LDS.  For I < J, block J is
// walked in chunks of 64: at step s lane l pairs its i-particles with j = (l + s) mod 64
// of the chunk and accumulates both the force on its i-particles and the force on that
// j in a register that moves to lane l-1 after every step (DPP wavefront rotation), so
// after 64 steps lane l holds the whole wavefront's force on j = l.  The four
// wavefronts' j-partials are added in LDS.  A diagonal pair I = J is done one-sided.
// The workgroup works in block I's frame: i-particles are block I's local coordinates,
// block J's enter as fl(loc_J + fl(o_J - o_I)).  Pairs with a flagged block take the DS form in
// the same launch, which stages both sides as hi + lo words of the FP64 differences from o_I.
//
// Results are partial fields part[K][p] (FP32, 3 per particle): particle p of block B
// receives one partial from every block K (K = B for its diagonal); k_reduce_sym adds
// them in FP64, in an order fixed by their count.  The j-side partials can go to a
// second array (SymOut): a pass over the block pairs of a band of columns J keeps only
// the band's slots (see direct_sym).
constexpr int kRotFromNext = 0x134;  // DPP wave_rol:1 -- lane l reads lane l+1 (mod 64)

__device__ __forceinline__ float rot_from_next(float v)
{
    // every lane has a source lane, so no "old" value is needed
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kRotFromNext, 0xf, 0xf,
                                                   false));
}

// Where the partial fields go: the i-side of an item to part[slot_i][p] (stride np_pad
// particles), the j-side to jpart[slot_j][p - joff] (stride jstride particles).  One
// array for both (jpart = part, jstride = np_pad, joff = 0) outside banded passes.
struct SymOut {
    float* part;
    float* jpart;
    int64_t jstride;
    int64_t joff;
};

// One block pair.  Work item {I, J, slot_i, slot_j}: global block indices I <= J (of
// one simulation), the partial slot the i-side field goes to (J's index within its
// simulation) and the slot of the j-side field (I's index within its simulation).
// UNI: the particles of block I all have mass mI and those of block J mass mJ, so the masses
// multiply the sums instead of every pair's factor: 15 instead of 17 VALU operations per
// pair.  nI, nJ: the particles of either block.  Wavefronts that hold only padding, and
// chunks of it, are left out: padding is massless, its terms are zeros.
template <int IPT, bool GUARD, bool DS, bool UNI>
__device__ __forceinline__ void sym_item(const float4* __restrict__ src,
                                         const double4* __restrict__ s64,
                                         const double4* __restrict__ frame, int64_t np_pad,
                                         int4 it, float eps2, float mI, float mJ, int nI,
                                         int nJ, const SymOut out, float4* tile, float (*jp)[3][64])
{
    constexpr int BLK = kBlock * IPT;
    constexpr int NCH = BLK / 64;
    // each 64-particle chunk of block J is stored twice in a row, so that lane l's rotating
    // index l + s needs no wrap-around; DS stores it once and its low words after all chunks
    constexpr int ROW = DS ? 64 : 128;
    float4* const tile_lo = tile + (DS ? BLK : 0);
    const int I = it.x, J = it.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t ibase = (int64_t)I * BLK + wave * 64 * IPT + lane;
    const int64_t jbase = (int64_t)J * BLK;
    eps2 = in_vgpr(eps2);
    const double4 oI = frame[I];

    float xi[IPT], yi[IPT], zi[IPT], mi[IPT], ax[IPT], ay[IPT], az[IPT];
    float xl[IPT], yl[IPT], zl[IPT];
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        if (DS) {
            const double4 q = s64[ibase + k * 64];
            split_ds(q.x - oI.x, xi[k], xl[k]);
            split_ds(q.y - oI.y, yi[k], yl[k]);
            split_ds(q.z - oI.z, zi[k], zl[k]);
            mi[k] = (float)q.w;
        } else {
            const float4 t = src[ibase + k * 64];
            xi[k] = t.x;
            yi[k] = t.y;
            zi[k] = t.z;
            mi[k] = t.w;
            xl[k] = yl[k] = zl[k] = 0.f;
        }
        ax[k] = ay[k] = az[k] = 0.f;
    }
    if (DS) {
        for (int q = threadIdx.x; q < BLK; q += kBlock) {
            const double4 v = s64[jbase + q];
            float4 h, l;
            split_ds(v.x - oI.x, h.x, l.x);
            split_ds(v.y - oI.y, h.y, l.y);
            split_ds(v.z - oI.z, h.z, l.z);
            h.w = (float)v.w;
            l.w = 0.f;
            tile[q] = h;
            tile_lo[q] = l;
        }
    } else {
        const double4 oJ = frame[J];
        const float offx = (float)(oJ.x - oI.x), offy = (float)(oJ.y - oI.y),
                    offz = (float)(oJ.z - oI.z);
        for (int q = threadIdx.x; q < NCH * 128; q += kBlock) {
            float4 v = src[jbase + (q >> 7) * 64 + (q & 63)];
            v.x += offx;
            v.y += offy;
            v.z += offz;
            tile[q] = v;
        }
    }
    __syncthreads();

    const bool live = wave * 64 * IPT < nI;
    const int chunks = (nJ + 63) / 64;
    if (I == J) {
        for (int c = 0; c < (live ? chunks : 0); c++) {
#pragma unroll(DS ? 1 : 8)
            for (int q = 0; q < 64; q++) {
                const float4 s = tile[c * ROW + q];
                float4 sl = make_float4(0.f, 0.f, 0.f, 0.f);
                if (DS) sl = tile_lo[c * ROW + q];
#pragma unroll
                for (int k = 0; k < IPT; k++) {
                    float dx = s.x - xi[k], dy = s.y - yi[k], dz = s.z - zi[k];
                    if (DS) {
                        dx = dx + (sl.x - xl[k]);
                        dy = dy + (sl.y - yl[k]);
                        dz = dz + (sl.z - zl[k]);
                    }
                    float r2 = __builtin_fmaf(dx, dx, eps2);
                    r2 = __builtin_fmaf(dy, dy, r2);
                    r2 = __builtin_fmaf(dz, dz, r2);
                    const float ri = __builtin_amdgcn_rsqf(r2);
                    float sc = UNI ? ri * (ri * ri) : (s.w * ri) * (ri * ri);
                    if (GUARD) sc = clamp_finite(sc);
                    ax[k] = __builtin_fmaf(dx, sc, ax[k]);
                    ay[k] = __builtin_fmaf(dy, sc, ay[k]);
                    az[k] = __builtin_fmaf(dz, sc, az[k]);
                }
            }
        }
    } else {
        for (int c = 0; c < chunks; c++) {
            float fx = 0.f, fy = 0.f, fz = 0.f;
            for (int s0 = 0; s0 < (live ? 64 : 0); s0 += 8) {
#pragma unroll(DS ? 1 : 8)
                for (int s = 0; s < 8; s++) {
                    const int q = c * ROW + (DS ? (lane + s0 + s) & 63 : lane + s0 + s);
                    const float4 sj = tile[q];
                    float4 sl = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (DS) sl = tile_lo[q];
#pragma unroll
                    for (int k = 0; k < IPT; k++) {
                        float dx = sj.x - xi[k], dy = sj.y - yi[k], dz = sj.z - zi[k];
                        if (DS) {
                            dx = dx + (sl.x - xl[k]);
                            dy = dy + (sl.y - yl[k]);
                            dz = dz + (sl.z - zl[k]);
                        }
                        float r2 = __builtin_fmaf(dx, dx, eps2);
                        r2 = __builtin_fmaf(dy, dy, r2);
                        r2 = __builtin_fmaf(dz, dz, r2);
                        const float ri = __builtin_amdgcn_rsqf(r2);
                        const float ri3 = ri * ri * ri;
                        float si = UNI ? ri3 : sj.w * ri3;
                        if (GUARD) si = clamp_finite(si);
                        ax[k] = __builtin_fmaf(dx, si, ax[k]);
                        ay[k] = __builtin_fmaf(dy, si, ay[k]);
                        az[k] = __builtin_fmaf(dz, si, az[k]);
                        float sm = UNI ? ri3 : mi[k] * ri3;
                        if (GUARD) sm = clamp_finite(sm);
                        fx = __builtin_fmaf(dx, sm, fx);
                        fy = __builtin_fmaf(dy, sm, fy);
                        fz = __builtin_fmaf(dz, sm, fz);
                    }
                    fx = rot_from_next(fx);
                    fy = rot_from_next(fy);
                    fz = rot_from_next(fz);
                }
            }
            // lane l now holds this wavefront's pull of its i-particles by j = l; the
            // force on j is the opposite
            jp[wave][0][lane] = fx;
            jp[wave][1][lane] = fy;
            jp[wave][2][lane] = fz;
            __syncthreads();
            if (threadIdx.x < 3 * 64) {
                const int comp = threadIdx.x >> 6, t = threadIdx.x & 63;
                float sacc = jp[0][comp][t];
#pragma unroll
                for (int w = 1; w < kBlock / 64; w++) sacc += jp[w][comp][t];
                out.jpart[((int64_t)it.w * out.jstride + (jbase - out.joff) + c * 64 + t) * 3 +
                          comp] = UNI ? -sacc * mI : -sacc;
            }
            __syncthreads();
        }
    }
    if (!live) return;
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        float* o = out.part + ((int64_t)it.z * np_pad + ibase + k * 64) * 3;
        o[0] = UNI ? ax[k] * mJ : ax[k];
        o[1] = UNI ? ay[k] * mJ : ay[k];
        o[2] = UNI ? az[k] * mJ : az[k];
    }
}

// One launch over a list of block pairs.  queue == nullptr: workgroup b takes item b.
// Otherwise the workgroups are persistent and take items from *queue (which must be 0 at
// launch) until the list is exhausted.
//  - Items with a flagged block take the DS form, about twice the time of another item; a
//    persistent launch takes them first, spread over the workgroups, so that none starts
//    last.  (As a launch of its own after the others the DS form ran at the length of one
//    item, 190 us in an ensemble of 32 spheres of 1024 to 16384 particles, whose outermost
//    blocks are flagged, and 4.6 us where no block is.)
//  - Items whose blocks each have one mass (umass, not NaN) take the UNI form in simulations
//    of at least kUniMin particles (nb_blk[b] or, where it is null, nb blocks), unless the
//    guard is needed, which bounds the factors with their masses.  Systems of unequal masses
//    gain nothing.  Measured (N = 262144, equal masses, per launch): 13.33 -> 11.98 ms.  Below
//    kUniMin results keep the bits of the general form, though there is as much to gain (us a
//    force: N = 16384 109 -> 104, 32768 319 -> 288, 65536 1029 -> 931, 98304 2083 -> 1874): the
//    sums are rounded elsewhere, and four steps move the velocities by up to 1e-7.
//  - Registers for six wavefronts per SIMD where a lane has one particle and five otherwise,
//    as LDS allows: N = 16384 118 -> 113 us a call, 32768 334 -> 319 (four lose 3 % at 65536
//    and beyond).  Padding left out: 128 spheres of 1024 to 65536 15.0 -> 14.6 ms a step.
constexpr int kUniMin = 131072;

template <int IPT, bool GUARD>
__global__ __launch_bounds__(kBlock, IPT == 1 ? 6 : 5) void k_direct_sym_f32(
    const float4* __restrict__ src, const double4* __restrict__ s64,
    const double4* __restrict__ frame, const int* __restrict__ flag,
    const int* __restrict__ nflag, const float* __restrict__ umass,
    const int* __restrict__ used, const int* __restrict__ nb_blk, int nb, int64_t np_pad, const int4* __restrict__ work,
    int64_t items, const float* __restrict__ eps2_blk, const SymOut out, int* __restrict__ queue)
{
    constexpr int NCH = kBlock * IPT / 64;
    __shared__ float4 tile[NCH * 128];
    __shared__ float jp[kBlock / 64][3][64];
    __shared__ int next;
    // the persistent launch's flagged items; k runs over this workgroup's share of the list
    const bool first = queue && *nflag != 0;
    int64_t k = blockIdx.x;
    for (bool flagged = first;;) {
        if (queue && !flagged) {
            if (threadIdx.x == 0) next = atomicAdd(queue, 1);
            __syncthreads();
            k = next;
            __syncthreads();
        }
        if (k >= items) {
            if (!flagged) break;
            flagged = false;
            continue;
        }
        const int4 it = work[k];
        const bool ds = (flag[it.x] | flag[it.y]) != 0;
        const float mI = umass[it.x], mJ = umass[it.y], eps2 = eps2_blk[it.x];
        const int blocks = nb_blk ? nb_blk[it.x] : nb;
        const int nI = used[it.x], nJ = used[it.y];
        if (ds && flagged == first)
            sym_item<IPT, GUARD, true, false>(nullptr, s64, frame, np_pad, it, eps2, 0.f, 0.f,
                                              nI, nJ, out, tile, jp);
        else if (!ds && !flagged && !GUARD && blocks >= kUniMin / (kBlock * IPT) && mI == mI &&
                 mJ == mJ)
            sym_item<IPT, GUARD, false, !GUARD>(src, nullptr, frame, np_pad, it, eps2, mI, mJ,
                                                nI, nJ, out, tile, jp);
        else if (!ds && !flagged)
            sym_item<IPT, GUARD, false, false>(src, nullptr, frame, np_pad, it, eps2, 0.f, 0.f,
                                               nI, nJ, out, tile, jp);
        if (!queue) break;
        __syncthreads();
        if (flagged) k += gridDim.x;
    }
}

// acc[perm[p]] = sum over the partial slots of p's simulation in FP64 (perm == nullptr:
// acc[p]).  nb_blk[b] (nullable): number of slots of the simulation that block b belongs
// to; otherwise every particle has nb slots.  Four consecutive components per lane, read
// as one 16-byte load per partial slab (each slab, 3 np_pad floats with np_pad a multiple
// of the block size, starts on a 16-byte boundary, and a group of four never straddles
// two blocks, as 3 x 256 is a multiple of 4).
__global__ __launch_bounds__(kBlock) void k_reduce_sym(const float* __restrict__ part, int nb,
                                                       const int* __restrict__ nb_blk,
                                                       int blk, int64_t np_pad, int64_t n3,
                                                       const u32* __restrict__ perm,
                                                       double* __restrict__ acc, StepUpdate up)
{
    // Each workgroup takes 64 groups of 4 floats, one per lane; its wavefront w adds the
    // slots w, w + kSlotLanes, ... in order (so each load reads 64 consecutive float4),
    // and the wavefronts' sums are added in a fixed order.  The order depends on the slot
    // count only, so an ensemble's particles sum exactly as they would alone.
    static_assert(kBlock == 64 * kSlotLanes, "one slice per wavefront");
    __shared__ double sh[kSlotLanes][4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t k0 = ((int64_t)blockIdx.x * 64 + lane) * 4;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (k0 < n3) {
        const int slots = nb_blk ? nb_blk[(k0 / 3) / blk] : nb;
        const float4* p = (const float4*)(part + k0);
        const int64_t stride = np_pad * 3 / 4;  // float4 per slab
        for (int b = w; b < slots; b += kSlotLanes) {
            const float4 v = p[(int64_t)b * stride];
            s[0] += (double)v.x;
            s[1] += (double)v.y;
            s[2] += (double)v.z;
            s[3] += (double)v.w;
        }
    }
    for (int j = 0; j < 4; j++) sh[w][j][lane] = s[j];
    __syncthreads();
    // wavefront w stores component w of its lanes' groups: (s0 + s1) + (s2 + s3)
    const int64_t k = k0 + w;
    if (k0 < n3 && k < n3) {
        const double t = (sh[0][w][lane] + sh[1][w][lane]) + (sh[2][w][lane] + sh[3][w][lane]);
        const int64_t q = k / 3;
        const int64_t at = perm ? 3 * (int64_t)perm[q] + (k - 3 * q) : k;
        if (up.v)
            update_one(up, at, t);
        else
            acc[at] = t;
    }
}

// One pass of the banded pair-once self field (direct_sym): the block pairs (I, J) with
// J in the band [c0, c0 + w) of blocks.  Particle p of block P has this pass's partials
// from partners q (blocks) in partner order: the j-side of (q, P) for q < P when P is
// in the band (partj[q][p - c0 blk], jw blocks of particles per slot), then the i-side
// of (P, q) for q >= P in the band (parti[q - c0][p]).  Their FP64 sum is added to
// acc[perm[p]] (written on the first pass).  w: the band's width in blocks.
__global__ __launch_bounds__(kBlock) void k_reduce_band(const float* __restrict__ parti,
                                                        const float* __restrict__ partj,
                                                        int blk, int c0, int w, int jw,
                                                        int64_t np_pad,
                                                        int64_t n3, const u32* __restrict__ perm,
                                                        bool first, double* __restrict__ acc)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= n3) return;
    const int64_t p = k / 3;
    const int comp = (int)(k - 3 * p);
    const int P = (int)(p / blk);
    double sum = 0.0;
    const bool in_band = P >= c0 && P < c0 + w;
    if (in_band) {
        const int64_t pj = p - (int64_t)c0 * blk;
        for (int q = 0; q < P; q++) sum += (double)partj[((int64_t)q * jw * blk + pj) * 3 + comp];
    }
    for (int q = P > c0 ? P : c0; q < c0 + w; q++)
        sum += (double)parti[((int64_t)(q - c0) * np_pad + p) * 3 + comp];
    const int64_t o = 3 * (int64_t)perm[p] + comp;
    acc[o] = first ? sum : acc[o] + sum;
}

// Sum of per-split partial fields (sorted target order), in split order, written to
// acc[perm[i]], or the particles' update with it.
__global__ __launch_bounds__(kBlock) void k_reduce_splits(const double* __restrict__ part,
                                                          int splits, int64_t n3,
                                                          const u32* __restrict__ perm,
                                                          double* __restrict__ acc,
                                                          StepUpdate up)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= n3) return;
    const int64_t q = k / 3;
    const int64_t at = 3 * (int64_t)perm[q] + (k - 3 * q);
    double s = part[k];
    int p = 1;
    for (; p + 4 <= splits; p += 4) {  // four loads in flight
        const double a = part[(int64_t)p * n3 + k], b = part[(int64_t)(p + 1) * n3 + k];
        const double d = part[(int64_t)(p + 2) * n3 + k], e = part[(int64_t)(p + 3) * n3 + k];
        s = (((s + a) + b) + d) + e;
    }
    for (; p < splits; p++) s += part[(int64_t)p * n3 + k];
    if (up.v)
        update_one(up, at, s);
    else
        acc[at] = s;
}

// (x, y, z, m) in input order, entries n..n_pad-1 massless at the origin
__global__ __launch_bounds__(kBlock) void k_pack_src64(const double* __restrict__ pos,
                                                       const double* __restrict__ mass,
                                                       int64_t n, int64_t n_pad,
                                                       double4* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n)
        out[i] = make_double4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], mass[i]);
    else if (i < n_pad)
        out[i] = make_double4(0.0, 0.0, 0.0, 0.0);
}

// ------------------------------------------------------------------------------
// dispatch
// ------------------------------------------------------------------------------
namespace {

struct F32Shape {
    int ipt;
    int splits;
};

// Targets per lane and source splits: enough workgroups for every CU, no more
// source splitting than needed.
F32Shape pick_shape(gh_ctx* c, int64_t nt, int64_t np_pad)
{
    int dev_cus = 256;
    (void)c;
    F32Shape sh{1, 1};
    if (nt >= (int64_t)kBlock * 2 * 2 * dev_cus) sh.ipt = 2;
    const int64_t wgs = (nt + (int64_t)kBlock * sh.ipt - 1) / ((int64_t)kBlock * sh.ipt);
    const int64_t want = 4LL * dev_cus;
    if (wgs < want) {
        int64_t sp = (want + wgs - 1) / wgs;
        const int64_t max_sp = np_pad / kBlock;  // at least one tile per split
        if (sp > max_sp) sp = max_sp;
        if (sp < 1) sp = 1;
        sh.splits = (int)sp;
    }
    return sh;
}

// The FP64 sums of targets from .. nt - 1 (self: of particles, from among all np).
struct F64Call {
    bool self;
    const double *pos, *mass;
    int64_t np;
    const double* tgt;
    int64_t from, nt;
    double eps2;
    double* acc;
    StepUpdate up;  // relay only
    hipStream_t s;
};

template <int P, int K>
void launch_relay(const F64Call& q)
{
    const dim3 grid((unsigned)((q.nt - q.from + P * K - 1) / (P * K))), block((P + 1) * 64);
    if (q.self)
        hipLaunchKernelGGL((k_direct_f64_relay<true, P, K>), grid, block, 0, q.s, q.pos, q.mass,
                           q.np, q.tgt, q.from, q.nt, q.eps2, q.acc, q.up);
    else
        hipLaunchKernelGGL((k_direct_f64_relay<false, P, K>), grid, block, 0, q.s, q.pos, q.mass,
                           q.np, q.tgt, q.from, q.nt, q.eps2, q.acc, q.up);
}

template <int W, int H>
void launch_ring(const F64Call& q)
{
    // 16 sources per lane and turn: passing the turn on takes about 390 cycles, the terms
    // of 8 sources 1900 (N = 16384: 433 us with 8, 398 with 16)
    constexpr int C = 16;
    const dim3 grid(blocks_for(q.nt - q.from, 64 / H)), block(64 * W);
    if (q.self)
        hipLaunchKernelGGL((k_direct_f64_ring<true, W, C, H>), grid, block, 0, q.s, q.pos,
                           q.mass, q.np, q.tgt, q.from, q.nt, q.eps2, q.acc);
    else
        hipLaunchKernelGGL((k_direct_f64_ring<false, W, C, H>), grid, block, 0, q.s, q.pos,
                           q.mass, q.np, q.tgt, q.from, q.nt, q.eps2, q.acc);
}

int launch_f64(gh_ctx* c, const F64Shape& sh, const F64Call& q)
{
    switch (sh.ring) {
    case F64Ring::none:
        switch (sh.targets) {
        case 1: launch_relay<1, 1>(q); break;
        case 3: launch_relay<3, 1>(q); break;
        case 4: launch_relay<4, 1>(q); break;
        case 6: launch_relay<3, 2>(q); break;
        case 8: launch_relay<4, 2>(q); break;
        case 9: launch_relay<3, 3>(q); break;
        case 16: launch_relay<8, 2>(q); break;
        default: launch_relay<4, 5>(q); break;
        }
        return check_launch(c, "k_direct_f64_relay");
    case F64Ring::w8_h2: launch_ring<8, 2>(q); break;
    case F64Ring::w8_h1: launch_ring<8, 1>(q); break;
    case F64Ring::w4_h2: launch_ring<4, 2>(q); break;
    default: launch_ring<4, 1>(q); break;
    }
    return check_launch(c, "k_direct_f64_ring");
}

template <int IPT>
void launch_f32(bool guard, dim3 grid, hipStream_t s, const double4* src64, int64_t np_pad,
                int64_t jps, const OrderBufs& t, int64_t nt, float eps2, double* out)
{
    const float4* tloc = t.loc.as<float4>();
    const double4* t64 = t.s64.as<double4>();
    const double4* fr = t.frame.as<double4>();
    const int* fl = t.flag.as<int>();
    const u32* perm = t.perm();
    if (guard)
        hipLaunchKernelGGL((k_direct_f32<IPT, true>), grid, dim3(kBlock), 0, s, src64,
                           np_pad, jps, tloc, t64, fr, fl, perm, nt, eps2, out);
    else
        hipLaunchKernelGGL((k_direct_f32<IPT, false>), grid, dim3(kBlock), 0, s, src64,
                           np_pad, jps, tloc, t64, fr, fl, perm, nt, eps2, out);
}

}  // namespace

// FP32 pair arithmetic needs the zero-separation guard whenever a coincident pair (or
// the self pair of the one-sided kernels) could produce 0 * inf: m / eps^3 overflows FP32
// for eps^2 below about 1e-15 once masses reach 1e15 Msun, and the guard is also what
// the reference does for targets at zero distance (:327-330).
bool fp32_guard(double eps)
{
    const float eps2 = (float)(eps * eps);
    return !(eps2 >= 1e-15f);
}

// Symmetric (pair-once) kernel for the self field: particles per lane, or 0 for the
// one-sided kernel.  Block pairs must number a few thousand to fill 256 CUs.
// The pair-once kernel keeps one FP32 partial field per block: 12 B x np x (np / block)
// of scratch, which grows as np^2 (12.9 GB at np = 2^20).  Above kSymScratchMax the
// block pairs are taken in bands of columns, one pass each, whose partials take at most
// that much (direct_sym).
constexpr double kSymScratchMax = 13.0 * (1 << 30);

int sym_ipt(gh_ctx* c, int64_t np)
{
    const int forced = c->tune[GH_TUNE_DIRECT_SELF];
    if (forced < 0) return 0;
    int ipt = 0;
    if (forced == 1 || forced == 2 || forced == 4)
        ipt = forced;
    else if (np >= 65536)
        ipt = 4;
    else if (np >= 32768)
        ipt = 2;
    else if (np >= 16384)
        ipt = 1;
    return ipt;
}

int launch_sym(gh_ctx* c, int ipt, bool guard, const float4* src, const double4* s64,
               const double4* frame, const int* flag, const int* nflag, const float* umass,
               const int* used, const int* nb_blk, int nb, int64_t np_pad, const int4* work, int64_t items,
               const float* eps2_blk, float* part,
               int* queue, unsigned persistent_grid, hipStream_t s, float* jpart, int64_t jstride,
               int64_t joff)
{
    SymOut out;
    out.part = part;
    out.jpart = jpart ? jpart : part;
    out.jstride = jpart ? jstride : np_pad;
    out.joff = jpart ? joff : 0;
    if (items > 0x7fffffff) return fail(c, GH_EARG, "too many block pairs for one launch");
    const unsigned grid = queue ? persistent_grid : (unsigned)items;
    if (grid == 0) return 0;
#define GH_SYM(IPT)                                                                            \
    case IPT:                                                                                  \
        if (guard)                                                                             \
            hipLaunchKernelGGL((k_direct_sym_f32<IPT, true>), dim3(grid), dim3(kBlock), 0, s,  \
                               src, s64, frame, flag, nflag, umass, used, nb_blk, nb, np_pad,  \
                               work, items, eps2_blk, out, queue);                             \
        else                                                                                   \
            hipLaunchKernelGGL((k_direct_sym_f32<IPT, false>), dim3(grid), dim3(kBlock), 0, s, \
                               src, s64, frame, flag, nflag, umass, used, nb_blk, nb, np_pad,  \
                               work, items, eps2_blk, out, queue);                             \
        break
    switch (ipt) {
        GH_SYM(1);
        GH_SYM(2);
        GH_SYM(4);
        default: return fail(c, GH_EARG, "unsupported particles-per-lane %d", ipt);
    }
#undef GH_SYM
    return check_launch(c, "k_direct_sym_f32");
}

int reduce_sym(gh_ctx* c, const float* part, int nb, const int* nb_blk, int blk,
               int64_t np_pad, int64_t n, const u32* perm, double* acc, hipStream_t s,
               const StepUpdate* up)
{
    if (n <= 0) return 0;
    if ((np_pad * 3) % 4 != 0 || (3 * blk) % 4 != 0)
        return fail(c, GH_EARG, "partial slabs are not 16-byte aligned");
    hipLaunchKernelGGL(k_reduce_sym, dim3(blocks_for((3 * n + 3) / 4, 64)), dim3(kBlock), 0, s,
                       part, nb, nb_blk, blk, np_pad, 3 * n, perm, acc, up ? *up : StepUpdate());
    return check_launch(c, "k_reduce_sym");
}

__global__ void k_fill_f32(float* __restrict__ p, int64_t n, float v)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}

int direct_sym(gh_ctx* c, const double* d_pos, const double* d_mass, int64_t np, int ipt,
               double eps, double* d_acc, hipStream_t s, const StepUpdate* up, bool* updated)
{
    const int64_t blk = (int64_t)kBlock * ipt;
    const int64_t np_pad = pad_to(np, blk);
    const int nb = (int)(np_pad / blk);
    // band width in blocks: all of them when one partial per block fits kSymScratchMax,
    // else as many as keep the band's partials (2 w np_pad of 12 bytes) within it
    int w = nb;
    if (c->tune[GH_TUNE_SYM_BAND] > 0)
        w = std::min(nb, c->tune[GH_TUNE_SYM_BAND]);
    else if (12.0 * (double)np_pad * nb > kSymScratchMax)
        w = (int)std::max<double>(1.0, std::floor(kSymScratchMax / (24.0 * (double)np_pad)));
    const int bands = (nb + w - 1) / w;
    const int64_t items = (int64_t)nb * (nb + 1) / 2;
    if (items > 0x7fffffff) return fail(c, GH_EARG, "too many particles for one launch");
    const size_t part_floats = bands == 1 ? 3 * (size_t)np_pad * nb : 6 * (size_t)np_pad * w;
    GH_TRY(ensure(c, c->scratch, sizeof(float) * part_floats));
    GH_TRY(ensure(c, c->eps_blk, sizeof(float) * (size_t)nb));
    const float eps2 = (float)(eps * eps);
    if (c->sym_nb != nb || c->sym_ipt != ipt || c->sym_w != w) {
        // block pairs (I, J), I <= J, band by band of columns J, then ordered by I;
        // slots: the partner block, within the band for the i-side
        std::vector<int4> wl((size_t)items);
        c->sym_band_start.assign(1, 0);
        size_t k = 0;
        for (int b = 0; b < bands; b++) {
            const int c0 = b * w, c1 = std::min(nb, c0 + w);
            for (int I = 0; I < c1; I++)
                for (int J = std::max(I, c0); J < c1; J++)
                    wl[k++] = make_int4(I, J, bands == 1 ? J : J - c0, I);
            c->sym_band_start.push_back((int64_t)k);
        }
        GH_TRY(ensure(c, c->work, sizeof(int4) * (size_t)items));
        GH_HIP(c, hipMemcpyAsync(c->work.p, wl.data(), sizeof(int4) * (size_t)items,
                                 hipMemcpyHostToDevice, s));
        GH_HIP(c, hipStreamSynchronize(s));
        c->sym_nb = nb;
        c->sym_ipt = ipt;
        c->sym_w = w;
        c->sym_eps2 = -1.f;
    }
    if (c->sym_eps2 != eps2) {  // the block list is rebuilt above whenever nb changes
        hipLaunchKernelGGL(k_fill_f32, dim3(blocks_for(nb, kBlock)), dim3(kBlock), 0, s,
                           c->eps_blk.as<float>(), (int64_t)nb, eps2);
        GH_TRY(check_launch(c, "k_fill_f32"));
        c->sym_eps2 = eps2;
    }
    OrderBufs& o = c->ord_p;
    GH_TRY(spatial_order(c, o, d_pos, np, s));
    GH_TRY(gather_frames(c, o, d_pos, d_mass, o.perm(), np, np_pad, (int)blk, nullptr, true, s));
    float* part = c->scratch.as<float>();
    const bool guard = fp32_guard(eps);
    if (bands == 1) {
        {
            TimedScope ts(c, s, GH_T_DIRECT_F32);
            GH_TRY(launch_sym(c, ipt, guard, o.loc.as<float4>(), o.s64.as<double4>(),
                              o.frame.as<double4>(), o.flag.as<int>(), o.nflag.as<int>(),
                              o.umass.as<float>(), o.used.as<int>(), nullptr, nb, np_pad,
                              c->work.as<int4>(), items, c->eps_blk.as<float>(), part, nullptr, 0, s));
        }
        if (up) *updated = true;
        return reduce_sym(c, part, nb, nullptr, (int)blk, np_pad, np, o.perm(), d_acc, s, up);
    }
    float* partj = part + 3 * (size_t)np_pad * w;
    for (int b = 0; b < bands; b++) {
        const int c0 = b * w, wb = std::min(nb, c0 + w) - c0;
        const int64_t i0 = c->sym_band_start[b], ni = c->sym_band_start[b + 1] - i0;
        {
            TimedScope ts(c, s, GH_T_DIRECT_F32);
            GH_TRY(launch_sym(c, ipt, guard, o.loc.as<float4>(), o.s64.as<double4>(),
                              o.frame.as<double4>(), o.flag.as<int>(), o.nflag.as<int>(),
                              o.umass.as<float>(), o.used.as<int>(), nullptr, nb, np_pad,
                              c->work.as<int4>() + i0, ni, c->eps_blk.as<float>(), part, nullptr, 0, s, partj,
                              (int64_t)w * blk, (int64_t)c0 * blk));
        }
        hipLaunchKernelGGL(k_reduce_band, dim3(blocks_for(3 * np, kBlock)), dim3(kBlock), 0, s,
                           part, partj, (int)blk, c0, wb, w, np_pad, 3 * np, o.perm(), b == 0,
                           d_acc);
        GH_TRY(check_launch(c, "k_reduce_band"));
    }
    return 0;
}

// One-sided FP32 field at nt targets.  src64: the sources as (x, y, z, m), np_pad of
// them (massless padding); t: the targets' spatial order and frames in groups of
// 256 x the chosen targets per lane.
static int direct_f32_onesided(gh_ctx* c, const double4* src64, int64_t np_pad, OrderBufs& t,
                               int64_t nt, const F32Shape& sh, double eps, double* d_acc,
                               hipStream_t s, const StepUpdate* up = nullptr,
                               bool* updated = nullptr)
{
    if (nt <= 0) return 0;
    if (np_pad % kBlock != 0) return fail(c, GH_EARG, "internal: source count not padded");
    const float eps2 = (float)(eps * eps);
    const bool guard = fp32_guard(eps);
    int64_t jps = pad_to((np_pad + sh.splits - 1) / sh.splits, kBlock);
    const int splits = (int)((np_pad + jps - 1) / jps);
    double* out = d_acc;
    if (splits > 1) {
        GH_TRY(ensure(c, c->scratch, sizeof(double) * 3 * (size_t)nt * splits));
        out = c->scratch.as<double>();
    }
    dim3 grid(blocks_for(nt, kBlock * sh.ipt), splits);
    {
        TimedScope ts(c, s, GH_T_DIRECT_F32);
        switch (sh.ipt) {
            case 1:
                launch_f32<1>(guard, grid, s, src64, np_pad, jps, t, nt, eps2, out);
                break;
            case 2:
                launch_f32<2>(guard, grid, s, src64, np_pad, jps, t, nt, eps2, out);
                break;
            case 4:
                launch_f32<4>(guard, grid, s, src64, np_pad, jps, t, nt, eps2, out);
                break;
            default: return fail(c, GH_EARG, "unsupported targets-per-lane %d", sh.ipt);
        }
        GH_TRY(check_launch(c, "k_direct_f32"));
    }
    if (splits > 1) {
        hipLaunchKernelGGL(k_reduce_splits, dim3(blocks_for(3 * nt, kBlock)), dim3(kBlock), 0,
                           s, out, splits, 3 * nt, t.perm(), d_acc, up ? *up : StepUpdate());
        if (up) *updated = true;
        GH_TRY(check_launch(c, "k_reduce_splits"));
    }
    return 0;
}

int direct_dev(gh_ctx* c, const double* d_pos, const double* d_mass, int64_t np,
               const double* d_fpos, int64_t nf, double eps, int precision, double* d_acc,
               hipStream_t s, const StepUpdate* up, bool* updated)
{
    // timed runs keep the update apart, in its own class
    if (c->timing) up = nullptr;
    const bool self = (d_fpos == nullptr);
    const double* tgt = self ? d_pos : d_fpos;
    const int64_t nt = self ? np : nf;
    if (np < 0 || nt < 0) return fail(c, GH_EARG, "negative particle count");
    if (nt == 0) return 0;
    if (np == 0) {
        return zero_dev(c, d_acc, 3 * nt, s);
    }
    if (precision == GH_FP64) {
        const double eps2 = eps * eps;
        F64Call q = {self, d_pos, d_mass, np, tgt, 0, nt, eps2, d_acc, StepUpdate(), s};
        F64Shape sh = f64_shape(c, np, nt);
        TimedScope ts(c, s, GH_T_DIRECT_F64);
        if (f64_few(c, np, nt)) {
            hipLaunchKernelGGL(k_direct_f64_few, dim3(blocks_for(nt, kBlock)), dim3(kBlock), 0, s,
                               d_pos, d_mass, (int)np, tgt, nt, eps2, d_acc);
            return check_launch(c, "k_direct_f64_few");
        }
        if (sh.ring == F64Ring::none) {
            if (up && up->xh_next != up->xh) {  // other workgroups read xh
                q.up = *up;
                *updated = true;
            }
        } else if (const int64_t whole = f64_whole_rounds(c, nt)) {
            q.nt = whole;
            GH_TRY(launch_f64(c, {0, whole == kF64Round ? F64Ring::w8_h1 : F64Ring::w4_h1}, q));
            if (whole == nt) return 0;
            q.from = whole;
            q.nt = nt;
            sh = f64_shape(c, np, nt - whole);
        }
        return launch_f64(c, sh, q);
    }
    if (precision != GH_FP32) return fail(c, GH_EARG, "unknown precision %d", precision);
    const int sym = self ? sym_ipt(c, np) : 0;
    if (sym > 0) return direct_sym(c, d_pos, d_mass, np, sym, eps, d_acc, s, up, updated);
    F32Shape sh = pick_shape(c, nt, pad_to(np, kBlock));
    const int forced = c->tune[GH_TUNE_DIRECT_IPT];
    if (forced == 1 || forced == 2 || forced == 4) sh.ipt = forced;
    const int group = kBlock * sh.ipt;
    const int64_t nt_pad = pad_to(nt, group);
    if (self) {
        // targets and sources are the particles: one order, the sorted FP64 particles
        // (massless padding at their group's origin) are the sources
        OrderBufs& o = c->ord_p;
        GH_TRY(spatial_order(c, o, d_pos, np, s));
        GH_TRY(gather_frames(c, o, d_pos, d_mass, o.perm(), np, nt_pad, group, nullptr, true, s));
        return direct_f32_onesided(c, o.s64.as<double4>(), nt_pad, o, nt, sh, eps, d_acc, s, up,
                                   updated);
    }
    const int64_t np_pad = pad_to(np, kBlock);
    GH_TRY(ensure(c, c->src64, sizeof(double4) * (size_t)np_pad));
    hipLaunchKernelGGL(k_pack_src64, dim3(blocks_for(np_pad, kBlock)), dim3(kBlock), 0, s, d_pos,
                       d_mass, np, np_pad, c->src64.as<double4>());
    GH_TRY(check_launch(c, "k_pack_src64"));
    OrderBufs& t = c->ord_t;
    GH_TRY(spatial_order(c, t, tgt, nt, s));
    GH_TRY(gather_frames(c, t, tgt, nullptr, t.perm(), nt, nt_pad, group, nullptr, true, s));
    return direct_f32_onesided(c, c->src64.as<double4>(), np_pad, t, nt, sh, eps, d_acc, s);
}

}  // namespace gh
