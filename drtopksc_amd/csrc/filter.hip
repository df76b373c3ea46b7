// filter.hip -- top-k of one vector for large k in six launches: a sample bounds the k-th key from
// below, one pass over the keys keeps those above the bound, and the selection runs on them.
//
// The delegate scheme pays for large k twice: its delegate stores (0.4 GB beside 4 GB of keys at
// 2^30, k = 2^24) and a concatenation that reads most subranges again.  Here the keys are read
// once and about 1.1 .. 2.6 k of them written.
//
//  k_fsample  m pseudo-random keys, one from each of m equal strata.
//  k_fsplit   t, the r'-th largest sample, with r' = r + 7 sqrt(r) + 12 above the expected rank
//             r = k m / n: fewer than k keys reach t with a probability below 1e-12 (the positions
//             do not depend on the keys).  Up to 254 samples of ranks r -+ (6 sqrt(r) + 8)
//             become splitters.
//  k_filter   keys > t with their indices, in index order, per unit of 2048 keys; how many
//             equal t (counted, never stored: any number of ties at t costs nothing); and the
//             exact counts between and at the splitters.
//  k_fpick    the kept keys of the k-th key's class, and per range of units how many lie above it.
//  k_fkth     the k-th key, and where each range's outputs start.
//  k_fwrite   the outputs in index order; ties at t are read from the keys again.
//
// At 2^30 keys, k = 2^22, the six take 7 + 29 + 735 + 22 + 20 .. 38 + 27 us (1028 us for the general
// pipeline, 855 for the call); the read alone takes 630.  At 2^24 keys, k = 2^16: 3 + 9 + 21 + 8 + 16 + 6 us
// (67 and 61 for the calls): there the launches, and the chains of round trips in the two
// one-workgroup kernels, are most of it.
//
// Should the bound fail after all, or a buffer not hold what it was sized for, k_fkth selects from
// the keys themselves with its one workgroup: slow (25 ms at 2^25 keys, 438 at 2^28), but exact.
// drtopk_select_route tells from the workspace that a call ended there.
#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "wgselect.hpp"

namespace drtopk {

constexpr int FS_NT = 1024;
constexpr u32 F_CLASSES = 512;  // 2b: between splitters b-1 and b; 2b+1: equal to splitter b; 511: above the window
constexpr u32 F_ABOVE = F_CLASSES - 1;
constexpr u32 F_SPLIT = 254;  // so that no splitter's class is 511
constexpr int F_REPS = 4;         // replicas of the class counters
constexpr u32 F_BATCH = WG * 8; // kept keys a workgroup takes at a time in k_fpick and k_fwrite
// Sorted or clustered keys fill the units of few ranges.  A range whose units of at least DENSE_UNIT kept keys
// hold more than DENSE_RANGE together is listed by k_filter, and its units are shared out over the waves of
// the whole grid: with a workgroup per range, one held all there was to do (2^30 ascending keys, k = 2^18:
// k_fpick 154 us, k_fwrite 431; at 2^26, k = 2^16, 25 and 66).  A unit with few kept keys is not worth a wave
// (2^28 keys, the top ones 1 in 256 of a sixteenth: 380 us for the call, 219 in batches).
constexpr u32 DENSE_UNIT = 256, DENSE_RANGE = 2 * F_BATCH;
constexpr u32 DENSE_ENTRY = 0x80000000u;  // a class entry of a dense range names its unit, others their range
// Samples above the bound that are put in order at once, each compared with all.  482 of them (k = n / 24 below 2^26
// keys) took the kernel 21 us, the selections and the sort of the splitters alone 14; 353 of them 16 and 15.
constexpr u32 F_SORT = 320;
constexpr u32 F_STAGE = 512;    // kept keys a wave stages in LDS
constexpr u32 F_LISTS = 64;     // sublists of the class, so that their cursors do not serialise

enum : u32 { F_CLASS = 0, F_AT_T = 1, F_DONE = 2 };

struct FilterState {
    u32 t, up, q;      // bound, upper end of the window, splitters
    u32 pool;          // entries taken from the spill pool
    u32 fail;          // a buffer was too small
    u32 K, gt, ties;   // the k-th key, keys above it, ties taken
    u32 kind;          // F_CLASS, F_AT_T (K == t), F_DONE (outputs written by k_fkth)
    u32 ndense;        // dense ranges listed
    u32 pad[6];
    u32 lcount[F_LISTS];
    u32 split[256];    // ascending, 0xFFFFFFFF past q
    u32 upr;           // units per range, which k_filter seldom needs
    u32 pad2[15];
    // the counters behind it: classes (F_REPS replicas), kept keys of the full units per range, dense ranges
    __host__ __device__ __forceinline__ u32* cls() const { return (u32*)(this + 1); }
    __host__ __device__ __forceinline__ u32* dtot() const { return cls() + F_REPS * F_CLASSES; }
    __host__ __device__ __forceinline__ u32* dlist() const { return dtot() + F_RANGES; }
};
size_t filter_state_bytes() { return sizeof(FilterState) + 4ull * (F_REPS * F_CLASSES + 2 * F_RANGES); }

// ---------------------------------------------------------------- sample
// Sample i is a key of stratum [i n / m, (i + 1) n / m), at a place mixed from i by xorshifts and multiplications
// with the shifts of xxHash's 32-bit finaliser and its first three primes.
__host__ __device__ __forceinline__ u32 sample_pos(u32 i, u64 n, int lm) {
    const u32 b = (u32)(((u64)i * n) >> lm), e = (u32)(((u64)(i + 1) * n) >> lm);
    u32 h = i * 0x9E3779B1u;
    h ^= h >> 15;
    h *= 0x85EBCA77u;
    h ^= h >> 13;
    h *= 0xC2B2AE3Du;
    h ^= h >> 16;
    return b + (u32)(((u64)h * (e - b)) >> 32);
}

// The stratum of the sample at slot s: those whose maximum is taken together lie far apart, as keys in a
// sorted or clustered vector are large together (2^28 ascending keys, k = 2^24: the list of k_fsplit took
// eight samples for each it needed and overflowed).
__device__ __forceinline__ u32 sample_stratum(u32 s, int lm) { return (s * 0x9E3779B1u) & ((1u << lm) - 1); }

template <class K>
__global__ __launch_bounds__(WG) void k_fsample(const u32* __restrict__ keys, u64 n, int lm, u32* __restrict__ sample,
                                                u32* __restrict__ sup, Ctrl* ctrl, FilterState* st,
                                                u32* __restrict__ rg, u32* __restrict__ rq, u32 upr) {
    const u32 g = blockIdx.x * WG + threadIdx.x;  // 2^lm / 4 threads, at least 2048
    u32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = keys[sample_pos(sample_stratum(4 * g + j, lm), n, lm)];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = K::to_ord(v[j]);
    *(u32x4*)(sample + 4 * g) = v;
    if (lm > 15) {  // the maxima of every 8 (2^17 samples) or 32 (2^19) of them
        const int lanes = lm == 17 ? 2 : 8;
        const u32 m = row_max_u32(max4(v), lanes);
        if ((threadIdx.x & (lanes - 1)) == 0) sup[g / lanes] = m;
    }
    static_assert(F_REPS * F_CLASSES <= 2048 && F_RANGES <= 2048 && sizeof(FilterState) / 4 <= 2048, "one counter per thread");
    if (g < F_REPS * F_CLASSES) st->cls()[g] = 0;
    if (g < F_RANGES) rg[g] = rq[g] = st->dtot()[g] = 0;
    if (g < sizeof(FilterState) / 4) ((u32*)st)[g] = g == offsetof(FilterState, upr) / 4 ? upr : 0u;
    if (g == 0) ws_head_begin(&ctrl->head);
}

// ---------------------------------------------------------------- bound and splitters
// LM 13, 15: the 2^LM samples in LDS.  Otherwise LG = LM - 14: 2^14 maxima of 2^LG samples each: their r'-th largest T0 is
// a lower bound of the samples', and those above it, 1.1 .. 1.4 r' for random samples, are all in
// ranges whose maximum exceeds T0.  The samples above T0 are listed in LDS and the bounds taken there.
template <int LM>
__global__ __launch_bounds__(FS_NT) void k_fsplit(const u32* __restrict__ sample, const u32* __restrict__ sup, u32 rp,
                                                  u32 rlo, u32 rhi, FilterState* st) {
    constexpr int LG = LM > 15 ? LM - 14 : 0;
    constexpr u32 HELD = LG ? 16384 : 1u << LM;
    __shared__ WgSel<FS_NT> L;
    __shared__ __align__(16) u32 el[wg_words<FS_NT>(HELD)];
    __shared__ __align__(16) u32 own_list[LG ? F_LIST_LDS : 1];
    __shared__ __align__(16) u32 srt[F_SORT];
    u32* list = LG ? own_list : el;
    const int t = threadIdx.x;
    wg_init<FS_NT>(L);
    constexpr int ni = HELD / (4 * FS_NT);
    wg_stage<FS_NT>(el, ni, [&](u32 e) { return *(const u32x4*)((LG ? sup : sample) + e); });
    u32 gt;
    const u32 T0 = wg_kth<FS_NT>([&](auto&& f) { wg_each(el, ni, f); }, rp, L, &gt);
    u32 hi = L.hi;
    if (t == 0) L.misc[8] = 0;
    __syncthreads();
    if constexpr (LG == 0) {  // from the samples again: the list takes their place in LDS
#pragma unroll 8
        for (u32 e = 4 * t; e < HELD; e += 4 * FS_NT) {
            const u32x4 x = *(const u32x4*)(sample + e);
            if (max4(x) > T0) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (x[j] > T0) list[atomicAdd(&L.misc[8], 1u)] = x[j];
            }
        }
    } else {
        u32 e = t * ni * 4;
        wg_each(el, ni, [&](const u32x4& m) {
#pragma unroll
            for (u32 j = 0; j < 4; ++j) {
                if (m[j] <= T0) continue;
                u32x4 x[(1 << LG) / 4];
#pragma unroll
                for (int i = 0; i < (1 << LG) / 4; ++i) x[i] = *(const u32x4*)(sample + ((e + j) << LG) + 4 * i);
#pragma unroll
                for (int i = 0; i < (1 << LG); ++i)
                    if (x[i / 4][i % 4] > T0) {
                        const u32 p = atomicAdd(&L.misc[8], 1u);
                        if (p < F_LIST_LDS) list[p] = x[i / 4][i % 4];
                    }
            }
            e += 4;
        });
    }
    __syncthreads();
    const u32 nl = LG ? min(L.misc[8], F_LIST_LDS) : L.misc[8];
    const bool all = nl == L.misc[8];  // else (tied or clustered samples) T0 is the bound, and any listed sample a splitter
    auto each = [&](auto&& f) {
        for (u32 i = t; i < nl; i += FS_NT) f(u32x4{list[i], 0, 0, 0});
    };
    if (all && nl <= F_SORT) {
        // few: all in descending order, two threads comparing one of them with half of the others.  At
        // 2^15 samples and 220 in the list this takes the place of two selections and a sort.
        if (t < 4 && nl + t < F_SORT) list[nl + t] = 0;
        __syncthreads();
        const u32 c = (u32)t >> 1, x = c < nl ? list[c] : 0u;
        u32 rank = 0;
        for (u32 j = 4 * ((u32)t & 1); j < nl; j += 8) {
            const u32x4 y = *(const u32x4*)(list + j);
#pragma unroll
            for (u32 i = 0; i < 4; ++i) rank += j + i < nl && (y[i] > x || (y[i] == x && j + i < c)) ? 1u : 0u;
        }
        rank += (u32)__builtin_amdgcn_mov_dpp((int)rank, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
        if ((t & 1) == 0 && c < nl) srt[rank] = x;
        __syncthreads();
        const u32 T = nl >= rp ? srt[rp - 1] : T0, tw = nl >= rhi ? srt[rhi - 1] : T;
        const u32 up = rlo >= 1 && nl >= rlo ? srt[rlo - 1] : hi;
        // each value of the window once: samples that tie at `up` may be as many as there are in the list,
        // and none would be left below them, where the k-th key lies
        const u32 y = (u32)t < nl ? srt[t] : 0u;
        const bool is = (u32)t < nl && y > T && y >= tw && y <= up && (t == 0 || srt[t - 1] != y);
        u32 q;
        const u32 p = wg_excl_scan<FS_NT>(is ? 1u : 0u, L.a, &q);
        q = min(q, F_SPLIT);
        if (is && p < q) st->split[q - 1 - p] = y;
        if (t < 256 && (u32)t >= q) st->split[t] = 0xFFFFFFFFu;
        if (t == 0) {
            st->t = T;
            st->up = up;
            st->q = q;
        }
        return;
    }
    __syncthreads();
    // the bound t; the window (tw, up] that almost surely holds the k-th key, where the splitters lie
    u32 T = T0, tw = T0, up = hi;
    if (all && nl >= rp) T = tw = wg_kth_between<FS_NT>(each, T0, hi, rp, L, &gt);
    __syncthreads();
    if (all && nl >= rhi) tw = wg_kth_between<FS_NT>(each, T, hi, rhi, L, &gt);
    __syncthreads();
    if (all && rlo >= 1 && nl >= rlo) up = wg_kth_between<FS_NT>(each, tw, hi, rlo, L, &gt);
    __syncthreads();
    // splitters: up to 254 samples of the window, in order.  Of those that tie at its ends, which may be
    // any number, one each; of the others first one from each of 252 equal parts of the window, so that
    // the classes come out alike, then any.
    if (t == 0) {
        u32 c = 0;
        if (up > T) L.cand[c++] = up;
        if (tw > T && tw < up) L.cand[c++] = tw;
        L.misc[8] = c;
    }
    __syncthreads();
    const float part = (float)(F_SPLIT - 2) / (float)max(up - tw, 1u);
    for (int pass = 0; pass < 2; ++pass) {
        for (u32 i = t; i < nl; i += FS_NT) {
            const u32 x = list[i];
            if (x <= tw || x >= up) continue;  // tw >= T
            u32* first = &L.hist[min((u32)((float)(x - tw) * part), F_SPLIT - 3)];  // 1 + the part's first sample
            if (pass ? *first == i + 1 : atomicCAS(first, 0u, i + 1) != 0) continue;
            const u32 p = atomicAdd(&L.misc[8], 1u);
            if (p < F_SPLIT) L.cand[p] = x;
        }
        __syncthreads();
    }
    const u32 q = min(L.misc[8], F_SPLIT);
    {  // the rank of each, four threads comparing it with a quarter of the others
        const u32 c = (u32)t >> 2, x = L.cand[c];
        u32 rank = 0;
        for (u32 j = 4 * ((u32)t & 3); j < q; j += 16) {
            const u32x4 y = *(const u32x4*)(L.cand + j);
#pragma unroll
            for (u32 i = 0; i < 4; ++i) rank += j + i < q && (y[i] < x || (y[i] == x && j + i < c)) ? 1u : 0u;
        }
        rank += (u32)__builtin_amdgcn_mov_dpp((int)rank, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
        rank += (u32)__builtin_amdgcn_mov_dpp((int)rank, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
        if ((t & 3) == 0) st->split[c < q ? rank : c] = c < q ? x : 0xFFFFFFFFu;
    }
    if (t == 0) {
        st->t = T;
        st->up = up;
        st->q = q;
    }
}

// ---------------------------------------------------------------- filter
// Classes of W kept keys x <= up at once (a search is a chain of LDS round trips): splitters below
// each, and whether it equals the next one.
template <int W>
__device__ __forceinline__ void class_of(const u32* sp, const u32* x, u32 (&c)[W]) {
#pragma unroll
    for (int u = 0; u < W; ++u) c[u] = 0;
#pragma unroll
    for (u32 step = 128; step; step >>= 1) {
        u32 s[W];
#pragma unroll
        for (int u = 0; u < W; ++u) s[u] = sp[c[u] + step - 1];
#pragma unroll
        for (int u = 0; u < W; ++u) c[u] += s[u] < x[u] ? step : 0u;
    }
    u32 s[W];
#pragma unroll
    for (int u = 0; u < W; ++u) s[u] = sp[c[u]];  // sp[255] is 0xFFFFFFFF, c <= q
#pragma unroll
    for (int u = 0; u < W; ++u) c[u] = 2 * c[u] + (s[u] == x[u] ? 1u : 0u);
}

// The compare domain of a raw key: unsigned for uint32.  A float32's bits compare as a signed integer
// against a bound that is not negative, whatever the key; below that the negative keys' low bits
// are flipped first.
template <class K>
struct FDomain;
template <>
struct FDomain<KeyU32> {
    using T = u32;
    static __device__ __forceinline__ T bound(u32 ord) { return ord; }
    static __device__ __forceinline__ u32 to_domain(u32 raw) { return raw; }
    static __device__ __forceinline__ bool converts(T) { return false; }
    static __device__ __forceinline__ u32 ordered(u32 x, bool) { return x; }
};
template <>
struct FDomain<KeyF32> {
    using T = int;
    static __device__ __forceinline__ T bound(u32 ord) { return (int)(ord ^ 0x80000000u); }
    static __device__ __forceinline__ u32 to_domain(u32 raw) { return raw ^ ((u32)((int)raw >> 31) & 0x7FFFFFFFu); }
    static __device__ __forceinline__ bool converts(T t) { return t < 0; }
    static __device__ __forceinline__ u32 ordered(u32 x, bool converted) {
        return converted ? x ^ 0x80000000u : KeyF32::to_ord(x);
    }
};

// Bound by the read stream where few keys are kept: a wave takes 2048 keys at a time (eight 16-byte
// loads per lane), and a 256-key load that holds none above t costs four instructions a lane.
// The others are counted with one ballot per key, placed in index order with one mask count per
// key and staged in the wave's LDS.  They leave, with their classes counted, when that is full:
// on this part a load is waited for together with the stores issued before it, so a wave that
// stored after every unit waited for a write's round trip each time (2^30 keys, 172 K kept: 694 us).
// A wave meets consecutive units, so sorted keys leave all they keep to a few of them, and what a full unit
// costs a wave shows in the call: it searches four classes at a time, and counts neighbours of one class
// with one atomic (2^26 ascending keys, k = 2^16: the pass 108 -> 87 us; 50 for random keys).
// Waves work alone, without a barrier in the loop.
template <class K>
__global__ __launch_bounds__(WG, 7) void k_filter(const u32* __restrict__ keys, u32 n, u32 nunits, int rounds, u32 wcap,
                                               u32 pool_at, u32 pool_cap, FilterState* st, u32* __restrict__ skeys,
                                               u32* __restrict__ sidx, u32* __restrict__ cnt, u32* __restrict__ base_of) {
    using D = FDomain<K>;
    using DT = typename D::T;
    __shared__ u32 sp[256], lh[F_CLASSES], sk[WG / WAVE][F_STAGE], si[WG / WAVE][F_STAGE];
    const int lane = threadIdx.x & (WAVE - 1), w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
    sp[threadIdx.x] = st->split[threadIdx.x];
    lh[threadIdx.x] = 0;
    lh[WG + threadIdx.x] = 0;
    const u32 t_ord = st->t, up = st->up;
    const DT t = D::bound(t_ord);
    const bool conv = D::converts(t);  // uniform
    u32 above = 0;
    __syncthreads();
    // the wave's share of the segments, filled from its start; what its units kept and where, one unit
    // per lane until 64 of them are written
    const u32 gbase = (blockIdx.x * (WG / WAVE) + w) * wcap;
    u32 gpos = 0, nrec = 0, my_unit = 0, my_cnt = 0, my_base = 0;
    u32 fill = 0, dst = 0, last = 0;  // staged keys, their first slot; what the last unit kept
    bool apart = false;               // the staged keys end where others were stored past the stage
    // classes of N keys per lane, those of `act` kept ones
    auto count_classes = [&](auto width, const u32* v, const bool* act, bool neighbours) {
        constexpr int N = decltype(width)::value;
        u32 c[N];
        class_of<N>(sp, v, c);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const bool in = act[u] && v[u] <= up;
            above += act[u] && v[u] > up ? 1u : 0u;
            if (neighbours) {  // of sorted keys share a class: the first lane's is counted with one atomic
                const u32 c0 = (u32)__builtin_amdgcn_readfirstlane((int)c[u]);
                const u64 same = __ballot(in && c[u] == c0);
                if (in && c[u] != c0) atomicAdd(&lh[c[u]], 1u);
                if (same && lane == 0) atomicAdd(&lh[c0], (u32)__popcll(same));
            } else if (in) {
                atomicAdd(&lh[c[u]], 1u);
            }
        }
    };
    auto flush = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own LDS writes
        __builtin_amdgcn_wave_barrier();
        for (u32 i0 = 0; i0 < fill; i0 += 2 * WAVE) {
            u32 v[2];
            bool act[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const u32 i = i0 + u * WAVE + lane;
                act[u] = i < fill;
                v[u] = act[u] ? sk[w][i] : 0u;
                if (act[u]) {
                    skeys[dst + i] = v[u];
                    sidx[dst + i] = si[w][i];
                }
            }
            count_classes(std::integral_constant<int, 2>(), v, act, false);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        fill = 0;
        apart = false;
    };
    auto write_units = [&]() {
        if ((u32)lane < nrec) {
            cnt[my_unit] = my_cnt;
            base_of[my_unit] = my_base;
            const u32 c = my_cnt & 0xFFFFu;
            if (c >= DENSE_UNIT) {
                const u32 r = my_unit / st->upr, had = atomicAdd(&st->dtot()[r], c);
                if (had <= DENSE_RANGE && had + c > DENSE_RANGE) st->dlist()[atomicAdd(&st->ndense, 1u)] = r;
            }
        }
        nrec = 0;
    };
    // a workgroup step is 4 * rounds consecutive units, the waves taking every fourth
    const u32 per = (u32)rounds * (WG / WAVE);
    for (u32 step = blockIdx.x; step * per < nunits; step += gridDim.x)
        for (int rd = 0; rd < rounds; ++rd) {
            const u32 unit = step * per + rd * (WG / WAVE) + w;
            if (unit >= nunits) break;  // uniform over the wave; no barrier in the loop
            if (nrec == WAVE) write_units();
            const u32 k0 = unit * F_UNIT;
            u32x4 x[8];
            u32 pads = 0;
            if (k0 + F_UNIT <= n) {  // uniform
#pragma unroll
                for (int b = 0; b < 8; ++b)
                    x[b] = __builtin_nontemporal_load((const u32x4*)(keys + k0) + b * WAVE + lane);
            } else {
                pads = k0 + F_UNIT - n;
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const u32 e = k0 + 4 * (b * WAVE + lane);
                    if (e + 4 <= n) x[b] = *(const u32x4*)(keys + e);
                    else
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[b][j] = e + j < n ? keys[e + j] : K::from_ord(0);  // the lowest key
                }
            }
            // behind the loads: what is waited for with them is the stores of the flush before
            if (apart || fill + last > F_STAGE) flush();
            if (conv) {
#pragma unroll
                for (int b = 0; b < 8; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[b][j] = D::to_domain(x[b][j]);
            }
            u32 c[8], kept = 0, eq = 0;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                c[b] = 0;
                const DT m = max(max((DT)x[b][0], (DT)x[b][1]), max((DT)x[b][2], (DT)x[b][3]));
                if (__ballot(m >= t)) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        c[b] += (u32)__popcll(__ballot((DT)x[b][j] > t));
                        eq += (DT)x[b][j] == t ? 1u : 0u;
                    }
                    kept += c[b];
                }
            }
            if (__ballot(eq)) {
                eq = (u32)__builtin_amdgcn_readlane((int)wave_incl_scan_u32(eq), WAVE - 1);
                if (t_ord == 0) eq -= pads;
            } else {
                eq = 0;
            }
            const bool spill = gpos + kept > wcap;  // rare: clustered keys go to the pool
            const bool staged = fill + kept <= F_STAGE && !spill;
            u32 base = gbase + gpos;
            last = kept;
            if (spill) {
                u32 at = 0;
                if (lane == 0) at = atomicAdd(&st->pool, kept);
                at = (u32)__builtin_amdgcn_readfirstlane((int)at);
                base = pool_at + at;
                if (at > pool_cap || kept > pool_cap - at) {
                    if (lane == 0) st->fail = 1;
                    kept = 0;
                }
            } else {
                gpos += kept;
            }
            if ((u32)lane == nrec) {
                my_unit = unit;
                my_cnt = kept | (eq << 16);
                my_base = kept ? base : 0u;
            }
            ++nrec;
            if (kept == 0) continue;
            if (!staged) apart = fill > 0;
            else if (fill == 0) dst = base;
            u32 at = staged ? fill : base;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                if (c[b] == 0) continue;
                u32 pos = at;  // this lane's first: the granule's kept keys of the lanes below
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const u64 m = __ballot((DT)x[b][j] > t);
                    pos = __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, pos));
                }
                u32 v[4];
                bool act[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    act[j] = (DT)x[b][j] > t;
                    v[j] = D::ordered(x[b][j], conv);
                    if (act[j]) {
                        const u32 id = k0 + 4 * (b * WAVE + lane) + j;
                        if (staged) {
                            sk[w][pos] = v[j];
                            si[w][pos] = id;
                        } else {
                            skeys[pos] = v[j];
                            sidx[pos] = id;
                        }
                        ++pos;
                    }
                }
                if (!staged) {
                    bool any = false;
#pragma unroll
                    for (int j = 0; j < 4; ++j) any |= act[j] && v[j] <= up;
                    if (__ballot(any)) count_classes(std::integral_constant<int, 4>(), v, act, true);
                    else above += (u32)act[0] + (u32)act[1] + (u32)act[2] + (u32)act[3];
                }
                at += c[b];
            }
            if (staged) fill += kept;
        }
    flush();
    write_units();
    above = wave_incl_scan_u32(above);
    if (lane == WAVE - 1 && above) atomicAdd(&lh[F_ABOVE], above);
    __syncthreads();
    u32* g = st->cls() + (blockIdx.x % F_REPS) * F_CLASSES;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const u32 c = lh[j * WG + threadIdx.x];
        if (c) atomicAdd(&g[j * WG + threadIdx.x], c);
    }
}

// ---------------------------------------------------------------- the k-th key's class
struct FClass {
    u32 kept;      // all kept keys
    u32 lo, hi;    // kept < k: K == t.  Otherwise the k-th key lies in (lo, hi], hi == lo + 1 once it is known
    u32 above, kk; // keys above hi, rank of the k-th key among those in (lo, hi]
    u32 in;        // keys in (lo, hi]
};
// Every thread of an NT-thread block; `lds` holds 8 words, `scratch` NT/64.  Ends with a barrier.
template <int NT>
__device__ __forceinline__ FClass find_class(const FilterState* st, u32 k, u32* lds, u32* scratch) {
    constexpr int PER = NT >= 512 ? 1 : (int)F_CLASSES / NT;
    u32 c[PER], s = 0, tot;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        c[j] = 0;
        const int b = (int)F_CLASSES - 1 - ((int)threadIdx.x * PER + j);
        if (b >= 0) {
            u32 r[F_REPS];
#pragma unroll
            for (int i = 0; i < F_REPS; ++i) r[i] = st->cls()[i * F_CLASSES + b];
#pragma unroll
            for (int i = 0; i < F_REPS; ++i) c[j] += r[i];
        }
        s += c[j];
    }
    u32 run = wg_excl_scan<NT>(s, scratch, &tot);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (run < k && run + c[j] >= k) {
            lds[0] = (u32)((int)F_CLASSES - 1 - ((int)threadIdx.x * PER + j));
            lds[1] = run;
            lds[2] = c[j];
        }
        run += c[j];
    }
    __syncthreads();
    FClass f;
    f.kept = tot;
    f.lo = f.hi = st->t;
    f.above = f.kk = f.in = 0;
    if (tot >= k) {
        const u32 b = lds[0], i = b >> 1;
        f.above = lds[1];
        f.in = lds[2];
        f.kk = k - f.above;
        if (b == F_ABOVE) {
            f.lo = st->up;
            f.hi = 0xFFFFFFFFu;
        } else if (b & 1) {
            f.hi = st->split[i];
            f.lo = f.hi - 1;
        } else {
            f.lo = i ? st->split[i - 1] : st->t;
            f.hi = i < st->q ? st->split[i] - 1 : st->up;
        }
    }
    return f;
}

// The kept keys of units [u0, u1) of a range, laid end to end (at most F_RUNITS units).
struct RangeLds {
    u32 pref[F_RUNITS + 1], base[F_RUNITS], eqp[F_RUNITS + 1];
    u32 scratch[WG / WAVE], lds[8];
};
// Fills the table; returns the keys kept (every thread).  Contains barriers.
__device__ __forceinline__ u32 range_open(RangeLds& R, const u32* __restrict__ cnt, const u32* __restrict__ base_of, u32 u0,
                                          u32 u1, u32* eq_out) {
    static_assert(F_RUNITS <= WG, "one unit per thread");
    const u32 u = u0 + threadIdx.x;
    const u32 c = u < u1 ? cnt[u] : 0u;
    if (threadIdx.x < F_RUNITS) R.base[threadIdx.x] = u < u1 ? base_of[u] : 0u;
    u32 tot, eq;
    const u32 ex = wg_excl_scan<WG>(c & 0xFFFFu, R.scratch, &tot);
    const u32 eqx = wg_excl_scan<WG>(c >> 16, R.scratch, &eq);
    if (threadIdx.x < F_RUNITS) {
        R.pref[threadIdx.x] = ex;
        R.eqp[threadIdx.x] = eqx;
    }
    if (threadIdx.x == 0) {
        R.pref[F_RUNITS] = tot;
        R.eqp[F_RUNITS] = eq;
    }
    __syncthreads();
    *eq_out = eq;
    return tot;
}
// Slots of the eight consecutive kept keys from e on (valid ones only below `tot`).
__device__ __forceinline__ void range_slots(const RangeLds& R, u32 e, u32 tot, u32 (&at)[8]) {
    u32 s = 0;
#pragma unroll
    for (u32 step = F_RUNITS / 2; step; step >>= 1)
        if (R.pref[s + step] <= e) s += step;
#pragma unroll
    for (u32 j = 0; j < 8; ++j) {
        const bool ok = e + j < tot;
        while (ok && R.pref[s + 1] <= e + j) ++s;
        at[j] = ok ? R.base[s] + (e + j - R.pref[s]) : 0u;
    }
}

// The units of the dense ranges, over the waves of the grid: f(range, unit, kept keys, first slot), every lane
// of the wave at once.
template <class F>
__device__ __forceinline__ void dense_units(const FilterState* st, u32 ndense, u32 nranges, u32 nunits, u32 upr,
                                            const u32* __restrict__ cnt, const u32* __restrict__ base_of, F&& f) {
    for (u32 j = blockIdx.x * (WG / WAVE) + threadIdx.x / WAVE; j < ndense * upr; j += nranges * (WG / WAVE)) {
        const u32 r = st->dlist()[j / upr], u = r * upr + j % upr;
        if (u < nunits) f(r, u, cnt[u] & 0xFFFFu, base_of[u]);
    }
}

// Writes, per range, the kept keys above the class (and those equal to it where it is one value); for the units
// of dense ranges the same in gq, above << 16 | equal.  2048 workgroups are one round of the chip at eight waves
// per SIMD, which more than 80 scalar registers do not allow (2^28 keys, k = 2^24: 49 us with 86, 40 with 80).
__global__ __launch_bounds__(WG) __attribute__((amdgpu_num_sgpr(80))) void k_fpick(FilterState* st, u32 k, u32 nranges, u32 nunits, u32 upr,
                                              const u32* __restrict__ cnt, const u32* __restrict__ base_of,
                                              const u32* __restrict__ skeys, u32* __restrict__ gq, u32* __restrict__ rg,
                                              u32* __restrict__ rq, u32 lcap, u32* __restrict__ lkey,
                                              u32* __restrict__ lrange) {
    __shared__ RangeLds R;
    const u32 r = blockIdx.x, u0 = r * upr, u1 = min(u0 + upr, nunits);
    const u32 ndense = st->ndense;
    const bool dense = ndense && st->dtot()[r] > DENSE_RANGE;  // uniform
    const FClass f = find_class<WG>(st, k, R.lds, R.scratch);
    u32 eq;
    const u32 tot = range_open(R, cnt, base_of, u0, u1, &eq);
    if (f.kept < k) {  // K == t, or the bound failed
        if (threadIdx.x == 0) {
            rg[r] = tot;
            rq[r] = eq;
        }
        return;
    }
    const bool known = f.hi - f.lo == 1;  // one value: counted, not listed
    u32 g = 0, q = 0;
    for (u32 e0 = dense ? tot : 0; e0 < tot; e0 += F_BATCH) {
        u32 at[8], x[8], in = 0;
        range_slots(R, e0 + 8 * threadIdx.x, tot, at);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = skeys[at[j]];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (e0 + 8 * threadIdx.x + j >= tot) x[j] = 0;
            g += x[j] > f.hi ? 1u : 0u;
            in += x[j] > f.lo && x[j] <= f.hi ? 1u : 0u;
        }
        q += in;
        if (known) continue;
        u32 n;
        const u32 ex = wg_excl_scan<WG>(in, R.scratch, &n);
        if (n == 0) continue;  // uniform
        const u32 list = (r + e0 / F_BATCH) % F_LISTS;
        if (threadIdx.x == 0) R.lds[4] = atomicAdd(&st->lcount[list], n);
        __syncthreads();
        u32 to = R.lds[4] + ex;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (x[j] > f.lo && x[j] <= f.hi) {
                if (to < lcap) {
                    lkey[list * lcap + to] = x[j];
                    lrange[list * lcap + to] = r;
                }
                ++to;
            }
        __syncthreads();
    }
    if (!dense) {
        u32 gs, qs;
        wg_excl_scan<WG>(g, R.scratch, &gs);
        wg_excl_scan<WG>(q, R.scratch, &qs);
        if (threadIdx.x == 0) {
            rg[r] = gs;
            rq[r] = known ? qs : 0u;
        }
    }
    const u32 lane = threadIdx.x & (WAVE - 1);
    dense_units(st, ndense, nranges, nunits, upr, cnt, base_of, [&](u32 rr, u32 unit, u32 c, u32 from) {
        u32 m = 0;  // above << 16 | in the class
        for (u32 j0 = 0; j0 < c; j0 += 8 * WAVE) {
            u32 x[8], in = 0;
#pragma unroll
            for (u32 u = 0; u < 8; ++u) x[u] = skeys[from + min(j0 + u * WAVE + lane, c - 1)];
#pragma unroll
            for (u32 u = 0; u < 8; ++u) {
                if (j0 + u * WAVE + lane >= c) x[u] = 0;  // neither above nor in the class
                m += x[u] > f.hi ? 0x10000u : 0u;
                in += x[u] > f.lo && x[u] <= f.hi ? 1u : 0u;
            }
            m += in;
            if (known) continue;
            const u32 inc = wave_incl_scan_u32(in), n = (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
            if (n == 0) continue;  // uniform over the wave
            const u32 list = (unit + j0 / (8 * WAVE)) % F_LISTS;
            u32 b = 0;
            if (lane == 0) b = atomicAdd(&st->lcount[list], n);
            u32 to = (u32)__builtin_amdgcn_readfirstlane((int)b) + inc - in;
#pragma unroll
            for (u32 u = 0; u < 8; ++u)
                if (x[u] > f.lo && x[u] <= f.hi) {
                    if (to < lcap) {
                        lkey[list * lcap + to] = x[u];
                        lrange[list * lcap + to] = DENSE_ENTRY | unit;
                    }
                    ++to;
                }
        }
        m = wave_incl_scan_u32(m);
        if (lane == WAVE - 1) {
            gq[unit] = known ? m : m & 0xFFFF0000u;
            if (m >> 16) atomicAdd(&rg[rr], m >> 16);
            if (known && (m & 0xFFFFu)) atomicAdd(&rq[rr], m & 0xFFFFu);
        }
    });
}

// ---------------------------------------------------------------- k-th key and range offsets
template <class K>
__global__ __launch_bounds__(FS_NT) void k_fkth(FilterState* st, u32 k, u32 nranges,
                                                u32* __restrict__ rg, u32* __restrict__ rq, u32 lcap,
                                                const u32* __restrict__ lkey, const u32* __restrict__ lrange, u32 upr,
                                                u32* __restrict__ gq, const u32* __restrict__ keys, u32 n,
                                                u32* __restrict__ out_keys, i64* __restrict__ out_idx,
                                                u32* __restrict__ d_kth) {
    __shared__ WgSel<FS_NT> L;
    __shared__ __align__(16) u32 el[wg_words<FS_NT>(32768)];
    __shared__ u32 lpref[F_LISTS + 1], lds[8];
    const int t = threadIdx.x, lane = t & (WAVE - 1), w = t / WAVE;
    wg_init<FS_NT>(L);
    constexpr int RPT = F_RANGES / FS_NT;
    static_assert(32768 + 2 * F_RANGES <= wg_words<FS_NT>(32768), "the ranges' counts behind the list");
    u32 g[RPT], q[RPT];  // loaded with the class counters: one round trip
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const u32 r = t * RPT + j;
        g[j] = r < nranges ? rg[r] : 0u;
        q[j] = r < nranges ? rq[r] : 0u;
    }
    const u32 in_list = t < (int)F_LISTS ? st->lcount[t] : 0u;
    const FClass f = find_class<FS_NT>(st, k, lds, L.a);
    u32 qs = 0, eqs;
#pragma unroll
    for (int j = 0; j < RPT; ++j) qs += q[j];
    wg_excl_scan<FS_NT>(qs, L.b, &eqs);
    u32 Kk = f.hi, gt = f.above, kind = F_CLASS;
    bool ok = st->fail == 0;
    if (f.kept < k) {
        kind = F_AT_T;
        gt = f.kept;
        ok = ok && (u64)f.kept + eqs >= k;
    } else if (f.hi - f.lo > 1) {
        if (t < (int)WAVE) {
            const u32 inc = wave_incl_scan_u32(in_list);
            lpref[t + 1] = inc;
            if (t == 0) lpref[0] = 0;
            lds[4 + 0] = 0;
        }
        __syncthreads();
        if (t < (int)F_LISTS && lpref[t + 1] - lpref[t] > lcap) lds[4] = 1;
        __syncthreads();
        const u32 m = lpref[F_LISTS];
        ok = ok && lds[4] == 0 && m == f.in;
        if (ok) {
            // f(i, slot, key) for every entry of the lists laid end to end, a wave per list, eight loads
            // in flight
            auto each_entry = [&](auto&& fn) {
                for (u32 l = w; l < F_LISTS; l += FS_NT / WAVE) {
                    const u32 c = lpref[l + 1] - lpref[l];
                    for (u32 i0 = 0; i0 < c; i0 += 8 * WAVE) {
                        u32 x[8];
#pragma unroll
                        for (u32 u = 0; u < 8; ++u) x[u] = lkey[l * lcap + min(i0 + u * WAVE + lane, c - 1)];
#pragma unroll
                        for (u32 u = 0; u < 8; ++u) {
                            const u32 i = i0 + u * WAVE + lane;
                            if (i < c) fn(lpref[l] + i, l * lcap + i, x[u]);
                        }
                    }
                }
            };
            const bool held = m <= 32768;
            if (held) {
                each_entry([&](u32 i, u32, u32 x) { el[i] = x; });
                __syncthreads();
            }
            Kk = wg_kth_between<FS_NT>(
                [&](auto&& fn) {
                    if (held)
                        for (u32 i = t; i < m; i += FS_NT) fn(u32x4{el[i], f.lo, f.lo, f.lo});
                    else
                        each_entry([&](u32, u32, u32 x) { fn(u32x4{x, f.lo, f.lo, f.lo}); });
                },
                f.lo + 1, f.hi, f.kk, L, &gt);
            gt += f.above;
            // the class's keys above K and equal to it, back to their ranges (and units of dense ones)
            u32* add = el + 32768;
            for (u32 i = t; i < 2 * F_RANGES; i += FS_NT) add[i] = 0;
            __syncthreads();
            each_entry([&](u32, u32 s, u32 x) {
                if (x < Kk) return;
                const bool gr = x > Kk;
                const u32 r = lrange[s];
                if (!(r & DENSE_ENTRY)) {
                    atomicAdd(&add[(gr ? 0u : F_RANGES) + r], 1u);
                    return;
                }
                // entries of a dense unit lie side by side: those of the first lane's together
                const u32 unit = r & ~DENSE_ENTRY, unit0 = (u32)__builtin_amdgcn_readfirstlane((int)unit), to = unit / upr;
                const u32 ng = (u32)__popcll(__ballot(unit == unit0 && gr)), nq = (u32)__popcll(__ballot(unit == unit0 && !gr));
                const bool lead = lane == __ffsll((unsigned long long)__ballot(true)) - 1;
                if (unit == unit0 && !lead) return;
                const u32 a = lead ? ng : (gr ? 1u : 0u), b = lead ? nq : (gr ? 0u : 1u);
                atomicAdd(&gq[unit], a << 16 | b);
                if (a) atomicAdd(&add[to], a);
                if (b) atomicAdd(&add[F_RANGES + to], b);
            });
            __syncthreads();
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                g[j] += add[t * RPT + j];
                q[j] += add[F_RANGES + t * RPT + j];
            }
        }
    }
    if (ok) {
        u32 gs = 0, tot;
        qs = 0;
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            gs += g[j];
            qs += q[j];
        }
        __syncthreads();
        u32 gr = wg_excl_scan<FS_NT>(gs, L.a, &tot), qr = wg_excl_scan<FS_NT>(qs, L.b, &tot);
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const u32 r = t * RPT + j;
            if (r < nranges) {
                rg[r] = gr;
                rq[r] = qr;
            }
            gr += g[j];
            qr += q[j];
        }
        if (t == 0) {
            st->K = Kk;
            st->gt = gt;
            st->ties = k - gt;
            st->kind = kind;
            if (d_kth) *d_kth = K::from_ord(Kk);
        }
        return;
    }
    // last resort: this workgroup selects from the keys, a wave per contiguous share of them
    __syncthreads();
    wg_init<FS_NT>(L);
    __syncthreads();
    const u32 share = (((n + FS_NT / WAVE - 1) / (FS_NT / WAVE)) + 255u) & ~255u;
    const u32 b0 = min(n, w * share), b1 = min(n, b0 + share);
    auto load = [&](u32 e) {  // a lane's four keys (0 past the share: its last granule may be partial)
        u32x4 x = {0, 0, 0, 0};
        if (e + 4 <= b1) {
            x = *(const u32x4*)(keys + e);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = K::to_ord(x[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e + j < b1) x[j] = K::to_ord(keys[e + j]);
        }
        return x;
    };
    Kk = wg_kth<FS_NT>(
        [&](auto&& fn) {
#pragma unroll 8
            for (u32 e = b0 + 4 * lane; e < b1; e += 4 * WAVE) fn(load(e));
        },
        k, L, &gt);
    if (t == 0) {
        st->kind = F_DONE;
        if (d_kth) *d_kth = K::from_ord(Kk);
    }
    if (!out_keys && !out_idx) return;
    u32 cg = 0, cq = 0;
    for (u32 e = b0 + 4 * lane; e < b1; e += 4 * WAVE) {
        const u32x4 x = load(e);
#pragma unroll
        for (u32 j = 0; j < 4; ++j) {
            cg += x[j] > Kk ? 1u : 0u;
            cq += e + j < b1 && x[j] == Kk ? 1u : 0u;
        }
    }
    cg = wave_incl_scan_u32(cg);
    cq = wave_incl_scan_u32(cq);
    __syncthreads();
    if (lane == WAVE - 1) {
        L.a[w] = cg;
        L.b[w] = cq;
    }
    __syncthreads();
    u32 tot;
    u32 gr = wave_totals_prefix<FS_NT>(L.a, &tot), qr = wave_totals_prefix<FS_NT>(L.b, &tot);
    const u32 ties = k - gt;
    for (u32 e0 = b0; e0 < b1; e0 += 4 * WAVE) {
        const u32 e = e0 + 4 * lane;
        const u32x4 x = load(e);
        u32 mg = 0, mq = 0;
#pragma unroll
        for (u32 j = 0; j < 4; ++j) {
            mg += x[j] > Kk ? 1u : 0u;
            mq += e + j < b1 && x[j] == Kk ? 1u : 0u;
        }
        const u32 mine = (mg << 16) | mq, inc = wave_incl_scan_u32(mine);
        u32 gb = gr + ((inc - mine) >> 16), qb = qr + ((inc - mine) & 0xFFFFu);
#pragma unroll
        for (u32 j = 0; j < 4; ++j) {
            const bool isg = x[j] > Kk, isq = e + j < b1 && x[j] == Kk;
            if (isg || (isq && qb < ties)) {
                const u32 p = gb + min(qb, ties);
                if (out_keys) out_keys[p] = K::from_ord(x[j]);
                if (out_idx) out_idx[p] = (i64)(e + j);
            }
            gb += isg ? 1u : 0u;
            qb += isq ? 1u : 0u;
        }
        const u32 all = (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
        gr += all >> 16;
        qr += all & 0xFFFFu;
    }
}

// ---------------------------------------------------------------- outputs
template <class K>
__global__ __launch_bounds__(WG) void k_fwrite(const FilterState* st, u32 nranges, u32 nunits, u32 upr,
                                               const u32* __restrict__ cnt, const u32* __restrict__ base_of,
                                               const u32* __restrict__ skeys, const u32* __restrict__ sidx,
                                               const u32* __restrict__ gq, const u32* __restrict__ rg,
                                               const u32* __restrict__ rq, const u32* __restrict__ keys, u32 n, u32 k,
                                               u32* __restrict__ out_keys, i64* __restrict__ out_idx) {
    __shared__ RangeLds R;
    __shared__ u32 sk[F_BATCH], si[F_BATCH];
    const u32 kind = st->kind, K0 = st->K, ties = st->ties, ndense = st->ndense;
    if (kind == F_DONE) return;
    u32 r = blockIdx.x, sub = 0, subs = 1;
    if (kind == F_AT_T) {
        // Only the ranges with outputs, several workgroups to each where they are few: ties at the
        // bound may all be taken from the first of the ranges.
        __shared__ u16 act[F_RANGES];
        constexpr u32 RPT = F_RANGES / WG;
        const u32 nr = nranges, r0 = threadIdx.x * RPT;
        u32 on = 0, na;
#pragma unroll
        for (u32 j = 0; j < RPT; ++j)
            if (r0 + j < nr) {
                const u32 at = r0 + j, nx = at + 1;
                if (nx == nr || rg[nx] != rg[at] || (rq[at] < ties && rq[nx] != rq[at])) on |= 1u << j;
            }
        u32 to = wg_excl_scan<WG>((u32)__popc(on), R.scratch, &na);
#pragma unroll
        for (u32 j = 0; j < RPT; ++j)
            if (on >> j & 1) act[to++] = (u16)(r0 + j);
        __syncthreads();
        subs = max(nr / na, 1u);  // na >= 1: the last range is in
        if (r >= na * subs) return;
        sub = r % subs;
        r = act[r / subs];
    }
    const u32 u0 = r * upr, u1 = min(u0 + upr, nunits);
    u32 g = rg[r], q = rq[r], eq;  // outputs before the next batch: above K0, and ties
    const u32 tot = range_open(R, cnt, base_of, u0, u1, &eq);
    if (kind == F_AT_T) {
        // Each unit by a wave alone.  Ties at the bound were counted, not kept: a unit that gives some
        // is read again; of the others all that was kept goes out.  (The workgroup in batches of 2048
        // keys, three barriers each, a range per workgroup: 23 us for 65536 ties among the first
        // 475 K of 2^24 keys.)
        const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
        for (u32 i = sub * (WG / WAVE) + w; i < u1 - u0; i += subs * (WG / WAVE)) {
            u32 gu = g + R.pref[i], qu = q + R.eqp[i];
            if (qu >= ties || R.eqp[i + 1] == R.eqp[i]) {
                const u32 c = R.pref[i + 1] - R.pref[i], to = gu + min(qu, ties), from = R.base[i];
                for (u32 j = lane; j < c && to + j < k; j += WAVE) {
                    if (out_keys) out_keys[to + j] = K::from_ord(skeys[from + j]);
                    if (out_idx) out_idx[to + j] = (i64)sidx[from + j];
                }
                continue;
            }
            const u32 k0 = (u0 + i) * F_UNIT + 4 * lane;
            u32x4 x[8];
#pragma unroll
            for (u32 b = 0; b < 8; ++b) {
                const u32 e = k0 + b * 4 * WAVE;
                if (e + 4 <= n) x[b] = *(const u32x4*)(keys + e);
                else
#pragma unroll
                    for (u32 j = 0; j < 4; ++j) x[b][j] = e + j < n ? keys[e + j] : 0u;
            }
#pragma unroll
            for (u32 b = 0; b < 8; ++b) {
                u32 mine = 0;  // above << 16 | ties
#pragma unroll
                for (u32 j = 0; j < 4; ++j) {
                    const u32 v = K::to_ord(x[b][j]);
                    mine += k0 + b * 4 * WAVE + j < n ? (v > K0 ? 0x10000u : (v == K0 ? 1u : 0u)) : 0u;
                }
                const u32 inc = wave_incl_scan_u32(mine);
                u32 gb = gu + ((inc - mine) >> 16), qb = qu + ((inc - mine) & 0xFFFFu);
#pragma unroll
                for (u32 j = 0; j < 4; ++j) {
                    const u32 v = K::to_ord(x[b][j]), e = k0 + b * 4 * WAVE + j;
                    const bool isg = e < n && v > K0, isq = e < n && v == K0;
                    if (isg || (isq && qb < ties)) {
                        const u32 p = gb + min(qb, ties);
                        if (p < k) {
                            if (out_keys) out_keys[p] = x[b][j];
                            if (out_idx) out_idx[p] = (i64)e;
                        }
                    }
                    gb += isg ? 1u : 0u;
                    qb += isq ? 1u : 0u;
                }
                const u32 all = (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
                gu += all >> 16;
                qu += all & 0xFFFFu;
            }
        }
        return;
    }
    const bool dense = ndense && st->dtot()[r] > DENSE_RANGE;  // uniform
    dense_units(st, ndense, nranges, nunits, upr, cnt, base_of, [&](u32 rr, u32 unit, u32 c, u32 from) {
        const u32 lane = threadIdx.x & (WAVE - 1), first = rr * upr, mine = gq[unit];
        if (mine == 0) return;
        u32 gs = 0, qs = 0;  // in the range's units before this one
        for (u32 i = lane; i < unit - first; i += WAVE) {
            const u32 m = gq[first + i];
            gs += m >> 16;
            qs += m & 0xFFFFu;
        }
        u32 gu = rg[rr] + (u32)__builtin_amdgcn_readlane((int)wave_incl_scan_u32(gs), WAVE - 1);
        u32 qu = rq[rr] + (u32)__builtin_amdgcn_readlane((int)wave_incl_scan_u32(qs), WAVE - 1);
        if (mine >> 16 == 0 && qu >= ties) return;
        for (u32 j0 = 0; j0 < c; j0 += 8 * WAVE) {
            u32 x[8], id[8];
#pragma unroll
            for (u32 u = 0; u < 8; ++u) {
                const u32 at = from + min(j0 + u * WAVE + lane, c - 1);
                x[u] = skeys[at];
                id[u] = sidx[at];
            }
#pragma unroll
            for (u32 u = 0; u < 8; ++u) {
                const bool ok = j0 + u * WAVE + lane < c, isg = ok && x[u] > K0, isq = ok && x[u] == K0;
                const unsigned long long mg = __ballot(isg), mq = __ballot(isq);
                const u32 gb = gu + __builtin_amdgcn_mbcnt_hi((u32)(mg >> 32), __builtin_amdgcn_mbcnt_lo((u32)mg, 0));
                const u32 qb = qu + __builtin_amdgcn_mbcnt_hi((u32)(mq >> 32), __builtin_amdgcn_mbcnt_lo((u32)mq, 0));
                if (isg || (isq && qb < ties)) {
                    const u32 p = gb + min(qb, ties);
                    if (p < k) {
                        if (out_keys) out_keys[p] = K::from_ord(x[u]);
                        if (out_idx) out_idx[p] = (i64)id[u];
                    }
                }
                gu += (u32)__popcll(mg);
                qu += (u32)__popcll(mq);
            }
        }
    });
    if (dense) return;
    q = min(q, ties);
    // a batch of 8 keys per thread in index order: those above K0 and the ties still to take
    auto emit = [&](const u32 (&x)[8], const u32 (&id)[8], u32 nv) {
        u32 c = 0;  // above << 16 | ties, among the thread's first nv keys
#pragma unroll
        for (u32 j = 0; j < 8; ++j) c += j < nv ? (x[j] > K0 ? 0x10000u : (x[j] == K0 ? 1u : 0u)) : 0u;
        u32 all;
        const u32 ex = wg_excl_scan<WG>(c, R.scratch, &all);
        const u32 rem = min(ties - q, F_BATCH);  // ties left for this batch
        u32 lg = ex >> 16, lq = ex & 0xFFFFu;
#pragma unroll
        for (u32 j = 0; j < 8; ++j) {
            if (j >= nv || x[j] < K0) continue;
            if (x[j] > K0 || lq < rem) {
                const u32 s = lg + min(lq, rem);
                sk[s] = K::from_ord(x[j]);
                si[s] = id[j];
            }
            lg += x[j] > K0 ? 1u : 0u;
            lq += x[j] == K0 ? 1u : 0u;
        }
        __syncthreads();
        const u32 took = min(all & 0xFFFFu, rem), m = (all >> 16) + took, to = g + q;
        for (u32 i = threadIdx.x; i < m && to + i < k; i += WG) {
            if (out_keys) out_keys[to + i] = sk[i];
            if (out_idx) out_idx[to + i] = (i64)si[i];
        }
        g += all >> 16;
        q += took;
        __syncthreads();
    };
    for (u32 e0 = 0; e0 < tot; e0 += F_BATCH) {
        const u32 e = e0 + 8 * threadIdx.x;
        u32 at[8], x[8], id[8];
        range_slots(R, e, tot, at);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] = skeys[at[j]];
            id[j] = sidx[at[j]];
        }
        emit(x, id, e < tot ? min(tot - e, 8u) : 0u);
    }
}

hipError_t filter_last_resort(const void* state, hipStream_t st, int* taken) {
    u32 kind = 0;
    hipError_t e = hipMemcpyAsync(&kind, &((const FilterState*)state)->kind, sizeof(kind), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    *taken = kind == F_DONE;
    return e;
}

hipError_t launch_filter(const FilterArgs& a, hipStream_t st) {
    FilterState* fs = (FilterState*)a.state;
    const u32 n = (u32)a.n, k = (u32)a.k;
    const u32 nunits = filter_units(a.n);
    // Units per range: about half a batch of kept keys, in 512 .. F_RANGES ranges (2^24 random keys, k = 2^16:
    // 61.6 us with 512, 64.1 with 1024; ascending ones 98 and 78), from 2^26 keys 1024 .. F_RANGES (95.6 and
    // 96.3; ascending 281 and 222).
    const u64 half = (u64)F_BATCH / 2 * nunits / std::max<u64>(a.kept, 1);
    const u64 fewest = nunits < (1u << 15) ? 512 : 1024;
    const u64 most = std::min<u64>((nunits + fewest - 1) / fewest, F_RUNITS);
    const u32 upr = (u32)std::max<u64>((nunits + F_RANGES - 1) / F_RANGES, std::min(most, half));
    const u32 nranges = (nunits + upr - 1) / upr;
    if (upr > F_RUNITS || (a.lm != 13 && a.lm != 15 && a.lm != 17 && a.lm != 19)) return hipErrorInvalidValue;
    const FilterGrid fg = filter_grid(a.n);
#define F_SPLIT_LAUNCH(LM)                                                                                          \
    hipLaunchKernelGGL((k_fsplit<LM>), dim3(1), dim3(FS_NT), 0, st, a.sample, a.sample + (1u << a.lm), a.rp, a.rlo, \
                       a.rhi, fs)
#define F_LAUNCH(K)                                                                                                     \
    do {                                                                                                                \
        hipLaunchKernelGGL((k_fsample<K>), dim3((1u << a.lm) / 4 / WG), dim3(WG), 0, st, a.keys, a.n, a.lm, a.sample,  \
                           a.sample + (1u << a.lm), a.ctrl, fs, a.rg, a.rq, upr);                                      \
        if (a.lm == 13) F_SPLIT_LAUNCH(13);                                                                            \
        else if (a.lm == 15) F_SPLIT_LAUNCH(15);                                                                       \
        else if (a.lm == 17) F_SPLIT_LAUNCH(17);                                                                       \
        else F_SPLIT_LAUNCH(19);                                                                                       \
        hipLaunchKernelGGL((k_filter<K>), dim3(fg.grid), dim3(WG), 0, st, a.keys, n, nunits, fg.rounds, a.wcap,        \
                           fg.grid * 4 * a.wcap, a.pool_cap, fs, a.skeys, a.sidx, a.cnt, a.base);                      \
        hipLaunchKernelGGL(k_fpick, dim3(nranges), dim3(WG), 0, st, fs, k, nranges, nunits, upr, a.cnt, a.base,        \
                           a.skeys, a.gq, a.rg, a.rq, a.lcap, a.lkey, a.lrange);                                       \
        hipLaunchKernelGGL((k_fkth<K>), dim3(1), dim3(FS_NT), 0, st, fs, k, nranges, a.rg, a.rq, a.lcap, a.lkey,       \
                           a.lrange, upr, a.gq, a.keys, n, (u32*)a.out_keys, a.out_idx, (u32*)a.d_kth);                \
        if (a.out_keys || a.out_idx)                                                                                   \
            hipLaunchKernelGGL((k_fwrite<K>), dim3(nranges), dim3(WG), 0, st, fs, nranges, nunits, upr, a.cnt, a.base, \
                               a.skeys, a.sidx, a.gq, a.rg, a.rq, a.keys, n, k, (u32*)a.out_keys, a.out_idx);          \
    } while (0)
    if (a.f32) F_LAUNCH(KeyF32);
    else F_LAUNCH(KeyU32);
#undef F_LAUNCH
#undef F_SPLIT_LAUNCH
    return hipGetLastError();
}

}  // namespace drtopk
