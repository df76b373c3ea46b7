// short.hip -- top-k of one vector in one to five launches, for calls in the library's own
// configuration (api.hip, short_plan): the delegate scheme of the general pipeline, with every
// selection done by one workgroup (wgselect.hpp) instead of a chain of histogram and select
// launches, each of which costs 4-5 us however little it does.
//
//  k_small   n <= 36864: the whole top-k in one workgroup.
//  otherwise delegate pass (sample.hip) -> [k_super ->] k_first -> k_collect -> k_final:
//  k_first   exact k-th largest delegate T and the k subranges that hold the top-k: every
//            delegate > T, then the lowest-id delegates == T (FindTopKRanges +
//            FillWithKElementsID, baseline+filter+beta+shuffle/radixselect.cuh:413-427,
//            :603-618).  More delegates than its LDS holds are selected through their own
//            delegates: the maxima of every 2^f consecutive ones (k_super), whose k largest
//            ranges hold the k largest delegates for the same reason that the k largest
//            subranges hold the k largest keys.
//  k_collect keys >= T of those subranges with their indices, a segment per workgroup
//            (CreateConcatenateRange_optimized, radixselect.cuh:1575-1607), counted into
//            buckets of their distance from T on the way.
//  k_final   second top-k over the concatenation and the index-ordered outputs
//            (radixselect.cuh:1411-1470, MultiGPU/radixselect.cuh:1355-1383), by one workgroup where
//            the concatenation fits its LDS; clustered and tied keys leave up to 2^24 of them, which
//            several workgroups first reduce to those that can be in the top k.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "wgselect.hpp"

namespace drtopk {

constexpr int SH_NT = 1024;

// ---------------------------------------------------------------- one workgroup
// Keys e .. e+3 of the input (n >= 4), ordered, 0 past n; the load is issued from a clamped address,
// so that no lane waits for it under a condition.
template <class K>
__device__ __forceinline__ u32x4 load_keys(const u32* __restrict__ keys, u32 e, u32 n) {
    u32x4 r = *(const u32x4*)(keys + (e + 4 <= n ? e : 0u));
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = e + j < n ? K::to_ord(r[j]) : 0u;
    if (e < n && e + 4 > n) {  // the partial last granule, key by key
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (e + j < n) r[j] = K::to_ord(keys[e + j]);
    }
    return r;
}

// The whole top-k of n <= CAP keys: one launch where the general pipeline takes thirteen or more.
template <class K, u32 CAP>
__global__ __launch_bounds__(SH_NT) void k_small(const u32* __restrict__ keys, u32 n, u32 k, WsHead* head,
                                                 u32* __restrict__ out_keys, i64* __restrict__ out_idx,
                                                 u32* __restrict__ d_kth) {
    __shared__ WgSel<SH_NT> L;
    __shared__ __align__(16) u32 el[wg_words<SH_NT>(CAP)];
    const int t = threadIdx.x;
    const int ni = wg_granules<SH_NT>(n);
    if (t == 0) ws_head_begin(head);
    wg_init<SH_NT>(L);
    if (n >= 4) {
        wg_stage<SH_NT>(el, ni, [&](u32 e) { return load_keys<K>(keys, e, n); });
    } else {
        u32x4 r = {0, 0, 0, 0};
        if (t == 0)
            for (u32 j = 0; j < n; ++j) r[j] = K::to_ord(keys[j]);
        *(u32x4*)(el + 4 * t) = r;
        __syncthreads();
    }
    u32 gt;
    const u32 K0 = wg_kth<SH_NT>([&](auto&& f) { wg_each(el, ni, f); }, k, L, &gt);
    if (t == 0 && d_kth) *d_kth = K::from_ord(K0);
    if (!out_keys && !out_idx) return;
    wg_emit<SH_NT>(el, ni, K0, gt, k - gt, L, [&](u32 p, u32 e, u32 x) {
        if (p >= k) return;
        if (out_keys) out_keys[p] = K::from_ord(x);
        if (out_idx) out_idx[p] = (i64)e;
    });
}

template <class K>
static void launch_small_t(const ShortArgs& a, hipStream_t st) {
#define SM_LAUNCH(C)                                                                                                \
    hipLaunchKernelGGL((k_small<K, C>), dim3(1), dim3(SH_NT), 0, st, a.keys, (u32)a.n, (u32)a.k, &a.ctrl->head, \
                       (u32*)a.out_keys, a.out_idx, (u32*)a.d_kth)
    if (a.n <= 4096) SM_LAUNCH(4096);
    else SM_LAUNCH(SMALL_N);
#undef SM_LAUNCH
}
hipError_t launch_small(const ShortArgs& a, hipStream_t st) {
    if (a.n > SMALL_N) return hipErrorInvalidValue;
    if (a.f32) launch_small_t<KeyF32>(a, st);
    else launch_small_t<KeyU32>(a, st);
    return hipGetLastError();
}

// ---------------------------------------------------------------- delegates of delegates
// Elements e .. e+3 of a workspace array of m elements whose allocation is padded to 16 bytes: one
// load from a clamped address, the elements at or past m read as 0.
__device__ __forceinline__ u32x4 load_padded(const u32* __restrict__ a, u32 e, u32 m) {
    u32x4 r = *(const u32x4*)(a + (e < m ? e : 0u));
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = e + j < m ? r[j] : 0u;
    return r;
}

// Maxima of every 2^f1 delegates, and of every 2^f2 of those (f2 > 0): 2 <= f1, f1 + f2 <= 8, a lane
// per four delegates.
__global__ __launch_bounds__(WG) void k_super(const u32* __restrict__ dvals, u32 S, int f1, u32* __restrict__ sup1,
                                              int f2, u32* __restrict__ sup2) {
    const u32 e = 4 * (blockIdx.x * WG + threadIdx.x);
    const int lane = threadIdx.x & (WAVE - 1);
    u32 m = max4(load_padded(dvals, e, S));
    for (int level = 0; level < 2; ++level) {
        const int f = level ? f1 + f2 : f1, g = 1 << (f - 2);  // lanes per range; its last lane gets the maximum
        m = group_max_last(m, g);
        if ((lane & (g - 1)) == g - 1 && ((e >> f) << f) < S) (level ? sup2 : sup1)[e >> f] = m;
        if (f2 == 0) break;
    }
}

// ---------------------------------------------------------------- first top-k and range selection
// Buckets that k_collect counts into, by the distance of a key from T; bucket 0 is T alone.  Equal ones of
// 2^sh values up to the largest delegate, which keep sorted keys apart; or, where few of the selected
// delegates lie in the upper 31/32 of that range (an outlier, a heavy tail: all other keys would share a
// bucket), 64 to each power of two (LOG_BUCKETS).
constexpr int DB_BITS = 6;
constexpr u32 LOG_BUCKETS = 64;
struct Buckets {
    int lo, hi;  // least and largest bits dropped from a distance
    __device__ __forceinline__ explicit Buckets(u32 sh)
        : lo(sh == LOG_BUCKETS ? 0 : (int)sh), hi(sh == LOG_BUCKETS ? 31 - DB_BITS : (int)sh) {}
    __device__ __forceinline__ u32 of(u32 d) const {  // d >= 1
        d -= 1;
        const int e = min(max(31 - DB_BITS - __clz((int)(d | 1u)), lo), hi);
        return min(1 + ((u32)(e - lo) << DB_BITS) + (d >> e), (u32)WS_BINS - 1);
    }
    // The least distance in bucket b, and the bucket's width less 1.
    __device__ __forceinline__ u32 from(u32 b, u32* span) const {
        *span = 0;
        if (b == 0) return 0;
        const u32 c = b - 1, e = lo == hi ? (u32)lo : (c >> (DB_BITS + 1) ? (c >> DB_BITS) - 1 : 0u);
        *span = ((b == WS_BINS - 1 ? 2u : 1u) << e) - 1;  // the last one takes what the range leaves over
        return 1 + ((c - ((e - (u32)lo) << DB_BITS)) << e);
    }
};
static_assert(((32 - DB_BITS + 1) << DB_BITS) + 1 < WS_BINS, "buckets of every distance");

// The k largest delegates, lowest ids first among equals.  With f1 == 0 from the S delegates at once;
// otherwise from the topmost maxima down (sup2 when f2 > 0, sup1, the delegates), each level
// selecting among the 2^f values of each of the k ranges the level above selected.  Every level has
// at most CAP values.  LISTK: the lists of selected ranges stay in LDS (k <= LISTK; a lone
// workgroup waits about 1 us for every trip to global memory and makes five a level without them);
// 0: in `tmp`, 3k words.
template <u32 CAP, u32 LISTK>
__global__ __launch_bounds__(SH_NT) void k_first(const u32* __restrict__ dvals, u32 S, int f1,
                                                 const u32* __restrict__ sup1, int f2, const u32* __restrict__ sup2,
                                                 u32 k, Ctrl* ctrl, u32* tmp, u32* sel_ids, u32* __restrict__ ghist) {
    __shared__ WgSel<SH_NT> L;
    __shared__ __align__(16) u32 el[wg_words<SH_NT>(CAP)];
    __shared__ u32 lists[LISTK ? 3 * LISTK : 1];
    const int t = threadIdx.x;
    if (t == 0) {
        ws_head_begin(&ctrl->head);
        ctrl->arrived = 0;
        ctrl->bin_lo = 0xFFFFFFFFu;
        ctrl->bin_hi = 0;
        L.misc[11] = 0;
    }
    wg_init<SH_NT>(L);
#pragma unroll
    for (int j = 0; j < WS_BINS / SH_NT; ++j) ghist[j * SH_NT + t] = 0;
    const int top = f2 ? 2 : (f1 ? 1 : 0);
    const u32 S1 = (S + (1u << f1) - 1) >> f1, S2 = (S1 + (1u << f2) - 1) >> f2;
    u32* picked = LISTK ? lists : tmp;  // numbers of a level's selected values
    const u32* list = nullptr;          // ranges the level above selected
    u32 T = 0;
    for (int level = top; level >= 0; --level) {
        const u32* a = level == 2 ? sup2 : (level == 1 ? sup1 : dvals);
        const u32 m = level == 2 ? S2 : (level == 1 ? S1 : S);
        const int f = level == top ? 0 : (level == 1 ? f2 : f1);
        const u32 X = level == top ? m : k << f;  // values of this level
        const int ni = wg_granules<SH_NT>(X);
        // value x is a[x] at the top, below it value x % 2^f of the list's range x >> f (f >= 2)
        auto id = [&](u32 x) { return level == top ? x : (list[x >> f] << f) + (x & ((1u << f) - 1)); };
        wg_stage<SH_NT>(el, ni, [&](u32 x) { return load_padded(a, x < X ? id(x) : m, m); });
        u32 gt;
        auto each = [&](auto&& f) { wg_each(el, ni, f); };
        if (level == top) T = wg_kth<SH_NT>(each, k, L, &gt);
        else T = wg_kth_between<SH_NT>(each, T, L.hi, k, L, &gt);  // the level above bounds this one's
        // the selected delegates in the upper 31/32 of their range
        const u32 range = L.hi - T;
        u32 far = 0;
        // the values' numbers first, then their ids all at once: reading the list where a value is
        // emitted would wait for it there
        u32* const to = top == 0 ? sel_ids : picked;
        wg_emit<SH_NT>(el, ni, T, gt, k - gt, L, [&](u32 p, u32 e, u32 x) {
            to[p] = e;
            far += x - T > range >> 5 ? 1u : 0u;
        });
        if (level == 0) {
            far = wave_incl_scan_u32(far);
            if ((t & (WAVE - 1)) == WAVE - 1 && far) atomicAdd(&L.misc[11], far);
        }
        __syncthreads();
        if (level == 0 && t == 0) {
            const u32 bits = range ? 32 - __clz((int)range) : 0;
            ctrl->first.result = T;
            ctrl->bucket_sh = L.misc[11] < k / 32 ? LOG_BUCKETS : (bits > 11 ? bits - 11 : 0);
        }
        if (top == 0) return;
        u32* next = picked + (level == 1 ? k : 2 * k);
        for (u32 p = t; p < k; p += SH_NT) (level == 0 ? sel_ids : next)[p] = id(picked[p]);
        list = next;
        __syncthreads();
    }
}

// ---------------------------------------------------------------- concatenation
// Workgroup s takes slots [s*4096, (s+1)*4096) of the selected subranges laid back to back (alpha >=
// 2), 16 consecutive slots per thread, and leaves the keys >= T in index order at [s*4096, ...), their
// count and how many equal T, and the largest of them.  The buckets leave out the keys equal to T, which
// would all go to one word (2^26 keys, one value and an outlier, k = 8192: 345 us for the call).
constexpr u32 COLLECT_TILE = 4096;

template <class K, bool IDX>
__global__ __launch_bounds__(WG) void k_collect(const u32* __restrict__ keys, u32 n, int alpha,
                                                const u32* __restrict__ sel_ids, u32 nsel, const Ctrl* ctrl,
                                                u32* __restrict__ skeys, u32* __restrict__ sidx,
                                                u32* __restrict__ cnt, u32* __restrict__ segmax,
                                                u32* __restrict__ ghist) {
    __shared__ u32 lh[WS_BINS];
    __shared__ u32 scratch[WG / WAVE], wmax[WG / WAVE];
    const u32 V = nsel << alpha, Lm = (1u << alpha) - 1;
    const u32 v0 = blockIdx.x * COLLECT_TILE + threadIdx.x * 16;
    u32 g[4];
    u32x4 r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const u32 vp = v0 + 4 * q;
        g[q] = (sel_ids[vp < V ? vp >> alpha : 0u] << alpha) + (vp & Lm);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = *(const u32x4*)(keys + (g[q] + 4 <= n ? g[q] : 0u));
    const u32 T = ctrl->first.result;
    const Buckets bk(ctrl->bucket_sh);
#pragma unroll
    for (int j = 0; j < WS_BINS / WG; ++j) lh[j * WG + threadIdx.x] = 0;
    u32 take = 0, eq = 0, mx = 0;  // take: bit per slot
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool in = v0 + 4 * q < V;  // V is a multiple of 4
        if (in && g[q] + 4 > n)          // the input's partial last granule
            for (u32 j = 0; j < 4; ++j)
                if (g[q] + j < n) r[q][j] = keys[g[q] + j];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32 o = K::to_ord(r[q][j]);
            r[q][j] = o;
            if (in && g[q] + j < n && o >= T) {
                take |= 1u << (4 * q + j);
                eq += o == T ? 1u : 0u;
                mx = max(mx, o);
            }
        }
    }
    u32 tot;  // survivors | keys equal to T << 16, at most 4096 each
    u32 slot = block_excl_scan_u32<WG>((u32)__popc(take) | (eq << 16), scratch, &tot) & 0xFFFFu;
    const u32 base = blockIdx.x * COLLECT_TILE;
    bool one = false;  // sorted or tied keys: the thread's are all in one bucket
    if (take == 0xFFFFu) {
        u32 mn = r[0][0];
#pragma unroll
        for (int q = 0; q < 4; ++q) mn = min(min(mn, min(r[q][0], r[q][1])), min(r[q][2], r[q][3]));
        const u32 b = mn != T ? bk.of(mn - T) : 0u;
        one = b ? b == bk.of(mx - T) : mx == T;
        if (one && b) atomicAdd(&lh[b], 16u);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (take & (1u << j)) {
            const u32 o = r[j >> 2][j & 3];
            skeys[base + slot] = o;
            if (IDX) sidx[base + slot] = g[j >> 2] + (u32)(j & 3);
            if (!one && o != T) atomicAdd(&lh[bk.of(o - T)], 1u);
            ++slot;
        }
    }
    mx = wave_max_last(mx);
    if ((threadIdx.x & (WAVE - 1)) == WAVE - 1) wmax[threadIdx.x / WAVE] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        cnt[blockIdx.x] = tot;
        segmax[blockIdx.x] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    }
#pragma unroll
    for (int j = 0; j < WS_BINS / WG; ++j) {
        const u32 c = lh[j * WG + threadIdx.x];
        if (c) atomicAdd(&ghist[j * WG + threadIdx.x], c);
    }
}

// ---------------------------------------------------------------- second top-k and extraction
constexpr u32 FIN_CAP = 12288;  // concatenation held in LDS (k <= 8192 random keys leave 11.4 K)
constexpr u32 FIN_WGS = 128;    // most workgroups of k_final
constexpr u32 FIN_ALONE = 32;   // segments from which one workgroup takes the keys it needs without the others

// One workgroup holds a concatenation of up to FIN_CAP keys in LDS, or, of a longer one, those from the k-th
// key's bucket up where they lie in few segments (sorted keys); the others then have nothing to do.  Else
// (up to 2^24 keys) all of them first reduce it: to the keys from the k-th key's bucket
// up, or, where fewer than k keys lie above T, to the outputs themselves, whose places the counts of the
// segments tell.  One workgroup alone read 2^19 .. 2^20 keys in 100 us and more (2^24 keys, a sixteenth of
// them large in one block, k = 8192: 203 us for the call).  The workgroup that arrives last goes on with
// what the others left; none waits.
template <class K>
__global__ __launch_bounds__(SH_NT) void k_final(u32* skeys, u32* sidx, const u32* __restrict__ cnt,
                                                 const u32* __restrict__ segmax, const u32* __restrict__ ghist, u32 nseg,
                                                 u32 k, Ctrl* ctrl, u32* rcnt, u32* __restrict__ out_keys,
                                                 i64* __restrict__ out_idx, u32* __restrict__ d_kth) {
    __shared__ WgSel<SH_NT> L;
    __shared__ u32 pref[SHORT_SEGS + 1];  // keys before each segment
    __shared__ __align__(16) u32 el[wg_words<SH_NT>(FIN_CAP)], ix[wg_words<SH_NT>(FIN_CAP)];
    const int t = threadIdx.x, lane = t & (WAVE - 1), w = t / WAVE;
    constexpr int SPT = SHORT_SEGS / SH_NT, PER = WS_BINS / SH_NT;
    const u32 T = ctrl->first.result;
    u32 hc[PER], pc[SPT];  // this thread's buckets and segments
#pragma unroll
    for (int j = 0; j < PER; ++j) hc[j] = ghist[WS_BINS - 1 - (t * PER + j)];
#pragma unroll
    for (int j = 0; j < SPT; ++j) pc[j] = (u32)(t * SPT + j) < nseg ? cnt[t * SPT + j] : 0u;
    if (t == 0) {
        L.misc[0] = 0xFFFFFFFFu;
        L.misc[8] = 0;
    }
    wg_init<SH_NT>(L);
    // keys before each segment, from the low halves of pc; returns their number
    auto set_pref = [&]() {
        u32 s = 0, tot;
#pragma unroll
        for (int j = 0; j < SPT; ++j) s += pc[j] & 0xFFFFu;
        u32 run = wg_excl_scan<SH_NT>(s, L.a, &tot);
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            pref[t * SPT + j] = run;
            run += pc[j] & 0xFFFFu;
        }
        if (t == SH_NT - 1) pref[SHORT_SEGS] = tot;
        return tot;
    };
    u32 C = set_pref(), Q, q = 0;  // entries, and those equal to T, which the buckets leave out
#pragma unroll
    for (int j = 0; j < SPT; ++j) q += pc[j] >> 16;
    wg_excl_scan<SH_NT>(q, L.b, &Q);
    if (t == SH_NT - 1) hc[PER - 1] += Q;
    wg_find_bin<SH_NT>(hc, k, L, L.misc);
    __syncthreads();
    if (C < k || L.misc[0] == 0xFFFFFFFFu) {  // not for valid input: every key of the top-k set is here
        if (t == 0 && blockIdx.x == 0) ctrl_fail(ctrl, ERR_CONCAT_SHORT);
        return;
    }
    const u32 kth_bin = L.misc[0], above = L.misc[1], in_bin = L.misc[2];
    __syncthreads();  // the selection below reuses misc, and no barrier need come before it
    const bool at_t = C - Q < k;  // fewer than k keys above T: ties at T fill the rest
    const u32 kk = k - above;
    u32 span;
    const u32 base = T + Buckets(ctrl->bucket_sh).from(kth_bin, &span);
    span = min(span, 0xFFFFFFFFu - base);
    // f(keys, indices, m, i) for every lane of each 256-slot step of segment s by one wave, `U` 16-byte
    // loads of each in flight; m the lane's valid keys from slot i on
    auto each_of = [&](u32 s, auto U, auto&& f) {
        constexpr u32 N = decltype(U)::value;
        const u32 c = pref[s + 1] - pref[s];
        const u32 *p = skeys + (u64)s * COLLECT_TILE, *pi = sidx + (u64)s * COLLECT_TILE;
        for (u32 i0 = 0; i0 < c; i0 += N * 4 * WAVE) {
            u32x4 x[N], y[N];
#pragma unroll
            for (u32 u = 0; u < N; ++u) {
                const u32 at = min(i0 + 4 * (u * WAVE + lane), COLLECT_TILE - 4);
                x[u] = *(const u32x4*)(p + at);
                y[u] = out_idx ? *(const u32x4*)(pi + at) : u32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (u32 u = 0; u < N; ++u) {
                const u32 i = i0 + 4 * (u * WAVE + lane);
                if (i0 + 4 * u * WAVE < c) f(x[u], y[u], i < c ? min(c - i, 4u) : 0u, i);
            }
        }
    };
    constexpr std::integral_constant<u32, 4> U4{};
    // the outputs of the segments first, first + step, .. for this wave: keys > K0, `gt` of them in all, and
    // the first ties; sg and sq hold the counts of each segment's keys above and equal to K0
    u32* sg = el;
    u32* sq = ix;
    auto write_segments = [&](u32 K0, u32 ties, u32 first, u32 step) {
        __syncthreads();
        {
            u32 g[SPT], q[SPT], gs = 0, qs = 0, tot;
#pragma unroll
            for (int j = 0; j < SPT; ++j) {
                g[j] = sg[t * SPT + j];
                q[j] = sq[t * SPT + j];
                gs += g[j];
                qs += q[j];
            }
            u32 gr = wg_excl_scan<SH_NT>(gs, L.a, &tot);
            u32 qr = wg_excl_scan<SH_NT>(qs, L.b, &tot);
#pragma unroll
            for (int j = 0; j < SPT; ++j) {
                // a segment with nothing to write is marked by an impossible first output
                const bool none = g[j] == 0 && (q[j] == 0 || qr >= ties);
                sg[t * SPT + j] = none ? 0xFFFFFFFFu : gr;
                sq[t * SPT + j] = qr;
                gr += g[j];
                qr += q[j];
            }
        }
        __syncthreads();
        for (u32 s = first; s < nseg; s += step) {
            u32 gr = sg[s], qr = sq[s];
            if (gr == 0xFFFFFFFFu) continue;
            each_of(s, U4, [&](const u32x4& x, const u32x4& y, u32 m, u32) {
                u32 mine = 0;  // above << 16 | ties
#pragma unroll
                for (u32 j = 0; j < 4; ++j) mine += j < m ? (x[j] > K0 ? 0x10000u : (x[j] == K0 ? 1u : 0u)) : 0u;
                if (__ballot(mine != 0) == 0) return;
                const u32 inc = wave_incl_scan_u32(mine);
                u32 gb = gr + ((inc - mine) >> 16), qb = qr + ((inc - mine) & 0xFFFFu);
#pragma unroll
                for (u32 j = 0; j < 4; ++j) {
                    if (j >= m || x[j] < K0) continue;
                    if (x[j] > K0 || qb < ties) {
                        const u32 p = gb + min(qb, ties);
                        if (out_keys && p < k) out_keys[p] = K::from_ord(x[j]);
                        if (out_idx && p < k) out_idx[p] = (i64)y[j];
                    }
                    gb += x[j] > K0 ? 1u : 0u;
                    qb += x[j] == K0 ? 1u : 0u;
                }
                const u32 all = (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
                gr += all >> 16;
                qr += all & 0xFFFFu;
            });
        }
    };
    bool held = C <= FIN_CAP, placed = false, tied = false;
    u32 f = 0, nv = 0;  // this thread's segments with a key >= base, and how many there are
    if (!held && !at_t) {
#pragma unroll
        for (int j = 0; j < SPT; ++j) f |= (u32)(t * SPT + j) < nseg && segmax[t * SPT + j] >= base ? 1u << j : 0u;
        f |= wg_excl_scan<SH_NT>((u32)__popc(f), L.a, &nv) << SPT;
        placed = above + in_bin <= FIN_CAP && nv <= FIN_ALONE;
    }
    if (held || placed) {
        if (blockIdx.x) return;
    }
    if (held) {
    } else if (placed) {
        // the keys from the bucket up fit and lie in few segments: counted per segment, then placed in order
        // as if they were the whole concatenation
        u32 at = f >> SPT;
#pragma unroll
        for (int j = 0; j < SPT; ++j)
            if (f >> j & 1) L.cand[at++] = (u32)(t * SPT + j);
        C = above + in_bin;
        const u32 ni = (u32)wg_granules<SH_NT>(C);
        for (u32 i = 0; i < ni; ++i) *(u32x4*)(el + 4 * (t * (ni | 1) + i)) = u32x4{0, 0, 0, 0};
        __syncthreads();
        for (u32 v = w; v < nv; v += SH_NT / WAVE) {
            u32 c = 0;
            each_of(L.cand[v], U4, [&](const u32x4& x, const u32x4&, u32 m, u32) {
#pragma unroll
                for (u32 j = 0; j < 4; ++j) c += j < m && x[j] >= base ? 1u : 0u;
            });
            c = wave_incl_scan_u32(c);
            if (lane == WAVE - 1) L.hist[v] = c;
        }
        __syncthreads();
        for (u32 v = w; v < nv; v += SH_NT / WAVE) {
            const u32 inc = wave_incl_scan_u32((u32)lane < v ? L.hist[lane & (FIN_ALONE - 1)] : 0u);
            u32 to = (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
            each_of(L.cand[v], U4, [&](const u32x4& x, const u32x4& y, u32 m, u32) {
                u32 c = 0;
#pragma unroll
                for (u32 j = 0; j < 4; ++j) c += j < m && x[j] >= base ? 1u : 0u;
                const u32 inc = wave_incl_scan_u32(c);
                u32 e = to + inc - c;
#pragma unroll
                for (u32 j = 0; j < 4; ++j)
                    if (j < m && x[j] >= base) {
                        const u32 o = e / (4 * ni), q = 4 * o * (ni | 1) + (e - 4 * ni * o);
                        el[q] = x[j];
                        ix[q] = y[j];
                        ++e;
                    }
                to += (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
            });
        }
        __syncthreads();
        wg_init<SH_NT>(L);
        __syncthreads();
        held = true;
    } else if (at_t) {
        if (t == 0 && blockIdx.x == 0 && d_kth) *d_kth = K::from_ord(T);
        if (!out_keys && !out_idx) return;
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            sg[t * SPT + j] = (pc[j] & 0xFFFFu) - (pc[j] >> 16);
            sq[t * SPT + j] = pc[j] >> 16;
        }
        write_segments(T, k - (C - Q), blockIdx.x * (SH_NT / WAVE) + w, gridDim.x * (SH_NT / WAVE));
        return;
    } else {
        // this workgroup's segments to their keys >= base, in place: a wave has read what it overwrites.  Counts
        // of keys | keys of the bucket << 16; its least and largest key tell whether it is one value.
        u32 blo = 0xFFFFFFFFu, bhi = 0;
        for (u32 s = blockIdx.x * (SH_NT / WAVE) + w; s < nseg; s += gridDim.x * (SH_NT / WAVE)) {
            u32 to = 0, b = 0;
            if (segmax[s] >= base) {
                u32 *p = skeys + (u64)s * COLLECT_TILE, *pi = sidx + (u64)s * COLLECT_TILE;
                each_of(s, U4, [&](const u32x4& x, const u32x4& y, u32 m, u32) {
                    u32 c = 0;
#pragma unroll
                    for (u32 j = 0; j < 4; ++j) c += j < m && x[j] >= base ? 1u : 0u;
                    const u32 inc = wave_incl_scan_u32(c);
                    u32 e = to + inc - c;
#pragma unroll
                    for (u32 j = 0; j < 4; ++j)
                        if (j < m && x[j] >= base) {
                            p[e] = x[j];
                            if (out_idx) pi[e] = y[j];
                            ++e;
                            if (x[j] - base <= span) {
                                ++b;
                                blo = min(blo, x[j]);
                                bhi = max(bhi, x[j]);
                            }
                        }
                    to += (u32)__builtin_amdgcn_readlane((int)inc, WAVE - 1);
                });
            }
            b = wave_incl_scan_u32(b);
            if (lane == WAVE - 1) rcnt[s] = to | b << 16;
        }
        bhi = wave_max_last(bhi);
        blo = ~wave_max_last(~blo);
        if (lane == WAVE - 1 && bhi >= base) {
            atomicMin(&ctrl->bin_lo, blo);
            atomicMax(&ctrl->bin_hi, bhi);
        }
        __threadfence();  // the keys and counts before the arrival
        __syncthreads();
        if (t == 0) L.misc[11] = atomicAdd(&ctrl->arrived, 1u);
        __syncthreads();
        if (L.misc[11] != gridDim.x - 1) return;
        __threadfence();
#pragma unroll
        for (int j = 0; j < SPT; ++j) pc[j] = (u32)(t * SPT + j) < nseg ? rcnt[t * SPT + j] : 0u;
        tied = __hip_atomic_load(&ctrl->bin_lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               __hip_atomic_load(&ctrl->bin_hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        C = set_pref();
        held = C <= FIN_CAP;
        __syncthreads();
    }
    // concatenation element e: its segment is the last one starting at or before e (an empty
    // segment shares its start with the next one, which is the one found)
    auto seg_of = [&](u32 e) {
        u32 lo = 0;
#pragma unroll 1
        for (u32 step = SHORT_SEGS / 2; step; step >>= 1)
            if (pref[lo + step] <= e) lo += step;
        return lo;
    };
    const int ni = wg_granules<SH_NT>(C);
    const u32 own = 4 * (u32)t * ((u32)ni | 1);  // this thread's elements in el and ix
    if (held && !placed) {  // every thread fetches its own consecutive elements
        const u32 e0 = 4 * (u32)(t * ni);
        u32 s = e0 < C ? seg_of(e0) : 0u;
#pragma unroll 2
        for (int i = 0; i < ni; ++i) {
            const u32 e = e0 + 4 * i;
            u32x4 x, y = {0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool ok = e + j < C;
                while (ok && pref[s + 1] <= e + j) ++s;
                const u32 at = ok ? s * COLLECT_TILE + (e + j - pref[s]) : 0u;
                x[j] = skeys[at];
                if (out_idx) y[j] = sidx[at];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = e + j < C ? x[j] : 0u;
            *(u32x4*)(el + own + 4 * i) = x;
            *(u32x4*)(ix + own + 4 * i) = y;
        }
    }
    u32 K0, gt;
    if (at_t) {
        K0 = T;
        gt = C - Q;
    } else if (span == 0 || tied) {
        K0 = tied ? __hip_atomic_load(&ctrl->bin_lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : base;
        gt = above;
    } else if (held && in_bin <= WgSel<SH_NT>::CAND) {
        // (base > T, so the zeros past the concatenation, which the bucket's count does not cover, are not in it)
#pragma unroll 1
        for (int i = 0; i < ni; ++i) wg_collect<SH_NT>(*(const u32x4*)(el + own + 4 * i), base, span, L);
        __syncthreads();
        u32 g;
        K0 = wg_rank<SH_NT>(in_bin, kk, L, &g);
        gt = above + g;
    } else {
        // more keys than can be ranked directly: from LDS, or read from memory on every pass
        K0 = wg_kth_between<SH_NT>(
            [&](auto&& f) {
                if (held) {
                    wg_each(el, ni, f);
                } else {
                    for (u32 s = w; s < nseg; s += SH_NT / WAVE)
                        each_of(s, U4, [&](const u32x4& x, const u32x4&, u32 m, u32) {
                            // (a key below the bucket, of which there are none left, for the slots past the end)
                            u32x4 v;
#pragma unroll
                            for (u32 j = 0; j < 4; ++j) v[j] = j < m ? x[j] : base - 1;
                            f(v);
                        });
                }
            },
            base, base + span, kk, L, &gt);
        gt += above;
    }
    if (t == 0 && d_kth) *d_kth = K::from_ord(K0);
    if (!out_keys && !out_idx) return;
    const u32 ties = k - gt;
    if (held) {
        __syncthreads();
        wg_emit<SH_NT>(el, ni, K0, gt, ties, L, [&](u32 p, u32 e, u32 x) {
            if (p >= k) return;
            if (out_keys) out_keys[p] = K::from_ord(x);
            if (out_idx) out_idx[p] = (i64)ix[own + (e - 4 * (u32)(t * ni))];
        });
        return;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        sg[t * SPT + j] = (pc[j] & 0xFFFFu) - (pc[j] >> 16);
        sq[t * SPT + j] = pc[j] >> 16;
    }
    if (span && !tied) {  // the bucket holds more than one value
        __syncthreads();
        for (u32 s = w; s < nseg; s += SH_NT / WAVE) {
            u32 g = 0, q = 0;
            each_of(s, U4, [&](const u32x4& x, const u32x4&, u32 m, u32) {
#pragma unroll
                for (u32 j = 0; j < 4; ++j) {
                    g += j < m && x[j] > K0 ? 1u : 0u;
                    q += j < m && x[j] == K0 ? 1u : 0u;
                }
            });
            g = wave_incl_scan_u32(g);
            q = wave_incl_scan_u32(q);
            if (lane == WAVE - 1) {
                sg[s] = g;
                sq[s] = q;
            }
        }
    }
    write_segments(K0, ties, w, SH_NT / WAVE);
}

u32 short_segments(u64 V) { return (u32)((V + COLLECT_TILE - 1) / COLLECT_TILE); }

hipError_t launch_short(const ShortArgs& a, hipStream_t st) {
    const u64 S = (a.n + (1ull << a.alpha) - 1) >> a.alpha, V = a.k << a.alpha;
    const u32 nseg = short_segments(V);
    const u64 S1 = (S + (1ull << a.f1) - 1) >> a.f1, S2 = (S1 + (1ull << a.f2) - 1) >> a.f2;
    if (a.k > SHORT_KMAX || a.alpha < 2 || nseg > SHORT_SEGS || S2 > SMALL_N || (a.k << a.f1) > SMALL_N ||
        (a.k << a.f2) > SMALL_N)
        return hipErrorInvalidValue;
    SampleArgs sa;
    sa.keys = a.keys; sa.n = a.n; sa.alpha = a.alpha; sa.beta = 1; sa.f32 = a.f32;
    sa.staged = 0; sa.posmode = 0; sa.fuse = 0;
    sa.dvals = a.dvals; sa.dpos = nullptr; sa.ghist = nullptr; sa.hshift = 0; sa.bins = 0; sa.ctrl = a.ctrl;
    hipError_t e = launch_sample(sa, st);
    if (e != hipSuccess) return e;
    if (a.f1)
        hipLaunchKernelGGL(k_super, dim3((unsigned)((S + 4 * WG - 1) / (4 * WG))), dim3(WG), 0, st, a.dvals, (u32)S,
                           a.f1, a.sup1, a.f2, a.sup2);
#define FI_LAUNCH(C, LK)                                                                                            \
    hipLaunchKernelGGL((k_first<C, LK>), dim3(1), dim3(SH_NT), 0, st, a.dvals, (u32)S, a.f1, a.sup1, a.f2, a.sup2, \
                       (u32)a.k, a.ctrl, a.skeys, a.sel_ids, a.ghist)
    // the concatenation's area (4k words at least), written after k_first, holds its lists
    const u64 most = std::max(S2, std::max(a.f1 ? a.k << a.f1 : 0, a.f2 ? a.k << a.f2 : 0));
    if (!a.f1 && S <= 12288) FI_LAUNCH(12288, 0);
    else if (a.f1 && most <= SHORT_LISTED && a.k <= SHORT_LISTED / 5) FI_LAUNCH(SHORT_LISTED, SHORT_LISTED / 5);
    else FI_LAUNCH(SMALL_N, 0);
#undef FI_LAUNCH
    const bool out = a.out_keys || a.out_idx;
    // a wave per segment, where there can be more keys than one workgroup holds
    const u32 fin = V <= FIN_CAP ? 1 : std::min(FIN_WGS, (nseg + SH_NT / WAVE - 1) / (SH_NT / WAVE));
#define CO_LAUNCH(K, I)                                                                                               \
    hipLaunchKernelGGL((k_collect<K, I>), dim3(nseg), dim3(WG), 0, st, a.keys, (u32)a.n, a.alpha, a.sel_ids, (u32)a.k, \
                       a.ctrl, a.skeys, a.sidx, a.cnt, a.segmax, a.ghist)
#define FN_LAUNCH(K)                                                                                                  \
    hipLaunchKernelGGL((k_final<K>), dim3(fin), dim3(SH_NT), 0, st, a.skeys, a.sidx, a.cnt, a.segmax, a.ghist, nseg, \
                       (u32)a.k, a.ctrl, a.rcnt, (u32*)a.out_keys, a.out_idx, (u32*)a.d_kth)
    if (a.f32) {
        if (out) CO_LAUNCH(KeyF32, true); else CO_LAUNCH(KeyF32, false);
        FN_LAUNCH(KeyF32);
    } else {
        if (out) CO_LAUNCH(KeyU32, true); else CO_LAUNCH(KeyU32, false);
        FN_LAUNCH(KeyU32);
    }
#undef CO_LAUNCH
#undef FN_LAUNCH
    return hipGetLastError();
}

}  // namespace drtopk
