// wgselect.hpp -- top-k by one workgroup: the k-th largest of an array in LDS, and the index-ordered
// emission of the top-k set.
//
// The k-th largest is found by linear buckets over the keys' own range: a pass counts
// (key - min) >> shift into 2048 LDS bins, so it resolves 11 bits of the range the keys really
// span (FindKBucket's refinement, bucketselect_combined.cuh:200-216, with power-of-two bucket
// widths).  One pass usually leaves a few dozen keys in the k-th key's bin; those are ranked
// against each other directly.  Tied or skewed keys refine the bin again, at most three passes
// in all.
//
// A CU issues one wave instruction a cycle, so what bounds a lone workgroup is instructions per key
// (about 20 here) and the fixed cost of barriers and LDS round trips (about 2 us per selection).
// Every thread owns consecutive elements, so that the emission ranks a thread's keys with one scan
// per workgroup; one scan per 256 keys took three times as long (13.6 K cycles for 32768 keys).
// Passes are short rolled loops: unrolled over keys in registers they ran no faster.
#pragma once

#include "common.hpp"

namespace drtopk {

constexpr int WS_BINS = 2048;

template <int NT>
struct WgSel {
    static constexpr int NW = NT / WAVE;
    static_assert(NW <= 16 && (NW & (NW - 1)) == 0, "wave totals are reduced within one 16-lane row");
    static constexpr u32 CAND = NT / 4;  // keys ranked directly once the k-th key's bin holds no more
    u32 hist[WS_BINS];
    __align__(16) u32 cand[CAND];  // zero past the candidates
    u32 a[NW], b[NW], c[NW];  // per-wave values
    u32 misc[12];      // two sets of (bin, keys above it, keys in it), then candidates, k-th key, keys above
    u32 hi;            // wg_kth: the largest key
};

__device__ __forceinline__ u32 max4(const u32x4& v) { return max(max(v[0], v[1]), max(v[2], v[3])); }

// Exclusive prefix over the wave totals a[0..NT/64) (NT/64 <= 16) at wave w, and their sum, without
// an unrolled loop over the waves.
template <int NT>
__device__ __forceinline__ u32 wave_totals_prefix(const u32* a, u32* total) {
    constexpr int NW = NT / WAVE;
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    const u32 x = lane < NW ? a[lane & (NW - 1)] : 0u;
    const u32 inc = wave_incl_scan_u32(x);
    *total = (u32)__builtin_amdgcn_readlane((int)inc, NW - 1);
    return (u32)__builtin_amdgcn_readlane((int)(inc - x), w);
}

// block_excl_scan_u32 in a third of its code.
template <int NT>
__device__ __forceinline__ u32 wg_excl_scan(u32 v, u32* scratch, u32* total) {
    const u32 inc = wave_incl_scan_u32(v);
    if ((threadIdx.x & (WAVE - 1)) == WAVE - 1) scratch[threadIdx.x / WAVE] = inc;
    __syncthreads();
    const u32 off = wave_totals_prefix<NT>(scratch, total);
    __syncthreads();
    return off + inc - v;
}

// A workgroup's m elements in LDS: thread t owns the ni = wg_granules(m) granules of four elements
// from element t*ni*4 on, at word t*stride*4; an odd number of granules between threads keeps a
// wave's 16-byte reads off each other's banks.  Elements past m are 0.
template <int NT>
__device__ __forceinline__ int wg_granules(u32 m) {
    return (int)((m + NT * 4 - 1) / (NT * 4));
}
// Words of LDS for up to m elements.
template <int NT>
constexpr u32 wg_words(u32 m) {
    const u32 ni = (m + NT * 4 - 1) / (NT * 4);
    return NT * 4 * (ni | 1);
}
// Fills `el` with m elements: fetch(e) returns elements e .. e+3 (e a multiple of 4, any value up to
// the 4 * NT * ni'th; 0 past m), called with consecutive e in consecutive lanes.
template <int NT, class F>
__device__ __forceinline__ void wg_stage(u32* el, int ni, F&& fetch) {
    const u32 inv = (1u << 18) / (u32)ni + 1, stride = (u32)ni | 1;  // exact for ni <= 15: g < 2^14
#pragma unroll 4
    for (int i = 0; i < ni; ++i) {
        const u32 g = (u32)(i * NT) + threadIdx.x, o = (g * inv) >> 18;
        *(u32x4*)(el + 4 * (o * stride + (g - o * (u32)ni))) = fetch(4 * g);
    }
    __syncthreads();
}

// Thread t's share of a histogram of WS_BINS bins, read from the top: bins WS_BINS-1 - t*PER
// downwards, c[] their counts.  Finds the bin that holds the key of rank kk from the top and stores
// (bin, keys above it, keys in it) in M[0..2], which stay as they are when the bins hold fewer keys.
// A barrier has to come before M is read.
template <int NT>
__device__ __forceinline__ void wg_find_bin(const u32 (&c)[WS_BINS / NT], u32 kk, WgSel<NT>& L, u32* M) {
    constexpr int PER = WS_BINS / NT;
    u32 s = 0, tot;
#pragma unroll
    for (int j = 0; j < PER; ++j) s += c[j];
    const u32 inc = wave_incl_scan_u32(s);
    if ((threadIdx.x & (WAVE - 1)) == WAVE - 1) L.c[threadIdx.x / WAVE] = inc;
    __syncthreads();
    u32 run = wave_totals_prefix<NT>(L.c, &tot) + inc - s;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (run < kk && run + c[j] >= kk) {
            M[0] = (u32)(WS_BINS - 1 - ((int)threadIdx.x * PER + j));
            M[1] = run;
            M[2] = c[j];
        }
        run += c[j];
    }
}

// The key of rank kk from the top among cand[0..cnt) (cnt <= CAND) and the candidates above it: four
// threads per candidate, each comparing it with a quarter of them.  Empties the list.
template <int NT>
__device__ __forceinline__ u32 wg_rank(u32 cnt, u32 kk, WgSel<NT>& L, u32* above) {
    const u32 c = threadIdx.x >> 2;
    if (c < cnt) {
        const u32 x = L.cand[c];
        u32 ge = 0;  // greater << 16 | equal; the zeros past cnt are neither (a bin of zeros alone is one value wide)
        for (u32 j = 4 * (threadIdx.x & 3); j < cnt; j += 16) {
            const u32x4 y = *(const u32x4*)(L.cand + j);
#pragma unroll
            for (int q = 0; q < 4; ++q) ge += y[q] > x ? 0x10000u : (y[q] == x ? 1u : 0u);
        }
        ge += (u32)__builtin_amdgcn_mov_dpp((int)ge, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
        ge += (u32)__builtin_amdgcn_mov_dpp((int)ge, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
        const u32 g = ge >> 16, e = ge & 0xFFFFu;
        if (g < kk && kk <= g + e) {  // equal candidates store the same values
            L.misc[9] = x;
            L.misc[10] = g;
        }
    }
    __syncthreads();
    if (threadIdx.x < WgSel<NT>::CAND) L.cand[threadIdx.x] = 0;
    *above = L.misc[10];
    return L.misc[9];
}

// Appends the keys of x in [base, base + span] to the candidates (no more than fit; the caller has
// counted them): one test for the four, as few granules hold any.
template <int NT>
__device__ __forceinline__ void wg_collect(const u32x4& x, u32 base, u32 span, WgSel<NT>& L) {
    if (min(min(x[0] - base, x[1] - base), min(x[2] - base, x[3] - base)) <= span) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (x[j] - base <= span) {
                const u32 p = atomicAdd(&L.misc[8], 1u);
                if (p < WgSel<NT>::CAND) L.cand[p] = x[j];
            }
    }
}

// Histogram and candidate list, zero between selections; a barrier has to follow.
template <int NT>
__device__ __forceinline__ void wg_init(WgSel<NT>& L) {
#pragma unroll
    for (int j = 0; j < WS_BINS / NT; ++j) L.hist[j * NT + threadIdx.x] = 0;
    if (threadIdx.x < WgSel<NT>::CAND) L.cand[threadIdx.x] = 0;
}

// The k-th largest key of the keys that it(f) passes to f, four at a time, in any order (it must
// visit the same keys every time and contain no barrier); at least k of them lie in [lo, hi], none
// above.  Every thread of the workgroup calls this; all return the same key, *gt = keys greater
// than it.  Keys outside [lo, hi] cost two instructions a pass.
template <int NT, class It>
__device__ __forceinline__ u32 wg_kth_between(It&& it, u32 lo, u32 hi, u32 k, WgSel<NT>& L, u32* gt) {
    constexpr int PER = WS_BINS / NT;
    const int t = threadIdx.x;
    u32 base = lo, span = hi - lo, above = 0, kk = k;
    for (int pass = 0; span; ++pass) {
        // alternate sets: a wave still reading one pass's result never meets the next pass's
        u32* M = L.misc + 4 * (pass & 1);
        const int bits = 32 - __clz((int)span);
        const int sh = bits > 11 ? bits - 11 : 0;
        // Ties, or keys that an outlier leaves in one bin, would queue on one LDS word, 128 cycles a wave
        // instruction: where a quarter of a wave's first keys share a bin, it counts that one in a register.
        const u32 bins = span >> sh;
        u32 heavy = 0, z = 0;
        int mode = -1;
        it([&](const u32x4& x) {
            if (mode < 0) {
                const u32 b = (x[0] - base) >> sh;
                heavy = (u32)__builtin_amdgcn_readfirstlane((int)b);
                mode = heavy <= bins && __popcll(__ballot(b == heavy)) >= WAVE / 4 ? 1 : 0;
            }
            if (mode) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const u32 d = x[j] - base, b = d >> sh;
                    const bool in = d <= span;
                    z += in && b == heavy ? 1u : 0u;
                    if (in && b != heavy) atomicAdd(&L.hist[b], 1u);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const u32 d = x[j] - base;
                    if (d <= span) atomicAdd(&L.hist[d >> sh], 1u);
                }
            }
        });
        if (__ballot(mode > 0)) {
            const u32 h0 = (u32)__builtin_amdgcn_readfirstlane((int)heavy);
            const u32 all = wave_incl_scan_u32(heavy == h0 ? z : 0u);
            if ((t & (WAVE - 1)) == WAVE - 1 && all) atomicAdd(&L.hist[h0], all);
            if (heavy != h0 && z) atomicAdd(&L.hist[heavy], z);  // lanes that `it` visits apart
        }
        if (t == 0) {
            M[0] = 0;
            L.misc[8] = 0;  // candidates collected
        }
        __syncthreads();
        u32 c[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int b = WS_BINS - 1 - (t * PER + j);
            c[j] = L.hist[b];
            L.hist[b] = 0;
        }
        wg_find_bin<NT>(c, kk, L, M);
        __syncthreads();
        above += M[1];
        kk -= M[1];
        const u32 cnt = M[2];
        base += M[0] << sh;
        span = min((1u << sh) - 1u, hi - base);  // a top bin past 2^32 must not wrap round to low keys
        if (span && cnt <= WgSel<NT>::CAND) {
            it([&](const u32x4& x) { wg_collect<NT>(x, base, span, L); });
            __syncthreads();
            u32 g;
            base = wg_rank<NT>(cnt, kk, L, &g);
            above += g;
            break;
        }
    }
    *gt = above;
    return base;
}

// The k-th largest of the keys that it(f) visits (1 <= k <= their number) and the largest, L.hi.
// Padding keys of value 0 may be visited: they rank below or equal to every key.
template <int NT, class It>
__device__ __forceinline__ u32 wg_kth(It&& it, u32 k, WgSel<NT>& L, u32* gt) {
    constexpr int NW = WgSel<NT>::NW;
    const int t = threadIdx.x, lane = t & (WAVE - 1), w = t / WAVE;
    // the range of the keys above 0 (0 - 1 wraps to the largest value and drops out of the minimum)
    // and how many they are
    u32 mx = 0, mn = 0xFFFFFFFFu, nz = 0;
    it([&](const u32x4& x) {
        mx = max(mx, max4(x));
        mn = min(min(mn, min(x[0] - 1u, x[1] - 1u)), min(x[2] - 1u, x[3] - 1u));
#pragma unroll
        for (int j = 0; j < 4; ++j) nz += x[j] ? 1u : 0u;
    });
    mx = wave_max_last(mx);
    mn = ~wave_max_last(~mn);
    const u32 inc = wave_incl_scan_u32(nz);
    if (lane == WAVE - 1) {
        L.a[w] = mx;
        L.b[w] = ~mn;
        L.c[w] = inc;
    }
    __syncthreads();
    const u32 hi = (u32)__builtin_amdgcn_readfirstlane((int)row_max_u32(L.a[lane & (NW - 1)], NW));
    const u32 lo = ~(u32)__builtin_amdgcn_readfirstlane((int)row_max_u32(L.b[lane & (NW - 1)], NW)) + 1u;
    u32 n;
    wave_totals_prefix<NT>(L.c, &n);
    if (t == 0) L.hi = hi;
    if (n < k) {  // the rest are zeros
        *gt = n;
        __syncthreads();
        return 0;
    }
    if (lo == hi) {  // one value (and zeros): the bins would serialise on one LDS address
        *gt = 0;
        __syncthreads();
        return hi;
    }
    return wg_kth_between<NT>(it, lo, hi, k, L, gt);
}

// This thread's staged elements, four at a time.
template <class F>
__device__ __forceinline__ void wg_each(const u32* el, int ni, F&& f) {
    const u32* mine = el + 4 * threadIdx.x * ((u32)ni | 1);
#pragma unroll 2
    for (int i = 0; i < ni; ++i) f(*(const u32x4*)(mine + 4 * i));
}

// Calls emit(pos, e, key) for every staged element > K and for the first `ties` elements == K (of
// all the elements, `gt` of them > K), pos = rank among the emitted ones in element order.  Every
// thread of the workgroup calls this; a barrier has to follow before L is used again.
template <int NT, class F>
__device__ __forceinline__ void wg_emit(const u32* el, int ni, u32 K, u32 gt, u32 ties, WgSel<NT>& L, F&& emit) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    u32 c = 0;
    wg_each(el, ni, [&](const u32x4& x) {
#pragma unroll
        for (int j = 0; j < 4; ++j) c += x[j] >= K ? 1u : 0u;
    });
    u32 inc = wave_incl_scan_u32(c);
    if (lane == WAVE - 1) L.a[w] = inc;
    __syncthreads();
    u32 tot;
    u32 pos = wave_totals_prefix<NT>(L.a, &tot) + inc - c;
    u32 e = threadIdx.x * (u32)ni * 4;
    if (tot == gt + ties) {  // uniform: every tie is taken
        wg_each(el, ni, [&](const u32x4& x) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (x[j] >= K) emit(pos++, e + (u32)j, x[j]);
            e += 4;
        });
        return;
    }
    u32 g = 0;
    wg_each(el, ni, [&](const u32x4& x) {
#pragma unroll
        for (int j = 0; j < 4; ++j) g += x[j] > K ? 1u : 0u;
    });
    inc = wave_incl_scan_u32(g);
    if (lane == WAVE - 1) L.b[w] = inc;
    __syncthreads();
    const u32 gb = wave_totals_prefix<NT>(L.b, &tot) + inc - g;
    u32 qb = pos - gb;  // ties before this thread's elements
    if (g == 0 && qb >= ties) return;
    pos = gb + min(qb, ties);
    wg_each(el, ni, [&](const u32x4& x) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (x[j] >= K) {
                if (x[j] > K || qb < ties) emit(pos++, e + (u32)j, x[j]);
                qb += x[j] == K ? 1u : 0u;
            }
        }
        e += 4;
    });
}

}  // namespace drtopk
