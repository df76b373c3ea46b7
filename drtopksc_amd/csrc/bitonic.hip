// bitonic.hip -- the bitonic top-k family of Dr.Top-k on gfx950.
//
// Restates the SIGMOD-style network of bitonic/bitonic_com.cuh: sort into k-runs of
// alternating direction (Combined_Sigmod_Merge*, :101-228 / :231-386), merge pairs of runs
// by elementwise max (:299-321), rebuild each run with a bitonic merge (:332-356), repeat
// until k elements remain.  Every element is a 64-bit composite (ordered key << 32 | ~index),
// so every comparison is strict: the top-k is by key, lowest index first among equal keys,
// and the result does not depend on how the network is scheduled.
//
// Scheduling on gfx950 (160 KB of LDS per CU):
//  - k <= 4096: a workgroup reduces a tile in LDS to its own top-k (sort into k-runs, then
//    merge + rebuild rounds); tiles are reduced level by level until one remains.  A compare step costs
//    an LDS round trip and a barrier, so a thread takes eight composites through three steps at once in
//    registers.  Unsorted input comes in tiles of 2048 (the 55 steps of k = 1024 on many CUs), sorted runs
//    in tiles of 8192 (few levels).  The first level builds its composites from the delegates or the
//    concatenation, the last one writes the results: in index order, after one more sort of the k
//    survivors.  The reference halves once per launch (bitonic_com.cuh:648-657).
//    2^26 keys, k = 1024: the 131072 delegates take 36 us and the 524288 concatenated keys with the results
//    56 (one step per round trip in tiles of 8192, with launches of their own for the composites, the
//    copy of the delegates and the sort by index: 270 in all).
//  - k = 8192: tiles of 16384 composites, one compare step per round trip.
//  - k > 8192 (the reference's largerK global-scratch variant): the network runs over a global
//    buffer; strides >= 16384 are global passes, all smaller strides of a stage are fused into
//    one LDS pass per 16384-composite tile.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace drtopk {

constexpr u32 BT_KMAX = 4096;    // largest k of the eight-at-once tiles
constexpr u32 BT = 16384;        // LDS tile for larger k and the global network (128 KB)
constexpr int BTT = 1024;

__device__ __forceinline__ void cmpx(u64* A, u32 i, u32 inc, bool up) {
    const u64 a = A[i], b = A[i + inc];
    if (up == (a > b)) {
        A[i] = b;
        A[i + inc] = a;
    }
}

// Steps inc = inc0 .. 1 of stage `len` on a tile of T elements whose first global index is
// `base`; the direction of a pair comes from bit 2*len of its global index.
template <int NT>
__device__ __forceinline__ void lds_steps(u64* A, u32 T, u64 base, u64 len, u64 inc0) {
    for (u64 inc = inc0; inc > 0; inc >>= 1) {
        for (u32 t = threadIdx.x; t < T / 2; t += NT) {
            const u32 low = t & (u32)(inc - 1), i = 2 * t - low;
            cmpx(A, i, (u32)inc, ((base + i) & (2 * len)) == 0);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- eight composites at once (k <= 4096)
struct BtArgs {
    u64 n;             // the level's input (a power of two); n of the last level may be below 8
    u32 kk, k;         // run length max(k, 8); results k
    int src;           // BT_RUNS: sorted runs of kk in A; BT_DELEG: dvals; BT_KEYS: V, or its subranges in D
    int fin;           // BT_LEVEL: tile top-kk to out; BT_FIRST: top-k delegates to out; BT_LAST: results
    const u64* A;
    const u32* dvals;
    u64 S;
    const u32* keys;
    u64 nkeys, nv;
    int alpha, f32;
    const u64* D;
    u64* out;
    u32* out_keys;
    i64* out_idx;
    u32* d_kth;
    Ctrl* ctrl;
};
enum { BT_RUNS, BT_DELEG, BT_KEYS };
enum { BT_LEVEL, BT_FIRST, BT_LAST };

// Word of element i: one word of padding per eight, so that neither eight consecutive elements per
// thread nor elements at a stride meet in the banks.
__device__ __forceinline__ u32 bt_at(u32 i) { return i + (i >> 3); }

__device__ __forceinline__ void bt_cx(u64& a, u64& b, bool up) {
    const bool sw = up == (a > b);
    const u64 x = sw ? b : a, y = sw ? a : b;
    a = x;
    b = y;
}
// Compare steps at distances d, d/2, .. 1 (d = 1, 2 or 4, uniform).
__device__ __forceinline__ void bt_steps(u64 (&x)[8], u32 d, bool up) {
    if (d >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) bt_cx(x[j], x[j + 4], up);
    }
    if (d >= 2) {
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
            bt_cx(x[j], x[j + 2], up);
            bt_cx(x[j + 1], x[j + 3], up);
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j += 2) bt_cx(x[j], x[j + 1], up);
}
// Strides top .. 1 of stage `len` over the T elements of S, up to three per round trip.  Ends with a
// barrier.
__device__ __forceinline__ void bt_stage(u64* S, u32 T, u32 top, u32 len) {
    for (; top; top >>= 3) {
        const u32 b = top >= 4 ? 29 - __clz((int)top) : 0;  // unit 2^b = top / 4
        const u32 t = threadIdx.x;
        if (t < T / 8) {
            const u32 i0 = ((t >> b) << (b + 3)) | (t & ((1u << b) - 1));
            u64 x[8];
#pragma unroll
            for (u32 j = 0; j < 8; ++j) x[j] = S[bt_at(i0 + (j << b))];
            bt_steps(x, top >> b, (i0 & (2 * len)) == 0);
#pragma unroll
            for (u32 j = 0; j < 8; ++j) S[bt_at(i0 + (j << b))] = x[j];
        }
        __syncthreads();
    }
}
// Sorts the T elements, eight consecutive ones in each thread's x, into alternating runs of kk (or
// one ascending run where T == kk) in S.  Ends with a barrier.
__device__ __forceinline__ void bt_sort_runs(u64* S, u64 (&x)[8], u32 T, u32 kk) {
    const u32 t = threadIdx.x;
    if (t < T / 8) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) bt_cx(x[j], x[j + 1], (j & 2) == 0);
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
            bt_cx(x[j], x[j + 2], j == 0);
            bt_cx(x[j + 1], x[j + 3], j == 0);
            bt_cx(x[j], x[j + 1], j == 0);
            bt_cx(x[j + 2], x[j + 3], j == 0);
        }
        bt_steps(x, 4, ((8 * t) & 8) == 0);
#pragma unroll
        for (u32 j = 0; j < 8; ++j) S[bt_at(8 * t + j)] = x[j];
    }
    __syncthreads();
    for (u32 len = 8; len < kk; len <<= 1) bt_stage(S, T, len, len);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_bt_tile(const BtArgs a) {
    constexpr u32 TILE = NT * 8;
    __shared__ u64 S[TILE + TILE / 8];
    __shared__ u32 cnt;
    const u32 t = threadIdx.x, kk = a.kk;
    const u32 T = (u32)(a.n < 8 ? 8 : (a.n < TILE ? a.n : TILE));
    const u64 base = (u64)blockIdx.x * TILE;
    if (t == 0) cnt = 0;
    // eight consecutive composites per thread
    u64 x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = 0;
    if (a.src == BT_RUNS) {
        if (t < T / 8) {  // odd runs reversed: alternating runs without sorting again
            const u32 i = 8 * t, r0 = i & ~(kk - 1);
            const bool rev = i & kk;
            const u64* p = a.A + base + (rev ? r0 + (kk - 8 - (i - r0)) : i);
#pragma unroll
            for (u32 j = 0; j < 8; ++j) S[bt_at(rev ? i + 7 - j : i + j)] = p[j];
        }
        __syncthreads();
    } else {
        u32 valid = 0;
        const u64 v0 = base + 8 * t;
        if (t < T / 8) {
            if (a.src == BT_DELEG) {
#pragma unroll
                for (u32 j = 0; j < 8; ++j)
                    if (v0 + j < a.S) x[j] = ((u64)a.dvals[v0 + j] << 32) | (u64)(0xFFFFFFFFu - (u32)(v0 + j));
            } else {
                u64 g0 = v0;
                if (a.D && a.alpha >= 3 && v0 < a.nv)  // the eight lie in one subrange
                    g0 = ((u64)(0xFFFFFFFFu - (u32)a.D[v0 >> a.alpha]) << a.alpha) + (v0 & ((1ull << a.alpha) - 1));
#pragma unroll
                for (u32 j = 0; j < 8; ++j) {
                    u64 g = g0 + j;
                    if (a.D && a.alpha < 3 && v0 + j < a.nv)
                        g = ((u64)(0xFFFFFFFFu - (u32)a.D[(v0 + j) >> a.alpha]) << a.alpha) +
                            ((v0 + j) & ((1ull << a.alpha) - 1));
                    if (v0 + j < a.nv && g < a.nkeys) {
                        const u32 key = a.keys[g];
                        x[j] = ((u64)(a.f32 ? KeyF32::to_ord(key) : key) << 32) | (u64)(0xFFFFFFFFu - (u32)g);
                        ++valid;
                    }
                }
            }
        }
        if (a.src == BT_KEYS) {  // the concatenation's size, a statistic
            valid = wave_incl_scan_u32(valid);
            __syncthreads();
            if ((t & (WAVE - 1)) == WAVE - 1 && valid) atomicAdd(&cnt, valid);
            __syncthreads();
            if (t == 0 && cnt) atomicAdd((unsigned long long*)&a.ctrl->concat_size, (unsigned long long)cnt);
        }
        bt_sort_runs(S, x, T, kk);
    }
    for (u32 cur = T / 2; cur >= kk; cur >>= 1) {
        // merge: element t of the halved tile = max of the pair (i, i + kk) of runs 2r, 2r + 1; and the
        // first three strides of the runs' rebuild
        const u32 b = 28 - __clz((int)kk);  // unit kk / 8
        const u32 i0 = ((t >> b) << (b + 3)) | (t & ((1u << b) - 1));
        if (t < cur / 8) {
#pragma unroll
            for (u32 j = 0; j < 8; ++j) {
                const u32 m = i0 + (j << b), i = 2 * m - (m & (kk - 1));
                const u64 p = S[bt_at(i)], q = S[bt_at(i + kk)];
                x[j] = p > q ? p : q;
            }
            bt_steps(x, 4, (i0 & kk) == 0);
        }
        __syncthreads();
        if (t < cur / 8) {
#pragma unroll
            for (u32 j = 0; j < 8; ++j) S[bt_at(i0 + (j << b))] = x[j];
        }
        __syncthreads();
        bt_stage(S, cur, kk >> 4, kk >> 1);
    }
    const u32 skip = kk - a.k;  // S[0..kk) ascending
    if (a.fin == BT_LEVEL) {
        for (u32 i = t; i < kk; i += NT) a.out[(u64)blockIdx.x * kk + i] = S[bt_at(i)];
        return;
    }
    const u32 K0 = (u32)(S[bt_at(skip)] >> 32);
    if (a.fin == BT_FIRST) {
        for (u32 i = t; i < a.k; i += NT) a.out[i] = S[bt_at(skip + i)];
        if (t == 0) {
            a.ctrl->first.result = K0;
            a.ctrl->first.done = 1;
            a.ctrl->selected = a.k;
        }
        return;
    }
    // results: (index << 32 | key) of the k survivors, sorted
    u32 gt = 0;
    if (t < kk / 8) {
#pragma unroll
        for (u32 j = 0; j < 8; ++j) {
            const u32 i = 8 * t + j;
            const u64 c = S[bt_at(i)];
            x[j] = i >= skip ? ((u64)(0xFFFFFFFFu - (u32)c) << 32) | (c >> 32) : ~0ull;  // the rest sorts last
            gt += i >= skip && (u32)(c >> 32) > K0 ? 1u : 0u;
        }
    }
    gt = wave_incl_scan_u32(gt);
    if (t == 0) cnt = 0;
    __syncthreads();
    if ((t & (WAVE - 1)) == WAVE - 1 && gt) atomicAdd(&cnt, gt);
    bt_sort_runs(S, x, kk, kk);
    for (u32 i = t; i < a.k; i += NT) {
        const u64 p = S[bt_at(i)];
        if (a.out_keys) a.out_keys[i] = a.f32 ? KeyF32::from_ord((u32)p) : (u32)p;
        if (a.out_idx) a.out_idx[i] = (i64)(p >> 32);
    }
    if (t == 0) {
        a.ctrl->count_gt = cnt;
        a.ctrl->ties = a.k - cnt;
        a.ctrl->kth = K0;
        a.ctrl->second.result = K0;
        a.ctrl->second.done = 1;
        if (a.d_kth) *a.d_kth = a.f32 ? KeyF32::from_ord(K0) : K0;
    }
}

// All levels of one top-k: a.n composites of a.src to a.fin; B0 and B1 take the levels' runs.
void bt_levels(BtArgs a, u64* B0, u64* B1, hipStream_t st) {
    const int fin = a.fin;
    u64* const result = a.out;
    for (;;) {
        const bool small = a.n <= 2048 ? a.kk <= 2048 : (a.src != BT_RUNS && 2 * a.kk <= 2048);
        const u64 tile = small ? 2048 : 8192, tiles = a.n > tile ? a.n / tile : 1;
        a.fin = tiles == 1 ? fin : BT_LEVEL;
        a.out = tiles == 1 ? result : B0;
        if (small) hipLaunchKernelGGL((k_bt_tile<256>), dim3((unsigned)tiles), dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_bt_tile<1024>), dim3((unsigned)tiles), dim3(1024), 0, st, a);
        if (tiles == 1) return;
        a.n = tiles * a.kk;
        a.src = BT_RUNS;
        a.A = B0;
        std::swap(B0, B1);
    }
}

// ---------------------------------------------------------------- tile reduction (k == 8192)
// Reduces tile b of A (T <= TILE elements) to its top-k, sorted ascending, at out[b*k, b*k + k).
// presorted: A holds runs of k each sorted ascending (a previous level's output); odd runs are
// loaded reversed, which gives the alternating k-runs the merge needs without sorting again.
template <u32 TILE, int NT>
__global__ __launch_bounds__(NT) void k_bt_tile_reduce(const u64* __restrict__ A, u32 T, u32 k, int presorted,
                                                       u64* __restrict__ out) {
    __shared__ u64 S[TILE];
    const u64 base = (u64)blockIdx.x * T;
    if (presorted) {
        for (u32 i = threadIdx.x; i < T; i += NT) {
            const u32 j = i & (k - 1), r0 = i - j;  // position in its run, first index of the run
            S[i] = A[base + ((i & k) ? r0 + (k - 1 - j) : i)];
        }
        __syncthreads();
    } else {
        for (u32 i = threadIdx.x; i < T; i += NT) S[i] = A[base + i];
        __syncthreads();
        // sort into alternating k-runs (tile-local directions)
        for (u64 len = 1; len < k; len <<= 1) lds_steps<NT>(S, T, 0, len, len);
    }
    u32 cur = T;
    while (cur > k) {
        // merge: element t of the halved tile = max of the pair (i, i+k) of runs 2r, 2r+1
        u64 m[TILE / 2 / NT];
#pragma unroll
        for (u32 j = 0; j < TILE / 2 / NT; ++j) {
            const u32 t = threadIdx.x + j * NT;
            if (t < cur / 2) {
                const u32 i = 2 * t - (t & (k - 1));
                m[j] = S[i] > S[i + k] ? S[i] : S[i + k];
            }
        }
        __syncthreads();
#pragma unroll
        for (u32 j = 0; j < TILE / 2 / NT; ++j) {
            const u32 t = threadIdx.x + j * NT;
            if (t < cur / 2) S[t] = m[j];
        }
        __syncthreads();
        cur >>= 1;
        // rebuild every run of k into sorted order (alternating)
        lds_steps<NT>(S, cur, 0, k >> 1, k >> 1);
    }
    for (u32 i = threadIdx.x; i < k; i += NT) out[(u64)blockIdx.x * k + i] = S[i];
}

// ---------------------------------------------------------------- global network (k > BT/2)
// Stages len < BT of the run sort, all in LDS (runs of up to BT).
__global__ __launch_bounds__(BTT) void k_bt_sort_lds(u64* __restrict__ A, u64 lenmax) {
    __shared__ u64 S[BT];
    const u64 base = (u64)blockIdx.x * BT;
    for (u32 i = threadIdx.x; i < BT; i += BTT) S[i] = A[base + i];
    __syncthreads();
    for (u64 len = 1; len <= lenmax; len <<= 1) lds_steps<BTT>(S, BT, base, len, len);
    for (u32 i = threadIdx.x; i < BT; i += BTT) A[base + i] = S[i];
}

// The strides < BT of stage `len` (inc = BT/2 .. 1), one LDS pass per tile.
__global__ __launch_bounds__(BTT) void k_bt_stage_lds(u64* __restrict__ A, u64 len) {
    __shared__ u64 S[BT];
    const u64 base = (u64)blockIdx.x * BT;
    for (u32 i = threadIdx.x; i < BT; i += BTT) S[i] = A[base + i];
    __syncthreads();
    lds_steps<BTT>(S, BT, base, len, BT / 2);
    for (u32 i = threadIdx.x; i < BT; i += BTT) A[base + i] = S[i];
}

// One stride >= BT of stage `len`, over all n/2 pairs.
__global__ __launch_bounds__(WG) void k_bt_step(u64* __restrict__ A, u64 n, u64 len, u64 inc) {
    const u64 stride = (u64)gridDim.x * WG;
    for (u64 t = (u64)blockIdx.x * WG + threadIdx.x; t < n / 2; t += stride) {
        const u64 low = t & (inc - 1), i = 2 * t - low;
        const bool up = (i & (2 * len)) == 0;
        const u64 a = A[i], b = A[i + inc];
        if (up == (a > b)) {
            A[i] = b;
            A[i + inc] = a;
        }
    }
}

// Merge: B[t] = max(A[i], A[i+k]) for the pair of runs holding t.
__global__ __launch_bounds__(WG) void k_bt_merge(const u64* __restrict__ A, u64 n, u64 k, u64* __restrict__ B) {
    const u64 stride = (u64)gridDim.x * WG;
    for (u64 t = (u64)blockIdx.x * WG + threadIdx.x; t < n / 2; t += stride) {
        const u64 i = 2 * t - (t & (k - 1));
        const u64 a = A[i], b = A[i + k];
        B[t] = a > b ? a : b;
    }
}

static unsigned grid_for(u64 items) { return (unsigned)std::max<u64>(1, std::min<u64>((items + WG - 1) / WG, 8192)); }

// Tile reduction levels with tiles of TILE composites: n -> k.
// Levels after the first read the sorted runs the previous one wrote.
template <u32 TILE, int NT>
u64* tile_levels(u64* A, u64* B, u64 n, u64 k, hipStream_t st) {
    int presorted = 0;
    while (n > TILE) {
        hipLaunchKernelGGL((k_bt_tile_reduce<TILE, NT>), dim3((unsigned)(n / TILE)), dim3(NT), 0, st, A, TILE,
                           (u32)k, presorted, B);
        n = (n / TILE) * k;
        std::swap(A, B);
        presorted = 1;
    }
    // last tile: n <= TILE elements -> k (also sorts when n == k)
    const u32 T = (u32)std::max<u64>(n, 1);
    hipLaunchKernelGGL((k_bt_tile_reduce<TILE, NT>), dim3(1), dim3(NT), 0, st, A, T, (u32)k, presorted, B);
    return B;
}

// Top-k (ascending, at A[0..k)) of the n composites in A (n a power of two, n >= k, k a power
// of two); B is scratch of n elements.  Returns the buffer holding the result.
u64* bitonic_topk(u64* A, u64* B, u64 n, u64 k, hipStream_t st) {
    if (k <= BT / 2) return tile_levels<BT, BTT>(A, B, n, k, st);
    // global network
    hipLaunchKernelGGL(k_bt_sort_lds, dim3((unsigned)(n / BT)), dim3(BTT), 0, st, A, (u64)(BT / 2));
    for (u64 len = BT; len < k; len <<= 1) {
        for (u64 inc = len; inc >= BT; inc >>= 1)
            hipLaunchKernelGGL(k_bt_step, dim3(grid_for(n / 2)), dim3(WG), 0, st, A, n, len, inc);
        hipLaunchKernelGGL(k_bt_stage_lds, dim3((unsigned)(n / BT)), dim3(BTT), 0, st, A, len);
    }
    while (n > k) {
        hipLaunchKernelGGL(k_bt_merge, dim3(grid_for(n / 2)), dim3(WG), 0, st, A, n, k, B);
        n >>= 1;
        std::swap(A, B);
        const u64 len = k >> 1;
        for (u64 inc = len; inc >= BT; inc >>= 1)
            hipLaunchKernelGGL(k_bt_step, dim3(grid_for(n / 2)), dim3(WG), 0, st, A, n, len, inc);
        hipLaunchKernelGGL(k_bt_stage_lds, dim3((unsigned)(n / BT)), dim3(BTT), 0, st, A, len);
    }
    return A;
}

// ---------------------------------------------------------------- composites
// Delegates: (max << 32) | ~s, zero padding up to npad.
__global__ __launch_bounds__(WG) void k_bt_comp_delegates(const u32* __restrict__ dvals, u64 S, u64* __restrict__ A,
                                                         u64 npad) {
    const u64 stride = (u64)gridDim.x * WG;
    for (u64 i = (u64)blockIdx.x * WG + threadIdx.x; i < npad; i += stride)
        A[i] = i < S ? (((u64)dvals[i] << 32) | (u64)(0xFFFFFFFFu - (u32)i)) : 0ull;
}

// Keys of the subranges named by the top-k delegate composites D[0..k) (whole subranges,
// CreateConcatenateRange bitonic_com.cuh:72-98), or of V itself when D is null.
template <class K>
__global__ __launch_bounds__(WG) void k_bt_comp_keys(const u32* __restrict__ keys, u64 n, int alpha,
                                                     const u64* __restrict__ D, u64 nv, u64* __restrict__ A, u64 npad,
                                                     Ctrl* ctrl) {
    __shared__ u64 red[WG / WAVE];
    const u64 L = 1ull << alpha;
    const u64 stride = (u64)gridDim.x * WG;
    u64 valid = 0;
    for (u64 v = (u64)blockIdx.x * WG + threadIdx.x; v < npad; v += stride) {
        u64 c = 0;
        if (v < nv) {
            u64 g = v;
            if (D) {
                const u32 sid = 0xFFFFFFFFu - (u32)D[v >> alpha];
                g = ((u64)sid << alpha) + (v & (L - 1));
            }
            if (g < n) {
                c = ((u64)K::to_ord(keys[g]) << 32) | (u64)(0xFFFFFFFFu - (u32)g);
                ++valid;
            }
        }
        A[v] = c;
    }
    valid = wave_sum_u64(valid);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) red[w] = valid;
    __syncthreads();
    if (threadIdx.x == 0 && ctrl) {
        u64 s = 0;
        for (int i = 0; i < WG / WAVE; ++i) s += red[i];
        if (s) atomicAdd((unsigned long long*)&ctrl->concat_size, (unsigned long long)s);
    }
}

// Threshold (k-th delegate) and the first-stage statistics.
__global__ void k_bt_first_done(const u64* __restrict__ D, u64 k, Ctrl* ctrl) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        ctrl->first.result = (u32)(D[0] >> 32);
        ctrl->first.done = 1;
        ctrl->selected = k;
    }
}

// Final stage: k-th key, counts, and (index << 32 | key) pairs for the index-order sort.
__global__ __launch_bounds__(WG) void k_bt_final(const u64* __restrict__ R, u64 k, u64* __restrict__ P, u64 npad,
                                                 Ctrl* ctrl) {
    __shared__ u64 red[WG / WAVE];
    const u32 K0 = (u32)(R[0] >> 32);
    const u64 stride = (u64)gridDim.x * WG;
    u64 gt = 0;
    for (u64 i = (u64)blockIdx.x * WG + threadIdx.x; i < npad; i += stride) {
        if (i < k) {
            const u64 c = R[i];
            const u32 key = (u32)(c >> 32), idx = 0xFFFFFFFFu - (u32)c;
            gt += key > K0;
            P[i] = ((u64)idx << 32) | key;
        } else {
            P[i] = ~0ull;  // sorts after every real pair
        }
    }
    gt = wave_sum_u64(gt);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) red[w] = gt;
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 s = 0;
        for (int i = 0; i < WG / WAVE; ++i) s += red[i];
        if (s) atomicAdd((unsigned long long*)&ctrl->count_gt, (unsigned long long)s);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->kth = K0;
        ctrl->second.result = K0;
        ctrl->second.done = 1;
    }
}

// Index-ordered outputs from the sorted pairs.
template <class K>
__global__ __launch_bounds__(WG) void k_bt_emit(const u64* __restrict__ P, u64 k, u32* __restrict__ out_keys,
                                                i64* __restrict__ out_idx, u32* __restrict__ d_kth, Ctrl* ctrl) {
    const u64 stride = (u64)gridDim.x * WG;
    for (u64 i = (u64)blockIdx.x * WG + threadIdx.x; i < k; i += stride) {
        const u64 p = P[i];
        if (out_keys) out_keys[i] = K::from_ord((u32)p);
        if (out_idx) out_idx[i] = (i64)(p >> 32);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->ties = k - ctrl->count_gt;
        if (d_kth) *d_kth = K::from_ord(ctrl->kth);
    }
}

hipError_t launch_bitonic(const BitonicArgs& a, hipStream_t st) {
    const u64 k = a.k;
    u64* A = a.bufA;
    u64* B = a.bufB;
    if (k <= BT_KMAX) {
        BtArgs t = {};
        t.k = (u32)k;
        t.kk = (u32)std::max<u64>(k, 8);
        t.dvals = a.dvals; t.S = a.S; t.keys = a.keys; t.nkeys = a.n; t.alpha = a.alpha; t.f32 = a.f32; t.ctrl = a.ctrl;
        t.nv = a.n;
        if (a.alpha > 0) {
            t.n = a.npad1; t.src = BT_DELEG; t.fin = BT_FIRST; t.out = a.dsel;
            bt_levels(t, A, B, st);
            t.D = a.dsel;
            t.nv = k << a.alpha;
        }
        t.n = a.npad2; t.src = BT_KEYS; t.fin = BT_LAST; t.out = nullptr;
        t.out_keys = (u32*)a.out_keys; t.out_idx = a.out_idx; t.d_kth = (u32*)a.d_kth;
        bt_levels(t, A, B, st);
        return hipGetLastError();
    }
    const u64* top = nullptr;  // top-k delegate composites
    u64 nv, npad;
    if (a.alpha > 0) {
        // first top-k over the delegates (bitonic_firstTopk, bitonic_com.cuh:610-666)
        npad = a.npad1;
        hipLaunchKernelGGL(k_bt_comp_delegates, dim3(grid_for(npad)), dim3(WG), 0, st, a.dvals, a.S, A, npad);
        top = bitonic_topk(A, B, npad, k, st);
        hipLaunchKernelGGL(k_bt_first_done, dim3(1), dim3(1), 0, st, top, k, a.ctrl);
        // keep the k delegate composites while the second stage reuses the buffers
        u64* D = a.dsel;
        hipError_t e = hipMemcpyAsync(D, top, k * sizeof(u64), hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return e;
        top = D;
        nv = k << a.alpha;
    } else {
        nv = a.n;
    }
    // second top-k over the concatenation (bitonic, bitonic_com.cuh:669-728) or over V
    npad = a.npad2;
    if (a.f32)
        hipLaunchKernelGGL((k_bt_comp_keys<KeyF32>), dim3(grid_for(npad)), dim3(WG), 0, st, a.keys, a.n, a.alpha, top,
                           nv, A, npad, a.ctrl);
    else
        hipLaunchKernelGGL((k_bt_comp_keys<KeyU32>), dim3(grid_for(npad)), dim3(WG), 0, st, a.keys, a.n, a.alpha, top,
                           nv, A, npad, a.ctrl);
    const u64* R = bitonic_topk(A, B, npad, k, st);
    // outputs in index order: sort (index << 32 | key) ascending over the k survivors
    u64* P = (R == A) ? B : A;
    const u64 kp = k;  // k is a power of two
    hipLaunchKernelGGL(k_bt_final, dim3(grid_for(kp)), dim3(WG), 0, st, R, k, P, kp, a.ctrl);
    u64* Q = (P == A) ? B : A;
    const u64* sorted = bitonic_topk(P, Q, kp, kp, st);  // one run of k: a full ascending sort
    if (a.f32)
        hipLaunchKernelGGL((k_bt_emit<KeyF32>), dim3(grid_for(k)), dim3(WG), 0, st, sorted, k, (u32*)a.out_keys,
                           a.out_idx, (u32*)a.d_kth, a.ctrl);
    else
        hipLaunchKernelGGL((k_bt_emit<KeyU32>), dim3(grid_for(k)), dim3(WG), 0, st, sorted, k, (u32*)a.out_keys,
                           a.out_idx, (u32*)a.d_kth, a.ctrl);
    return hipGetLastError();
}

}  // namespace drtopk
