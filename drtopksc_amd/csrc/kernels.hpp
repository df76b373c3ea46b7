// kernels.hpp -- host-side launchers of the device kernels (one per .hip file group).
#pragma once

#include "common.hpp"

namespace drtopk {

// A segmented array: segment s holds len(s) elements at [s*segcap, s*segcap + len(s)).
// len(s) = cnt[s], or min(segcap, n - s*segcap) when cnt is null (a flat array in tiles).
struct Seg {
    const u32* keys;
    const u32* idx;
    const u32* cnt;
    u64 segcap;
    u64 nseg;
    u64 n;
};

struct SampleArgs {
    const u32* keys;   // raw keys (uint32 or float32 bits)
    u64 n;
    int alpha, beta;
    int f32;           // keys are float32
    int staged;        // LDS-staged variant (alpha <= 5)
    int posmode;       // 0 none, 1 absolute positions, 2 packed offsets (beta >= 2)
    int fuse;          // 0 none, 1 radix top-digit histogram, 2 min/max
    u32* dvals;        // [beta*S] ordered delegates
    void* dpos;        // positions / packed offsets
    u32* ghist;        // fused histogram (fuse == 1)
    int hshift, bins;  // fused histogram: bin = delegate >> hshift, bins bins
    Ctrl* ctrl;
    // beta 2: when set, dvals[s] holds the first delegate and the 16-bit word s of dtop the top
    // byte of the second (all a beta-path threshold on the top 8-bit digit needs of it) and,
    // above it, the first's offset in the subrange (0xFF without positions); dpos unused
    u8* dtop = nullptr;
};
hipError_t launch_sample(const SampleArgs& a, hipStream_t st);

// Compute units of the current device (cached per device).
unsigned device_cus();

// Selection machinery -------------------------------------------------------------------
// mode 0: radix digits (prefix match + digit); mode 1: bucket levels (range + linear map)
hipError_t launch_init(Ctrl* ctrl, const Ctrl& init, u32* zero_begin, u64 zero_words, hipStream_t st);
hipError_t launch_hist(int mode, const u32* arr, SelState* sel, u32* ghist, int bins, unsigned grid,
                       hipStream_t st);
hipError_t launch_hist_raw(int mode, int f32, const u32* keys, SelState* sel, u32* ghist, int bins,
                           unsigned grid, hipStream_t st);
hipError_t launch_hist_seg(int mode, const Seg& seg, SelState* sel, u32* ghist, int bins, unsigned grid,
                           hipStream_t st);
// segcnt / nseg: first pass over a segmented concatenation; the kernel then also sets its size
// (concat_size, sel->m and the too-short error) from the segment counts, and with `part` first
// sums the beta concatenation's npart per-workgroup records (beta_part_total).
hipError_t launch_select(int mode, u32* ghist, int bins, SelState* sel, Ctrl* ctrl, hipStream_t st,
                         const u32* segcnt = nullptr, u64 nseg = 0, const u64* part = nullptr, u64 npart = 0);
hipError_t launch_bucket_begin(SelState* sel, Ctrl* ctrl, int from_ctrl_minmax, hipStream_t st);
hipError_t launch_minmax(const u32* arr, SelState* sel, Ctrl* ctrl, unsigned grid, hipStream_t st);
hipError_t launch_minmax_raw(int f32, const u32* keys, SelState* sel, Ctrl* ctrl, unsigned grid,
                             hipStream_t st);
hipError_t launch_minmax_seg(const Seg& seg, SelState* sel, unsigned grid, hipStream_t st);
hipError_t launch_find(const u32* arr, int raw_f32, SelState* sel, unsigned grid, hipStream_t st);
hipError_t launch_find_seg(const Seg& seg, SelState* sel, unsigned grid, hipStream_t st);

// compact.hip -------------------------------------------------------------------------
// Ordered compactions run as count pass -> single-workgroup scan -> write pass, with no
// waiting between workgroups.
hipError_t launch_scan(const u64* in, u64 nseg, u64* out_excl, u64* total, hipStream_t st);

// FindTopKRanges + FillWithKElementsID: exactly k subrange ids, ascending.
struct RangeArgs {
    const u32* dvals;
    u64 S;
    u64 k;
    int fullcmp;       // 1: compare full keys (bucket), 0: radix prefix of the first top-k
    SelState* sel;     // first top-k state
    Ctrl* ctrl;
    u32* sel_ids;      // [k]
    u64* cnt;          // per-tile packed (greater, equal) counts
    u64* off;          // their exclusive prefix
};
hipError_t launch_range(const RangeArgs& a, hipStream_t st);
__host__ __device__ inline u64 range_tiles(u64 S) { return (S + 4095) / 4096; }

// Default-path concatenation, staged per 4096-key tile of the selected subranges.
struct GatherArgs {
    const u32* keys;
    u64 n;
    int alpha, f32, filter;
    const u32* sel_ids;
    u64 nsel;
    Ctrl* ctrl;
    u32* skeys;        // segment t at [t*GATHER_TILE, ...)
    u32* sidx;         // or nullptr
    u32* cnt;          // [nseg]
    u32* ghist2;       // fused top-digit histogram of the concatenation, or nullptr
    int hshift2, bins2;
    u64 seg_limit = 0; // entries a segment may hold (0: its capacity); beyond it the error is raised
};
hipError_t launch_gather(const GatherArgs& a, hipStream_t st);
u64 gather_segcap(u64 V);   // segment capacity / count for V = nsel << alpha virtual keys
u64 gather_nseg(u64 V);

// Beta-path range selection + concatenation, staged per 1024-subrange tile.
struct BetaGatherArgs {
    const u32* keys;
    u64 n;
    int alpha, beta, f32, filter;  // filter: bit 0 keep keys >= threshold, bit 1 drop lonely delegates below it
    const u32* dvals;
    const void* doff;
    Ctrl* ctrl;
    u32* skeys;        // segment t at [t*segcap, ...)
    u32* sidx;
    u32* cnt;
    u32* ghist2;
    int hshift2, bins2;
    const u8* dtop = nullptr;  // beta 2: delegates in the sampler's dtop form (dvals[s] first, 16-bit dtop words)
    u64 seg_limit = 0;         // entries a segment may hold (0: its capacity)
    u64* part = nullptr;       // [beta_grid] per-workgroup records (selected, lonely, lonely delegates, dropped)
};
constexpr int BETA_SUBS_PER_THREAD = 4;  // 4 measured faster than 8 (fewer VGPRs, more resident workgroups)
constexpr u64 BETA_TILE_SUBS = 256 * BETA_SUBS_PER_THREAD;  // subranges per chunk of the beta gather
hipError_t launch_beta_gather(const BetaGatherArgs& a, hipStream_t st);
u64 beta_segcap(u64 S, int alpha);
u64 beta_nseg(u64 S, int alpha);
u64 beta_grid(u64 S, int alpha);  // workgroups of the beta gather = records it writes

// concatenation size = sum of segment counts -> ctrl->concat_size, second.m (with `part`: the
// beta concatenation's per-workgroup records summed into the Ctrl counts first)
hipError_t launch_seg_total(const u32* cnt, u64 nseg, Ctrl* ctrl, hipStream_t st, const u64* part = nullptr,
                            u64 npart = 0);

// findTopk + FillTopk: keys above the k-th largest, then the lowest-index ties, index order.
struct ExtractArgs {
    Seg seg;           // concatenation, or V itself (cnt == nullptr, raw keys)
    int direct;        // 1: seg is V (raw keys, index = position)
    int f32;
    u64 k;
    SelState* sel;     // second top-k state
    Ctrl* ctrl;
    void* out_keys;
    i64* out_idx;
    u64* cnt;          // [nseg] packed (greater, equal)
    u64* off;
    bool finalize = false;  // also do k_finalize's work (k-th key out, greater / tie counts)
    void* d_kth = nullptr;
};
constexpr u64 DIRECT_TILE = 16384;
hipError_t launch_extract(const ExtractArgs& a, hipStream_t st);
hipError_t launch_finalize(SelState* sel, Ctrl* ctrl, int f32, void* d_kth, u64 k, hipStream_t st);

// short.hip ---------------------------------------------------------------------------
// One-workgroup selections: the whole top-k (launch_small, n <= SMALL_N), or delegate pass ->
// first top-k -> concatenation -> second top-k and outputs in four or five launches.
constexpr u32 SMALL_N = 36864;     // keys, or values of one selection, that one workgroup holds in LDS
constexpr u32 SHORT_KMAX = 8192;   // largest k of launch_short
constexpr u32 SHORT_LISTED = 20480;  // values a level may have for its lists to stay in LDS, with k <= 4096
constexpr u32 SHORT_SEGS = 4096;   // most concatenation segments it reads
struct ShortArgs {
    const u32* keys;   // 16-byte aligned
    u64 n, k;
    int alpha, f32;    // alpha >= 2
    int f1, f2;        // log2 of the delegates per range of the first top-k's second level, and of
                       // those ranges per range of the third (0: no such level; f1 + f2 <= 8)
    Ctrl* ctrl;
    u32* dvals;        // [S] delegates, padded to 16 bytes
    u32* sup1;         // maxima of every 2^f1 delegates, padded to 16 bytes
    u32* sup2;         // maxima of every 2^f2 of those
    u32* sel_ids;      // [k]
    u32* ghist;        // [2048]
    u32* skeys;        // concatenation: short_segments x 4096 keys
    u32* sidx;         // and indices
    u32* cnt;          // [short_segments]
    u32* segmax;       // [short_segments]
    u32* rcnt;         // [short_segments] counts of the reduced segments: the delegates' area, dead by then
    void* out_keys;
    i64* out_idx;
    void* d_kth;
};
hipError_t launch_small(const ShortArgs& a, hipStream_t st);
hipError_t launch_short(const ShortArgs& a, hipStream_t st);
u32 short_segments(u64 V);         // concatenation segments of V = k << alpha slots

// filter.hip --------------------------------------------------------------------------
// Large k: a sampled lower bound of the k-th key, one filter pass, selection of what it keeps.
constexpr u32 F_UNIT = 2048;     // keys per unit: one segment of kept keys
constexpr u32 F_RANGES = 2048;   // most ranges of units (workgroups of the passes over kept keys)
constexpr u32 F_RUNITS = 256;    // most units per range (n <= 2^30)
constexpr u32 F_LIST_LDS = 17408;  // samples above the first bound of 2^17 or 2^19
inline u32 filter_units(u64 n) { return (u32)((n + F_UNIT - 1) / F_UNIT); }
// Workgroups of the filter pass and the consecutive 8192-key rounds each takes per step.  2^30 keys, no
// key kept: 693 us with 1 round, 633 with 4, 619 with 8 (8192 workgroups); small inputs need the
// workgroups more.
struct FilterGrid {
    u32 grid;
    int rounds;
};
inline FilterGrid filter_grid(u64 n) {
    const u32 units = filter_units(n);
    u32 r = units / (4 * 2048);
    r = r < 1 ? 1 : (r > 8 ? 8 : r);
    const u32 steps = (units + 4 * r - 1) / (4 * r);
    return {steps < 8192 ? steps : 8192, (int)r};
}
size_t filter_state_bytes();
struct FilterArgs {
    const u32* keys;   // 16-byte aligned, n >= 2^15
    u64 n, k;
    int f32;
    int lm;            // log2 of the samples: 13, 15, 17 or 19; n >= 2^lm
    u32 rp;            // sample rank bounding the k-th key from below
    u32 rlo, rhi;      // sample ranks between which the k-th key almost surely lies (rlo 0: the largest)
    u64 kept;          // keys expected above the bound
    u32 wcap;          // kept keys a wave's own segment holds
    u32 pool_cap;      // and the pool behind the segments, for units that find it full
    u32 lcap;          // entries of each of the 64 sublists of the k-th key's class
    Ctrl* ctrl;
    void* state;       // filter_state_bytes()
    u32* sample;       // [2^lm + 2^14]
    u32* cnt;          // [units] kept | equal to the bound << 16
    u32* base;         // [units] first slot of the unit's kept keys
    u32* gq;           // [units] of dense ranges: keys above the k-th | equal to it, low half
    u32 *rg, *rq;      // [F_RANGES]
    u32 *lkey, *lrange;  // [64 * lcap]: the class's keys, and the range (or unit) of each
    u32 *skeys, *sidx;   // [4 * workgroups * wcap + pool_cap]
    void* out_keys;
    i64* out_idx;
    void* d_kth;
};
hipError_t launch_filter(const FilterArgs& a, hipStream_t st);
// Whether the last call on this state ended in the one-workgroup selection from all keys.  Synchronises.
hipError_t filter_last_resort(const void* state, hipStream_t st, int* taken);

// bitonic.hip ---------------------------------------------------------------------------
// Bitonic family: first top-k over the delegates, whole-subrange concatenation, second
// top-k, index-ordered outputs.  alpha == 0: one top-k over V.
struct BitonicArgs {
    const u32* keys;
    u64 n;
    int alpha, f32;
    u64 k, S;
    const u32* dvals;  // delegates (alpha > 0)
    Ctrl* ctrl;
    u64* bufA;         // max(npad1, npad2) composites each
    u64* bufB;
    u64* dsel;         // k composites
    u64 npad1, npad2;  // next powers of two of S and of k << alpha (or n)
    void* out_keys;
    i64* out_idx;
    void* d_kth;
};
hipError_t launch_bitonic(const BitonicArgs& a, hipStream_t st);
hipError_t launch_to_user(const u32* ord, u64 m, int f32, void* out, hipStream_t st);

}  // namespace drtopk
