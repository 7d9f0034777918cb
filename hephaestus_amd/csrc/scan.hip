// Prefix scans for gfx950: ScanOps (crates/hephaestus-core/src/domain/
// scan.rs:197-264), extended with the exclusive form and rank-1 operands.
//
// The reference launches ONE 256-lane block per scan line; each lane walks a
// contiguous chunk serially, lane 0 folds the chunk totals, and a second sweep
// re-reads and re-writes the output (core accelerator/scan.rs:56-155).  A 1-D
// scan of 2^28 elements therefore runs on one CU.  Here every line is cut
// into tiles that all CUs process in a single pass (32768 elements for long
// lines, 2048 to 8192 for few lines of middling length; of many lines one of
// up to 32768 elements is one tile of the smallest shape that holds it, see
// tile_shape):
//
//   * block b scans tile b.  The tile is loaded with 16-byte vectors,
//     wave-striped: step j of wave w holds 256 contiguous elements, lane l
//     four of them; each step is a 4-element register scan plus a 6-step
//     wave64 scan of the lane totals;
//   * the tile aggregate is published, wave 0 looks back for the tile's
//     exclusive prefix and publishes the tile's inclusive prefix;
//   * every element is read once and written once, 16-byte vectors again.
//
// The look-back has two levels.  Tiles are grouped in superblocks of 64; the
// last tile of a superblock also publishes the superblock's aggregate (as
// soon as its 63 predecessors have published theirs) and later its
// inclusive prefix.  A tile first folds its own superblock's predecessors
// (one poll of 64 lanes) and then whole superblocks, 64 per poll.  With ~2000
// tiles in flight, a flat look-back walks up to ~32 sequential polls to
// reach a published prefix; the two levels need about two.
//
// Forward progress does not depend on the order in which the hardware
// dispatches blocks: when a status stays unpublished for p.spin_limit polls
// (its block may not be running yet), the waiting wave computes the missing
// value itself -- a tile aggregate from the input with the owner's
// arithmetic, a superblock value from its tiles' statuses -- and publishes
// it ("decoupled fallback", Smith, Levien and Owens 2024).  There is no
// tile-ticket counter: one same-address device-scope atomic per tile
// serialises at ~11 ns on MI355X, which alone cost 745 us for 65536 tiles.
//
// Status words carry a 14-bit per-launch tag (set by the host), so a launch
// never clears the status array and needs no end-of-launch bookkeeping.
// Integer scans publish (tag, flag, value) in ONE 64-bit word.  f32 scans
// carry the inter-tile prefix in f64 (every output stays within a few ulp of
// the f32-rounded exact prefix at 2^30 elements) in ONE 16-byte slot, read
// and written with one 16-byte access; each of its four dwords carries the
// tag and flag next to 16 bits of the value.
#include "hx_device.hpp"
#include "hx_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace hx {
namespace {

constexpr int kBlock = 256;                          // column-scan kernels
constexpr int kWaves = 8;                            // waves per tile block (long lines)
constexpr int kSteps = 16;                           // 16-byte vectors per lane (long lines)
constexpr int kSuper = 64;                           // tiles per superblock
constexpr uint32_t kInvalid = 0, kAggregate = 1, kPrefix = 2;

__device__ __forceinline__ uint64_t status_word(uint32_t tag, uint32_t flag, uint32_t v) {
    return ((uint64_t)status_word_hi(tag, flag) << 32) | (uint64_t)v;
}

// Tile statuses sit one per 128-byte line.  Tiles publish their statuses
// at about the same moment from CUs all over the chip, through to memory;
// packed densely, 16 of them shared a line.  Measured on MI355X, 2^28 u32
// exclusive scan, one process: status stride 8 bytes 336.3 us, 16: 334.7,
// 32: 332.6, 64: 331.6, 128: 328.8, 256: 328.5; 2^30 f32 inclusive scan,
// 16-byte slots: 1313.6 us, 128-byte stride 1291.0.  The column look-back
// (lanes across lines, polled as one contiguous run) keeps dense words.
constexpr uint64_t kTileStatusBytes = 128;

// (tag, flag, value) in one 64-bit word: [63:34] tag, [33:32] flag, [31:0]
// value; entry t at word t * STRIDE.
template <uint32_t STRIDE> struct PackedStatusT {
    using C = uint32_t;
    uint64_t *words;
    __device__ __forceinline__ uint64_t *at(uint64_t t) const { return words + t * STRIDE; }
    __device__ __forceinline__ void publish(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        st_relaxed(at(t), status_word(tag, flag, v));
    }
    // Fallback publication: never overwrites a word of this launch (so a
    // published inclusive prefix is never downgraded to an aggregate).
    __device__ __forceinline__ void publish_if_unset(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        uint64_t cur = ld_relaxed(at(t));
        if ((uint32_t)(cur >> 34) == tag) return;
        __hip_atomic_compare_exchange_strong(at(t), &cur, status_word(tag, flag, v), __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // Tile-level owner publication (same single store).
    __device__ __forceinline__ void publish_tile(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        publish(t, tag, flag, v);
    }
    __device__ __forceinline__ void read(uint64_t t, uint32_t tag, uint32_t &flag, C &v) const {
        const uint64_t w = ld_relaxed(at(t));
        const uint32_t hi = (uint32_t)(w >> 32);
        flag = ((hi >> 2) == tag) ? (hi & 3u) : kInvalid;
        v = (uint32_t)w;
    }
};
using PackedStatus = PackedStatusT<1>;                             // column look-back
using TilePackedStatus = PackedStatusT<kTileStatusBytes / 8>;      // tile scans

// f64 carries of the tile scans: one 16-byte slot per entry (at the start of
// the entry's 128-byte line; adjacent slots for row-tile columns), overwritten by
// its single writer (aggregate, then inclusive prefix) and read with ONE
// 16-byte load per lane.  Dword i of the slot is (check << 16) | bits
// [63-16i : 48-16i] of the f64, with check = (tag << 2) | flag (tags below
// 2^14; slot16_encode / slot16_decode).  A reader accepts the slot only when the four checks agree with
// each other and carry this launch's tag, so only 32-bit single-copy
// atomicity is assumed: a read that mixes dwords of two writes (aggregate
// and prefix, or an earlier launch's words) never has four equal checks.
// Words of the packed and partial-slot formats left in the same area read as
// not ready: their high halves are below 2^16, a check dword is at least
// 2^18.  Measured against two self-tagged 8-byte words read with two loads,
// 2^30 f32 inclusive scan on MI355X: 1360 -> 1315 us; the number of loads
// per poll, not their cache scope, set the difference (agent and system
// scope both 1360 us).
template <uint32_t STRIDE> struct F64QuadStatusT {
    using C = double;
    typedef uint32_t slot_t __attribute__((ext_vector_type(4)));
    uint64_t *words;
    __device__ __forceinline__ volatile __attribute__((address_space(1))) slot_t *slot(uint64_t t) const {
        return (volatile __attribute__((address_space(1))) slot_t *)(words + t * STRIDE);
    }
    __device__ __forceinline__ void publish(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        uint32_t w[4];
        slot16_encode(tag, flag, __builtin_bit_cast(uint64_t, v), w);
        slot_t q;
        q.x = w[0];
        q.y = w[1];
        q.z = w[2];
        q.w = w[3];
        *slot(t) = q;
    }
    __device__ __forceinline__ void publish_tile(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        publish(t, tag, flag, v);
    }
    // Slots have one writer: waiters that compute a missing value keep it
    // to themselves (SharedFallback).
    __device__ __forceinline__ void publish_if_unset(uint64_t, uint32_t, uint32_t, C) const {}
    __device__ __forceinline__ void read(uint64_t t, uint32_t tag, uint32_t &flag, C &v) const {
        const slot_t q = *slot(t);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        uint64_t b;
        flag = slot16_decode(tag, w, b);
        v = __builtin_bit_cast(double, b);
    }
};
using F64QuadStatus = F64QuadStatusT<kTileStatusBytes / 8>; // tile scans: one slot per 128-byte line
using F64QuadDense = F64QuadStatusT<2>;                     // row-tile columns: adjacent slots

// f64 values for the single-pass column scan: one slot of two self-tagged
// words (high and low halves) per entry, which the owner writes twice --
// aggregate, then inclusive prefix.  A reader accepts the slot only when both
// halves carry this launch's tag and the same flag; a half-updated slot reads
// as not ready.  Every slot has exactly one writer (waiters that give up
// compute the value themselves and do not publish it), so halves of
// different values can only meet transiently.
struct F64PairStatus {
    using C = double;
    uint64_t *words;
    __device__ __forceinline__ void publish_tile(uint64_t t, uint32_t tag, uint32_t flag, C v) const {
        const uint64_t b = __builtin_bit_cast(uint64_t, v);
        st_relaxed(&words[2 * t], status_word(tag, flag, (uint32_t)(b >> 32)));
        st_relaxed(&words[2 * t + 1], status_word(tag, flag, (uint32_t)b));
    }
    __device__ __forceinline__ void publish_if_unset(uint64_t, uint32_t, uint32_t, C) const {}
    __device__ __forceinline__ void read(uint64_t t, uint32_t tag, uint32_t &flag, C &v) const {
        const uint64_t hi = ld_relaxed(&words[2 * t]), lo = ld_relaxed(&words[2 * t + 1]);
        const uint32_t h = (uint32_t)(hi >> 32), l = (uint32_t)(lo >> 32);
        flag = (h == l && (h >> 2) == tag) ? (h & 3u) : kInvalid;
        v = __builtin_bit_cast(double, (hi << 32) | (lo & 0xFFFFFFFFull));
    }
};

// Whether waiters that compute a missing status publish it for others
// (publish_if_unset, a CAS on a single word) or keep it to themselves.
template <typename S> struct SharedFallback { static constexpr bool value = true; };
template <uint32_t STRIDE> struct SharedFallback<F64QuadStatusT<STRIDE>> { static constexpr bool value = false; };

struct ScanParams {
    const void *in;
    void *out;
    uint64_t lines, len, tiles_per_line, total_tiles, supers_per_line;
    int64_t in_line_stride, in_elem_stride;
    int64_t out_line_stride, out_elem_stride;
    uint64_t in_offset, out_offset;
    uint32_t tag;        // this launch's status tag
    uint32_t spin_limit; // polls before a waiter computes a missing value (64)
    uint64_t tile0;      // tile of block 0 (tile kernels launched in batches)
    uint32_t head;       // tile lines: elements [0, head) of the line are virtual (scan_out_head)
};

// The four elements of one lane and step (logical index e..e+3 of the
// line), identity past the end and, with HEAD, before p.head.
template <typename T, bool VEC, bool REV, bool NT, bool HEAD>
__device__ __forceinline__ void load4(const ScanParams &p, const T *in, int64_t ib, uint64_t e, T ident,
                                      T (&v)[4]) {
    const uint64_t head = HEAD ? p.head : 0u;
    if constexpr (VEC) {
        if (e + 3 < p.len && e >= head) {
            using V = typename Vec4A4<T>::type;
            if constexpr (REV) {
                // Logical e..e+3 are physical len-1-e down to len-4-e.
                const V q = load_a4<NT>((const V *)(in + ib + (int64_t)(p.len - 4 - e)));
                v[0] = (T)q.w;
                v[1] = (T)q.z;
                v[2] = (T)q.y;
                v[3] = (T)q.x;
            } else {
                const V q = load_a4<NT>((const V *)(in + ib + (int64_t)e));
                v[0] = (T)q.x;
                v[1] = (T)q.y;
                v[2] = (T)q.z;
                v[3] = (T)q.w;
            }
            return;
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint64_t i = e + c;
        const uint64_t li = REV ? (p.len - 1 - i) : i;
        v[c] = (i < p.len && i >= head) ? in[ib + (int64_t)li * p.in_elem_stride] : ident;
    }
}

// A lane's left-to-right fold of its four elements; the owner and the
// fallback both build step totals from it the same way.
template <typename T, typename Op>
__device__ __forceinline__ T lane_fold(const T (&v)[4]) {
    return Op::combine(Op::combine(Op::combine(v[0], v[1]), v[2]), v[3]);
}

// Aggregate of tile `u` computed by ONE wave, step by step, with the same
// operations and order as the four owner waves (fallback path).
template <typename T, typename Op, bool VEC, bool REV, bool NT, int STEPS, int WAVES, bool HEAD>
__device__ T tile_aggregate(const ScanParams &p, uint64_t u) {
    constexpr int kWaveElems = kWave * 4 * STEPS;
    constexpr int kTileElems = WAVES * kWaveElems;
    const T ident = Op::template identity<T>();
    const uint64_t line = u / p.tiles_per_line;
    const uint64_t tin = u - line * p.tiles_per_line;
    const int64_t ib = (int64_t)p.in_offset + (int64_t)line * p.in_line_stride;
    const T *in = (const T *)p.in;
    T agg = ident;
    for (int w = 0; w < WAVES; ++w) {
        T carry = ident;
        for (int j = 0; j < STEPS; ++j) {
            T v[4];
            load4<T, VEC, REV, NT, HEAD>(p, in, ib,
                                   tin * kTileElems + (uint64_t)w * kWaveElems + (uint64_t)j * (kWave * 4) +
                                       (uint64_t)lane_id() * 4,
                                   ident, v);
            const T incl = wave_inclusive_scan<Op, T>(lane_fold<T, Op>(v));
            carry = Op::combine(carry, read_lane(incl, kWave - 1));
        }
        agg = Op::combine(agg, carry);
    }
    return agg;
}

// The look-back reaches the tile's own aggregate through a hook: poll() runs
// on every spin, agg() yields the aggregate.  KnownAgg: the aggregate is
// already computed and published when the look-back starts.  (A variant
// whose fifth wave starts looking back while the data waves still load, and
// publishes the aggregate from poll(), measured 19% slower at 2^28 u32: the
// extra wave's registers cut occupancy and its polls span the whole load.)
template <typename C> struct KnownAgg {
    C a;
    __device__ __forceinline__ void poll() {}
    __device__ __forceinline__ C agg() { return a; }
};

// Wave-wide fold of the look-back values.  f64 carries fold with DPP moves
// (no lane-address registers, which the shuffle form keeps live across the
// whole look-back); 32-bit values keep the shuffle butterfly.
template <typename Op, typename C> __device__ __forceinline__ C lookback_reduce(C v) {
    if constexpr (sizeof(C) == 8)
        return group_reduce<64>(v, [](C a, C b) { return Op::combine(a, b); });
    else
        return wave_reduce<Op, C>(v);
}

// Fold of the statuses of the `count` (<= 64) tiles just before tile
// `tile_end`, nearest first, stopping at the first inclusive prefix; `found`
// tells whether one was met.  Lane l reads the tile at distance l.  A tile
// that stays unpublished is computed by tile_aggregate: published for every
// waiter where the status takes shared fallbacks, else kept in the lane that
// reads that tile.
template <typename T, typename Op, typename Status, bool VEC, bool REV, bool NT, int STEPS, int WAVES, bool HEAD,
          typename Hook>
__device__ typename Status::C fold_tiles(const ScanParams &p, const Status &st, uint64_t tile_end, int count,
                                         bool &found, Hook &hook) {
    using C = typename Status::C;
    const int lane = lane_id();
    const C ident = Op::template identity<C>();
    uint32_t flag;
    C val;
    uint32_t spins = 0;
    constexpr bool kShared = SharedFallback<Status>::value;
    bool own = false; // this lane's tile aggregate, computed by this wave
    C own_val = ident;
    for (;;) {
        flag = kAggregate; // lanes past `count`: valid, not a prefix, identity
        val = ident;
        if (lane < count) st.read(tile_end - 1 - lane, p.tag, flag, val);
        if constexpr (!kShared) {
            if (own && flag == kInvalid) {
                flag = kAggregate;
                val = own_val;
            }
        }
        const uint64_t pm = ballot(flag == kPrefix);
        const uint64_t im = ballot(flag == kInvalid);
        // Every status up to and including the nearest prefix is needed.
        const uint64_t need = pm ? (((pm & (~pm + 1ull)) << 1) - 1ull) : ~0ull;
        const uint64_t missing = im & need;
        if (missing == 0ull) break;
        hook.poll();
        if (++spins >= p.spin_limit) {
            const int k = __ffsll((long long)missing) - 1;
            const uint64_t u = tile_end - 1 - (uint64_t)k;
            const T a = tile_aggregate<T, Op, VEC, REV, NT, STEPS, WAVES, HEAD>(p, u);
            if constexpr (kShared) {
                if (lane == 0) st.publish_if_unset(u, p.tag, kAggregate, (C)a);
            } else if (lane == k) {
                own = true;
                own_val = (C)a;
            }
            spins = 0;
            continue;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    const uint64_t pm = ballot(flag == kPrefix);
    const int first = pm ? (__ffsll((long long)pm) - 1) : kWave;
    found = pm != 0ull;
    return lookback_reduce<Op, C>((lane <= first) ? val : ident);
}

// Exclusive prefix of tile `tile` (position `tin` in its line), computed by
// one wave.  The last tile of a superblock publishes the superblock
// aggregate on the way (it needs the tile's own aggregate: hook.agg()).
template <typename T, typename Op, typename Status, bool VEC, bool REV, bool NT, int STEPS, int WAVES, bool HEAD,
          typename Hook>
__device__ typename Status::C lookback(const ScanParams &p, const Status &st, const Status &st1, uint64_t tile,
                                       uint64_t line, uint64_t tin, Hook &hook) {
    using C = typename Status::C;
    const int lane = lane_id();
    const C ident = Op::template identity<C>();
    const int pos = (int)(tin % kSuper);
    const uint64_t sb = tin / kSuper;
    const uint64_t line_super = line * p.supers_per_line;
    const bool last_in_super = pos == kSuper - 1 && tin + 1 < p.tiles_per_line;

    // Level 0: predecessors in the tile's own superblock.
    bool found = false;
    C excl = pos > 0 ? fold_tiles<T, Op, Status, VEC, REV, NT, STEPS, WAVES, HEAD>(p, st, tile, pos, found, hook) : ident;
    if (found) return excl; // superblock 0 always ends here (tile 0 is a prefix)
    if (last_in_super) {
        const C a = hook.agg();
        if (lane == 0) st1.publish(line_super + sb, p.tag, kAggregate, Op::combine(excl, a));
    }

    // Level 1: whole superblocks, nearest first.
    int64_t pred = (int64_t)(line_super + sb) - 1;
    for (;;) {
        const int64_t idx = pred - lane;
        const bool in_line = idx >= (int64_t)line_super;
        uint32_t flag;
        C val;
        uint32_t spins = 0;
        constexpr bool kShared = SharedFallback<Status>::value;
        uint32_t own_flag = kInvalid; // this lane's superblock, rebuilt by this wave
        C own_val = ident;
        for (;;) {
            flag = kPrefix; // before the line's first superblock: identity
            val = ident;
            if (in_line) st1.read((uint64_t)idx, p.tag, flag, val);
            if constexpr (!kShared) {
                if (flag == kInvalid && own_flag != kInvalid) {
                    flag = own_flag;
                    val = own_val;
                }
            }
            const uint64_t pm = ballot(flag == kPrefix);
            const uint64_t im = ballot(flag == kInvalid);
            const uint64_t need = pm ? (((pm & (~pm + 1ull)) << 1) - 1ull) : ~0ull;
            const uint64_t missing = im & need;
            if (missing == 0ull) break;
            hook.poll();
            if (++spins >= p.spin_limit) {
                // Rebuild the missing superblock's value from its 64 tiles:
                // an inclusive prefix if one of them has one, else the sum.
                const int k = __ffsll((long long)missing) - 1;
                const uint64_t s = (uint64_t)(pred - k);
                const uint64_t s_end = line * p.tiles_per_line + (s - line_super + 1) * kSuper;
                bool f = false;
                const C v = fold_tiles<T, Op, Status, VEC, REV, NT, STEPS, WAVES, HEAD>(p, st, s_end, kSuper, f, hook);
                if constexpr (kShared) {
                    if (lane == 0) st1.publish_if_unset(s, p.tag, f ? kPrefix : kAggregate, v);
                } else if (lane == k) {
                    own_flag = f ? kPrefix : kAggregate;
                    own_val = v;
                }
                spins = 0;
                continue;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        const uint64_t pm = ballot(flag == kPrefix);
        const int first = pm ? (__ffsll((long long)pm) - 1) : kWave;
        excl = Op::combine(excl, lookback_reduce<Op, C>((lane <= first) ? val : ident));
        if (pm) break;
        pred -= kWave;
    }
    return excl;
}

template <typename T, typename C, typename Op>
__device__ __forceinline__ T finalize(C tile_excl, T within) {
    if constexpr (std::is_same<T, float>::value) {
        return (float)Op::combine(tile_excl, (double)within);
    } else {
        return Op::combine((T)tile_excl, within);
    }
}

// The tile's exclusive prefix applied to an element's in-tile prefix.
// Integers: one combine.  f32 with an f64 carry: the carry is split once per
// tile into f32 hi + lo (lo = the f32 rounding of carry - hi, exact to
// ~2^-48 relative) and each output is hi + (within + lo) (sums) or
// fma(hi, within, lo * within) (products), about one ulp from the f64
// combine rounded to f32 and far inside 2 ceil(log2 n) eps sum|x|.  The f64
// form converts every element to f64: the compiler hoists those conversions
// above the store branch and holds 96 extra registers, which kept f32 tiles
// at one block per CU.  A non-finite hi takes lo = 0 (hi + w then gives the
// f64 form's inf or NaN).
template <typename T, typename C, typename Op> struct TileCarry {
    T c;
    __device__ __forceinline__ explicit TileCarry(C v) : c((T)v) {}
    __device__ __forceinline__ T apply(T within) const { return Op::combine(c, within); }
};
template <typename Op> struct TileCarry<float, double, Op> {
    float hi, lo;
    __device__ __forceinline__ explicit TileCarry(double v) {
        hi = (float)v;
        lo = __builtin_isfinite(hi) ? (float)(v - (double)hi) : 0.0f;
    }
    __device__ __forceinline__ float apply(float w) const {
        if constexpr (std::is_same<Op, OpSum>::value) {
            return hi + (w + lo);
        } else {
            // lo * w is not finite only where w is infinite or NaN, or the
            // product overflows; hi * w then gives the f64 form's inf, NaN
            // or sign (fma(hi, w, -inf) would turn +inf into NaN or -inf).
            const float lw = lo * w;
            return __builtin_isfinite(lw) ? __builtin_fmaf(hi, w, lw) : hi * w;
        }
    }
};

// Full tiles of unit-stride lines (every tile but a line's ragged last one;
// the vectors need only 4-byte alignment): a block-uniform base pointer plus one 32-bit lane offset,
// so each step is a single base + offset + immediate vector access with no
// bounds check and no per-step 64-bit address held in registers.
// A whole tile of a reverse scan is a mirrored block of memory: logical
// elements e..e+3 of a lane's step are one 16-byte vector in reversed order,
// at byte (tile_bytes - 16 - lane_off - j * 1024) from the block's lowest
// address (always >= 0).
// Tiles are held to 128 VGPRs, two 8-wave blocks per CU: the integer
// inclusive forms (131 VGPRs unconstrained, one block per CU) spill a few
// words of look-back state and still gain ~3% (2^28 u32 inclusive 0.388 ->
// 0.378 ms).  f32 tiles fit in 121 with no spill through three changes: the
// split carry (TileCarry), the DPP look-back fold (lookback_reduce), and wave
// 0's 64 data registers parked in LDS while it looks back (ParkTile), with
// the wave's exclusive offset read only after the look-back.  Before them
// f32 tiles needed ~150 and ran one 12-wave block per CU.
template <typename T> struct ScanWavesPerEu { static constexpr int value = 4; };

// f32 tiles park wave 0's data in LDS during the look-back (16 KiB per
// block).  Integer tiles fit without it (116 VGPRs); parking measured 0.4%
// slower there.
template <typename T> struct ParkTile { static constexpr bool value = false; };
template <> struct ParkTile<float> { static constexpr bool value = true; };

// Paced tiles (integer scans).  Two blocks share each CU, and the memory
// instructions of all their waves queue through the CU's one vector-memory
// path in issue order.  A block that has its carry issues its 16 stores per
// wave back to back, and the other block's loads -- the next tile's, which
// set the pace of the whole stream -- wait behind them.  So:
//   * a block whose tile has predecessors (it will look back) runs at wave
//     priority 3 from its start and drops to 0 for its stores: when waves of
//     both blocks are ready to issue, the loads go first;
//   * stores leave 32 idle cycles (four s_nop 7) between each other, so a
//     load that becomes ready during a block's store phase is issued at the
//     next gap instead of after the whole burst.
// Measured on MI355X, 2^28 u32 exclusive scan, one process: burst stores
// 356.9 us; gaps only 350.7-353.8; priority only 344.9; both 335.6 (gaps of
// s_sleep 1: 336.4, two or three s_nop 7: 336.5-336.8, six or eight: 335.7-
// 335.8, every second store only: 339.2; priority 3 for the loads and 1 for
// the look-back: 338.6).  At 2^30: 1405.5 -> 1323.2 us.  Lines of one tile
// (row-wise scans) never look back; for them the gaps alone pay (the same
// kernel without look-back: burst 363.9 us, gaps 341.1; with the priority as
// well 349.5), so they keep the default priority.  f32 tiles, two blocks
// per CU as well, gain the same way (2^30 f32: 1382.8 us unpaced, 1315.6
// paced).

__device__ __forceinline__ void store_gap() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }

template <typename T, bool NT, int STEPS>
__device__ __forceinline__ void load_full_tile_rev(const T *base, uint32_t rev_off, T (&x)[STEPS][4]) {
    using V = typename Vec4A4<T>::type;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const V q = load_a4<NT>((const V *)((const char *)base + rev_off - (uint32_t)j * (kWave * 16)));
        x[j][0] = (T)q.w;
        x[j][1] = (T)q.z;
        x[j][2] = (T)q.y;
        x[j][3] = (T)q.x;
    }
}

template <typename T, bool NT, int STEPS>
__device__ __forceinline__ void load_full_tile(const T *base, uint32_t lane_off, T (&x)[STEPS][4]) {
    using V = typename Vec4A4<T>::type;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const V q = load_a4<NT>((const V *)((const char *)base + lane_off + (uint32_t)j * (kWave * 16)));
        x[j][0] = (T)q.x;
        x[j][1] = (T)q.y;
        x[j][2] = (T)q.z;
        x[j][3] = (T)q.w;
    }
}

// STEPS vectors per lane: a tile is 4 waves * 64 lanes * 4 * STEPS elements.
// VEC: unit-stride lines (16-byte vector loads and stores at any 4-byte
// aligned start).  REV:
// suffix scan (logical element i is physical len-1-i).  NT: non-temporal
// vector accesses.
template <typename T, typename Op, typename Status, bool EXCL, bool VEC, bool REV, int STEPS = kSteps,
          bool NT = true, int WAVES = kWaves, bool HEAD = false>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(ScanWavesPerEu<T>::value)))
void scan_tiles_kernel(ScanParams p, Status st, Status st1) {
    using C = typename Status::C;
    constexpr int kWaveElems = kWave * 4 * STEPS;
    constexpr int kTileElems = WAVES * kWaveElems;
    __shared__ T s_wave_tot[WAVES];
    __shared__ C s_excl;
    constexpr bool kPark = ParkTile<T>::value;
    __shared__ T s_park[kPark ? STEPS * 4 * kWave : 1];

    const bool looks_back = p.tiles_per_line > 1;
    if (looks_back) __builtin_amdgcn_s_setprio(3);

    const uint64_t tile = p.tile0 + blockIdx.x;
    const uint64_t line = tile / p.tiles_per_line;
    const uint64_t tin = tile - line * p.tiles_per_line;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = lane_id();
    const int64_t ib = (int64_t)p.in_offset + (int64_t)line * p.in_line_stride;
    const int64_t ob = (int64_t)p.out_offset + (int64_t)line * p.out_line_stride;
    const uint64_t e0 = tin * kTileElems + (uint64_t)w * kWaveElems + (uint64_t)lane * 4;
    const T *in = (const T *)p.in;
    T *out = (T *)p.out;
    const T ident = Op::template identity<T>();

    // Wave index made explicitly uniform so lane offsets stay 32-bit.
    const uint32_t lane_off =
        ((uint32_t)__builtin_amdgcn_readfirstlane(w) * kWaveElems + (uint32_t)lane * 4) * (uint32_t)sizeof(T);
    const bool full = VEC && (tin + 1) * kTileElems <= p.len && (!HEAD || tin > 0);
    // Reverse: the tile's lowest physical element, and the mirrored offset.
    const int64_t rev_tile = REV ? (int64_t)(p.len - (tin + 1) * kTileElems) : 0;
    const uint32_t rev_off = (uint32_t)(kTileElems - 4) * (uint32_t)sizeof(T) - lane_off;
    T x[STEPS][4];
    if (full) {
        if constexpr (REV)
            load_full_tile_rev<T, NT, STEPS>(in + ib + rev_tile, rev_off, x);
        else
            load_full_tile<T, NT, STEPS>(in + ib + (int64_t)(tin * kTileElems), lane_off, x);
        // All STEPS loads are issued before any arithmetic is scheduled.
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
            load4<T, VEC, REV, NT, HEAD>(p, in, ib, e0 + (uint64_t)j * (kWave * 4), ident, x[j]);
    }

    // Per step: register scan of 4, wave scan of lane totals, running carry.
    T carry = ident;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const T p0 = x[j][0];
        const T p1 = Op::combine(p0, x[j][1]);
        const T p2 = Op::combine(p1, x[j][2]);
        const T p3 = Op::combine(p2, x[j][3]);
        const T incl = wave_inclusive_scan<Op, T>(p3);
        const T lex = wave_shift_right<Op, T>(incl);
        const T base = Op::combine(carry, lex);
        if constexpr (EXCL) {
            x[j][0] = base;
            x[j][1] = Op::combine(base, p0);
            x[j][2] = Op::combine(base, p1);
            x[j][3] = Op::combine(base, p2);
        } else {
            x[j][0] = Op::combine(base, p0);
            x[j][1] = Op::combine(base, p1);
            x[j][2] = Op::combine(base, p2);
            x[j][3] = Op::combine(base, p3);
        }
        carry = Op::combine(carry, read_lane(incl, kWave - 1));
    }
    if (lane == 0) s_wave_tot[w] = carry;
    __syncthreads();
    // Wave totals are combined in wave order for the tile aggregate and each
    // wave's exclusive offset.  f32 tiles read the offset after the look-back
    // (nothing of it is held across the look-back) and park wave 0's data in
    // LDS meanwhile, so its registers are free for the look-back; the empty
    // asm statements keep the compiler from forwarding the parked values.
    T wave_excl = ident;
    T tile_agg = ident;
    if constexpr (!kPark) {
#pragma unroll
        for (int k = 0; k < WAVES; ++k) {
            if (k < w) wave_excl = Op::combine(wave_excl, s_wave_tot[k]);
            tile_agg = Op::combine(tile_agg, s_wave_tot[k]);
        }
    }

    if (w == 0) {
        if constexpr (kPark) {
#pragma unroll
            for (int k = 0; k < WAVES; ++k) tile_agg = Op::combine(tile_agg, s_wave_tot[k]);
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                using V = typename Vec4A4<T>::type;
                V v;
                v.x = x[j][0];
                v.y = x[j][1];
                v.z = x[j][2];
                v.w = x[j][3];
                *(V *)&s_park[(j * kWave + lane) * 4] = v;
            }
            asm volatile("" ::: "memory");
        }
        const C agg = (C)tile_agg;
        C excl = Op::template identity<C>();
        if (tin == 0) {
            // A line of one tile has no successor to read it (its status
            // area is not even allocated: scan_bytes).
            if (lane == 0 && looks_back) st.publish_tile(tile, p.tag, kPrefix, agg);
        } else {
            if (lane == 0) st.publish_tile(tile, p.tag, kAggregate, agg);
            KnownAgg<C> hook{agg};
            excl = lookback<T, Op, Status, VEC, REV, NT, STEPS, WAVES, HEAD>(p, st, st1, tile, line, tin, hook);
            // A line of one superblock needs no prefixes: every tile folds
            // all of its predecessors' aggregates in one poll, always the same
            // way, so f32 results are reproducible bit for bit (as they are
            // for lines of one tile).
            if (lane == 0 && p.tiles_per_line > kSuper)
                st.publish_tile(tile, p.tag, kPrefix, Op::combine(excl, agg));
        }
        if (lane == 0 && tin % kSuper == kSuper - 1 && tin + 1 < p.tiles_per_line)
            st1.publish(line * p.supers_per_line + tin / kSuper, p.tag, kPrefix, Op::combine(excl, agg));
        if (lane == 0) s_excl = excl;
        if constexpr (kPark) {
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                using V = typename Vec4A4<T>::type;
                const V v = *(const V *)&s_park[(j * kWave + lane) * 4];
                x[j][0] = v.x;
                x[j][1] = v.y;
                x[j][2] = v.z;
                x[j][3] = v.w;
            }
        }
    }
    __syncthreads();
    const TileCarry<T, C, Op> tile_carry(s_excl);
    if constexpr (kPark) {
#pragma unroll
        for (int k = 0; k < WAVES; ++k)
            if (k < w) wave_excl = Op::combine(wave_excl, s_wave_tot[k]);
    }
    if (looks_back) __builtin_amdgcn_s_setprio(0);

    if (full) {
        using V = typename Vec4A4<T>::type;
        if constexpr (REV) {
            const auto orsrc = stream_rsrc(out + ob + rev_tile, kTileElems * (uint32_t)sizeof(T));
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                V v;
                v.w = tile_carry.apply(Op::combine(wave_excl, x[j][0]));
                v.z = tile_carry.apply(Op::combine(wave_excl, x[j][1]));
                v.y = tile_carry.apply(Op::combine(wave_excl, x[j][2]));
                v.x = tile_carry.apply(Op::combine(wave_excl, x[j][3]));
                stream_store(v, orsrc, rev_off - (uint32_t)j * (kWave * 16));
                store_gap();
            }
        } else {
            const auto orsrc = stream_rsrc(out + ob + (int64_t)(tin * kTileElems), kTileElems * (uint32_t)sizeof(T));
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                V v;
                v.x = tile_carry.apply(Op::combine(wave_excl, x[j][0]));
                v.y = tile_carry.apply(Op::combine(wave_excl, x[j][1]));
                v.z = tile_carry.apply(Op::combine(wave_excl, x[j][2]));
                v.w = tile_carry.apply(Op::combine(wave_excl, x[j][3]));
                stream_store(v, orsrc, lane_off + (uint32_t)j * (kWave * 16));
                store_gap();
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const uint64_t e = e0 + (uint64_t)j * (kWave * 4);
        T r[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            // Opaque to the optimizer: the ragged tile's outputs are not
            // merged with the whole-tile path's and hoisted above the branch
            // (which kept every output of the tile live at once).
            T xv = x[j][c];
            asm volatile("" : "+v"(xv));
            r[c] = tile_carry.apply(Op::combine(wave_excl, xv));
        }
        if constexpr (VEC) {
            if (e + 3 < p.len && e >= (HEAD ? p.head : 0u)) {
                using V = typename Vec4A4<T>::type;
                V v;
                if constexpr (REV) {
                    v.w = r[0];
                    v.z = r[1];
                    v.y = r[2];
                    v.x = r[3];
                    store_a4<NT>(v, (V *)(out + ob + (int64_t)(p.len - 4 - e)));
                } else {
                    v.x = r[0];
                    v.y = r[1];
                    v.z = r[2];
                    v.w = r[3];
                    store_a4<NT>(v, (V *)(out + ob + (int64_t)e));
                }
                continue;
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint64_t i = e + c;
            const uint64_t li = REV ? (p.len - 1 - i) : i;
            if (i < p.len && i >= (HEAD ? p.head : 0u)) out[ob + (int64_t)li * p.out_elem_stride] = r[c];
        }
    }
}

// Short dense lines: a scan along lines of fewer than 256 elements packed
// back to back (line stride = length, element stride 1, input and output).
// One tile per line (scan_tiles_kernel) left most of a block idle and made
// the launch block-bound: [2^24, 4] u32 along axis 1 took 4.0 ms.  Here the
// operand is one flat range of lines x len elements, cut into tiles of
// WAVES x 64 x 4 x STEPS elements in logical order (a reverse scan mirrors
// the range), loaded and stored as 16-byte vectors exactly like a 1-D scan,
// and scanned with a segmented scan that restarts at every line start
// (logical index k with k % len == 0):
//
//   * per lane, the four elements' running values restart at a line start;
//   * across the wave, (flag, value) pairs -- flag: a line starts in the
//     span -- take a six-step DPP scan under the segmented combine
//     (f1, v1) . (f2, v2) = (f1 | f2, f2 ? v2 : v1 + v2), which is
//     associative; across steps a register carry, across waves LDS;
//   * the line open at the tile start takes the fold of its elements in the
//     previous tile (at most len - 1 < 255 of them), which wave 0 re-reads,
//     so no tile waits for another: no look-back and no status words.
//
// Line starts are tracked with an incremental remainder, no division per
// element.  f32 lines scan in f32 (a line holds fewer than 256 elements).
// Small tiles: no tile waits for another, so a block that holds little lets
// the CU overlap many blocks' loads, scans and stores, and small operands
// fill the chip.  4 waves x 2 steps (2048 elements) for small operands and for
// lines of a few elements, 4 x 4 beyond (short_tiles_small); us, 4 x 2 / 4 x 4
// / 8 x 16 tiles: f32 [13635, 48] 3.1 / 4.1 / 18.9; u32 [60000, 100] 7.8 / 7.3 /
// 12.2, [300000, 40] 15.8 / 17.0 / 17.4; f32 [100000, 200] 29.6 / 27.7 / 36.7,
// [500000, 250] 163 / 165 / 184, [2684354, 100] 341 / 350 / 385, [1052688, 255]
// 433 / 367 / 384 (the f32 form of 8 x 16 tiles spilled under the 128-VGPR
// cap; 8 x 4 tiles 382 / 378 at the last two).
struct ShortParams {
    const void *in;
    void *out;
    uint64_t n;      // lines * len
    uint64_t in_offset, out_offset;
    uint64_t tile0;  // tile of block 0 (launched in batches)
    uint32_t len;    // elements per line, 1..255
};

// The segmented combine on (flag, value) pairs.
template <typename Op, typename T>
__device__ __forceinline__ void seg_combine(uint32_t fa, T va, uint32_t &fb, T &vb) {
    vb = fb ? vb : Op::combine(va, vb);
    fb |= fa;
}

// Inclusive segmented scan across the 64 lanes (Hillis-Steele on DPP moves,
// as wave_inclusive_scan; lanes with no source take (0, identity)).
template <typename Op, typename T> __device__ __forceinline__ void wave_seg_scan(uint32_t &f, T &v) {
    const T id = Op::template identity<T>();
#define HX_SEG_STEP(CTRL, MASK)                                                                                      \
    {                                                                                                                \
        const T vs = dpp_move<CTRL, MASK>(id, v);                                                                    \
        const uint32_t fs = dpp_move<CTRL, MASK>(0u, f);                                                             \
        seg_combine<Op, T>(fs, vs, f, v);                                                                            \
    }
    HX_SEG_STEP(kDppRowShr1, 0xf)
    HX_SEG_STEP(kDppRowShr2, 0xf)
    HX_SEG_STEP(kDppRowShr4, 0xf)
    HX_SEG_STEP(kDppRowShr8, 0xf)
    HX_SEG_STEP(kDppRowBcast15, 0xa)
    HX_SEG_STEP(kDppRowBcast31, 0xc)
#undef HX_SEG_STEP
}

template <typename T, typename Op, bool EXCL, bool REV, int STEPS, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(4)))
void scan_short_lines_kernel(ShortParams p) {
    constexpr uint32_t kWaveElems = kWave * 4 * STEPS;
    constexpr uint32_t kTileElems = WAVES * kWaveElems;
    __shared__ uint32_t s_wf[WAVES];
    __shared__ T s_wv[WAVES];
    __shared__ T s_carry;

    const T ident = Op::template identity<T>();
    const uint64_t tile = p.tile0 + blockIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = lane_id();
    const uint32_t L = p.len;
    const T *in = (const T *)p.in + p.in_offset;
    T *out = (T *)p.out + p.out_offset;
    const uint64_t k0 = tile * kTileElems;                                // tile's first logical element
    const uint64_t wbase = k0 + (uint64_t)w * kWaveElems;
    const bool full = k0 + kTileElems <= p.n;
    // Logical element k lives at in[k] (forward) or in[n - 1 - k] (reverse).
    const uint32_t lane_off = ((uint32_t)w * kWaveElems + (uint32_t)lane * 4) * (uint32_t)sizeof(T);

    T x[STEPS][4];
    if (full) {
        using V = typename Vec4A4<T>::type;
        if constexpr (REV) {
            const char *base = (const char *)(in + (p.n - k0 - kTileElems));
            const uint32_t rev = (kTileElems - 4) * (uint32_t)sizeof(T) - lane_off;
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                const V q = load_a4<true>((const V *)(base + rev - (uint32_t)j * (kWave * 16)));
                x[j][0] = (T)q.w;
                x[j][1] = (T)q.z;
                x[j][2] = (T)q.y;
                x[j][3] = (T)q.x;
            }
        } else {
            const char *base = (const char *)(in + k0);
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                const V q = load_a4<true>((const V *)(base + lane_off + (uint32_t)j * (kWave * 16)));
                x[j][0] = (T)q.x;
                x[j][1] = (T)q.y;
                x[j][2] = (T)q.z;
                x[j][3] = (T)q.w;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint64_t k = wbase + (uint64_t)j * (kWave * 4) + (uint64_t)lane * 4 + c;
                x[j][c] = k < p.n ? in[REV ? p.n - 1 - k : k] : ident;
            }
    }

    // The line open at the tile start: the fold of its elements before k0.
    const uint32_t m = (uint32_t)(k0 % L);
    if (w == 0) {
        T a = ident;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t i = (uint32_t)lane + 64u * q;
            if (i < m) {
                const uint64_t k = k0 - m + i;
                a = Op::combine(a, in[REV ? p.n - 1 - k : k]);
            }
        }
        a = wave_reduce<Op, T>(a);
        if (lane == 0) s_carry = a;
    }

    // Remainder of this lane's first element modulo L, then per step.
    const uint32_t wrem = (uint32_t)(wbase % L);
    uint32_t r = (wrem + (uint32_t)lane * 4u) % L;
    const uint32_t step_inc = (kWave * 4u) % L;
    uint32_t fs = 0u; // step carry: (flag, value)
    T vs = ident;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        // flags of the four elements: remainder 0 marks a line start
        uint32_t rc = r, f[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            f[c] = rc == 0u;
            rc += 1u;
            rc = rc >= L ? rc - L : rc;
        }
        T pl[4];
        pl[0] = x[j][0];
#pragma unroll
        for (int c = 1; c < 4; ++c) pl[c] = f[c] ? x[j][c] : Op::combine(pl[c - 1], x[j][c]);
        uint32_t fl = f[0] | f[1] | f[2] | f[3];
        T vl = pl[3];
        wave_seg_scan<Op, T>(fl, vl); // lane inclusive over the wave's step
        // lane exclusive: the previous lane's inclusive value
        uint32_t fe = dpp_move<kDppWaveShr1>(0u, fl);
        T ve = dpp_move<kDppWaveShr1>(ident, vl);
        // this lane's incoming value within the wave: step carry, then lanes before
        const T vin = fe ? ve : Op::combine(vs, ve);
        uint32_t seen = 0u; // a line start at or before element c in this lane
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            seen |= f[c];
            x[j][c] = seen ? pl[c] : Op::combine(vin, pl[c]);
        }
        if constexpr (EXCL) {
            // exclusive: identity at a line start, else the inclusive value
            // of the element before (the lane's incoming value for c = 0)
#pragma unroll
            for (int c = 3; c >= 1; --c) x[j][c] = f[c] ? ident : x[j][c - 1];
            x[j][0] = f[0] ? ident : vin;
        }
        // carry to the next step: the wave's inclusive (flag, value) at lane 63
        const uint32_t f63 = read_lane(fl, kWave - 1);
        const T v63 = read_lane(vl, kWave - 1);
        vs = f63 ? v63 : Op::combine(vs, v63);
        fs |= f63;
        r += step_inc;
        r = r >= L ? r - L : r;
        // One step at a time: interleaving steps' scans (the scheduler's
        // choice) spilled the f32 forms at 16 steps.
        __builtin_amdgcn_sched_barrier(0);
    }
    if (lane == 0) {
        s_wf[w] = fs;
        s_wv[w] = vs;
    }
    __syncthreads();
    // This wave's incoming value: the open line's carry, then waves before.
    T win = s_carry;
    for (int q = 0; q < w; ++q) win = s_wf[q] ? s_wv[q] : Op::combine(win, s_wv[q]);
    // Elements before the wave's first line start take win.
    const uint64_t first_start = wbase + (uint64_t)((L - wrem) % L);

    if (full) {
        using V = typename Vec4A4<T>::type;
        const auto orsrc = stream_rsrc(REV ? (void *)(out + (p.n - k0 - kTileElems)) : (void *)(out + k0),
                                       kTileElems * (uint32_t)sizeof(T));
        const uint32_t rev = (kTileElems - 4) * (uint32_t)sizeof(T) - lane_off;
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            const uint64_t k = wbase + (uint64_t)j * (kWave * 4) + (uint64_t)lane * 4;
            T y[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) y[c] = k + c >= first_start ? x[j][c] : Op::combine(win, x[j][c]);
            V v;
            if constexpr (REV) {
                v.w = y[0];
                v.z = y[1];
                v.y = y[2];
                v.x = y[3];
                stream_store(v, orsrc, rev - (uint32_t)j * (kWave * 16));
            } else {
                v.x = y[0];
                v.y = y[1];
                v.z = y[2];
                v.w = y[3];
                stream_store(v, orsrc, lane_off + (uint32_t)j * (kWave * 16));
            }
            store_gap();
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint64_t k = wbase + (uint64_t)j * (kWave * 4) + (uint64_t)lane * 4 + c;
            T xv = x[j][c];
            asm volatile("" : "+v"(xv)); // not merged with the whole-tile stores (see scan_tiles_kernel)
            if (k < p.n) out[REV ? p.n - 1 - k : k] = k >= first_start ? xv : Op::combine(win, xv);
        }
}

// Column scans: many strided lines whose starts are adjacent in memory
// (axis-0 scan of a row-major matrix).  Lines that ascend in memory in both
// operands take the strips below (col_strip_kernel), very wide integer ones
// and those that descend the single-pass col_lookback_kernel; this chunked
// reduce-then-scan serves fewer than 256 descending lines and many short
// lines (col_scan_kernel alone).  Lanes run across lines -- a wave owns 64*V
// adjacent lines, V = 4 giving every lane one 16-byte load per step -- and the scan
// axis is cut into chunks so that thousands of waves share the work however
// tall the matrix is:
//   col_totals_kernel  chunk totals of every line (one read of the input);
//   col_carry_kernel   per line, an exclusive scan of its chunk totals in
//                      place (chunks x lines words, a thread per line);
//   col_scan_kernel    every chunk rescanned from its carry, outputs written.
// With one chunk only col_scan_kernel runs (carry = identity).  Each lane
// walks its lines serially; f32 accumulates in f64, integers wrap in u32.
template <typename T> struct ColAcc { using type = uint32_t; };
template <> struct ColAcc<float> { using type = double; };

struct ColShape {
    int V = 1;
    uint64_t groups = 0, chunk = 0;
    uint32_t nchunks = 1;
};

template <typename T, int V> struct ColIO;
template <typename T> struct ColIO<T, 1> {
    using A = typename ColAcc<T>::type;
    static __device__ __forceinline__ void load(const T *p, A (&x)[1]) { x[0] = (A)__builtin_nontemporal_load(p); }
    static __device__ __forceinline__ void store(T *p, const A (&y)[1]) { __builtin_nontemporal_store((T)y[0], p); }
    static __device__ __forceinline__ void load_n(const T *p, uint32_t, A, A (&x)[1]) { load(p, x); }
    static __device__ __forceinline__ void store_n(T *p, uint32_t, const A (&y)[1]) { store(p, y); }
};
template <typename T> struct ColIO<T, 4> {
    using A = typename ColAcc<T>::type;
    using Vt = typename Vec4A4<T>::type;
    static __device__ __forceinline__ void load(const T *p, A (&x)[4]) {
        const Vt v = __builtin_nontemporal_load((const Vt *)p);
        x[0] = (A)v.x;
        x[1] = (A)v.y;
        x[2] = (A)v.z;
        x[3] = (A)v.w;
    }
    static __device__ __forceinline__ void store(T *p, const A (&y)[4]) {
        Vt v;
        v.x = (T)y[0];
        v.y = (T)y[1];
        v.z = (T)y[2];
        v.w = (T)y[3];
        __builtin_nontemporal_store(v, (Vt *)p);
    }
    // The lane of a partial group (the last nv < 4 lines, when the line
    // count is not a multiple of 4) moves its lines one by one; the others
    // read as `ident` and are never stored.
    static __device__ __forceinline__ void load_n(const T *p, uint32_t nv, A ident, A (&x)[4]) {
        if (nv >= 4) {
            load(p, x);
            return;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) x[v] = (uint32_t)v < nv ? (A)__builtin_nontemporal_load(p + v) : ident;
    }
    static __device__ __forceinline__ void store_n(T *p, uint32_t nv, const A (&y)[4]) {
        if (nv >= 4) {
            store(p, y);
            return;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if ((uint32_t)v < nv) __builtin_nontemporal_store((T)y[v], p + v);
    }
};

// Lines of this lane's group that exist (V, or fewer in the last group).
__device__ __forceinline__ uint32_t col_valid_lines(uint64_t lines, uint64_t line0, int V) {
    return lines - line0 < (uint64_t)V ? (uint32_t)(lines - line0) : (uint32_t)V;
}

// Wave w -> (line group g, chunk k); adjacent waves take adjacent groups of
// the same chunk.  Returns false for lanes with no line.
struct ColWork {
    uint64_t line0, k, i0, i1;
};
__device__ __forceinline__ bool col_work(const ScanParams &p, uint64_t chunk, uint32_t nchunks, uint64_t groups,
                                         int V, ColWork *w) {
    const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
    if (wave >= groups * nchunks) return false;
    const uint64_t g = wave % groups;
    w->k = wave / groups;
    w->line0 = (g * kWave + (uint64_t)lane_id()) * V;
    if (w->line0 >= p.lines) return false;
    w->i0 = w->k * chunk;
    w->i1 = w->i0 + chunk < p.len ? w->i0 + chunk : p.len;
    return true;
}

template <typename T, typename Op, int V, bool REV>
__global__ __launch_bounds__(kBlock) void col_totals_kernel(ScanParams p, typename ColAcc<T>::type *totals,
                                                            uint64_t chunk, uint32_t nchunks, uint64_t groups) {
    using A = typename ColAcc<T>::type;
    constexpr int kU = V == 4 ? 8 : 16;
    ColWork w;
    if (!col_work(p, chunk, nchunks, groups, V, &w)) return;
    const T *in = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)w.line0 * p.in_line_stride);
    const uint32_t nv = col_valid_lines(p.lines, w.line0, V);
    const A aid = Op::template identity<A>();
    A acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = aid;
    uint64_t i = w.i0;
    for (; i + kU <= w.i1; i += kU) {
        A x[kU][V];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint64_t li = REV ? p.len - 1 - (i + u) : i + u;
            ColIO<T, V>::load_n(in + (int64_t)li * p.in_elem_stride, nv, aid, x[u]);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v] = Op::combine(acc[v], x[u][v]);
    }
    for (; i < w.i1; ++i) {
        const uint64_t li = REV ? p.len - 1 - i : i;
        A x[V];
        ColIO<T, V>::load_n(in + (int64_t)li * p.in_elem_stride, nv, aid, x);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = Op::combine(acc[v], x[v]);
    }
#pragma unroll
    for (int v = 0; v < V; ++v)
        if ((uint32_t)v < nv) totals[w.k * p.lines + w.line0 + v] = acc[v];
}

// Exclusive scan of each line's chunk totals, in place.  A block owns 16 lines
// and cuts the chunks into 64 contiguous slices, one to every 16 lanes: a lane
// totals its slice, kCarryBatch loads together (one batch, kept for the
// rewrite, up to 512 chunks), folds the earlier slices' totals through LDS and
// rewrites its slice.  The order depends on the chunk count alone.  With
// slices of a sixteenth of the chunks and one load at a time, [65536, 100] f32
// in three launches took 33.4 us against 25.4.
constexpr int kCarryWaves = 16, kCarryLines = 16, kCarryBatch = 8;
constexpr int kCarrySlices = kCarryWaves * (kWave / kCarryLines);

template <typename A, typename Op>
__global__ __launch_bounds__(kWave *kCarryWaves) void col_carry_kernel(A *totals, uint64_t lines, uint32_t nchunks) {
    __shared__ A sh[kCarrySlices][kCarryLines];
    const int q = threadIdx.x % kCarryLines;
    const uint32_t s = threadIdx.x / kCarryLines;
    const uint64_t line = (uint64_t)blockIdx.x * kCarryLines + q;
    const uint32_t per = (nchunks + kCarrySlices - 1) / kCarrySlices;
    const uint32_t k0 = s * per < nchunks ? s * per : nchunks;
    const uint32_t k1 = k0 + per < nchunks ? k0 + per : nchunks;
    const bool live = line < lines;
    const A id = Op::template identity<A>();
    A v[kCarryBatch];
    auto load = [&](uint32_t k) {
#pragma unroll
        for (uint32_t u = 0; u < kCarryBatch; ++u)
            v[u] = live && k + u < k1 ? totals[(uint64_t)(k + u) * lines + line] : id;
    };
    A sum = id;
    for (uint32_t k = k0; k < k1; k += kCarryBatch) {
        load(k);
#pragma unroll
        for (uint32_t u = 0; u < kCarryBatch; ++u) sum = Op::combine(sum, v[u]);
    }
    sh[s][q] = sum;
    __syncthreads();
    A acc = id;
#pragma unroll 8
    for (uint32_t t = 0; t < s; ++t) acc = Op::combine(acc, sh[t][q]);
    for (uint32_t k = k0; k < k1; k += kCarryBatch) {
        if (per > (uint32_t)kCarryBatch) load(k);
#pragma unroll
        for (uint32_t u = 0; u < kCarryBatch; ++u) {
            if (live && k + u < k1) totals[(uint64_t)(k + u) * lines + line] = acc;
            acc = Op::combine(acc, v[u]);
        }
    }
}

template <typename T, typename Op, int V, bool EXCL, bool REV, bool CARRY>
__global__ __launch_bounds__(kBlock) void col_scan_kernel(ScanParams p, const typename ColAcc<T>::type *carries,
                                                          uint64_t chunk, uint32_t nchunks, uint64_t groups) {
    using A = typename ColAcc<T>::type;
    constexpr int kU = V == 4 ? 8 : 16;
    ColWork w;
    if (!col_work(p, chunk, nchunks, groups, V, &w)) return;
    const T *in = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)w.line0 * p.in_line_stride);
    T *out = (T *)p.out + ((int64_t)p.out_offset + (int64_t)w.line0 * p.out_line_stride);
    const uint32_t nv = col_valid_lines(p.lines, w.line0, V);
    const A aid = Op::template identity<A>();
    A acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = CARRY && (uint32_t)v < nv ? carries[w.k * p.lines + w.line0 + v] : aid;
    auto step = [&](uint64_t li, const A (&x)[V]) {
        A y[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if constexpr (EXCL) {
                y[v] = acc[v];
                acc[v] = Op::combine(acc[v], x[v]);
            } else {
                acc[v] = Op::combine(acc[v], x[v]);
                y[v] = acc[v];
            }
        }
        ColIO<T, V>::store_n(out + (int64_t)li * p.out_elem_stride, nv, y);
    };
    uint64_t i = w.i0;
    for (; i + kU <= w.i1; i += kU) {
        A x[kU][V];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint64_t li = REV ? p.len - 1 - (i + u) : i + u;
            ColIO<T, V>::load_n(in + (int64_t)li * p.in_elem_stride, nv, aid, x[u]);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) step(REV ? p.len - 1 - (i + u) : i + u, x[u]);
    }
    for (; i < w.i1; ++i) {
        const uint64_t li = REV ? p.len - 1 - i : i;
        A x[V];
        ColIO<T, V>::load_n(in + (int64_t)li * p.in_elem_stride, nv, aid, x);
        step(li, x);
    }
}

// Row-tile column scans: axis 0 of a dense row-major [R, C] matrix of 2 to 24
// columns, where a strip's lanes would mostly be idle.  A tile of `rows`
// whole rows (a multiple of 4, at most kRowTileElems elements) moves between
// HBM and LDS as coalesced 16-byte vectors.  In LDS, thread j owns column j
// mod C over row group j / C, one of G = 512 / C contiguous groups of `rpg`
// rows: it folds its group, the group totals are scanned along the groups
// (row_group_scan), whose last group holds the tile's column totals, and
// after the look-back it rescans its rows in place from the tile's carry and
// the earlier groups' totals before the tile is stored.  Every combination
// runs in ColAcc (f64 for f32).  Mirrored scans take tiles from row R - 1
// down and walk each tile's rows upwards in LDS.  The strided per-line path
// gave these shapes one lane per line (2^28 u32, C = 3: 2.3 ms; C = 12:
// 10 ms).
constexpr int kRowTileThreads = 512;
constexpr uint32_t kRowTileElems = 16384;
constexpr int kRowTileVecsPerThread = (int)(kRowTileElems / 4 / kRowTileThreads);

struct RowTileShape {
    uint64_t R = 0, tiles = 0;
    uint32_t C = 0;
    uint32_t rows = 0;   // rows per tile
    uint32_t groups = 0; // row groups (threads) per column
    uint32_t rpg = 0;    // rows per group
};

RowTileShape row_tile_shape(uint64_t C, uint64_t R) {
    RowTileShape s;
    s.R = R;
    s.C = (uint32_t)C;
    // Whole 128-byte lines per tile (rows * C a multiple of 32), so every
    // tile of an aligned matrix starts on a line: 2^28 u32, C = 3 / 5 / 7 /
    // 10: 465 / 452 / 472 / 472 us -> 453 / 447 / 456 / 466.
    uint32_t m = 32;
    while (m > 4 && C % (32 / m * 2) == 0) m /= 2;
    s.rows = (uint32_t)(kRowTileElems / C) / m * m; // C < 256: at least 64
    s.groups = (uint32_t)(kRowTileThreads / C);
    // An odd group length keeps the lanes of one wave (64 / C groups, C * rpg
    // elements apart in LDS) off a common bank: with C = 2 and 32 rows per
    // group every lane of a wave hit one bank (2^28 u32: 1081 us).
    s.rpg = ((s.rows + s.groups - 1) / s.groups) | 1u;
    s.tiles = ceil_div(R, (uint64_t)s.rows);
    return s;
}

// Tile t's physical rows [r0, r0 + n).
template <bool REV>
__device__ __forceinline__ void row_tile_span(const RowTileShape &s, uint64_t t, uint64_t &r0, uint32_t &n) {
    const uint64_t a = t * s.rows;
    const uint64_t b = a + s.rows < s.R ? a + s.rows : s.R;
    n = (uint32_t)(b - a);
    r0 = REV ? s.R - b : a;
}

// ne elements from src (4-byte aligned) straight into the 16-byte aligned LDS
// tile (tile_load_lds): no register round trip and no LDS write
// instructions (2^28 u32 scans, 2-4% faster than loads into registers and
// 16-byte LDS writes: C = 4 437 -> 422 us, C = 24 514 -> 502).
template <typename T> __device__ __forceinline__ void row_tile_load(const T *src, uint32_t ne, T *tile) {
    tile_load_lds<kRowTileThreads, kRowTileVecsPerThread>(src, ne, tile);
}

template <typename T> __device__ __forceinline__ void row_tile_store(const T *tile, uint32_t ne, T *dst) {
    using VA = typename Vec4A4<T>::type;
    using VL = typename Vec4<T>::type;
    const uint32_t nv = ne / 4;
#pragma unroll
    for (int u = 0; u < kRowTileVecsPerThread; ++u) {
        const uint32_t v = threadIdx.x + (uint32_t)u * kRowTileThreads;
        if (v < nv) store_a4<true>((VA)(*(const VL *)(tile + 4 * v)), (VA *)(dst + 4 * v));
    }
    const uint32_t e = 4 * nv + threadIdx.x;
    if (e < ne) __builtin_nontemporal_store(tile[e], dst + e);
}

// Fold of column c over logical rows [lo, hi) of a tile of n rows (logical
// row i is physical row n - 1 - i when mirrored), eight LDS reads in flight.
template <typename T, typename Op, bool REV>
__device__ __forceinline__ typename ColAcc<T>::type row_group_fold(const T *tile, uint32_t n, uint32_t C, uint32_t c,
                                                                  uint32_t lo, uint32_t hi) {
    using A = typename ColAcc<T>::type;
    A acc = Op::template identity<A>();
    uint32_t i = lo;
    for (; i + 8 <= hi; i += 8) {
        T x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = tile[(REV ? n - 1 - (i + u) : i + u) * C + c];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = Op::combine(acc, (A)x[u]);
    }
    for (; i < hi; ++i) acc = Op::combine(acc, (A)tile[(REV ? n - 1 - i : i) * C + c]);
    return acc;
}

// Inclusive scan of the group totals gtot[g * C + c] along the groups of
// each column, in place: Hillis-Steele steps over LDS, two barriers each,
// in an order fixed by the shape.  Folding the earlier groups one LDS read
// at a time took a thread up to 169 dependent reads (C = 3) per tile.  Every
// thread of the block calls it.
template <typename A, typename Op>
__device__ __forceinline__ void row_group_scan(A *gtot, uint32_t groups, uint32_t C, uint32_t j, bool owner,
                                               uint32_t g) {
    for (uint32_t d = 1; d < groups; d <<= 1) {
        const bool take = owner && g >= d;
        A o = Op::template identity<A>();
        if (take) o = gtot[j - d * C];
        __syncthreads();
        if (take) gtot[j] = Op::combine(o, gtot[j]);
        __syncthreads();
    }
}

// Rescan of column c over logical rows [lo, hi) in place from `pre` (the
// carry into the group), eight rows read before they are rewritten.
template <typename T, typename Op, bool EXCL, bool REV>
__device__ __forceinline__ void row_group_rescan(T *tile, uint32_t n, uint32_t C, uint32_t c, uint32_t lo,
                                                 uint32_t hi, typename ColAcc<T>::type pre) {
    using A = typename ColAcc<T>::type;
    auto step = [&](T &slot, T x) {
        if constexpr (EXCL) {
            slot = (T)pre;
            pre = Op::combine(pre, (A)x);
        } else {
            pre = Op::combine(pre, (A)x);
            slot = (T)pre;
        }
    };
    uint32_t i = lo;
    for (; i + 8 <= hi; i += 8) {
        T x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = tile[(REV ? n - 1 - (i + u) : i + u) * C + c];
#pragma unroll
        for (int u = 0; u < 8; ++u) step(tile[(REV ? n - 1 - (i + u) : i + u) * C + c], x[u]);
    }
    for (; i < hi; ++i) {
        T &slot = tile[(REV ? n - 1 - i : i) * C + c];
        step(slot, slot);
    }
}

// Single-pass row-tile column scan: the row tiles above with a decoupled
// look-back over C-wide carries, so every element is read once and written
// once.  Status entry (tile u, column c) is u * C + c.  After its groups'
// totals, tile t publishes its column aggregates (threads c < C), and the
// whole block looks back in rounds: thread j reads predecessor k = j / C
// (tile t - 1 - base - k) in column c = j mod C, so a round covers 512 / C
// predecessors; per column the nearest inclusive prefix of the round is an
// LDS atomicMin of k; entries up to it that are not ready are polled again,
// and after p.spin_limit polls the waiter rebuilds that predecessor's column
// aggregate from the input (rowtile_column_aggregate: the same group sums,
// folded in group order, so integers match the owner's bits and f32 its value
// to rounding) and uses it, so progress never depends on dispatch order.  The round's needed values fold over k through an LDS tree
// into the column carry, which is published with the tile's aggregate as the
// inclusive prefix.  Tile 0's value is always its prefix; an only tile
// publishes nothing.  f32 carries are
// f64 in 16-byte slots (F64QuadDense), integers packed words.  An f32
// carry's f64 rounding depends on which predecessors had published prefixes:
// results agree with the f64 scan to within its bound, not bit for bit across
// runs.  2^28 u32, us, against totals, carries and a rescan in three
// launches: C = 2 556 -> 474, 3 599 -> 471, 7 608 -> 473, 12 606 -> 468, 24
// 579 -> 514; at C = 48 / 100 / 255 (a round covering 10 / 5 / 2
// predecessors) one pass of these tiles took 622 / 800 / 1093.
template <typename T, typename Op, bool REV>
__device__ __forceinline__ typename ColAcc<T>::type rowtile_column_aggregate(const ScanParams &p, const RowTileShape &s,
                                                                         uint64_t u, uint32_t c) {
    using A = typename ColAcc<T>::type;
    const uint32_t C = s.C;
    uint64_t r0;
    uint32_t n;
    row_tile_span<REV>(s, u, r0, n);
    const T *base = (const T *)p.in + p.in_offset + r0 * C + c;
    A tot = Op::template identity<A>();
    for (uint32_t g = 0; g < s.groups; ++g) {
        const uint32_t lo = g * s.rpg < n ? g * s.rpg : n;
        const uint32_t hi = lo + s.rpg < n ? lo + s.rpg : n;
        A acc = Op::template identity<A>();
        for (uint32_t i = lo; i < hi; ++i) acc = Op::combine(acc, (A)base[(uint64_t)(REV ? n - 1 - i : i) * C]);
        tot = Op::combine(tot, acc);
    }
    return tot;
}

template <typename T, typename Op, typename Status, bool EXCL, bool REV>
__global__ __launch_bounds__(kRowTileThreads) __attribute__((amdgpu_waves_per_eu(4)))
void col_rowtile_lookback_kernel(ScanParams p, RowTileShape s, Status st) {
    using A = typename ColAcc<T>::type;
    __shared__ __attribute__((aligned(16))) T tile[kRowTileElems];
    __shared__ A gtot[kRowTileThreads];
    __shared__ A lb_val[kRowTileThreads];
    __shared__ A s_agg[256], s_carry[256];
    __shared__ uint32_t s_first[256], s_done[256];
    __shared__ uint32_t s_rows;
    const uint64_t t = p.tile0 + blockIdx.x; // scan order: the look-back needs dispatch order
    const uint32_t C = s.C;
    const A aid = Op::template identity<A>();
    uint64_t r0;
    uint32_t n;
    row_tile_span<REV>(s, t, r0, n);
    row_tile_load<T>((const T *)p.in + p.in_offset + r0 * C, n * C, tile);
    __syncthreads();
    const uint32_t j = threadIdx.x, g = j / C, c = j - g * C;
    const bool owner = g < s.groups;
    const uint32_t lo = g * s.rpg < n ? g * s.rpg : n;
    const uint32_t hi = lo + s.rpg < n ? lo + s.rpg : n;
    if (owner) gtot[j] = row_group_fold<T, Op, REV>(tile, n, C, c, lo, hi);
    __syncthreads();
    row_group_scan<A, Op>(gtot, s.groups, C, j, owner, g);
    if (j < C) {
        const A tot = gtot[(s.groups - 1) * C + j];
        s_agg[j] = tot;
        if (s.tiles > 1) st.publish_tile(t * C + j, p.tag, t == 0 ? kPrefix : kAggregate, tot);
        s_carry[j] = aid;
        s_done[j] = t == 0 ? 1u : 0u;
    }
    __syncthreads();
    if (t > 0) {
        const uint32_t KP = kRowTileThreads / C; // predecessors per round
        const uint32_t k = j / C, kc = j - k * C;
        // Lanes of this wave below this one in the same column (l - C,
        // l - 2C, ...): of a wave's prefix flags in one column only the
        // lowest lane's goes to LDS, so the atomics on a column's word stay
        // at one per wave (one per thread took C = 3 scans from 456 to
        // about 580 us).
        const int lane = lane_id();
        uint64_t below = 0;
        for (int l = lane - (int)C; l >= 0; l -= (int)C) below |= 1ull << l;
        uint64_t base = 0;
        for (;;) {
            const bool item = k < KP && base + k < t && s_done[kc] == 0u;
            const uint64_t u = t - 1 - base - k;
            uint32_t flag = kInvalid;
            A val = aid;
            if (item) st.read(u * C + kc, p.tag, flag, val);
            uint32_t spins = 0;
            bool need;
            for (;;) {
                if (j < C) s_first[j] = KP;
                if (j == 0) s_rows = 0;
                __syncthreads();
                const bool pre = item && flag == kPrefix;
                const uint64_t pm = ballot(pre);
                if (pre && (pm & below) == 0ull) atomicMin(&s_first[kc], k);
                __syncthreads();
                need = item && k <= s_first[kc];
                const bool missing = need && flag == kInvalid;
                if (!__syncthreads_or(missing)) break;
                if (++spins >= p.spin_limit) {
                    if (missing) {
                        val = rowtile_column_aggregate<T, Op, REV>(p, s, u, kc);
                        flag = u == 0 ? kPrefix : kAggregate; // tile 0's aggregate is its prefix
                    }
                    spins = 0;
                } else {
                    __builtin_amdgcn_s_sleep(1);
                    if (missing) st.read(u * C + kc, p.tag, flag, val);
                }
            }
            // Fold the round's needed values over k (rows of a [KP][C]
            // array) in a fixed tree as deep as the deepest needed row, then
            // into the column carries.
            lb_val[j] = need ? val : aid;
            const uint32_t deep =
                group_reduce<64>(need ? k + 1 : 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
            if (lane == 0 && deep > 0) atomicMax(&s_rows, deep);
            __syncthreads();
            for (uint32_t cur = s_rows; cur > 1;) {
                const uint32_t half = (cur + 1) / 2;
                if (j < (cur - half) * C) lb_val[j] = Op::combine(lb_val[j], lb_val[j + half * C]);
                __syncthreads();
                cur = half;
            }
            bool pending = false;
            if (j < C && s_done[j] == 0u) {
                s_carry[j] = Op::combine(s_carry[j], lb_val[j]);
                if (s_first[j] < KP) s_done[j] = 1u;
                else pending = true;
            }
            if (!__syncthreads_or(pending)) break;
            base += KP;
        }
        if (j < C) st.publish_tile(t * C + j, p.tag, kPrefix, Op::combine(s_carry[j], s_agg[j]));
        __syncthreads();
    }
    if (owner) {
        A pre = s_carry[c];
        if (g > 0) pre = Op::combine(pre, gtot[j - C]);
        row_group_rescan<T, Op, EXCL, REV>(tile, n, C, c, lo, hi, pre);
    }
    __syncthreads();
    row_tile_store<T>(tile, n * C, (T *)p.out + p.out_offset + r0 * C);
}

// Single-pass column scan.  A block owns a tile of kColTileRows scan steps x
// 64*V adjacent lines.  Its kColDataWaves data waves each hold kColRows
// steps of the tile in registers (lane l: lines 64*V*g + V*l .. +V-1), scan
// them per line, and combine their totals through LDS.  The block's last
// wave holds no data: it runs the decoupled look-back, lane l for its V
// lines, polling kColPoll earlier chunks of the same line group per round
// trip and folding aggregates until each line meets an inclusive prefix.
// Integer scans publish one packed word per line and chunk; f32 scans an
// f64 carry in a two-word slot (F64PairStatus), with the tile's steps
// scanned in f32 and the carries and outputs formed in f64.
// Data and look-back waves run separate code paths (wave-uniform), so the
// tile's registers are not live during the look-back.  Status entry of
// (chunk c, line j) is c * lpad + j.  Every element is read once and written
// once.  A predecessor that stays unpublished for p.spin_limit rounds has its
// aggregate rebuilt from the input by the waiter with the owner's arithmetic
// (f32: per-wave f32 prefix from the identity, then f64 over the waves in
// order) and used directly, so progress never depends on dispatch order.
constexpr int kColWaves = 16;
constexpr int kColDataWaves = kColWaves - 1;
constexpr int kColRows = 16;
constexpr uint64_t kColTileRows = (uint64_t)kColDataWaves * kColRows;
// Predecessor chunks polled per round trip.  Status reads are device-scope
// and uncached, and wider polls cost more than the round trips they save
// (u32, 65536 x 4096 / 1048576 x 256: 1 chunk 0.352 / 0.462 ms; 2: 0.354 /
// 0.491; 4: 0.361 / 0.568; 8: 0.384 / 0.762).
constexpr int kColPoll = 1;

template <typename T, int V>
__device__ __forceinline__ void col_load_t(const T *p, T (&x)[V]) {
    if constexpr (V == 4) {
        using Vt = typename Vec4A4<T>::type;
        const Vt v = __builtin_nontemporal_load((const Vt *)p);
        x[0] = (T)v.x;
        x[1] = (T)v.y;
        x[2] = (T)v.z;
        x[3] = (T)v.w;
    } else {
        x[0] = __builtin_nontemporal_load(p);
    }
}

template <typename T, int V>
__device__ __forceinline__ void col_store_t(T *p, const T (&y)[V]) {
    if constexpr (V == 4) {
        using Vt = typename Vec4A4<T>::type;
        Vt v;
        v.x = y[0];
        v.y = y[1];
        v.z = y[2];
        v.w = y[3];
        __builtin_nontemporal_store(v, (Vt *)p);
    } else {
        __builtin_nontemporal_store(y[0], p);
    }
}

// The same for the lane of a partial group: its nv < V lines one by one,
// the others read as `ident` and never stored.
template <typename T, int V>
__device__ __forceinline__ void col_load_n(const T *p, uint32_t nv, T ident, T (&x)[V]) {
    if (V == 1 || nv >= (uint32_t)V) {
        col_load_t<T, V>(p, x);
        return;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) x[v] = (uint32_t)v < nv ? __builtin_nontemporal_load(p + v) : ident;
}

template <typename T, int V>
__device__ __forceinline__ void col_store_n(T *p, uint32_t nv, const T (&y)[V]) {
    if (V == 1 || nv >= (uint32_t)V) {
        col_store_t<T, V>(p, y);
        return;
    }
#pragma unroll
    for (int v = 0; v < V; ++v)
        if ((uint32_t)v < nv) __builtin_nontemporal_store(y[v], p + v);
}

// Aggregate of chunk c for the V lines starting at line0, exactly as the
// owner computes it (the decoupled fallback).
template <typename T, typename Op, int V, bool REV>
__device__ void col_tile_aggregate(const ScanParams &p, uint64_t c, uint64_t line0,
                                   typename ColAcc<T>::type (&agg)[V]) {
    using A = typename ColAcc<T>::type;
    const T *in = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)line0 * p.in_line_stride);
    const uint32_t nv = col_valid_lines(p.lines, line0, V);
#pragma unroll
    for (int v = 0; v < V; ++v) agg[v] = Op::template identity<A>();
    // Rolled loops: this rare path must not add register pressure to the
    // kernel, whose tile stays live in registers across the look-back.
#pragma unroll 1
    for (int q = 0; q < kColDataWaves; ++q) {
        T run[V];
#pragma unroll
        for (int v = 0; v < V; ++v) run[v] = Op::template identity<T>();
#pragma unroll 1
        for (int r = 0; r < kColRows; ++r) {
            const uint64_t i = c * kColTileRows + (uint64_t)q * kColRows + r;
            if (i >= p.len) break;
            const uint64_t li = REV ? p.len - 1 - i : i;
            T x[V];
            col_load_n<T, V>(in + (int64_t)li * p.in_elem_stride, nv, Op::template identity<T>(), x);
#pragma unroll
            for (int v = 0; v < V; ++v) run[v] = Op::combine(run[v], x[v]);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) agg[v] = Op::combine(agg[v], (A)run[v]);
    }
}

// Addressing of a line group: a wave-uniform element base (the group's
// lowest address on every step) and one 32-bit byte offset per lane, so each
// access is a scalar base plus a vector offset and no per-step 64-bit address
// stays live across the look-back.
struct ColGroupAddr {
    int64_t base;      // element offset of the group's lowest line, step 0
    uint32_t lane_off; // bytes from there to this lane's first line
};

template <int V, typename T>
__device__ __forceinline__ ColGroupAddr col_group_addr(uint64_t g, int lane, int64_t line_stride, uint64_t offset) {
    constexpr int64_t kGroup = (int64_t)kWave * V;
    ColGroupAddr a;
    if (line_stride > 0) {
        a.base = (int64_t)offset + (int64_t)g * kGroup;
        a.lane_off = (uint32_t)(lane * V) * (uint32_t)sizeof(T);
    } else { // -1: lines run downwards in memory (one line per lane)
        a.base = (int64_t)offset - ((int64_t)g * kGroup + kGroup - 1);
        a.lane_off = (uint32_t)(kGroup - 1 - lane * V) * (uint32_t)sizeof(T);
    }
    return a;
}

// The look-back wave: publishes the tile's aggregate, folds its
// predecessors' statuses per line (kColPoll chunks per round trip, consumed
// in order and in step for all of the lane's lines, so no status is counted
// twice), publishes the inclusive prefix and leaves the carry in s_carry.
template <typename T, typename Op, typename Status, int V, bool REV>
__device__ void col_lookback_wave(const ScanParams &p, const Status &st, uint64_t c, uint64_t lpad, uint64_t line0,
                                  bool active, const typename ColAcc<T>::type (&agg)[V],
                                  typename ColAcc<T>::type (&excl)[V]) {
    using A = typename ColAcc<T>::type;
    constexpr int P = kColPoll;
    const A aid = Op::template identity<A>();
#pragma unroll
    for (int v = 0; v < V; ++v) excl[v] = aid;
    if (!active) return;
    const uint64_t e = c * lpad + line0;
    if (c == 0) {
#pragma unroll
        for (int v = 0; v < V; ++v) st.publish_tile(e + v, p.tag, kPrefix, agg[v]);
        return;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) st.publish_tile(e + v, p.tag, kAggregate, agg[v]);
    bool done[V];
#pragma unroll
    for (int v = 0; v < V; ++v) done[v] = false;
    uint64_t pos = c - 1; // next predecessor to consume
    uint32_t spins = 0;
    for (;;) {
        uint32_t flag[P][V];
        A val[P][V];
#pragma unroll
        for (int k = 0; k < P; ++k)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                flag[k][v] = kInvalid;
                val[k][v] = aid;
                if (!done[v] && (uint64_t)k <= pos) st.read((pos - k) * lpad + line0 + v, p.tag, flag[k][v], val[k][v]);
            }
        // The next predecessor not ready for some line: wait, and after
        // p.spin_limit polls take its aggregate from the input (the owner's
        // arithmetic) and use it directly -- so progress never depends on
        // dispatch order.  Publishing it is only a courtesy to other
        // waiters, and is skipped where a status slot must keep one writer.
        bool ready0 = true;
#pragma unroll
        for (int v = 0; v < V; ++v) ready0 = ready0 && (done[v] || flag[0][v] != kInvalid);
        if (!ready0) {
            if (++spins < p.spin_limit) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            A fb[V];
            col_tile_aggregate<T, Op, V, REV>(p, pos, line0, fb);
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (!done[v] && flag[0][v] == kInvalid) {
                    st.publish_if_unset(pos * lpad + line0 + v, p.tag, kAggregate, fb[v]);
                    flag[0][v] = kAggregate;
                    val[0][v] = fb[v];
                }
        }
        spins = 0;
        int used = 0;
        bool finished = false;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (finished || used < k || (uint64_t)k > pos) break;
            bool ready = true;
#pragma unroll
            for (int v = 0; v < V; ++v) ready = ready && (done[v] || flag[k][v] != kInvalid);
            if (!ready) break;
            // Chunk 0's aggregate is its inclusive prefix: a fallback may
            // have published it as an aggregate, and consuming it still
            // finishes the line.
            const bool first_chunk = (uint64_t)k == pos;
            bool all = true;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if (done[v]) continue;
                excl[v] = Op::combine(val[k][v], excl[v]);
                if (flag[k][v] == kPrefix || first_chunk) done[v] = true;
                else all = false;
            }
            used = k + 1;
            finished = all;
        }
        if (finished) break;
        pos -= (uint64_t)used; // used >= 1 (entry pos was ready); chunk 0 finishes every line
    }
#pragma unroll
    for (int v = 0; v < V; ++v) st.publish_tile(e + v, p.tag, kPrefix, Op::combine(excl[v], agg[v]));
}

template <typename T, typename Op, typename Status, int V, bool EXCL, bool REV>
__global__ __launch_bounds__(kColWaves *kWave) void col_lookback_kernel(ScanParams p, Status st, uint64_t groups,
                                                                        uint64_t lpad) {
    using A = typename ColAcc<T>::type;
    constexpr int kLines = kWave * V;
    __shared__ A s_agg[kColDataWaves][kLines];
    __shared__ A s_carry[kLines];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = lane_id();
    const uint64_t tile = blockIdx.x;
    const uint64_t g = tile % groups, c = tile / groups;
    const uint64_t line0 = (g * kWave + (uint64_t)lane) * V;
    const bool active = line0 < p.lines;
    const uint32_t nv = active ? col_valid_lines(p.lines, line0, V) : 0u;
    const A aid = Op::template identity<A>();

    if (w == kColDataWaves) {
        __syncthreads(); // the data waves' totals
        A agg[V], excl[V];
#pragma unroll
        for (int v = 0; v < V; ++v) agg[v] = aid;
#pragma unroll 1
        for (int q = 0; q < kColDataWaves; ++q)
#pragma unroll
            for (int v = 0; v < V; ++v) agg[v] = Op::combine(agg[v], s_agg[q][lane * V + v]);
        col_lookback_wave<T, Op, Status, V, REV>(p, st, c, lpad, line0, active, agg, excl);
#pragma unroll
        for (int v = 0; v < V; ++v) s_carry[lane * V + v] = excl[v];
        __syncthreads(); // the carry
        return;
    }

    const uint64_t i0 = c * kColTileRows + (uint64_t)w * kColRows;
    const ColGroupAddr ia = col_group_addr<V, T>(g, lane, p.in_line_stride, p.in_offset);
    const ColGroupAddr oa = col_group_addr<V, T>(g, lane, p.out_line_stride, p.out_offset);
    const T tid = Op::template identity<T>();

    // The wave's steps, scanned per line from the identity.
    T x[kColRows][V];
#pragma unroll
    for (int r = 0; r < kColRows; ++r) {
        const uint64_t i = i0 + r;
        if (active && i < p.len) {
            const int64_t li = (int64_t)(REV ? p.len - 1 - i : i);
            const char *row = (const char *)((const T *)p.in + (ia.base + li * p.in_elem_stride));
            col_load_n<T, V>((const T *)(row + ia.lane_off), nv, tid, x[r]);
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) x[r][v] = tid;
        }
    }
#pragma unroll
    for (int r = 0; r < kColRows; ++r)
#pragma unroll
        for (int v = 0; v < V; ++v) x[r][v] = Op::combine(r == 0 ? tid : x[r - 1][v], x[r][v]);
#pragma unroll
    for (int v = 0; v < V; ++v) s_agg[w][lane * V + v] = (A)x[kColRows - 1][v];
    __syncthreads(); // totals to the look-back wave
    __syncthreads(); // its carry
    if (!active) return;

    A carry[V];
#pragma unroll
    for (int v = 0; v < V; ++v) carry[v] = s_carry[lane * V + v];
#pragma unroll 1
    for (int q = 0; q < w; ++q)
#pragma unroll
        for (int v = 0; v < V; ++v) carry[v] = Op::combine(carry[v], s_agg[q][lane * V + v]);
#pragma unroll
    for (int r = 0; r < kColRows; ++r) {
        const uint64_t i = i0 + r;
        if (i >= p.len) break;
        T y[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if constexpr (EXCL)
                y[v] = r == 0 ? finalize<T, A, Op>(carry[v], tid) : finalize<T, A, Op>(carry[v], x[r - 1][v]);
            else
                y[v] = finalize<T, A, Op>(carry[v], x[r][v]);
        }
        const int64_t li = (int64_t)(REV ? p.len - 1 - i : i);
        char *row = (char *)((T *)p.out + (oa.base + li * p.out_elem_stride));
        col_store_n<T, V>((T *)(row + oa.lane_off), nv, y);
    }
}

// Strip column scans: many lines adjacent in memory (axis 0 of a row-major
// matrix), read and written once.  The lines are cut into strips of W (32 or
// 64) and the scan axis into chunks; a block owns one chunk of one strip.  Its
// data waves put W / 4 lanes on a row (one 16-byte vector of four lines each)
// and 256 / W rows on a load instruction; a lane takes STEPS consecutive rows
// and keeps them in registers.  The lanes' totals go to LDS, and the block's
// last wave, which holds no data, turns them into the lanes' exclusive
// prefixes (a lane per line), publishes the chunk's totals and looks back over
// the strip's earlier chunks, P statuses per line in flight, while the data
// waves wait at the barrier; each lane then rescans its rows from the carry.
// Integers wrap in u32; f32 totals, carries and running values are all f64.
//
// Why strips: a look-back's length is the number of chunks that load at the
// same time, and its cost one round trip (1.5 to 2.5 us) per P chunks.  A
// strip of 64 lines leaves room for 448 rows in a block of 8 waves, against
// 240 rows of 256 lines in the 16-wave tiles of col_lookback_kernel, and gives
// a matrix four times as many chains.  Below 256 lines it replaces three
// passes (totals, carries, rescan), 12 bytes an element instead of 8.
// Measured on MI355X, 2^26 elements, u32 / f32, us: [2^21, 32] 138 / 142 ->
// 86 / 119; [2^20, 64] 142 / 144 -> 86 / 120; [2^19, 128] 143 / 145 -> 86 / 109;
// [65536, 1024] 102 / 130 -> 91 / 92; smaller, u32: [510, 659] 11.9 -> 5.3,
// [1146, 90] 11.8 -> 5.6, [4096, 1024] 15.6 -> 7.2.  (f32 below 256 lines looks
// back in order; 103, 106 and 95 for the first three without.)
//
// Whole 128-byte lines (row pitch and output start multiples of 128 bytes)
// are stored non-temporally.  Elsewhere neighbouring strips share the lines
// at their edges, and a non-temporal store of part of a line costs a
// read-modify-write in memory: such strips store through the L2, and the
// blocks are dealt so that the strips that share lines run on one XCD, whose
// L2 then merges the parts (StripDeal).  [700001, 100] u32: 193 us
// non-temporal, 139 through the L2, 105 with the deal (three passes: 148);
// [165595, 486] f32 229, 185, 136 (184).
enum StripDeal : uint32_t {
    kDealRows = 0,   // block b: strip b mod groups of chunk b / groups
    kDealChunks = 1, // every chunk's strips on one XCD, chunks round robin
    kDealStrips = 2, // an eighth of the strips on each XCD
};

constexpr int kStripWaves = 8;
template <int W, int STEPS> struct StripGeom {
    static_assert(W == 32 || W == 64, "strips of 32 or 64 lines");
    static constexpr int kDataWaves = kStripWaves - 1;
    static constexpr int kLanesPerRow = W / 4;
    static constexpr int kSub = kWave / kLanesPerRow; // rows per load instruction
    static constexpr int kParts = kDataWaves * kSub;  // lanes along the axis
    static constexpr uint64_t kRows = (uint64_t)kParts * STEPS;
};

// Statuses in flight per line: the f32 slots are 16 bytes, and four of them
// a line took [2^19, 128] from 99 us to 103, [8192, 256] from 9.9 to 11.0.
template <typename T> struct StripPolls { static constexpr int value = 4; };
template <> struct StripPolls<float> { static constexpr int value = 2; };

// The last wave's look-back: lane l < W (live where the line exists) folds
// its line's statuses of the chunks before `c`, nearest first, P per round
// trip, consumed in order and in step for the whole wave, and publishes the
// line's inclusive prefix.  Entry (chunk, line) of the status array is
// chunk * lpad + entry.  A chunk that stays unpublished for p.spin_limit polls
// is totalled from the input by the waiter, so progress never depends on the
// dispatch order; the value is not published (every slot has one writer).
// `base` is the line's total before the launch's first chunk (the identity,
// but for a scan cut into several launches).  A launch of one chunk publishes nothing (its status area is not allocated).
template <typename T, typename Op, typename Status, uint64_t ROWS, bool REV>
__device__ void strip_lookback(const ScanParams &p, const Status &st, uint64_t c, uint64_t chunks, uint64_t lpad,
                               uint64_t line, uint64_t entry, bool live, typename ColAcc<T>::type base,
                               typename ColAcc<T>::type agg, typename ColAcc<T>::type &excl) {
    using A = typename ColAcc<T>::type;
    constexpr int P = StripPolls<T>::value;
    if (c == 0) {
        excl = base;
        if (live && chunks > 1) st.publish_tile(entry, p.tag, kPrefix, Op::combine(excl, agg));
        return;
    }
    excl = Op::template identity<A>();
    if (live) st.publish_tile(c * lpad + entry, p.tag, kAggregate, agg);
    bool done = !live;
    uint64_t pos = c - 1; // next chunk to consume
    uint32_t spins = 0;
    for (;;) {
        uint32_t flag[P];
        A val[P];
        // Every lane reads (chunk 0 past the start): straight-line loads stay
        // in flight together.
#pragma unroll
        for (int k = 0; k < P; ++k)
            st.read((pos >= (uint64_t)k ? pos - k : 0) * lpad + entry, p.tag, flag[k], val[k]);
        uint32_t used = 0;
        bool finished = false;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (finished || used != (uint32_t)k || pos < (uint64_t)k) continue;
            if (ballot(!done && flag[k] == kInvalid) != 0ull) continue;
            if (!done) {
                excl = Op::combine(val[k], excl);
                done = flag[k] == kPrefix || pos == (uint64_t)k; // chunk 0 ends every line
            }
            used = k + 1;
            finished = ballot(!done) == 0ull;
        }
        if (finished) break;
        pos -= used; // chunk 0 finishes, so used <= pos here
        if (used != 0) {
            spins = 0;
            continue;
        }
        if (++spins < p.spin_limit) {
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        spins = 0;
        A t = Op::template identity<A>();
        if (live) {
            const T *in = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)line);
#pragma unroll 8
            for (uint64_t i = pos * ROWS; i < (pos + 1) * ROWS; ++i) // earlier chunks are whole
                t = Op::combine(t, (A)in[(int64_t)(REV ? p.len - 1 - i : i) * p.in_elem_stride]);
        }
        if (!done) {
            const bool missing = flag[0] == kInvalid;
            if (pos == 0) t = Op::combine(base, t); // chunk 0 publishes its prefix
            excl = Op::combine(missing ? t : val[0], excl);
            done = (!missing && flag[0] == kPrefix) || pos == 0;
        }
        if (ballot(!done) == 0ull) break;
        pos -= 1;
    }
    if (live) st.publish_tile(c * lpad + entry, p.tag, kPrefix, Op::combine(excl, agg));
}

// The ordered look-back of f32 matrices below kOrderedMaxLines: results are
// the same bits in every run.  (In the walk above an f64 sum's grouping
// depends on the prefix that was met first.)  Chunks form groups of kStripGroup.  A chunk publishes its total, never a
// prefix.  The last chunk of a group also publishes the group's total, and
// then the line's total through the group, its prefix.  A chunk folds the
// totals of its group's earlier chunks, from the first on, and then walks back
// over whole groups, nearest first, to the first prefix and folds forward from
// there.  So each prefix is the fold, from the left, of all group totals
// before it, whichever prefixes the look-backs met.  A group's entries lie
// after the chunks', (group, line) like (chunk, line).
//
// A status that stays unpublished for p.spin_limit polls is rebuilt by the
// waiter with its owner's arithmetic: a chunk's total from the input, a
// group's from its chunks.  One loop over chunks serves both: a launch fetches
// its code cold, and with the loop in three places [240, 64] took 5.4 us
// against 5.1.
//
// f32, us, first prefix met / prefixes of chunks, every total kept and folded
// forward / groups: [16384, 64] 12.3 / 17.1 / 15.0, [524288, 64] 57.5 / 188 / 65.3,
// [2097152, 64] 199 / 782 / 225.
constexpr int kStripGroup = 16;
constexpr int kStripChunkPolls = 3, kStripGroupPolls = 2; // statuses in flight per line

// 64-bit words of a status.
template <typename T> constexpr uint64_t kStripSlotWords = std::is_same<T, float>::value ? 2 : 1;

template <typename T, typename Op, typename Status, int PARTS, int STEPS, bool REV>
__device__ typename ColAcc<T>::type strip_ordered_lookback(const ScanParams &p, const Status &st, uint64_t c,
                                                           uint64_t count, uint64_t lpad, uint64_t line,
                                                           uint64_t entry, bool live, typename ColAcc<T>::type base,
                                                           typename ColAcc<T>::type own) {
    using A = typename ColAcc<T>::type;
    const Status groups{st.words + count * lpad * kStripSlotWords<T>};
    const A id = Op::template identity<A>();
    if (live && count > 1) st.publish_tile(c * lpad + entry, p.tag, kAggregate, own);
    const uint64_t g = c / kStripGroup;
    const bool ends = c % kStripGroup == kStripGroup - 1 && c + 1 < count; // its group, with more to come
    uint64_t lo = g * kStripGroup, hi = c; // chunks to fold
    A before = id, through = id; // own group's total before and after this chunk
    A prefix = id;               // the line's total through group g - 1
    uint64_t at = g;             // group under way: back down to a prefix, then forward to g - 1
    uint64_t found = 0;          // the group whose prefix this lane met
    bool own_group = true, back = true, done = !live;
    for (;;) {
        // Fold of the totals of chunks [lo, hi), in order.
        A sum = id;
        uint32_t spins = 0;
        while (lo < hi) {
            constexpr int P = kStripChunkPolls;
            uint32_t flag[P];
            A val[P];
            // Straight-line loads stay in flight together (past the end: the
            // last one again); a wait polls one status.
#pragma unroll
            for (int k = 0; k < P; ++k) {
                flag[k] = kInvalid;
                if (k == 0 || spins == 0) st.read((lo + k < hi ? lo + k : hi - 1) * lpad + entry, p.tag, flag[k], val[k]);
            }
            uint32_t used = 0;
#pragma unroll
            for (int k = 0; k < P; ++k) {
                if (used != (uint32_t)k || lo + k >= hi) continue;
                if (ballot(live && flag[k] == kInvalid) != 0ull) continue;
                sum = Op::combine(sum, val[k]);
                used = k + 1;
            }
            lo += used;
            if (used != 0) {
                spins = 0;
            } else if (++spins < p.spin_limit) {
                __builtin_amdgcn_s_sleep(1);
            } else {
                // The total with its owner's arithmetic: each lane's STEPS
                // rows, the lanes' totals in order.
                A t = id;
                if (live) {
                    const T *in = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)line);
                    for (int e = 0; e < PARTS; ++e) {
                        A part = id;
#pragma unroll 4
                        for (int k = 0; k < STEPS; ++k) {
                            const uint64_t i = (lo * PARTS + e) * STEPS + k; // earlier chunks are whole
                            part = Op::combine(part, (A)in[(int64_t)(REV ? p.len - 1 - i : i) * p.in_elem_stride]);
                        }
                        t = Op::combine(t, part);
                    }
                }
                sum = Op::combine(sum, flag[0] == kInvalid ? t : val[0]);
                ++lo;
                spins = 0;
            }
        }
        // A rebuilt value of group `at`, and whether there is one.
        A rebuilt = id;
        bool have = false;
        if (own_group) {
            own_group = false;
            before = sum;
            through = Op::combine(before, own);
            if (g == 0) {
                if (live && ends) groups.publish_tile(entry, p.tag, kPrefix, Op::combine(base, through));
                return Op::combine(base, before);
            }
            if (live && ends) groups.publish_tile(g * lpad + entry, p.tag, kAggregate, through);
            at = g - 1;
        } else {
            rebuilt = at == 0 ? Op::combine(base, sum) : sum;
            have = true;
        }
        // Groups, until the walk ends or one has to be rebuilt.
        spins = 0;
        bool rebuild = false;
        while (!rebuild) {
            constexpr int P = kStripGroupPolls;
            uint32_t flag[P];
            A val[P];
#pragma unroll
            for (int k = 0; k < P; ++k) {
                flag[k] = kInvalid;
                const uint64_t u = back ? (at >= (uint64_t)k ? at - k : 0) : (at + k < g ? at + k : g - 1);
                if (k == 0 || (spins == 0 && !have)) groups.read(u * lpad + entry, p.tag, flag[k], val[k]);
            }
            if (have && flag[0] == kInvalid) {
                flag[0] = at == 0 ? kPrefix : kAggregate; // group 0 publishes only its prefix
                val[0] = rebuilt;
            }
            have = false;
            uint32_t used = 0;
#pragma unroll
            for (int k = 0; k < P; ++k) {
                if (used != (uint32_t)k) continue;
                if (back) {
                    if (at < (uint64_t)k || ballot(!done) == 0ull) continue;
                    if (ballot(!done && flag[k] == kInvalid) != 0ull) continue;
                    if (!done) found = at - k;
                    done = done || flag[k] == kPrefix;
                } else {
                    if (at + k >= g) continue;
                    const bool need = live && at + k >= found;
                    if (ballot(need && flag[k] == kInvalid) != 0ull) continue;
                    if (need) prefix = flag[k] == kPrefix ? val[k] : Op::combine(prefix, val[k]);
                }
                used = k + 1;
            }
            if (back) {
                if (ballot(!done) == 0ull) {
                    // Forward from the group that the furthest lane met; with
                    // one round the values are here.
                    if (at == g - 1) {
#pragma unroll
                        for (int k = P - 1; k >= 0; --k) {
                            if (!live || found + k > at) continue;
                            prefix = found + k == at ? val[k] : Op::combine(prefix, val[k]);
                        }
                        at = g;
                    } else {
                        at = g - 1 - group_reduce<64>(live ? (uint32_t)(g - 1 - found) : 0u,
                                                      [](uint32_t a, uint32_t b) { return a > b ? a : b; });
                    }
                    back = false;
                    used = 1; // no wait
                } else {
                    at -= used;
                }
            } else {
                at += used;
            }
            if (!back && at >= g) break;
            if (used != 0) {
                spins = 0;
            } else if (++spins < p.spin_limit) {
                __builtin_amdgcn_s_sleep(1);
            } else {
                rebuild = true;
            }
        }
        if (!rebuild) break;
        lo = at * kStripGroup;
        hi = lo + kStripGroup;
    }
    if (live && ends) groups.publish_tile(g * lpad + entry, p.tag, kPrefix, Op::combine(prefix, through));
    return Op::combine(prefix, before);
}

struct StripParams {
    uint32_t groups, width; // strips, lines per strip (a multiple of 4, at most W)
    uint32_t deal;          // StripDeal
    uint32_t cached;        // stores go through the L2 (else non-temporal)
    uint64_t lpad;          // status entries per chunk
    uint64_t chunks;        // of this launch
    uint32_t pass;          // StripPass
    void *totals;           // a value a status entry, or (kPassTakes, kPassLeaves) two rows of them
};
// A launch looks back (0) or is one of three that leave the chunks' totals,
// (col_carry_kernel in between) and start from them.  A scan cut along the
// axis takes a launch's line totals on to the next, rows alternating.
// PASSES launches know these forms; the others' look-back is the whole of it
// (what they skip costs a two-chunk scan 0.4 us of cold instruction fetches:
// [240, 100] u32 5.06 us against 4.64).
enum StripPass : uint32_t {
    kPassTotals = 1,  // only leave the chunks' totals
    kPassCarries = 2, // the chunks' carries are there
    kPassTakes = 4,   // row 0 (kPassOdd: 1) holds the lines' totals so far
    kPassLeaves = 8,  // leave them in row 1 (kPassOdd: 0)
    kPassOdd = 16,
};

template <typename T, typename Op, typename Status, int W, int STEPS, bool EXCL, bool REV, bool ORDERED, bool PASSES>
__global__ __launch_bounds__(kStripWaves *kWave) __attribute__((amdgpu_waves_per_eu(ORDERED && STEPS == 8 ? 8 : 4)))
void col_strip_kernel(ScanParams p, StripParams sp, Status st) {
    using A = typename ColAcc<T>::type;
    using G = StripGeom<W, STEPS>;
    using Vt = typename Vec4A4<T>::type;
    __shared__ A s_part[G::kParts][W]; // lane totals, then their exclusive prefixes
    __shared__ A s_carry[W];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = lane_id();
    // Predecessor chunks always have lower block indices.
    uint32_t g;
    uint64_t c;
    if (sp.deal == kDealRows) {
        g = blockIdx.x % sp.groups;
        c = blockIdx.x / sp.groups;
    } else {
        const uint32_t xcd = blockIdx.x % kXcds, q = blockIdx.x / kXcds;
        if (sp.deal == kDealChunks) {
            g = q % sp.groups;
            c = (uint64_t)(q / sp.groups) * kXcds + xcd;
        } else {
            const uint32_t per = (sp.groups + kXcds - 1) / kXcds;
            g = xcd * per + q % per;
            c = q / per;
        }
        if (g >= sp.groups || c >= sp.chunks) return; // the deal's padding
    }
    const uint64_t first = (uint64_t)g * sp.width; // the strip's first line
    const uint32_t cnt = p.lines - first < sp.width ? (uint32_t)(p.lines - first) : sp.width;
    const A aid = Op::template identity<A>();

    const uint32_t pass = PASSES ? sp.pass : 0u;
    if (w == G::kDataWaves) {
        __syncthreads(); // the lanes' totals
        const int l = lane & (W - 1);
        A run = aid;
        if (lane < W) {
#pragma unroll 14
            for (int e = 0; e < G::kParts; ++e) {
                const A v = s_part[e][l];
                s_part[e][l] = run;
                run = Op::combine(run, v);
            }
        }
        const uint64_t entry = (uint64_t)g * W + l;
        const bool live = lane < (int)cnt;
        A *totals = (A *)sp.totals;
        if (pass & kPassTotals) {
            if (live) totals[c * sp.lpad + entry] = run;
            return;
        }
        const uint64_t odd = pass & kPassOdd ? sp.lpad : 0;
        A excl;
        if (pass & kPassCarries) {
            excl = live ? totals[c * sp.lpad + entry] : aid;
        } else {
            A base = aid;
            if ((pass & kPassTakes) && live) base = totals[odd + entry];
            if constexpr (ORDERED)
                excl = strip_ordered_lookback<T, Op, Status, G::kParts, STEPS, REV>(p, st, c, sp.chunks, sp.lpad, first + l,
                                                                                    entry, live, base, run);
            else
                strip_lookback<T, Op, Status, G::kRows, REV>(p, st, c, sp.chunks, sp.lpad, first + l, entry, live, base,
                                                             run, excl);
        }
        if (lane < W) s_carry[l] = excl;
        __syncthreads(); // the carry
        if ((pass & kPassLeaves) && live && c + 1 == sp.chunks) totals[sp.lpad - odd + entry] = Op::combine(excl, run);
        return;
    }

    const uint32_t sub = (uint32_t)lane / G::kLanesPerRow, q = (uint32_t)lane % G::kLanesPerRow;
    // Lane q's lines l0 .. l0 + nv - 1 of the strip.  Where the strip's line
    // count is no multiple of 4 its last lane moves back to a whole vector: the
    // lines it shares with its neighbour get the same values twice.
    const bool active = 4 * q < cnt;
    const uint32_t l0 = cnt < 4 ? 0u : 4 * q + 4 <= cnt ? 4 * q : cnt - 4;
    const uint32_t nv = active ? (cnt < 4 ? cnt : 4u) : 0u;
    const uint32_t part = (uint32_t)w * G::kSub + sub;
    const uint64_t i0 = c * G::kRows + (uint64_t)part * STEPS;
    const bool whole = (c + 1) * G::kRows <= p.len;
    const T tid = Op::template identity<T>();
    T x[STEPS][4];
    {
        const T *src = (const T *)p.in + ((int64_t)p.in_offset + (int64_t)(first + l0) +
                                          (int64_t)(REV ? p.len - 1 - i0 : i0) * p.in_elem_stride);
        const int64_t step = REV ? -p.in_elem_stride : p.in_elem_stride;
        if (whole && nv == 4) {
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                col_load_t<T, 4>(src, x[j]);
                src += step;
            }
        } else {
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                if (active && i0 + j < p.len) {
                    col_load_n<T, 4>(src, nv, tid, x[j]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v) x[j][v] = tid;
                }
                src += step;
            }
        }
    }
    {
        A tot[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) tot[v] = aid;
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) tot[v] = Op::combine(tot[v], (A)x[j][v]);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if ((uint32_t)v < nv) s_part[part][l0 + v] = tot[v];
    }
    __syncthreads(); // totals to the last wave
    if (pass & kPassTotals) return;
    __syncthreads(); // its prefixes and carry
    if (!active) return;
    A run[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const uint32_t l = (uint32_t)v < nv ? l0 + v : l0;
        run[v] = Op::combine(s_carry[l], s_part[part][l]);
    }
    T *dst = (T *)p.out + ((int64_t)p.out_offset + (int64_t)(first + l0) +
                           (int64_t)(REV ? p.len - 1 - i0 : i0) * p.out_elem_stride);
    const int64_t step = REV ? -p.out_elem_stride : p.out_elem_stride;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        if (!whole && i0 + j >= p.len) break;
        T y[4];
        // Opaque: the totals' f64 conversions are not kept for this second
        // use (they would hold 128 registers across the look-back).
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "+v"(x[j][v]));
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if constexpr (EXCL) y[v] = (T)run[v];
            run[v] = Op::combine(run[v], (A)x[j][v]);
            if constexpr (!EXCL) y[v] = (T)run[v];
        }
        if (!sp.cached) {
            col_store_n<T, 4>(dst, nv, y);
        } else if (nv == 4) {
            Vt v;
            v.x = y[0];
            v.y = y[1];
            v.z = y[2];
            v.w = y[3];
            *(Vt *)dst = v;
        } else {
#pragma unroll
            for (int v = 0; v < 3; ++v)
                if ((uint32_t)v < nv) dst[v] = y[v];
        }
        dst += step;
    }
}

// 16 waves per CU: on a 65536 x 4096 u32 column scan 4096 waves of 256 steps
// took 164 + 12 + 386 us (totals, carry, rescan); 8192 waves 202 + 23 + 512.
constexpr uint64_t kColTargetWaves = 4096;
constexpr uint64_t kColMinChunk = 32;      // scan steps per chunk

bool column_mode(const ScanArgs &a) {
    const bool contiguous = a.in_elem_stride == 1 && a.out_elem_stride == 1;
    const bool adjacent = (a.in_line_stride == 1 || a.in_line_stride == -1) &&
                          (a.out_line_stride == 1 || a.out_line_stride == -1);
    return !contiguous && adjacent && a.lines >= 16;
}

ColShape column_shape(const ScanArgs &a) {
    ColShape s;
    const uintptr_t ibase = (uintptr_t)a.in + 4u * a.in_offset; // every element type is 4 bytes
    const uintptr_t obase = (uintptr_t)a.out + 4u * a.out_offset;
    // A lane's four adjacent lines are one 16-byte vector per step; the
    // vectors need only 4-byte alignment (Vec4A4), so any element stride and
    // start qualify.  When the line count is not a multiple of 4, the lane
    // of the last group moves its 1-3 lines one by one (col_load_n,
    // ColIO::load_n): u32 [8191, 8191] and [1023, 65537] along axis 0 took
    // 189 and 293 us with one line per lane everywhere.
    const bool vec = a.in_line_stride == 1 && a.out_line_stride == 1 && ibase % 4 == 0 && obase % 4 == 0;
    s.V = vec ? 4 : 1;
    s.groups = ceil_div(a.lines, (uint64_t)kWave * s.V);
    uint64_t k = 1;
    if (s.groups < kColTargetWaves) {
        k = ceil_div(kColTargetWaves, s.groups);
        const uint64_t kmax = ceil_div(a.len, kColMinChunk);
        if (k > kmax) k = kmax;
    }
    if (k <= 1) {
        s.chunk = a.len;
        s.nchunks = 1;
    } else {
        s.chunk = ceil_div(a.len, k);
        s.nchunks = (uint32_t)ceil_div(a.len, s.chunk);
    }
    return s;
}

// Single-pass column scans (col_lookback_kernel): line groups, padded line
// count of the status array, chunks of kColTileRows steps.
struct ColLbShape {
    int V = 1;
    uint64_t groups = 0, lpad = 0, chunks = 0;
};

ColLbShape col_lb_shape(const ScanArgs &a) {
    ColLbShape s;
    s.V = column_shape(a).V;
    s.groups = ceil_div(a.lines, (uint64_t)kWave * s.V);
    s.lpad = s.groups * kWave * s.V;
    s.chunks = ceil_div(a.len, kColTileRows);
    return s;
}

// col_lookback_kernel needs whole line groups: with fewer than 256 lines
// every tile leaves lanes idle and all tiles form one long look-back chain
// (measured, u32: 4194304 x 64 1.63 ms single-pass against 0.75 ms chunked;
// 1048576 x 256 0.46 against 0.71; 65536 x 4096 0.35 against 0.54).
constexpr uint64_t kSinglePassMinLines = 256;
// Many short lines: a scan of at most kColShortMaxLen steps whose chunked
// form needs one chunk over at least kColShortMinGroups line groups reads and
// writes each element once in col_scan_kernel, with no carries and no
// look-back.  The single pass's tiles hold 240 steps, so at 4 steps a
// sixteenth of its waves had data: u32 [4, 2^24] along axis 0 took 760 us
// single-pass and takes 85 this way ([16, 2^22] 207 -> 131, [64, 2^20] 109
// -> 100).  Longer lines keep the single pass ([240, 2^20]: 373 us against
// 435), and so do fewer groups, which leave the chip too few waves for
// serial steps ([32, 2^16]: 5.3 us against 7.5).
constexpr uint64_t kColShortMaxLen = 64;
constexpr uint64_t kColShortMinGroups = 1024;
bool column_short_lines(const ScanArgs &a) {
    if (!column_mode(a) || a.lines < kSinglePassMinLines) return false;
    const ColShape s = column_shape(a);
    return s.nchunks == 1 && a.len <= kColShortMaxLen && s.groups >= kColShortMinGroups;
}
// Where col_lookback_kernel's 1 KiB rows beat the strips' 256 bytes:
//   Large integer matrices from 1024 lines where the rows are whole 128-byte
//   lines and from 4096 where they are whole 16-byte vectors: u32, us, rows of
//   1 KiB / strips: [32768, 4096] 182 / 195, [131072, 1024] 189 / 201, [49152,
//   2048] 146 / 153, [26541, 4532] 205 / 211; but [524288, 256] 250 / 200, [65536,
//   1024] 102 / 91.
//   Matrices beyond the caches whose strips share 128-byte lines, from 8192
//   lines: u32 / f32, us, [2048, 50001] 189 / 238, [4096, 32001] 242 / 338 and 250 /
//   323, [512, 200001] 184 / 234 and 197 / 239; more lines have few rows, and f32
//   strips keep those: [400, 300001] u32 231 / 286, [300, 400001] f32 252 / 196.
//   One round of blocks, one to a CU, with half their rows or more: u32 / f32,
//   us, [240, 65536] 19.0 / 24.4 and 20.3 / 26.7, [200, 50001] 17.0 / 20.0 and 18.1 /
//   20.2, but [128, 50001] 11.3 / 12.4 and 12.6 / 11.8; two rounds of whole lines that
//   nearly fill the chip: u32 [300, 65536] 27.9 / 34.4, f32 [480, 65536] 44.7 / 56.1,
//   but [350, 40000] u32 21.9 / 20.9.
constexpr uint64_t kWideLines = 1024, kWideVectorLines = 4096;
constexpr uint64_t kWideElems = 1ull << 26;
constexpr uint64_t kWideSharedLines = 8192, kWideSharedMaxInt = 1ull << 19, kWideSharedMaxF32 = 1ull << 18;
constexpr uint64_t kWideSharedElemsInt = 5ull << 24, kWideSharedElemsF32 = 3ull << 25;
constexpr uint64_t kWideBlocks = 256, kWideRoundElems = 1ull << 23;
bool whole_line_rows(const ScanArgs &a) {
    return ((uintptr_t)a.out + 4u * a.out_offset) % 128 == 0 && a.out_elem_stride % 32 == 0; // 4-byte elements
}
bool column_wide(const ScanArgs &a) {
    const uint64_t n = a.len * a.lines;
    const bool f32 = a.dtype == HX_DTYPE_F32, whole = whole_line_rows(a);
    const ColLbShape s = col_lb_shape(a);
    if (s.groups <= kWideBlocks && s.chunks <= 2 && n > s.chunks * kWideRoundElems)
        return s.chunks == 1 || (whole && s.groups > kWideBlocks * 3 / 4);
    if (!whole && a.lines >= kWideSharedLines && a.lines <= (f32 ? kWideSharedMaxF32 : kWideSharedMaxInt) &&
        n > (f32 ? kWideSharedElemsF32 : kWideSharedElemsInt))
        return true;
    if (f32 || n <= kWideElems) return false;
    return (a.lines >= kWideLines && whole) || (a.lines >= kWideVectorLines && a.out_elem_stride % 4 == 0);
}
bool column_single_pass(const ScanArgs &a) {
    return column_mode(a) && a.lines >= kSinglePassMinLines && !column_short_lines(a) &&
           (column_shape(a).V == 1 || column_wide(a));
}

uint64_t column_bytes(const ScanArgs &a) {
    const ColShape s = column_shape(a);
    if (s.nchunks <= 1 || a.lines == 0) return 0;
    return (uint64_t)s.nchunks * a.lines * (a.dtype == HX_DTYPE_F32 ? 8u : 4u);
}

template <typename T, typename Op, int V, bool EXCL, bool REV>
hx_status launch_column_v(const ScanParams &p, const ColShape &s, void *ws, hipStream_t stream) {
    using A = typename ColAcc<T>::type;
    A *totals = (A *)ws;
    const uint64_t blocks = ceil_div(s.groups * s.nchunks, kBlock / kWave);
    if (blocks > 0x7FFFFFFFull) return fail(HX_ERR_DISPATCH_FAILED, "column scan exceeds the grid range");
    const dim3 grid((uint32_t)blocks), block(kBlock);
    if (s.nchunks <= 1) {
        hipLaunchKernelGGL((col_scan_kernel<T, Op, V, EXCL, REV, false>), grid, block, 0, stream, p,
                           (const A *)nullptr, s.chunk, s.nchunks, s.groups);
        return check_launch("col_scan_kernel");
    }
    hipLaunchKernelGGL((col_totals_kernel<T, Op, V, REV>), grid, block, 0, stream, p, totals, s.chunk, s.nchunks,
                       s.groups);
    HX_TRY(check_launch("col_totals_kernel"));
    hipLaunchKernelGGL((col_carry_kernel<A, Op>), dim3((uint32_t)ceil_div(p.lines, kCarryLines)),
                       dim3(kWave * kCarryWaves), 0, stream, totals, p.lines, s.nchunks);
    HX_TRY(check_launch("col_carry_kernel"));
    hipLaunchKernelGGL((col_scan_kernel<T, Op, V, EXCL, REV, true>), grid, block, 0, stream, p, (const A *)totals,
                       s.chunk, s.nchunks, s.groups);
    return check_launch("col_scan_kernel");
}

template <typename T, typename Op, typename Status, int V, bool EXCL, bool REV>
hx_status launch_col_lookback_v(const ScanParams &p, const ColLbShape &s, const Status &st, hipStream_t stream) {
    hipLaunchKernelGGL((col_lookback_kernel<T, Op, Status, V, EXCL, REV>), dim3((uint32_t)(s.groups * s.chunks)),
                       dim3(kColWaves * kWave), 0, stream, p, st, s.groups, s.lpad);
    return check_launch("col_lookback_kernel");
}

template <typename T, typename Op, typename Status, int V>
hx_status launch_col_lookback_s(const ScanParams &p, const ColLbShape &s, const Status &st, bool excl, bool rev,
                                hipStream_t stream) {
    if (excl)
        return rev ? launch_col_lookback_v<T, Op, Status, V, true, true>(p, s, st, stream)
                   : launch_col_lookback_v<T, Op, Status, V, true, false>(p, s, st, stream);
    return rev ? launch_col_lookback_v<T, Op, Status, V, false, true>(p, s, st, stream)
               : launch_col_lookback_v<T, Op, Status, V, false, false>(p, s, st, stream);
}

template <typename T, typename Op>
hx_status launch_col_lookback(const ScanParams &p, const ColLbShape &s, bool excl, bool rev, void *status,
                              hipStream_t stream) {
    if constexpr (std::is_same<T, float>::value) {
        // Ascending f32 lines take the strips (column_single_pass).
        const F64PairStatus st{(uint64_t *)status};
        return s.V == 4 ? launch_col_lookback_s<T, Op, F64PairStatus, 4>(p, s, st, excl, rev, stream)
                        : launch_col_lookback_s<T, Op, F64PairStatus, 1>(p, s, st, excl, rev, stream);
    } else {
        const PackedStatus st{(uint64_t *)status};
        return s.V == 4 ? launch_col_lookback_s<T, Op, PackedStatus, 4>(p, s, st, excl, rev, stream)
                        : launch_col_lookback_s<T, Op, PackedStatus, 1>(p, s, st, excl, rev, stream);
    }
}

template <typename T, typename Op, bool EXCL>
hx_status launch_column(const ScanParams &p, const ColShape &s, bool rev, void *ws, hipStream_t stream) {
    if (s.V == 4)
        return rev ? launch_column_v<T, Op, 4, EXCL, true>(p, s, ws, stream)
                   : launch_column_v<T, Op, 4, EXCL, false>(p, s, ws, stream);
    return rev ? launch_column_v<T, Op, 1, EXCL, true>(p, s, ws, stream)
               : launch_column_v<T, Op, 1, EXCL, false>(p, s, ws, stream);
}

// One 128-byte line per tile or superblock entry (a packed u32 word or a
// 16-byte f64 slot at its start).
uint64_t status_bytes(uint64_t entries) { return entries * kTileStatusBytes; }

// Tile shapes (waves x 16-byte steps per lane).  Of many lines, one up to
// 32768 elements is one tile: the smallest shape that holds it, so a block never
// carries idle waves and a row-wise scan needs no look-back.  Longer lines
// take 8 x 16 tiles chained by the look-back.  Measured on 2^28 u32 (f32)
// inclusive scans as 65536 x 4096: 1316 us (2329) with 8 x 16 tiles, whose
// waves 1-7 held no elements, against 334 (333) with 4 x 4; 262144 x 1024:
// 3404 (6047) against 331 (339) with 2 x 2; 16384 x 16384: 4 x 16 360 us,
// 8 x 8 410; 1048576 x 256: 1 x 1 351 us, 2 x 2 636; 524288 x 512: 1 x 2
// 339, 2 x 2 434.
struct TileShape {
    int waves, steps;
    uint64_t elems() const { return (uint64_t)waves * kWave * 4 * steps; }
};
// Lines longer than one 8 x 16 tile: the tiles chained by the look-back.
// f32 lines took 12 x 16 tiles (one block per CU) before f32 tiles fit in
// 128 VGPRs; 8 x 16 at two blocks per CU: 2^30 f32 1373.1 -> 1315.6 us.
constexpr int kLongWaves = 8, kLongSteps = 16;
// Few lines of more than 4096 elements leave most of the chip idle in tiles
// that large (up to 4096 one tile is as fast as a chain or faster: u32 lines of
// 3000 elements 3.2 us against 3.7, 3 lines of 4096 3.3 against 3.8): a block
// moves its 128 KiB at one CU's rate, and 2^20 elements
// are 32 blocks.  Fewer than 256 lines take smaller tiles and chain them,
// while the tiles number about four or five a CU: 2048 elements up to 2^17,
// 4096 up to 2^22, 8192 up to kMid8192Elems (2^23 where the outputs do not
// start on a 128-byte line: the larger tiles then run on the output's grid,
// scan_out_head).  u32 inclusive (f32), us, one size of tile for all -> now:
// 10^5 elements 7.4 (8.4) -> 4.0 (4.1), 10^6 7.2 (7.9) -> 5.1 (5.9), 3 * 10^6
// 9.1 (9.5) -> 6.4 (7.2), 10^7 15.4 (14.9) -> 14.5 (13.8); 16 * 10^6 in 8192s 26.8
// against 20.4.
// Chained tiles have status words.  Where a launch of its own clears them
// (ScanArgs::clears) a line that one tile holds keeps it up to kClearOneTile
// elements, and beyond where it fills the tile: a graph node of u32 lines of
// 5000 / 8192 / 32768 elements 4.1 / 3.1 / 5.1 us against 5.3 / 5.1 / 5.3 for clear
// and scan, but 12000 6.2 against 5.2 (a tile that is not full loads element
// by element).
constexpr uint64_t kMidMaxLines = 255;
constexpr uint64_t kMid2048Elems = 1ull << 17, kMid4096Elems = 1ull << 22, kMid8192Elems = 10ull << 20;
constexpr uint64_t kClearOneTile = 8192;
inline TileShape line_tile_shape(uint64_t len) {
    if (len <= 256) return {1, 1};
    if (len <= 512) return {1, 2};
    if (len <= 1024) return {2, 2};
    if (len <= 2048) return {2, 4};
    if (len <= 4096) return {4, 4};
    if (len <= 8192) return {4, 8};
    if (len <= 16384) return {4, 16};
    if (len <= 32768) return {kWaves, kSteps};
    return TileShape{kLongWaves, kLongSteps};
}
inline TileShape tile_shape(const ScanArgs &a) {
    const uint64_t len = a.len, n = a.len * a.lines;
    const TileShape one = line_tile_shape(len);
    const bool keep_one = a.clears && len <= one.elems() && (len <= kClearOneTile || len == one.elems());
    if (len > 4096 && !keep_one && a.lines <= kMidMaxLines && a.in_elem_stride == 1 && a.out_elem_stride == 1) {
        const bool grid = ((uintptr_t)a.out + 4u * a.out_offset + (a.reverse ? 4u * len : 0u)) % 128 == 0;
        if (n <= kMid2048Elems) return {2, 4};
        if (n <= kMid4096Elems) return {4, 4};
        if (n <= (grid ? kMid8192Elems : 1ull << 23)) return {4, 8};
    }
    return one;
}
bool long_tiles(const TileShape &s) { return s.waves == kLongWaves && s.steps == kLongSteps; }

// A launch's work-items (blocks x block size) must stay below 2^32, so many
// short lines (2^26 lines of at most 512 elements, 2^24 of at most 8192)
// take several launches of consecutive tiles, in order.  A later batch's
// look-back reads an earlier batch's statuses, published under the same tag
// before that launch ended; lines of one tile publish none.
template <typename T, typename Op, typename Status, bool EXCL, int STEPS, int WAVES>
hx_status launch_tiles_shaped(ScanParams p, const Status &st, const Status &st1, bool vec, bool rev,
                              hipStream_t stream) {
    const uint64_t max_blocks = std::min<uint64_t>(0x7FFFFFFFull, 0xFFFFFFFFull / (WAVES * kWave));
    const uint64_t total = p.total_tiles;
    for (uint64_t t0 = 0; t0 < total; t0 += max_blocks) {
        p.tile0 = t0;
        const dim3 grid((uint32_t)std::min<uint64_t>(max_blocks, total - t0)), block(WAVES * kWave);
        if (p.head != 0) {
            // Only long lines of 16-byte accesses run on virtual lines
            // (scan_out_head); the bounds cost the other launches registers,
            // so they have kernels of their own.
            if constexpr (STEPS == kSteps && WAVES == kWaves) {
                if (!vec) return fail(HX_ERR_DISPATCH_FAILED, "virtual line heads need 16-byte accesses");
                if (rev)
                    hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, true, true, STEPS, true, WAVES, true>),
                                       grid, block, 0, stream, p, st, st1);
                else
                    hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, true, false, STEPS, true, WAVES, true>),
                                       grid, block, 0, stream, p, st, st1);
                HX_TRY(check_launch("scan_tiles_kernel"));
                continue;
            } else {
                return fail(HX_ERR_DISPATCH_FAILED, "virtual line heads need the long-line tiles");
            }
        }
        if (vec && rev)
            hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, true, true, STEPS, true, WAVES>), grid, block,
                               0, stream, p, st, st1);
        else if (vec)
            hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, true, false, STEPS, true, WAVES>), grid, block,
                               0, stream, p, st, st1);
        else if (rev)
            hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, false, true, STEPS, true, WAVES>), grid, block,
                               0, stream, p, st, st1);
        else
            hipLaunchKernelGGL((scan_tiles_kernel<T, Op, Status, EXCL, false, false, STEPS, true, WAVES>), grid, block,
                               0, stream, p, st, st1);
        HX_TRY(check_launch("scan_tiles_kernel"));
    }
    return HX_OK;
}

template <typename T, typename Op, typename Status, bool EXCL>
hx_status launch_tiles(const ScanParams &p, const Status &st, const Status &st1, bool vec, bool rev,
                       const TileShape &shape, hipStream_t stream) {
    switch (shape.waves * 100 + shape.steps) {
    case 101: return launch_tiles_shaped<T, Op, Status, EXCL, 1, 1>(p, st, st1, vec, rev, stream);
    case 102: return launch_tiles_shaped<T, Op, Status, EXCL, 2, 1>(p, st, st1, vec, rev, stream);
    case 202: return launch_tiles_shaped<T, Op, Status, EXCL, 2, 2>(p, st, st1, vec, rev, stream);
    case 204: return launch_tiles_shaped<T, Op, Status, EXCL, 4, 2>(p, st, st1, vec, rev, stream);
    case 404: return launch_tiles_shaped<T, Op, Status, EXCL, 4, 4>(p, st, st1, vec, rev, stream);
    case 408: return launch_tiles_shaped<T, Op, Status, EXCL, 8, 4>(p, st, st1, vec, rev, stream);
    case 416: return launch_tiles_shaped<T, Op, Status, EXCL, 16, 4>(p, st, st1, vec, rev, stream);
    default: break;
    }
    static_assert(kLongWaves == kWaves && kLongSteps == kSteps, "long lines take the 32768-element tile");
    return launch_tiles_shaped<T, Op, Status, EXCL, kSteps, kWaves>(p, st, st1, vec, rev, stream);
}

// Short dense lines (scan_short_lines_kernel): fewer than 256 elements per
// line, lines packed back to back in input and output.
constexpr uint64_t kShortLineMax = 256;
constexpr int kShortWaves = 4;
constexpr uint64_t kShortSmallElems = 1ull << 22;
constexpr uint64_t kShortFewLen = 48, kShortFewElems = 1ull << 25;
bool short_tiles_small(const ShortParams &p) {
    return p.n <= kShortSmallElems || (p.len <= kShortFewLen && p.n <= kShortFewElems);
}
bool short_line_scan(const ScanArgs &a) {
    return a.len >= 1 && a.len < kShortLineMax && a.lines >= 2 && a.in_elem_stride == 1 &&
           a.out_elem_stride == 1 && a.in_line_stride == (int64_t)a.len && a.out_line_stride == (int64_t)a.len;
}

template <typename T, typename Op, bool EXCL, bool REV, int STEPS>
hx_status launch_short_steps(ShortParams p, hipStream_t stream) {
    constexpr uint64_t kTile = (uint64_t)kShortWaves * kWave * 4 * STEPS;
    const uint64_t tiles = ceil_div(p.n, kTile);
    const uint64_t max_blocks = std::min<uint64_t>(0x7FFFFFFFull, 0xFFFFFFFFull / (kShortWaves * kWave));
    for (uint64_t t0 = 0; t0 < tiles; t0 += max_blocks) {
        p.tile0 = t0;
        hipLaunchKernelGGL((scan_short_lines_kernel<T, Op, EXCL, REV, STEPS, kShortWaves>),
                           dim3((uint32_t)std::min<uint64_t>(max_blocks, tiles - t0)), dim3(kShortWaves * kWave), 0,
                           stream, p);
        HX_TRY(check_launch("scan_short_lines_kernel"));
    }
    return HX_OK;
}

template <typename T, typename Op, bool EXCL, bool REV>
hx_status launch_short_dir(const ShortParams &p, hipStream_t stream) {
    return short_tiles_small(p) ? launch_short_steps<T, Op, EXCL, REV, 2>(p, stream)
                                : launch_short_steps<T, Op, EXCL, REV, 4>(p, stream);
}

template <typename T, typename Op>
hx_status launch_short(const ScanArgs &a, hipStream_t stream) {
    ShortParams p{};
    p.in = a.in;
    p.out = a.out;
    p.n = a.lines * a.len;
    p.in_offset = a.in_offset;
    p.out_offset = a.out_offset;
    p.len = (uint32_t)a.len;
    if (a.exclusive)
        return a.reverse ? launch_short_dir<T, Op, true, true>(p, stream) : launch_short_dir<T, Op, true, false>(p, stream);
    return a.reverse ? launch_short_dir<T, Op, false, true>(p, stream) : launch_short_dir<T, Op, false, false>(p, stream);
}

// Row-tile column scans (col_rowtile_lookback_kernel): dense matrices of at
// most kRowTileMaxCols columns.  A look-back round covers 512 / C
// predecessors; wider matrices take strips.
constexpr uint64_t kRowTileMaxCols = 24;
bool rowtile_column_scan(const ScanArgs &a) {
    const uint64_t c = a.lines;
    const uintptr_t ibase = (uintptr_t)a.in + 4u * a.in_offset; // every element type is 4 bytes
    const uintptr_t obase = (uintptr_t)a.out + 4u * a.out_offset;
    return c >= 2 && c <= kRowTileMaxCols && a.in_line_stride == 1 && a.out_line_stride == 1 &&
           a.in_elem_stride == (int64_t)c && a.out_elem_stride == (int64_t)c && ibase % 4 == 0 && obase % 4 == 0;
}

uint64_t rowtile_lb_bytes(const ScanArgs &a) {
    const RowTileShape s = row_tile_shape(a.lines, a.len);
    if (s.tiles <= 1) return 0; // no look-back, no status words
    return kLookbackOffset + s.tiles * a.lines * (a.dtype == HX_DTYPE_F32 ? 16u : 8u);
}

template <typename T, typename Op, typename Status, bool EXCL>
hx_status launch_rowtile_lb_dir(const ScanParams &p, const RowTileShape &s, const Status &st, bool rev,
                                hipStream_t stream) {
    const dim3 grid((uint32_t)s.tiles), block(kRowTileThreads);
    if (rev)
        hipLaunchKernelGGL((col_rowtile_lookback_kernel<T, Op, Status, EXCL, true>), grid, block, 0, stream, p, s, st);
    else
        hipLaunchKernelGGL((col_rowtile_lookback_kernel<T, Op, Status, EXCL, false>), grid, block, 0, stream, p, s, st);
    return check_launch("col_rowtile_lookback_kernel");
}

template <typename T, typename Op>
hx_status launch_rowtile_lb(const ScanArgs &a, ScanParams p, void *ws, uint64_t ws_bytes, LookbackState &lb,
                            hipStream_t stream) {
    const RowTileShape s = row_tile_shape(a.lines, a.len);
    if (s.tiles > 0x7FFFFFFFull) return fail(HX_ERR_DISPATCH_FAILED, "column scan exceeds the grid range");
    if (ws_bytes < rowtile_lb_bytes(a))
        return fail(HX_ERR_DISPATCH_FAILED, "scan workspace of %llu bytes is too small", (unsigned long long)ws_bytes);
    if (s.tiles > 1) HX_TRY(next_lookback_launch(lb, ws, ws_bytes, stream, &p.tag));
    p.tile0 = 0;
    uint64_t *words = (uint64_t *)((char *)ws + kLookbackOffset);
    hx_status r;
    if constexpr (std::is_same<T, float>::value) {
        const F64QuadDense st{words};
        r = a.exclusive ? launch_rowtile_lb_dir<T, Op, F64QuadDense, true>(p, s, st, a.reverse, stream)
                        : launch_rowtile_lb_dir<T, Op, F64QuadDense, false>(p, s, st, a.reverse, stream);
    } else {
        const PackedStatus st{words};
        r = a.exclusive ? launch_rowtile_lb_dir<T, Op, PackedStatus, true>(p, s, st, a.reverse, stream)
                        : launch_rowtile_lb_dir<T, Op, PackedStatus, false>(p, s, st, a.reverse, stream);
    }
    if (r == HX_OK && s.tiles > 1) commit_lookback_launch(lb);
    return r;
}

// Strip column scans (col_strip_kernel): lines adjacent in memory in both
// operands, any row pitch.
//
// Width: 64 lines, 32 for matrices of at most 32, and for those below 64
// unless they are large integer ones (u32 / f32, us, 64 and 32 lines wide:
// [100000, 33] 15.7 / 19.6 and 14.2 / 17.4; [1000003, 48] 73 / 98 and 83 / 92).
//
// Rows per lane: 16, and 8 where the matrix is small and its chains stay
// short (u32, us, 8 / 16 rows: [510, 659] 5.2 / 6.4, [16384, 512] 12.8 / 14.5,
// [8192, 2048] 26.5 / 28.2, but [100000, 64] 17.5 / 15.5), where many strips share
// lines (below), and where 8 rows a lane hold the lines and 16 would leave
// waves without a row (f32, us, 8 / 16 rows: [40, 1000001] 68 / 147, [72, 400001]
// 43 / 69, [128, 200001] 41 / 48); beyond the caches only up to half of them
// ([224, 400001] 194 / 153).
constexpr uint64_t kStripOneChunk = StripGeom<64, 8>::kRows;
constexpr uint64_t kStripSmallElems = 1ull << 24;
constexpr uint64_t kStripSmallLen = 1ull << 16;
// Stores of whole lines that go through the L2 all the same: sizes from
// kStripSmallElems to this, several strips.  u32, us, through the L2 against
// non-temporal: [65536, 1024] 91 / 102, [16384, 4096] 86 / 101, but [4096,
// 1024] 8.8 / 8.3, [131072, 1024] 212 / 201 and one strip, [2^20, 64], 88 / 85.
constexpr uint64_t kStripCachedElems = 1ull << 26;
// Where strips share lines: chunks dealt to XCDs, if there are enough of
// them to fill the eight evenly, else strips.  u32, rows / chunks / strips,
// us: [40000, 1001] 82 / 66 / 75, [100000, 333] 71 / 56 / 83, [12000, 3001]
// (27 chunks) 68.5 / 63.0 / 62.2, [3782, 5485] (9 chunks) 36.2 / 43.9 / 30.6.
constexpr uint64_t kStripDealChunks = 32;
constexpr uint64_t kStripDealStrips = 16;
// Two blocks on a CU for dealt chunks (by their LDS): with three, the 32 CUs'
// outputs push half-written lines out of the XCD's 4 MB L2.  With many strips
// to a chunk, half the rows per block do the same again.  u32, three blocks
// of 16 rows / two of 16 / two of 8, us: [70000, 2001] 350 / 274 / 224, [140000,
// 1001] 355 / 270 / 210, [300000, 500] 350 / 256 / 226, [500000, 257] 274 / 217 /
// 225 (col_lookback_kernel 260, 247, 258, 356).  f32 needs twice the strips:
// [140000, 1001] - / 249 / 231, [300000, 500] - / 237 / 255.
constexpr uint32_t kStripDealLds = 54 * 1024;
constexpr uint64_t kStripDealManyInt = 8, kStripDealManyF32 = 16;
// f32 matrices below this many lines give the same bits in every run: they
// look back in order (strip_ordered_lookback), or, where the chain of chunks is
// long and the matrix stays in the caches for a second read, take three
// launches.  f32, us, first prefix met (other bits every run) / ordered / three
// launches / three passes of row tiles, as it was before strips: [2048, 64] 7.0 /
// 8.0 / - / 13.1, [4096, 64] 8.5 / 11.8 / 11.5 / 13.3, [16384, 64] 12.3 / 15.0 / 12.0 / 13.5,
// [65536, 64] 19.0 / 22.5 / 14.9 / 13.9, [131072, 128] 30.1 / 37.3 / 43.0 / 36.1,
// [524288, 64] 57.5 / 65.3 / 79.0 / 74.2.  Three launches always take 8 rows a
// lane, and as many blocks to a CU as fit: they do not wait for each other.
constexpr uint64_t kOrderedMaxLines = 256;
constexpr uint64_t kStripCarryLen = 4096, kStripCarryMaxLen = 1ull << 18, kStripCarryElems = 1ull << 24;

struct StripShape {
    int W = 64, steps = 16;
    StripParams sp{};
    uint64_t chunks = 0;   // of the axis; sp.chunks a launch
    uint64_t launches = 1;
    bool ordered = false; // strip_ordered_lookback
    bool carries = false; // three launches: totals, carries, rescan
    uint32_t lds = 0; // dynamic LDS, for the blocks per CU alone
};

uint64_t strip_entry_bytes(const ScanArgs &a) { return a.dtype == HX_DTYPE_F32 ? 16u : 8u; }
uint64_t strip_total_bytes(const ScanArgs &a) { return a.dtype == HX_DTYPE_F32 ? 8u : 4u; }
// Groups of chunks with more chunks after them, which have statuses.
uint64_t strip_groups(const StripShape &s, uint64_t chunks) { return s.ordered ? (chunks - 1) / kStripGroup : 0; }
// Status words of a launch, and between launches two rows of line totals
// (read by one launch, written by the next); nothing for one chunk.
uint64_t strip_bytes(const ScanArgs &a, const StripShape &s) {
    if (s.chunks <= 1) return 0;
    if (s.carries) return s.chunks * s.sp.lpad * strip_total_bytes(a);
    return kLookbackOffset + (s.sp.chunks + strip_groups(s, s.sp.chunks)) * s.sp.lpad * strip_entry_bytes(a) +
           (s.launches > 1 ? 2 * s.sp.lpad * strip_total_bytes(a) : 0);
}
// Rows of a chunk.
uint64_t strip_rows(const StripShape &s) {
    return s.steps == 8 ? (s.W == 32 ? StripGeom<32, 8>::kRows : StripGeom<64, 8>::kRows)
                        : (s.W == 32 ? StripGeom<32, 16>::kRows : StripGeom<64, 16>::kRows);
}
// Blocks of a launch of `chunks` chunks.
uint64_t strip_blocks(const StripShape &s, uint64_t chunks) {
    switch (s.sp.deal) {
    case kDealChunks: return ceil_div(chunks, (uint64_t)kXcds) * kXcds * s.sp.groups;
    case kDealStrips: return chunks * ceil_div((uint64_t)s.sp.groups, (uint64_t)kXcds) * kXcds;
    default: return chunks * s.sp.groups;
    }
}

StripShape strip_shape(const ScanArgs &a) {
    StripShape s;
    const uint64_t n = a.len * a.lines;
    const bool f32 = a.dtype == HX_DTYPE_F32;
    s.W = a.lines <= 32 || (a.lines < 64 && (f32 || n <= kStripSmallElems)) ? 32 : 64;
    // The lines are shared out evenly, in whole 16-byte vectors, so that no
    // strip is left with a few lines (and a block with a few lanes).
    const uint64_t strips = ceil_div(a.lines, (uint64_t)s.W);
    s.sp.width = (uint32_t)(ceil_div(ceil_div(a.lines, strips), 4) * 4);
    s.sp.groups = (uint32_t)ceil_div(a.lines, (uint64_t)s.sp.width);
    s.sp.lpad = (uint64_t)s.sp.groups * s.W;
    auto cut = [&](int steps) {
        s.steps = steps;
        s.chunks = ceil_div(a.len, strip_rows(s));
        s.sp.chunks = s.chunks;
    };
    const bool small = n <= kStripSmallElems && a.len <= kStripSmallLen;
    const bool few_rows = a.len <= kStripOneChunk && (a.len <= kStripOneChunk / 2 || n <= kStripCachedElems);
    cut(small || few_rows ? 8 : 16);
    const bool lines128 = whole_line_rows(a) && s.sp.width % 32 == 0;
    s.sp.cached = !lines128 || (s.sp.groups > 1 && n > kStripSmallElems && n <= kStripCachedElems) ? 1u : 0u;
    s.sp.deal = kDealRows;
    if (!lines128 && s.sp.groups > 1) {
        if (s.sp.chunks >= kStripDealChunks) {
            s.sp.deal = kDealChunks;
            s.lds = kStripDealLds;
            if (s.sp.groups >= (f32 ? kStripDealManyF32 : kStripDealManyInt)) cut(8);
        } else if (s.sp.groups >= kStripDealStrips) {
            s.sp.deal = kDealStrips;
        }
    }
    s.ordered = f32 && a.lines < kOrderedMaxLines;
    s.carries = s.ordered && a.len > kStripCarryLen && a.len <= kStripCarryMaxLen && n < kStripCarryElems;
    if (s.carries) {
        cut(8);
        s.lds = 0;
        return s;
    }
    // A fixed workspace too small for the statuses: 16 rows a lane halves
    // them, and what is still too long goes in several launches, each from
    // the totals the one before left.  The 8 MiB scratch, us, chunked
    // (totals, carries, rescan) / so: f32 [4194304, 64] 1417 / 403, [2097152,
    // 128] 929 / 378, u32 [8388608, 64] 1441 / 663.
    if (strip_bytes(a, s) > a.workspace_limit && s.steps == 8) cut(16);
    if (strip_bytes(a, s) > a.workspace_limit) {
        const uint64_t row = s.sp.lpad * strip_entry_bytes(a);
        const uint64_t fixed = kLookbackOffset + 2 * s.sp.lpad * strip_total_bytes(a);
        // n chunks and their groups take at most n + n / kStripGroup rows.
        s.sp.chunks = a.workspace_limit > fixed ? (a.workspace_limit - fixed) / row * kStripGroup / (kStripGroup + 1) : 0;
        if (s.sp.chunks > kXcds) s.sp.chunks = s.sp.chunks / kXcds * kXcds;
        s.launches = s.sp.chunks > 0 ? ceil_div(s.chunks, s.sp.chunks) : 0; // 0: no room for one chunk
    }
    return s;
}

bool strip_column_scan(const ScanArgs &a) {
    if (!column_mode(a) || a.in_line_stride != 1 || a.out_line_stride != 1) return false;
    if (rowtile_column_scan(a) || column_short_lines(a)) return false;
    if (column_wide(a) || a.lines >= (1ull << 31)) return false;
    const StripShape s = strip_shape(a);
    return s.launches > 0 && strip_blocks(s, s.sp.chunks) * (kStripWaves * kWave) <= 0xFFFFFFFFull;
}

template <typename T, typename Op, typename Status, int W, int STEPS, bool ORDERED, bool PASSES>
hx_status launch_strip_dir(const ScanParams &p, const StripShape &s, const Status &st, bool excl, bool rev,
                           hipStream_t stream) {
    const dim3 grid((uint32_t)strip_blocks(s, s.sp.chunks)), block(kStripWaves * kWave);
    if (excl && rev)
        hipLaunchKernelGGL((col_strip_kernel<T, Op, Status, W, STEPS, true, true, ORDERED, PASSES>), grid, block, s.lds,
                           stream, p, s.sp, st);
    else if (excl)
        hipLaunchKernelGGL((col_strip_kernel<T, Op, Status, W, STEPS, true, false, ORDERED, PASSES>), grid, block, s.lds,
                           stream, p, s.sp, st);
    else if (rev)
        hipLaunchKernelGGL((col_strip_kernel<T, Op, Status, W, STEPS, false, true, ORDERED, PASSES>), grid, block, s.lds,
                           stream, p, s.sp, st);
    else
        hipLaunchKernelGGL((col_strip_kernel<T, Op, Status, W, STEPS, false, false, ORDERED, PASSES>), grid, block,
                           s.lds, stream, p, s.sp, st);
    return check_launch("col_strip_kernel");
}

template <typename T, typename Op, typename Status, int W, bool ORDERED>
hx_status launch_strip_steps(const ScanParams &p, const StripShape &s, const Status &st, bool excl, bool rev,
                             hipStream_t stream) {
    // Several launches: three (ordered), or 16 rows a lane below 256 lines.
    constexpr bool kMayPass8 = ORDERED, kMayPass16 = ORDERED || !std::is_same<T, float>::value;
    const bool passes = s.carries || s.launches > 1;
    if (s.steps == 8) {
        if constexpr (kMayPass8)
            if (passes) return launch_strip_dir<T, Op, Status, W, 8, ORDERED, true>(p, s, st, excl, rev, stream);
        if (!passes) return launch_strip_dir<T, Op, Status, W, 8, ORDERED, false>(p, s, st, excl, rev, stream);
    } else {
        if constexpr (kMayPass16)
            if (passes) return launch_strip_dir<T, Op, Status, W, 16, ORDERED, true>(p, s, st, excl, rev, stream);
        if (!passes) return launch_strip_dir<T, Op, Status, W, 16, ORDERED, false>(p, s, st, excl, rev, stream);
    }
    return fail(HX_ERR_DISPATCH_FAILED, "a column scan of this shape takes one launch");
}

template <typename T, typename Op, typename Status>
hx_status launch_strip_shaped(const ScanParams &p, const StripShape &s, const Status &st, bool excl, bool rev,
                              hipStream_t stream) {
    constexpr bool kMayOrder = std::is_same<T, float>::value; // strips of 32 lines are always ordered there
    if (s.W == 32) return launch_strip_steps<T, Op, Status, 32, kMayOrder>(p, s, st, excl, rev, stream);
    if constexpr (kMayOrder)
        if (s.ordered) return launch_strip_steps<T, Op, Status, 64, true>(p, s, st, excl, rev, stream);
    return launch_strip_steps<T, Op, Status, 64, false>(p, s, st, excl, rev, stream);
}

template <typename T, typename Op>
hx_status launch_strip(const ScanArgs &a, ScanParams p, void *ws, uint64_t ws_bytes, LookbackState &lb,
                       hipStream_t stream) {
    StripShape s = strip_shape(a);
    if (ws_bytes < strip_bytes(a, s))
        return fail(HX_ERR_DISPATCH_FAILED, "scan workspace of %llu bytes is too small", (unsigned long long)ws_bytes);
    uint64_t *words = (uint64_t *)((char *)ws + kLookbackOffset);
    auto launch = [&] {
        if constexpr (std::is_same<T, float>::value)
            return launch_strip_shaped<T, Op>(p, s, F64QuadDense{words}, a.exclusive, a.reverse, stream);
        else
            return launch_strip_shaped<T, Op>(p, s, PackedStatus{words}, a.exclusive, a.reverse, stream);
    };
    if (s.carries) {
        using A = typename ColAcc<T>::type;
        s.sp.totals = ws;
        s.sp.pass = kPassTotals;
        HX_TRY(launch());
        hipLaunchKernelGGL((col_carry_kernel<A, Op>), dim3((uint32_t)ceil_div(s.sp.lpad, kCarryLines)),
                           dim3(kWave * kCarryWaves), 0, stream, (A *)ws, s.sp.lpad, (uint32_t)s.chunks);
        HX_TRY(check_launch("col_carry_kernel"));
        s.sp.pass = kPassCarries;
        return launch();
    }
    const uint64_t per = s.sp.chunks, rows = strip_rows(s);
    s.sp.totals = (char *)words + (per + strip_groups(s, per)) * s.sp.lpad * strip_entry_bytes(a);
    for (uint64_t k = 0; k < s.launches; ++k) {
        // Launch k scans what the earlier ones left of the lines (a mirrored
        // line's end is its far end: the offsets stay).
        const uint64_t done = k * per * rows;
        p.len = a.len - done;
        if (!a.reverse) {
            p.in_offset = a.in_offset + (uint64_t)((int64_t)done * a.in_elem_stride);
            p.out_offset = a.out_offset + (uint64_t)((int64_t)done * a.out_elem_stride);
        }
        s.sp.chunks = std::min(per, s.chunks - k * per);
        s.sp.pass = (k > 0 ? kPassTakes : 0u) | (k + 1 < s.launches ? kPassLeaves : 0u) | (k % 2 ? kPassOdd : 0u);
        if (s.chunks > 1) HX_TRY(next_lookback_launch(lb, ws, ws_bytes, stream, &p.tag));
        HX_TRY(launch());
        if (s.chunks > 1) commit_lookback_launch(lb);
    }
    return HX_OK;
}

// 16-byte scans of lines longer than one tile whose outputs start off a
// 128-byte boundary (by the same amount on every line) run on virtual lines
// `head` (1-31) elements longer, the virtual elements (logical [0, head))
// read as the identity and never stored, so that every whole tile's stores
// cover whole lines.  Forward lines gain the elements before their start
// (both offsets move back by head), reverse lines after their end (logical
// index 0 is the physical last).  2^28 u32 exclusive scans, output (and
// input) at element offset k, tiles on the line's own grid: k = 0, 16, 32:
// 331-336 us; k = 1, 4, 5, 8: 418-428.  Stores that start 16 or 32 bytes
// into a 64-byte segment cost as much as unaligned ones; misaligned loads
// cost nothing measurable (input offset 1, output aligned: 333 us).
constexpr uint64_t kOutGrid = 32; // elements: 128 bytes
uint32_t scan_out_head(const ScanArgs &a) {
    if (a.len <= 32768 || a.in_elem_stride != 1 || a.out_elem_stride != 1 || !long_tiles(tile_shape(a))) return 0;
    if (a.lines > 1 && a.out_line_stride % (int64_t)kOutGrid != 0) return 0;
    const uintptr_t ibase = (uintptr_t)a.in + 4u * a.in_offset; // every element type is 4 bytes
    const uintptr_t obase = (uintptr_t)a.out + 4u * a.out_offset;
    if (ibase % 4 != 0 || obase % 4 != 0) return 0;
    const uint64_t first = obase / 4;
    return a.reverse ? (uint32_t)((kOutGrid - (first + a.len) % kOutGrid) % kOutGrid)
                     : (uint32_t)(first % kOutGrid);
}

uint64_t scan_bytes(const ScanArgs &a) {
    if (short_line_scan(a)) return 0;
    if (rowtile_column_scan(a)) return rowtile_lb_bytes(a);
    if (strip_column_scan(a)) return strip_bytes(a, strip_shape(a));
    if (column_mode(a) && column_single_pass(a)) {
        const ColLbShape c = col_lb_shape(a);
        return kLookbackOffset + c.chunks * c.lpad * (a.dtype == HX_DTYPE_F32 ? 16u : 8u);
    }
    if (column_mode(a)) return column_bytes(a);
    const uint64_t vlen = a.len + scan_out_head(a);
    const uint64_t tpl = ceil_div(vlen, tile_shape(a).elems());
    // Lines of one tile never look back and publish no status.
    if (tpl <= 1) return kLookbackOffset;
    return kLookbackOffset + status_bytes(tpl * a.lines) + status_bytes(ceil_div(tpl, kSuper) * a.lines);
}

// The size by which a caller that cannot allocate (hx_scan_noalloc) takes or
// rejects a scan: its workspace, except for strips, which are cut to fit any
// workspace.  Theirs is a figure of the matrix alone, however they are cut:
// one status a line per 240 rows from 256 lines up (16 rows a lane need no
// more than that); below, one word a line per tile of 32768 elements (32, 64
// and 128 dense lines) or of whole rows up to 16384, or the chunk totals of
// padded rows.
uint64_t fixed_workspace_bytes(const ScanArgs &a) {
    if (!strip_column_scan(a)) return scan_bytes(a);
    const uint64_t word = a.dtype == HX_DTYPE_F32 ? 8u : 4u;
    if (a.lines >= kSinglePassMinLines)
        return kLookbackOffset + ceil_div(a.len, kColTileRows) * ceil_div(a.lines, 256) * 256 * 2 * word;
    if (a.in_elem_stride != (int64_t)a.lines || a.out_elem_stride != (int64_t)a.lines) return column_bytes(a);
    const bool pow2 = a.lines >= 32 && (a.lines & (a.lines - 1)) == 0;
    const uint64_t tiles = pow2 ? ceil_div(a.len * a.lines, 32768) : row_tile_shape(a.lines, a.len).tiles;
    return tiles <= 1 ? 0 : tiles * a.lines * word;
}

template <typename T, typename Op>
hx_status launch_op(const ScanArgs &a, void *ws, uint64_t ws_bytes, LookbackState &lb, hipStream_t stream) {
    ScanParams p{};
    p.in = a.in;
    p.out = a.out;
    p.lines = a.lines;
    p.len = a.len;
    const TileShape shape = tile_shape(a);
    p.tiles_per_line = ceil_div(a.len, shape.elems());
    p.total_tiles = p.tiles_per_line * a.lines;
    p.supers_per_line = ceil_div(p.tiles_per_line, kSuper);
    p.in_line_stride = a.in_line_stride;
    p.in_elem_stride = a.in_elem_stride;
    p.out_line_stride = a.out_line_stride;
    p.out_elem_stride = a.out_elem_stride;
    p.in_offset = a.in_offset;
    p.out_offset = a.out_offset;
    p.spin_limit = lookback_poll_limit();
    if (a.lines == 0 || a.len == 0) return HX_OK;

    if (short_line_scan(a)) return launch_short<T, Op>(a, stream);
    if (rowtile_column_scan(a)) return launch_rowtile_lb<T, Op>(a, p, ws, ws_bytes, lb, stream);
    if (strip_column_scan(a)) return launch_strip<T, Op>(a, p, ws, ws_bytes, lb, stream);
    if (column_mode(a) && column_single_pass(a)) {
        const ColLbShape cs = col_lb_shape(a);
        if (cs.groups * cs.chunks > 0x7FFFFFFFull)
            return fail(HX_ERR_DISPATCH_FAILED, "column scan exceeds the grid range");
        if (ws_bytes < scan_bytes(a))
            return fail(HX_ERR_DISPATCH_FAILED, "scan workspace of %llu bytes is too small",
                        (unsigned long long)ws_bytes);
        HX_TRY(next_lookback_launch(lb, ws, ws_bytes, stream, &p.tag));
        hx_status s = launch_col_lookback<T, Op>(p, cs, a.exclusive, a.reverse, (char *)ws + kLookbackOffset, stream);
        if (s == HX_OK) commit_lookback_launch(lb);
        return s;
    }
    if (column_mode(a)) {
        const ColShape cs = column_shape(a);
        if (cs.nchunks > 1 && ws_bytes < column_bytes(a))
            return fail(HX_ERR_DISPATCH_FAILED, "scan workspace of %llu bytes is too small",
                        (unsigned long long)ws_bytes);
        return a.exclusive ? launch_column<T, Op, true>(p, cs, a.reverse, ws, stream)
                           : launch_column<T, Op, false>(p, cs, a.reverse, ws, stream);
    }
    if (ws_bytes < scan_bytes(a))
        return fail(HX_ERR_DISPATCH_FAILED, "scan workspace of %llu bytes is too small", (unsigned long long)ws_bytes);
    const uint32_t head = scan_out_head(a);
    if (head != 0) {
        // Virtual lines head elements longer.  Forward: both offsets move
        // back by head, so virtual element head is each line's first.
        // Reverse: the virtual elements lie past the line's physical end.
        p.head = head;
        p.len = a.len + head;
        if (!a.reverse) {
            p.in_offset = a.in_offset - head;
            p.out_offset = a.out_offset - head;
        }
        p.tiles_per_line = ceil_div(p.len, shape.elems());
        p.total_tiles = p.tiles_per_line * a.lines;
        p.supers_per_line = ceil_div(p.tiles_per_line, kSuper);
    }
    HX_TRY(next_lookback_launch(lb, ws, ws_bytes, stream, &p.tag));
    const bool contiguous = a.in_elem_stride == 1 && a.out_elem_stride == 1;
    const uintptr_t ibase = (uintptr_t)((const T *)a.in + a.in_offset);
    const uintptr_t obase = (uintptr_t)((T *)a.out + a.out_offset);
    // Vector accesses need only 4-byte alignment (Vec4A4), which every
    // 4-byte element has: contiguous lines take the vector path wherever
    // they start, forward or mirrored.
    const bool vec = contiguous && ibase % 4 == 0 && obase % 4 == 0;
    uint64_t *level0 = (uint64_t *)((char *)ws + kLookbackOffset);
    uint64_t *level1 = (uint64_t *)((char *)level0 + status_bytes(p.total_tiles));
    hx_status s;
    if constexpr (std::is_same<T, float>::value) {
        F64QuadStatus st{level0}, st1{level1};
        s = a.exclusive ? launch_tiles<T, Op, F64QuadStatus, true>(p, st, st1, vec, a.reverse, shape, stream)
                        : launch_tiles<T, Op, F64QuadStatus, false>(p, st, st1, vec, a.reverse, shape, stream);
    } else {
        TilePackedStatus st{level0}, st1{level1};
        s = a.exclusive ? launch_tiles<T, Op, TilePackedStatus, true>(p, st, st1, vec, a.reverse, shape, stream)
                        : launch_tiles<T, Op, TilePackedStatus, false>(p, st, st1, vec, a.reverse, shape, stream);
    }
    if (s == HX_OK) commit_lookback_launch(lb);
    return s;
}

} // namespace

uint64_t scan_workspace_bytes(const ScanArgs &a) { return scan_bytes(a); }
uint64_t scan_fixed_workspace_bytes(const ScanArgs &a) { return fixed_workspace_bytes(a); }

bool scan_uses_lookback(const ScanArgs &a) {
    if (short_line_scan(a)) return false;
    if (rowtile_column_scan(a)) return scan_bytes(a) > 0; // one tile: none
    if (strip_column_scan(a)) return scan_bytes(a) > 0 && !strip_shape(a).carries; // one chunk: none
    return !column_mode(a) || column_single_pass(a);
}

hx_status launch_scan(const ScanArgs &a, void *ws, uint64_t ws_bytes, LookbackState &lb, hipStream_t stream) {
    const bool prod = a.op == HX_OP_PROD;
    switch (a.dtype) {
    case HX_DTYPE_F32:
        return prod ? launch_op<float, OpProd>(a, ws, ws_bytes, lb, stream)
                    : launch_op<float, OpSum>(a, ws, ws_bytes, lb, stream);
    case HX_DTYPE_U32:
    case HX_DTYPE_I32:
        // Two's complement: i32 sums and products have the bits of u32 ones.
        return prod ? launch_op<uint32_t, OpProd>(a, ws, ws_bytes, lb, stream)
                    : launch_op<uint32_t, OpSum>(a, ws, ws_bytes, lb, stream);
    }
    return fail(HX_ERR_INVALID_CONFIGURATION, "unknown dtype %d", (int)a.dtype);
}

} // namespace hx

// Host-side checks of the f32 scan slot codec (the device code uses the same
// inline functions).
extern "C" void hx_debug_slot16_encode(uint32_t tag, uint32_t flag, uint64_t bits, uint32_t *dwords) {
    uint32_t q[4];
    hx::slot16_encode(tag, flag, bits, q);
    for (int i = 0; i < 4; ++i) dwords[i] = q[i];
}
extern "C" uint32_t hx_debug_slot16_decode(uint32_t tag, const uint32_t *dwords, uint64_t *bits) {
    const uint32_t q[4] = {dwords[0], dwords[1], dwords[2], dwords[3]};
    uint64_t b = 0;
    const uint32_t flag = hx::slot16_decode(tag, q, b);
    *bits = b;
    return flag;
}
