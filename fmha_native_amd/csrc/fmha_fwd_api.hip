// fmha_fwd_api.hip — C-ABI launcher for the gfx950 D64 BF16 FMHA forward.
//
// Replaces the reference's launch sites (src/bench_fmha_fwd.cpp:174-191,
// tests/test_fmha_fwd_d64.cpp:563-578): pick one of the four entries (varlen
// <=> seqstart_q set; causal flag), build the (nhead_q, ceil(seqlen_q/kM0),
// batch) grid and launch on the caller's stream.  Unlike the reference it
// validates its arguments and returns hipError_t instead of exiting.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <numeric>

#include "fmha_fwd.h"
#include "fmha_internal.h"

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int kMaxGridYZ = 65535;  // largest grid y / z dimension

// Largest byte offset touched inside one (batch, head) of a tensor with `rows`
// rows must fit the 31-bit buffer offsets the kernel uses.  Row indices run
// past the last row by at most one 64-key tile (K/V loaders) or, for Q and O,
// by the rest of the block's M-tiles: up to 2*kM0 - 1 rows for the pair form's
// second M-tile.  Such rows are zero-filled or dropped by the descriptor bound,
// but their offsets are still computed in 32-bit arithmetic.
bool offsets_fit(int rows, int stride) {
    const int64_t max_rows = (int64_t)rows + FMHA_KN0 + 2 * FMHA_KM0;
    return max_rows * (int64_t)stride * 2 + 256 < ((int64_t)1 << 31);
}

}  // namespace

extern "C" hipError_t fmha_fwd_d64_bf16_check(const FmhaFwdParams* p, int batch, int causal) {
    if (p == nullptr) return hipErrorInvalidValue;
    if (batch < 0 || (causal != 0 && causal != 1)) return hipErrorInvalidValue;
    if (p->q == nullptr || p->k == nullptr || p->v == nullptr || p->o == nullptr) return hipErrorInvalidValue;
    if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->o)) return hipErrorInvalidValue;
    if (p->lse != nullptr && (reinterpret_cast<uintptr_t>(p->lse) & 3u)) return hipErrorInvalidValue;
    if (p->seqlen_q < 0 || p->seqlen_k < 0) return hipErrorInvalidValue;
    // the running max assumes a positive scale (a larger score is a larger
    // probability); NaN fails this comparison too
    if (!(p->scale > 0.0f) || p->scale > 3.402823466e38f) return hipErrorInvalidValue;
    if (p->nhead_q <= 0 || p->nhead_k <= 0 || p->nhead_q % p->nhead_k != 0) return hipErrorInvalidValue;
    const int strides[12] = {p->stride_q, p->nhead_stride_q, p->batch_stride_q, p->stride_k, p->nhead_stride_k,
                             p->batch_stride_k, p->stride_v, p->nhead_stride_v, p->batch_stride_v, p->stride_o,
                             p->nhead_stride_o, p->batch_stride_o};
    for (int s : strides)
        if (s < 0 || (s & 7) != 0) return hipErrorInvalidValue;
    // a row must hold the 64 head-dim elements (rows never overlap)
    if (p->stride_q < FMHA_HEAD_DIM || p->stride_k < FMHA_HEAD_DIM || p->stride_v < FMHA_HEAD_DIM ||
        p->stride_o < FMHA_HEAD_DIM)
        return hipErrorInvalidValue;
    if ((p->seqstart_q == nullptr) != (p->seqstart_k == nullptr)) return hipErrorInvalidValue;
    if (!offsets_fit(p->seqlen_q, p->stride_q) || !offsets_fit(p->seqlen_k, p->stride_k) ||
        !offsets_fit(p->seqlen_k, p->stride_v) || !offsets_fit(p->seqlen_q, p->stride_o))
        return hipErrorInvalidValue;
    if (p->seqstart_q != nullptr && p->lse != nullptr && p->nhead_stride_q % p->stride_q != 0)
        return hipErrorInvalidValue;  // varlen LSE head stride is nhead_stride_q / stride_q
    // grid (nhead_q, ceil(seqlen_q / kM0), batch): y and z are at most 65535
    if ((p->seqlen_q + FMHA_KM0 - 1) / FMHA_KM0 > kMaxGridYZ || batch > kMaxGridYZ) return hipErrorInvalidValue;
    return hipSuccess;
}

namespace {

// What the launch rules read from the current device, cached per device
// ordinal: compute units, XCDs and each XCD's L2 (MI355X: 256, 8, 4 MiB,
// also the values used when a query fails).
struct DeviceShape {
    int cus, xccs, l2_bytes;
};
DeviceShape device_shape() {
    static std::atomic<int> cache[64][3];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return {256, 8, 4 << 20};
    int v[3];
    const hipDeviceAttribute_t attr[3] = {hipDeviceAttributeMultiprocessorCount, hipDeviceAttributeNumberOfXccs,
                                          hipDeviceAttributeL2CacheSize};
    const int fallback[3] = {256, 8, 4 << 20};
    for (int i = 0; i < 3; ++i) {
        v[i] = cache[dev][i].load(std::memory_order_relaxed);
        if (v[i] == 0) {
            if (hipDeviceGetAttribute(&v[i], attr[i], dev) != hipSuccess || v[i] <= 0) v[i] = fallback[i];
            cache[dev][i].store(v[i], std::memory_order_relaxed);
        }
    }
    return {v[0], v[1], v[2]};
}
int device_cus() { return device_shape().cus; }

// Form choice from the grid (measured on MI355X, 256 CUs, all forms on one
// box; blocks = regular-grid blocks, pairs = pair-grid blocks):
//  * split-KV (two 4-wave groups per M-tile, one block per CU, each group
//    walking half of the keys): when the regular grid cannot fill the GPU and
//    the M-tiles are long (seqlen_k >= 2048) — blocks <= CUs (+8-14% at
//    64-256 blocks with 4096 keys), and for causal grids, whose heaviest
//    M-tile is the critical path, below 1.5 blocks per CU (+16% at 384 = 1.5
//    per CU) or up to 2 per CU with seqlen_k >= 8192 (+6% at 512).  Elsewhere
//    it loses 2-17% to the regular form; with few key tiles the halves are
//    too short to pay for the merge (1024 keys: -2 to +1%; <= 512 keys: -4
//    to -20%, down to the two-block grid B1 H2 S128).
//  * pair (two adjacent M-tiles per 8-wave block, one block per CU): the two
//    blocks a CU holds in the regular form progress unevenly, so each CU's
//    last block runs alone; a pair block has no such tail, but pays a barrier
//    across 8 waves.  It wins when the pair blocks fill whole rounds of the
//    CUs: dense from seqlen_k >= 2048 (+1.3-5 % at 1-4 rounds, 2048-32768
//    keys; the dense B4 H16 S2048 benchmark grid +1.4-2.6 %); causal at
//    exactly two rounds from 8192 keys (+3.1-4.5 %, the causal B1 H16 S8192
//    benchmark grid +3.4-3.7 %: each CU gets one heavy and one light pair,
//    heaviest first), or at any whole number from 32768 (+1 % at four).
//    Causal at one round loses ~20 % (split-KV takes those grids), at three
//    4-5 %, at four up to 4096 keys 1-4 %; dense at 1024 keys -3.5 to +2.6 %;
//    any partial last round 8-17 %.
//  * regular: everything else.
int pick_variant(int64_t blocks, int64_t pairs, int causal, int seqlen_k, int64_t cus) {
    // blocks (up to ~2^63) is only compared, never multiplied; cus < 2^31
    if (seqlen_k >= 2048) {
        if (blocks <= cus) return FMHA_VARIANT_SPLITKV;
        if (causal && (blocks <= 3 * cus / 2 || (blocks <= 2 * cus && seqlen_k >= 8192))) return FMHA_VARIANT_SPLITKV;
    }
    const bool whole_rounds = pairs >= cus && pairs % cus == 0;
    if (!causal && whole_rounds && seqlen_k >= 2048) return FMHA_VARIANT_PAIR;
    if (causal && ((pairs == 2 * cus && seqlen_k >= 8192) || (whole_rounds && seqlen_k >= 32768)))
        return FMHA_VARIANT_PAIR;
    return FMHA_VARIANT_REGULAR;
}

// Causal dense grids of more than one batch run on the tile-major entries
// (grid (nhead_q, batch, tiles): every batch's heaviest M-tiles start first)
// instead of batch after batch, while the K/V one XCD serves stays within
// twice its L2 (MI355X: 4 MiB per XCD, 8 XCDs).  Heads go to the XCDs round
// robin, so an XCD serves batch x ceil(nhead_k / XCDs) x seqlen_k x 256 bytes
// of K/V.  Beyond that the interleaved batches push each sequence's K/V out
// of L2 before its later M-tiles run.  Measured on causal grids (regular
// form): +19% B8 H16 S1024, +8% B4 H16 S2048, +6% B16 H8 S2048, +2-6% B2 H16
// S4096/S8192, and -1 to -5% above 8 MiB.
bool use_tilemajor(const FmhaFwdParams* p, int batch, int causal, const DeviceShape& d) {
    if (!causal || batch < 2 || p->seqstart_q != nullptr) return false;
    // batch x heads-per-XCD x seqlen_k <= 2 x L2 / 256 B, evaluated without overflow
    const int64_t limit = 2 * (int64_t)d.l2_bytes / 256;
    const int64_t rows = (int64_t)batch * (((int64_t)p->nhead_k + d.xccs - 1) / d.xccs);  // <= 2^16 * 2^31
    return p->seqlen_k == 0 || (rows <= limit && rows * p->seqlen_k <= limit);
}

// Block order of causal launches.  Dense batches: the reference's (batch
// after batch) or the tile-major entries (use_tilemajor).  Varlen launches of
// at most 64 sequences in the regular form: the reference's order (sequence
// after sequence in the caller's order, the blocks past each short sequence's
// end dispatched between live ones) or one of the compact entries on the same
// grid, whose blocks take the live (sequence, M-tile) items in the level
// order (highest M-tile index first across all sequences) or the sequence
// order (longest sequence first, each heaviest M-tile first), the grid's
// ranks past the live items last.
enum Order : int { kOrderAuto = 0, kOrderReference = 1, kOrderTileMajor = 2, kOrderSequence = 3 };
constexpr int kOrderFlags = FMHA_VARIANT_REFERENCE_ORDER | FMHA_VARIANT_TILE_MAJOR_ORDER | FMHA_VARIANT_SEQUENCE_ORDER;
// the order a variant's flags ask for; -1 for more than one
int order_of(int variant) {
    const int f = variant & kOrderFlags;
    return f == 0                               ? kOrderAuto
           : f == FMHA_VARIANT_REFERENCE_ORDER  ? kOrderReference
           : f == FMHA_VARIANT_TILE_MAJOR_ORDER ? kOrderTileMajor
           : f == FMHA_VARIANT_SEQUENCE_ORDER   ? kOrderSequence
                                                : -1;
}
constexpr int kCompactMaxSeqs = 64;
bool compact_applies(const FmhaFwdParams* p, int batch, int causal) {
    return causal && p->seqstart_q != nullptr && batch >= 1 && batch <= kCompactMaxSeqs;
}
// The varlen order of a regular-form causal launch: kOrderReference,
// kOrderTileMajor (level order) or kOrderSequence.  Automatic: the sequence
// order for at most 8 sequences on a grid of at most 8 rounds of the resident
// blocks (2 per CU), else the reference's.  Each block of a compact entry
// finds its item in a loop over the sequences (~15 instructions each, in
// dead blocks too), which the short M-tiles of many-sequence launches do not
// repay.  Interleaved A/B in one process, H = nhead_q (reference order /
// level / sequence): cfg4's eight lengths at H4 -3.6 % / +15 %, H8 +16 % /
// +13 %, H16 -3.3 % / +2.2 %, H32 -15 % / -2.5 %; 16 lengths 100-4000 H8
// +2.6 % / +5.1 %, H16 -12 % / -2.3 %; 32 and 64 sequences of 16-2048 tokens
// H16 -17 to -29 % / -12 to -41 %; 16 x 512 H16 -1.1 % / -9.7 %.
int varlen_order(const FmhaFwdParams* p, int batch, int causal, int order, int64_t cus) {
    if (!compact_applies(p, batch, causal) || order == kOrderReference) return kOrderReference;
    if (order != kOrderAuto) return order;
    const int64_t blocks = (int64_t)p->nhead_q * ((p->seqlen_q + kM0 - 1) / kM0) * batch;  // the grid: a bound
    return batch <= 8 && blocks <= 16 * cus ? kOrderSequence : kOrderReference;
}
// Dense causal batches on the tile-major entries?
bool dense_tile_major(const FmhaFwdParams* p, int batch, int causal, int order, const DeviceShape& d) {
    if (order == kOrderReference || order == kOrderSequence) return false;
    if (order == kOrderTileMajor) return causal && batch >= 2 && p->seqstart_q == nullptr;
    return use_tilemajor(p, batch, causal, d);
}

// Keys up to which the automatic choice takes the short form: on every grid
// of two blocks' worth of query rows per compute unit, and causal on grids of
// eight.
constexpr int kShortKeys = 3 * FMHA_KN0, kShortKeysCausal = 6 * FMHA_KN0;

// blocks of the regular grid and of the pair grid
int64_t grid_blocks(const FmhaFwdParams* p, int batch) {
    return (int64_t)p->nhead_q * ((p->seqlen_q + kM0 - 1) / kM0) * batch;
}
int64_t pair_blocks(const FmhaFwdParams* p, int batch) {
    return (int64_t)p->nhead_q * (((p->seqlen_q + kM0 - 1) / kM0 + 1) / 2) * batch;
}

// The automatic form: the short form when its keys fit three tiles and the
// launch has at least two blocks' worth of query rows per compute unit, or,
// causal, up to 384 keys with at least eight; else the grid-shape rule above.
// For varlen launches seqlen_k and seqlen_q are the caller's bounds (the rows
// counted here are an upper bound); the short form reads each sequence's own
// lengths like the other forms, so the bounds steer the choice only.
// Kernel trace, H16, ~262,144 query rows, against the regular form: the
// short form is 12-29 % faster at 64-128 keys (dense S128 22.7 against 25.9
// us, causal S64 24.8 against 35.1 us); back to back, H16, 65,536-262,144 rows: 8-14 % faster dense at
// 160-192 keys, 3 % at 224, -6 to +1 % at 256-320, 2-8 % slower at 384;
// causal 12-21 % faster at 160-192 keys at every size, 7-11 % at 224-384
// keys from 262,144 rows, 1-9 % at 229,376-258,048 rows (7 x CUs x 128; it
// skips the key halves a wave cannot see) and -14 to +2 % below (S384 at
// 196,608 rows -7 %; S512-S640 -5 to -6 % at any size).  On smaller grids one
// block's latency sets the launch time and the regular form wins (B1 H2
// S128: 4.6 against 5.6 us).  Varlen batches of 256-2048 sequences of 16-192
// tokens, H16: 13-33 % faster.  Past a few key tiles the regular form's
// software pipeline (GEMM0 of the next tile beside the softmax of this one)
// catches up with the short form's four blocks per compute unit; causal
// grids keep the short form longer (their light M-tiles are short).
int pick_form(const FmhaFwdParams* p, int batch, int causal, int64_t cus) {
    const int64_t rows = (int64_t)batch * p->nhead_q * p->seqlen_q;
    if (p->seqlen_k <= kShortKeys && rows >= 2 * cus * kM0) return FMHA_VARIANT_SHORT;
    if (causal && p->seqlen_k <= kShortKeysCausal && rows >= 7 * cus * kM0) return FMHA_VARIANT_SHORT;
    return pick_variant(grid_blocks(p, batch), pair_blocks(p, batch), causal, p->seqlen_k, cus);
}

}  // namespace

namespace {

// Key tiles of causal M-tile mt (pipeline.hpp:168-193, as the kernel).
int causal_ntiles(const FmhaFwdParams* p, int mt) {
    const int sq = p->seqlen_q, sk = p->seqlen_k;
    const int last = std::min(mt * kM0 + kM0 - 1, sq - 1);
    const int e = last + (sk - sq) + 1;
    const int kv_end = e < 0 ? 0 : (e > sk ? sk : e);
    return (kv_end + kN0 - 1) / kN0;
}

// Plan of a balanced causal launch on `cus` compute units.  Work units are
// M-tiles (two resident blocks per CU) or, in pair mode, M-tile pairs (one
// 8-wave block per CU); the units whose key tiles exceed a fraction of the
// average work per resident block (half; pairs 0.7) are split into two key
// halves (so none outlasts the average much), and the items are ordered by
// work, heaviest first (longest processing time first; ties: later unit,
// first half).  In the automatic mode (over M-tiles) the plan is taken only
// where balanced_pays() says it measured faster.  Returns false when there is
// no plan (not causal dense, too many items for the table); fills `a` (table,
// split range in M-tiles, pair flag) when given.
//
// Modes: the automatic rule, or forced over single M-tiles
// (FMHA_VARIANT_BALANCED) or over M-tile pairs (FMHA_VARIANT_BALANCED_PAIR).
enum PlanMode : int { kPlanAuto = 0, kPlanSingle = 1, kPlanPair = 2 };
bool balanced_plan_build(const FmhaFwdParams* p, int batch, int causal, int64_t cus, int xccs, int mode,
                         FmhaBalancedArgs* a, int64_t* ws_bytes);

// The plan depends on the launch's shape only, so the last one built on a
// thread is kept: a serving loop relaunching one shape skips the sort (about
// 10 us of host time for cfg5's 531 items).
bool balanced_plan(const FmhaFwdParams* p, int batch, int causal, int64_t cus, int xccs, int mode,
                   FmhaBalancedArgs* a, int64_t* ws_bytes) {
    struct Key {
        int seqlen_q, seqlen_k, nhead_q, batch, causal, varlen, mode, xccs;
        int64_t cus;
        bool operator==(const Key& o) const {
            return seqlen_q == o.seqlen_q && seqlen_k == o.seqlen_k && nhead_q == o.nhead_q && batch == o.batch &&
                   causal == o.causal && varlen == o.varlen && mode == o.mode && xccs == o.xccs && cus == o.cus;
        }
    };
    thread_local Key last_key{-1, -1, -1, -1, -1, -1, -1, -1, -1};
    thread_local bool last_ok = false;
    thread_local int64_t last_bytes = 0;
    thread_local FmhaBalancedArgs last_plan;
    const Key key{p->seqlen_q, p->seqlen_k, p->nhead_q, batch, causal, p->seqstart_q != nullptr ? 1 : 0,
                  mode, xccs, cus};
    if (!(key == last_key)) {
        last_ok = balanced_plan_build(p, batch, causal, cus, xccs, mode, &last_plan, &last_bytes);
        last_key = key;
    }
    if (!last_ok) return false;
    if (ws_bytes) *ws_bytes = last_bytes;
    if (a) {
        a->split_from = last_plan.split_from;
        a->n_split = last_plan.n_split;
        a->n_items = last_plan.n_items;
        a->pair = last_plan.pair;
        std::copy(last_plan.item, last_plan.item + last_plan.n_items, a->item);
    }
    return true;
}

// Whether the automatic choice takes a balanced plan: where the balanced form
// measured faster than the launch without a workspace (split-KV or the
// regular form; all three on one box, causal, 256 CUs, blocks = regular-grid
// blocks, heaviest = key tiles of the last M-tile, avg = key tiles per
// resident block).  It pays for its second launch, the split M-tiles' extra
// prologues and the partials' traffic only when the M-tiles are long:
//  * at most one block per CU: heaviest >= 64 (+10-41 % at 4096-8192 keys),
//    or >= 32 at up to half a block per CU (+16 % B1 H8 S2048); shorter
//    M-tiles lose 15-50 % (B2-B16 H16 S256-S1024);
//  * up to 1.5 blocks per CU: heaviest >= 128 (+8.5 % B1 H5 S8192; 64:
//    -2.5 %);
//  * 1.5-2 blocks per CU: never (split-KV or regular are 1.4-7 % faster at
//    4096-32768 keys);
//  * more: a partial second round whose heaviest M-tile outlasts 1.5x the
//    average, with heaviest >= 128 (cfg5 B1 H2 S40000 +13 %; +0.5-15 % at
//    564-672 blocks with 8192-80000 keys; 64: -7 %; at 768 blocks, where the
//    heaviest is ~1.3x the average, -11 % to +0.7 %).
bool balanced_pays(int64_t blocks, int heaviest, double avg, int64_t cus) {
    if (heaviest <= avg) return false;  // the heaviest-first order balances already
    if (blocks <= cus) return heaviest >= 64 || (2 * blocks <= cus && heaviest >= 32);
    if (2 * blocks <= 3 * cus) return heaviest >= 128;
    if (blocks <= 2 * cus) return false;
    return heaviest >= 128 && heaviest > 1.5 * avg;
}

// Dispatch order of a plan's items (sorted heaviest first) that lets each
// XCD's L2 serve items reading the same keys.  Workgroup i of a launch runs
// on XCD i % xccs, and table entry z is block (h, b, z) of every (batch,
// head), linear id h + nhead_q * (b + batch * z); when hb = nhead_q * batch
// divides xccs into g = xccs / hb >= 2 groups, entry z runs on the XCDs of
// group z % g only.  Blocks are dispatched in order, one group after the
// other, so every run of g consecutive entries (one per group) must keep
// items of about equal work, or a group with busy slots holds back the
// dispatch of the others (a list schedule that gave each group its own run
// of heaviest items measured 20-29 % slower on B1 H1 S40000 and B1 H2
// S16384).  Within each such run the items are therefore only re-ordered by
// the first key tile they read (first halves and whole M-tiles, which start
// at key 0, to the lower groups; second halves, which start half-way, to the
// higher ones), so each group keeps taking items that start at the same key.
// Otherwise (hb not a divisor of xccs, or xccs <= 1) the order stays
// heaviest first.  Allocates nothing.
template <class Start>
void xcd_order(int n, int xccs, int64_t hb, Start start, int* order) {
    for (int i = 0; i < n; ++i) order[i] = i;
    if (xccs <= 1 || hb >= xccs || xccs % hb != 0) return;
    const int g = (int)(xccs / hb);
    for (int r = 0; r < n; r += g) {
        const int e = std::min(n, r + g);
        std::sort(order + r, order + e, [&](int x, int y) {
            const int sx = start(x), sy = start(y);
            return sx != sy ? sx < sy : x < y;
        });
    }
}

bool balanced_plan_build(const FmhaFwdParams* p, int batch, int causal, int64_t cus, int xccs, int mode,
                         FmhaBalancedArgs* a, int64_t* ws_bytes) {
    if (!causal || p->seqstart_q != nullptr || batch <= 0 || p->seqlen_q <= 0 || cus <= 0) return false;
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    if (m_tiles > FMHA_BALANCED_MAX_ITEMS) return false;
    double total = 0.0;
    for (int mt = 0; mt < m_tiles; ++mt) total += causal_ntiles(p, mt);
    total *= (double)p->nhead_q * batch;
    const int heaviest = causal_ntiles(p, m_tiles - 1);
    if (mode == kPlanAuto &&
        !balanced_pays((int64_t)m_tiles * p->nhead_q * batch, heaviest, total / (2.0 * (double)cus), cus))
        return false;
    // work units: M-tiles (two resident blocks per CU) or M-tile pairs (one
    // 8-wave block per CU), each unit's key tiles those of its last M-tile
    const bool pair = mode == kPlanPair;
    const int units = pair ? (m_tiles + 1) / 2 : m_tiles;
    auto work = [&](int u) { return causal_ntiles(p, pair ? std::min(2 * u + 1, m_tiles - 1) : u); };
    double unit_total = total;
    if (pair) {
        unit_total = 0.0;
        for (int u = 0; u < units; ++u) unit_total += work(u);
        unit_total *= (double)p->nhead_q * batch;
    }
    // key tiles per resident block (two per CU; a pair block alone on its CU)
    const double avg = unit_total / ((pair ? 1.0 : 2.0) * (double)cus);
    // units with more key tiles than this are split: half the average (pairs:
    // 0.7 of it; B1 H2 S40000 causal measured 0.6-0.7 best, 0.5 -4 %, 1.0 -25 %)
    const double limit = std::max(2.0, avg * (pair ? 0.7 : 0.5));
    int split_u = units;  // key tiles grow with the unit: the split ones are a suffix
    while (split_u > 0 && work(split_u - 1) > limit) --split_u;
    const int split_from = pair ? std::min(2 * split_u, m_tiles) : split_u;
    const int n_split = m_tiles - split_from;
    const int n_items = split_u + 2 * (units - split_u);
    if (n_items > FMHA_BALANCED_MAX_ITEMS) return false;
    if (ws_bytes) *ws_bytes = (int64_t)n_split * p->nhead_q * batch * 2 * FMHA_BALANCED_PART_BYTES;
    if (a) {
        // a fixed table and an in-place sort: the plan allocates nothing (the
        // allocation-free entry point runs it too); the order is total, so
        // std::sort needs no stability
        struct It {
            int w, u, half;
        };
        It items[FMHA_BALANCED_MAX_ITEMS];
        int n = 0;
        for (int u = 0; u < units; ++u) {
            const int kt = work(u);
            if (u < split_u) {
                items[n++] = {kt, u, 0};
            } else {
                items[n++] = {(kt + 1) / 2, u, 0};
                items[n++] = {kt / 2, u, 1};
            }
        }
        std::sort(items, items + n, [](const It& x, const It& y) {
            if (x.w != y.w) return x.w > y.w;
            if (x.u != y.u) return x.u > y.u;
            return x.half < y.half;
        });
        // the first key tile an item reads (a second half starts past the first)
        int order[FMHA_BALANCED_MAX_ITEMS];
        xcd_order(n, xccs, (int64_t)p->nhead_q * batch,
                  [&](int i) { return items[i].half ? (work(items[i].u) + 1) / 2 : 0; }, order);
        for (int i = 0; i < n_items; ++i)
            a->item[i] = (unsigned short)(items[order[i]].u | (items[order[i]].half << 15));
        a->split_from = split_from;
        a->n_split = n_split;
        a->n_items = n_items;
        a->pair = pair ? 1 : 0;
    }
    return true;
}

// ---- chunk form (kModeChunk in fmha_fwd_kernel.hip) ----
//
// Dense launches of at most 5/8 M-tile per compute unit, with a workspace.
// What bounds them is one block's chain of key tiles (split-KV halves it,
// the balanced form too), so M-tiles of more than `tiles` key tiles are cut
// into equal chunks that run as blocks of their own, all resident at once, and
// a second launch merges the partial results.  Measured on 256 CUs over 29
// shapes (16-144 M-tiles of 11-313 key tiles, 12 chunk lengths each), a launch
// of I chunk blocks, the longest of w tiles, at most c per M-tile, takes
//     6.1 + k (w + 1) + 0.0127 I + 0.3 c   us,
// (w over all M-tiles: causal ones just below the chunk length stay whole),
// k = 0.55 up to one block per CU and 0.9 up to two (rms error 8 %): shorter
// chunks trade the chain against the partials' traffic and the merge's.  The
// forms without chunks take 9.5 + 0.275 n us (balanced), 6 + 0.435 n
// (split-KV) or 3.9 + 0.55 n (regular) for their longest M-tile's n tiles.
// The rule takes the chunk length with the least estimate where that is below
// the other form's.  Start / chunks: B1 H16 512 x 16384 causal 78 / 46 us,
// H16 100 x 8192 43 / 18, H2 S4096 causal 26 / 17, H1 S16384 causal 80 / 53,
// H4 S4096 34 / 29, H6 S2500 23.7 / 21.5; H16 S1024 (128 M-tiles of 16 tiles)
// stays regular, 12.5 / 14, and H72 256 x 2048 causal (M-tiles of 30 and 32
// tiles: cutting the longer ones alone leaves 30) split-KV, 20.3 / 26.0.
struct ChunkChoice {
    int tiles;  // key tiles per chunk
    double us;  // estimate
};
int chunk_count(int n, int tiles) { return std::max(1, (n + tiles - 1) / tiles); }
// Key tiles of M-tile mt.
int mtile_tiles(const FmhaFwdParams* p, int causal, int mt) {
    return causal ? causal_ntiles(p, mt) : (p->seqlen_k + kN0 - 1) / kN0;
}
// Chunk blocks of a launch (M-tiles kept whole among them).
int64_t chunk_items(const FmhaFwdParams* p, int causal, int m_tiles, int64_t hb, int tiles) {
    if (!causal) return hb * m_tiles * chunk_count(mtile_tiles(p, 0, 0), tiles);
    int64_t n = 0;
    for (int mt = 0; mt < m_tiles; ++mt) n += chunk_count(causal_ntiles(p, mt), tiles);
    return hb * n;
}
// Key tiles of the longest chunk.
int chunk_longest(const FmhaFwdParams* p, int causal, int m_tiles, int tiles) {
    int w = 0;
    for (int mt = causal ? 0 : m_tiles - 1; mt < m_tiles; ++mt) {
        const int n = mtile_tiles(p, causal, mt), c = std::min(FMHA_CHUNK_MAX_CHUNKS, chunk_count(n, tiles));
        w = std::max(w, (n + c - 1) / c);
    }
    return w;
}
// The chunk length for at most `slots` blocks at k us per tile.
ChunkChoice chunk_choice(const FmhaFwdParams* p, int causal, int m_tiles, int64_t hb, int longest, double total,
                         int64_t slots, double k) {
    // the estimate's minimum over the length, then as long as the blocks fit
    int lo = std::max(4, (int)std::sqrt((0.0127 * total + 0.3 * longest) / k));
    int hi = longest;  // every M-tile whole: fewer blocks than CUs (the caller's condition)
    if (lo < hi && chunk_items(p, causal, m_tiles, hb, lo) > slots) {
        while (hi - lo > 1) {  // items(lo) > slots >= items(hi)
            const int mid = (lo + hi) / 2;
            (chunk_items(p, causal, m_tiles, hb, mid) > slots ? lo : hi) = mid;
        }
        lo = hi;
    }
    if (lo >= longest) return {0, 0.0};
    const int c = std::min(FMHA_CHUNK_MAX_CHUNKS, chunk_count(longest, lo));
    const double w = chunk_longest(p, causal, m_tiles, lo);
    return {lo, 6.1 + k * (w + 1.0) + 0.0127 * (double)chunk_items(p, causal, m_tiles, hb, lo) + 0.3 * c};
}
// The M-tile forms' estimate for launches of at most one block per CU, and
// the chunk length (0: no chunks).
ChunkChoice mtile_us(const FmhaFwdParams* p, int batch, int causal, int64_t cus, bool workspace) {
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    const int64_t hb = (int64_t)p->nhead_q * batch;
    const int longest = mtile_tiles(p, causal, m_tiles - 1);
    ChunkChoice best{0, p->seqlen_k >= 2048 ? 6.0 + 0.435 * longest : std::max(6.7, 3.9 + 0.55 * longest)};
    if (!workspace || p->seqstart_q != nullptr || hb > cus || hb * m_tiles > cus) return best;
    double total = 0.0;
    for (int mt = 0; mt < m_tiles; ++mt) total += mtile_tiles(p, causal, mt);
    total *= (double)hb;
    if (causal && balanced_pays(hb * m_tiles, longest, total / (2.0 * (double)cus), cus))
        best.us = 9.5 + 0.275 * longest;
    if (8 * hb * m_tiles > 5 * cus || m_tiles > FMHA_CHUNK_MAX_MTILES) return best;  // chunks: the measured range
    for (const ChunkChoice& c : {chunk_choice(p, causal, m_tiles, hb, longest, total, cus, 0.55),
                                 chunk_choice(p, causal, m_tiles, hb, longest, total, 2 * cus, 0.9)})
        if (c.tiles > 0 && c.us < (best.tiles == 0 ? 0.97 : 1.0) * best.us) best = c;
    return best;
}

// ---- decode form (fmha_decode.hip) ----
// The packed rows of a KV head (its query heads x the queries) and the blocks
// of an unsplit launch.
int64_t decode_rows(const FmhaFwdParams* p) { return (int64_t)(p->nhead_q / p->nhead_k) * p->seqlen_q; }
int64_t decode_items(const FmhaFwdParams* p, int batch) {
    const int64_t tiles = (decode_rows(p) + FMHA_DECODE_ROWS - 1) / FMHA_DECODE_ROWS;
    const double n = (double)batch * p->nhead_k * (double)tiles;  // up to ~2^79
    return n < 1e15 ? (int64_t)batch * p->nhead_k * tiles : (int64_t)1e15;
}
// Fills `a` but its workspace pointers for at most `chunks` key chunks per
// (sequence, KV head), whole steps each; returns the workspace bytes.
int64_t decode_plan(const FmhaFwdParams* p, int batch, int causal, int chunks, int64_t cus, FmhaDecodeArgs* a) {
    const int steps = std::max(1, (p->seqlen_k + FMHA_DECODE_KEY_STEP - 1) / FMHA_DECODE_KEY_STEP);
    const int per = (steps + chunks - 1) / chunks;
    a->p = *p;
    a->part = a->ml = nullptr;
    a->chunk_keys = per * FMHA_DECODE_KEY_STEP;
    a->n_chunks = (steps + per - 1) / per;
    a->rows = (int)decode_rows(p);
    // what the M-tile form it replaces computes: whole M-tiles, pairs of them in the pair form
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    a->grid_rows = kM0 * (p->seqstart_q != nullptr && pick_form(p, batch, causal, cus) == FMHA_VARIANT_PAIR
                              ? 2 * ((m_tiles + 1) / 2)
                              : m_tiles);
    const int64_t pairs = (int64_t)batch * p->nhead_k;
    const int64_t blocks = pairs * a->n_chunks * ((a->rows + FMHA_DECODE_ROWS - 1) / FMHA_DECODE_ROWS);
    // eight waves (one block per CU) halve a block's serial chain; short key
    // ranges on more blocks than CUs take two four-wave blocks per CU, whose
    // prologues and epilogues overlap (B64 H16/16 1 x 128: 14.9 / 10.8 us with
    // 8 / 4 waves; 1 x 2048 on 320 blocks 36.2 / 34.7; 1 x 8000 varlen on 320
    // 80.6 / 96.6)
    a->waves = p->seqlen_k <= (blocks > cus ? 2048 : 128) ? 4 : 8;
    return a->n_chunks == 1 ? 0 : pairs * a->n_chunks * a->rows * (FMHA_HEAD_DIM + 2) * (int64_t)sizeof(float);
}
// Key chunks of a launch with a workspace: none where the pairs fill half the
// CUs (B16 H32/8 1 x 4100, 128 blocks: 28.7 us whole, 29.2 in two chunks; B64
// H8/2 1 x 2048 13.4 / 16.2) or the chain is at most five steps (the merge
// launch costs ~3 us, a step 0.6: B1 H8 4 x 4096, 16 steps, 15.7 whole, 9.8 in
// eight chunks); else as many as fit the CUs in one round (12 sequences to
// 16,000 keys, 24 pairs: 10 chunks 16.3 us, 16 chunks, a partial second round,
// 19.7).
int decode_chunks(const FmhaFwdParams* p, int batch, int64_t cus) {
    const int64_t items = decode_items(p, batch);
    if (items <= 0 || 2 * items >= cus || p->seqlen_k <= 5 * FMHA_DECODE_KEY_STEP) return 1;
    return (int)std::min<int64_t>(FMHA_DECODE_MAX_CHUNKS, cus / items);
}
// Whether a launch runs it: the automatic choice without an order flag (those
// ask for the M-tile grid); the bounds steer varlen launches.  Two regions:
//  * decode proper, at most 32 queries and 128 packed rows, bound by the K/V
//    stream.  M-tile forms / decode, us, one box (dense caches, LSE): B16 H32/8
//    1 x 4100 82 / 28, B1 H32/8 1 x 32768 312 / 18, B2 H16/2 16 x 16384 77 / 13,
//    B64 H16/16 1 x 128 11.5 / 10.8.  Packed sequences of up to 64 queries too,
//    from 1024 keys and at most one row tile per compute unit (0.17-1.02x over
//    35 launches).  Past 32 queries a head has two row tiles that each walk its
//    keys, and past one round the M-tile forms are ahead (their waves without
//    rows cost nothing): dense B32 H16/16 64 x 1024 29.5 / 33.0, B76 H6 64 x 1787
//    causal 42.8 / 62.0, packed 0.77-1.56x over 24 launches.  Where the short form
//    would run (two blocks' worth of query rows per compute unit, few keys: both
//    compute-bound) it takes about 1.2 x row tiles / query heads of a KV head
//    times as long: B128 H16/16 32 x 128 18.1 / 24.1, one head per KV head
//    1.05-1.47x over 33 launches, four 0.3-0.7x up to 64 rows and 0.8-1.2x at
//    128, eight 0.17-0.65x.
//  * dense launches of at most one 32-row tile per compute unit, bound by one
//    block's chain of key tiles, which the decode form splits over eight waves:
//    5.9 + 0.65 us per 256-key step (0.8 above half a block per CU, where two
//    waves share a SIMD's matrix core with nothing left over) + 3.2 for the
//    merge of a split launch, and no less than 4 us + K and V once at 5.4 TB/s or
//    once per XCD that a head's row tiles fall on (heads and chunks go round
//    robin) at 7 TB/s (rms error 10 % over 880 launches above 10 us, 21 % without
//    it: B14 H6 40 x 7106 causal took 45.0, the chain's estimate 28.3, the balanced
//    form 41.8), against the estimates of the other forms.  H8
//    S512 8.0 / 6.9, H4 S1024 12.3 / 7.8, H8 S1024 causal 12.9 / 7.9, H2 S2048
//    19.6 / 10.8, H4 256 x 8192 17.4 / 12.8, B8 H16/2 64 x 1000 13.2 / 8.3, H16
//    100 x 8192 17.9 / 14.5 (chunks / decode); up to 256 keys both take one
//    launch's latency (H2 S128 6.7 / 6.5 and 7.0 / 7.3 on two boxes) and the
//    M-tile forms stay; H16/4 512 x 16384 stays in chunks (46 / 56).
//
// `split`: a workspace holds the split launch's partials; `workspace`: there
// is one at all (the balanced and chunk forms' estimates count).
struct DecodeAsk {
    int seqlen_q, seqlen_k, nhead_q, nhead_k, batch, causal, split, workspace, cus, xccs;
    bool operator==(const DecodeAsk& o) const {
        return seqlen_q == o.seqlen_q && seqlen_k == o.seqlen_k && nhead_q == o.nhead_q && nhead_k == o.nhead_k &&
               batch == o.batch && causal == o.causal && split == o.split && workspace == o.workspace &&
               cus == o.cus && xccs == o.xccs;
    }
};
bool decode_faster(const FmhaFwdParams* p, const DecodeAsk& a) {
    const int64_t items = decode_items(p, a.batch);
    if (items > a.cus) return false;
    const int chunks = a.split ? decode_chunks(p, a.batch, a.cus) : 1;
    const int steps = (p->seqlen_k + FMHA_DECODE_KEY_STEP - 1) / FMHA_DECODE_KEY_STEP;
    const int per = (steps + chunks - 1) / chunks, n_chunks = (steps + per - 1) / per;
    const int64_t row_tiles = (decode_rows(p) + FMHA_DECODE_ROWS - 1) / FMHA_DECODE_ROWS;
    const int64_t copies = std::min<int64_t>(row_tiles, a.xccs / std::gcd(p->nhead_k * n_chunks, a.xccs));
    const double kv = 256e-6 * a.batch * p->nhead_k * (double)p->seqlen_k;  // MB
    const double us = std::max(5.9 + (2 * items > a.cus ? 0.8 : 0.65) * per,
                               4.0 + std::max(kv / 5.4, kv * (double)copies / 7.0)) + (chunks > 1 ? 3.2 : 0.0);
    return us < 0.97 * mtile_us(p, a.batch, a.causal, a.cus, a.workspace != 0).us;
}
bool takes_decode(const FmhaFwdParams* p, int batch, int causal, const DeviceShape& d, bool split, bool workspace) {
    // a grid holds fewer than 2^32 threads, and a decode block up to 512
    if (p->seqlen_k < 128 || p->nhead_k > (int)(UINT32_MAX / 512)) return false;
    if (decode_rows(p) <= 128 && p->seqlen_q <= 32) {
        const int64_t tiles = (decode_rows(p) + FMHA_DECODE_ROWS - 1) / FMHA_DECODE_ROWS;
        return pick_form(p, batch, causal, d.cus) != FMHA_VARIANT_SHORT || 4 * tiles <= 3 * (p->nhead_q / p->nhead_k);
    }
    if (p->seqstart_q != nullptr)
        return decode_rows(p) <= 128 && p->seqlen_q <= 64 && p->seqlen_k >= 1024 && decode_items(p, batch) <= d.cus;
    // the estimates walk the M-tiles: a thread's last answers with and without
    // a workspace are kept (they depend on the shape only)
    struct Kept {
        DecodeAsk ask{-1, -1, -1, -1, -1, -1, -1, -1, -1, -1};
        bool answer = false;
    };
    thread_local Kept kept[2];
    Kept& last = kept[workspace ? 1 : 0];
    const DecodeAsk ask{p->seqlen_q, p->seqlen_k, p->nhead_q, p->nhead_k, batch, causal,
                        split, workspace, d.cus, d.xccs};
    if (!(ask == last.ask)) {
        last.answer = decode_faster(p, ask);
        last.ask = ask;
    }
    return last.answer;
}

hipError_t decode_launch(const FmhaDecodeArgs& a, int batch, int causal, hipStream_t stream) {
    using Entry = void (*)(FmhaDecodeArgs);
    static const Entry walk[2][2][2] = {
        {{fmha_fwd_d64_bf16_decode_msk0, fmha_fwd_d64_bf16_decode_msk0_varlen},
         {fmha_fwd_d64_bf16_decode_msk1, fmha_fwd_d64_bf16_decode_msk1_varlen}},
        {{fmha_fwd_d64_bf16_decode4_msk0, fmha_fwd_d64_bf16_decode4_msk0_varlen},
         {fmha_fwd_d64_bf16_decode4_msk1, fmha_fwd_d64_bf16_decode4_msk1_varlen}}};
    static const Entry merge[2][2] = {
        {fmha_fwd_d64_bf16_decode_merge_msk0, fmha_fwd_d64_bf16_decode_merge_msk0_varlen},
        {fmha_fwd_d64_bf16_decode_merge_msk1, fmha_fwd_d64_bf16_decode_merge_msk1_varlen}};
    const int c = causal ? 1 : 0, v = a.p.seqstart_q != nullptr ? 1 : 0;
    hipLaunchKernelGGL(walk[a.waves == 4 ? 1 : 0][c][v],
                       dim3(a.p.nhead_k * a.n_chunks, (a.rows + FMHA_DECODE_ROWS - 1) / FMHA_DECODE_ROWS, batch),
                       dim3(64 * a.waves), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.n_chunks == 1) return e;
    hipLaunchKernelGGL(merge[c][v],
                       dim3((a.rows + FMHA_DECODE_MERGE_ROWS - 1) / FMHA_DECODE_MERGE_ROWS, a.p.nhead_k, batch),
                       dim3(64 * FMHA_DECODE_MERGE_ROWS), 0, stream, a);
    return hipGetLastError();
}
// Workspace bytes of the split launch (0: never split).
int64_t decode_bytes(const FmhaFwdParams* p, int batch, int64_t cus) {
    if (decode_items(p, batch) > INT32_MAX) return 0;
    FmhaDecodeArgs a;
    return decode_plan(p, batch, 0, decode_chunks(p, batch, cus), cus, &a);
}
// The launch with as many chunks as the workspace holds: the plan's, or one.
hipError_t decode_run(const FmhaFwdParams* p, int batch, int causal, int64_t cus, void* workspace,
                      int64_t workspace_bytes, hipStream_t stream) {
    FmhaDecodeArgs a;
    if (decode_plan(p, batch, causal, decode_chunks(p, batch, cus), cus, &a) > workspace_bytes)
        decode_plan(p, batch, causal, 1, cus, &a);
    if (a.n_chunks > 1) {
        a.part = (float*)workspace;
        a.ml = a.part + (int64_t)batch * p->nhead_k * a.n_chunks * a.rows * FMHA_HEAD_DIM;
    }
    return decode_launch(a, batch, causal, stream);
}

bool chunk_plan_build(const FmhaFwdParams* p, int batch, int causal, int64_t cus, FmhaChunkArgs* a, int64_t* bytes) {
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    if ((int64_t)p->nhead_q * batch > cus || (int64_t)p->nhead_q * batch * m_tiles > cus) return false;
    const int tiles = mtile_us(p, batch, causal, cus, true).tiles;
    if (tiles == 0) return false;
    const int longest = mtile_tiles(p, causal, m_tiles - 1);
    a->tiles = tiles;
    a->max_chunks = std::min(FMHA_CHUNK_MAX_CHUNKS, chunk_count(longest, tiles));
    // the heaviest M-tiles first, each one's chunks together
    int n = 0, slots = 0;
    unsigned short first[FMHA_CHUNK_MAX_MTILES];
    for (int mt = m_tiles - 1; mt >= 0; --mt) {
        const int nc = std::min(a->max_chunks, chunk_count(mtile_tiles(p, causal, mt), tiles));
        if (n + nc + m_tiles > FMHA_CHUNK_TABLE) return false;
        first[mt] = (unsigned short)slots;
        slots += nc > 1 ? nc : 0;
        for (int c = 0; c < nc; ++c) a->tab[n++] = (unsigned short)(mt << 6 | c);
    }
    std::copy(first, first + m_tiles, a->tab + n);
    a->n_items = n;
    a->n_slots = slots;
    *bytes = (int64_t)batch * p->nhead_q * slots * FMHA_BALANCED_PART_BYTES;
    return true;
}
// The plan of an automatic launch without an order flag; fills `a` but its
// workspace pointer.  It depends on the shape only, so the last one built on a
// thread is kept, as the balanced form's.
bool chunk_plan(const FmhaFwdParams* p, int batch, int causal, int64_t cus, FmhaChunkArgs* a, int64_t* bytes) {
    if (p->seqstart_q != nullptr) return false;
    struct Key {
        int seqlen_q, seqlen_k, nhead_q, batch, causal;
        int64_t cus;
        bool operator==(const Key& o) const {
            return seqlen_q == o.seqlen_q && seqlen_k == o.seqlen_k && nhead_q == o.nhead_q && batch == o.batch &&
                   causal == o.causal && cus == o.cus;
        }
    };
    thread_local Key last_key{-1, -1, -1, -1, -1, -1};
    thread_local bool last_ok = false;
    thread_local int64_t last_bytes = 0;
    thread_local FmhaChunkArgs last;
    const Key key{p->seqlen_q, p->seqlen_k, p->nhead_q, batch, causal, cus};
    if (!(key == last_key)) {
        last_ok = chunk_plan_build(p, batch, causal, cus, &last, &last_bytes);
        last_key = key;
    }
    if (!last_ok) return false;
    *bytes = last_bytes;
    if (a != nullptr) {
        *a = last;
        a->p = *p;
    }
    return true;
}
hipError_t chunk_launch(const FmhaChunkArgs& a, int batch, int causal, hipStream_t stream) {
    const dim3 block(kBlockSize), walk(a.p.nhead_q, batch, a.n_items),
        merge(a.p.nhead_q, 4 * ((a.p.seqlen_q + kM0 - 1) / kM0), batch);
    if (causal)
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_chunk_msk1, walk, block, 0, stream, a);
    else
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_chunk_msk0, walk, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (causal)
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_chunk_merge_msk1, merge, block, 0, stream, a);
    else
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_chunk_merge_msk0, merge, block, 0, stream, a);
    return hipGetLastError();
}

// Whether the automatic choice takes the wide form (64 rows per wave, 256 per
// block): dense layouts whose M-tile form would be the regular or the pair form
// (`form`).
//  * Blocks of about equal work (no mask, or a causal key range much longer
//    than the queries): a CU with two blocks takes 1.86 us per key tile of both
//    and one block alone 1.08 (regular 1.12 and 0.60 for half the rows, pair
//    1.065), so with k blocks on the fullest CU the launch takes 1.86 (k / 2) +
//    1.08 (k % 2) us per key tile, and the estimates are compared.  Over 26
//    shapes (S256-S8192, 192-3,072 blocks, us, other / wide): k = 2 B4 H16 S2048
//    71 / 65, B64 H8 S256 17.2 / 15.5; k = 3 full B6 H16 S2048 108 / 98, B12 H16
//    S1000 58 / 52; partial last rounds lose: B3 H16 S2048 (1.5 rounds) 56 / 60,
//    B9 H16 S900 43.6 / 44.9, B8 H16 S1030 (an odd M-tile) 47.1 / 48.5; causal, the
//    regular form's at its mean M-tile: B28 H8/1 703 x 4872 220 / 208, B58 H8/2 S193
//    (M-tiles of two and four tiles) 14.9 / 15.2.
//    k = 1 is one wave per SIMD against the regular form's two: 2-5 % slower at the
//    quartiles of 260 unmasked shapes, 2-29 % of 50 masked ones (H40 1024 x 512
//    11.7 / 12.4, H32 2048 x 256 8.6 / 9.6), but where a head's two M-tiles fall on different XCDs (heads go
//    round robin) and its keys are few, one block reads them once: B26 H6 153 x
//    848 20.0 / 17.6, B54 H4/1 132 x 1159 27.1 / 24.3, B14 H12 238 x 238 10.5 /
//    9.4; past 20 key tiles 0.86-1.10x, up to two 0.84-1.07x (H129 256 x 64 5.7 /
//    6.1), where the heads divide by the XCDs 0.95-1.12x.
//  * Causal squares: the heaviest-first order levels the blocks from four per CU,
//    and the waves' different diagonals (up to three tiles of a block's) cost
//    little from 2,560 keys: H32 S8192 283 / 262, H16 S16384 543 / 501, B12 H32
//    S3000 519 / 478, B4 H32 S4096 304 / 290; B16 H16 S2048 179 / 178, B16 H16
//    S1024 56 / 63, H24 S6000 (576 blocks) 122 / 130, H16 S8192 (512) 142 / 155.
bool takes_wide(const FmhaFwdParams* p, int batch, int causal, int form, const DeviceShape& d) {
    if (p->seqstart_q != nullptr || p->seqlen_k <= 0) return false;
    const int64_t cus = d.cus;
    if (form != FMHA_VARIANT_REGULAR && form != FMHA_VARIANT_PAIR) return false;
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    const int longest = mtile_tiles(p, causal, m_tiles - 1);
    const int lightest = mtile_tiles(p, causal, std::min(1, m_tiles - 1));
    const int64_t wide = pair_blocks(p, batch), regular = grid_blocks(p, batch);
    if (4 * (int64_t)lightest < 3 * (int64_t)longest) return wide >= 4 * cus && longest >= 40;
    if (wide <= cus && (causal || m_tiles != 2 || p->nhead_q % d.xccs == 0 || longest < 3 || longest > 20))
        return false;
    auto us = [cus](int64_t blocks, double two, double one) {
        const int64_t k = (blocks + cus - 1) / cus;  // blocks of the fullest CU
        return two * (double)(k / 2) + one * (double)(k % 2);
    };
    // the regular form's M-tiles walk their own tiles, a wide block its last row's
    const double mean = 0.5 * (mtile_tiles(p, causal, 0) + longest);
    double other = us(regular, 1.12, 0.60) * (mean / longest);
    if (form == FMHA_VARIANT_PAIR) other = std::min(other, 1.065 * (double)(wide / cus));
    return us(wide, 1.86, 1.08) < 0.97 * other;
}

// The plan mode of a form that runs a balanced plan (AUTO: might), or -1.
int plan_mode(int v) {
    return v == FMHA_VARIANT_AUTO            ? kPlanAuto
           : v == FMHA_VARIANT_BALANCED      ? kPlanSingle
           : v == FMHA_VARIANT_BALANCED_PAIR ? kPlanPair
                                             : -1;
}
// The XCD count a balanced plan is ordered for: the reference-order flag keeps
// the plain heaviest-first table (the results are the same bit for bit: the
// items do not change).
int plan_xccs(int order, const DeviceShape& d) { return order == kOrderReference ? 1 : d.xccs; }

// A launch's parts, once: the form, the block order and the device they were
// decided for.  The launch and fmha_fwd_d64_bf16_form() take it from here.
struct Launch {
    int form = -1;  // FMHA_VARIANT_* or FMHA_FORM_*; 0: nothing to launch; -1: rejected
    int order = kOrderAuto;
    bool plan_auto = false;  // a balanced form the automatic choice took
    DeviceShape dev{};
};
// `workspace`: the call has a workspace argument (of `bytes` bytes); the forms
// that need one are rejected without.
Launch decide(const FmhaFwdParams* p, int batch, int causal, int variant, bool workspace, int64_t bytes) {
    Launch l;
    l.order = order_of(variant);
    if (l.order < 0) return l;  // more than one order flag
    const int v = variant & ~kOrderFlags;
    const bool varlen = p->seqstart_q != nullptr;
    const bool empty = batch == 0 || p->seqlen_q == 0;
    switch (v) {  // 4 is a retired value
        case FMHA_VARIANT_PAIR_STREAM:
            if (varlen) return l;  // dense layouts only
            [[fallthrough]];
        case FMHA_VARIANT_REGULAR:
        case FMHA_VARIANT_SPLITKV:
        case FMHA_VARIANT_PAIR:
        case FMHA_VARIANT_SHORT:
            l.form = empty ? 0 : v;
            if (!empty) l.dev = device_shape();
            return l;
        case FMHA_VARIANT_BALANCED:
        case FMHA_VARIANT_BALANCED_PAIR:
            if (!workspace) return l;
            break;
        case FMHA_VARIANT_AUTO: break;
        default: return l;
    }
    if (empty) {
        l.form = 0;
        return l;
    }
    l.dev = device_shape();
    const int64_t cus = l.dev.cus;
    int64_t need = 0;
    if (v == FMHA_VARIANT_AUTO) {
        if (l.order == kOrderAuto) {
            if (takes_decode(p, batch, causal, l.dev, decode_bytes(p, batch, cus) <= bytes, bytes > 0)) {
                l.form = FMHA_FORM_DECODE;
                return l;
            }
            if (bytes > 0 && chunk_plan(p, batch, causal, cus, nullptr, &need) && need <= bytes) {
                l.form = FMHA_FORM_CHUNK;
                return l;
            }
        }
        // an automatic plan always splits something, so it needs a workspace
        l.plan_auto = bytes > 0 && balanced_plan(p, batch, causal, cus, plan_xccs(l.order, l.dev), kPlanAuto, nullptr,
                                                 &need) && need <= bytes;
        l.form = l.plan_auto ? FMHA_VARIANT_BALANCED : pick_form(p, batch, causal, cus);
        if (!l.plan_auto && l.order == kOrderAuto && takes_wide(p, batch, causal, l.form, l.dev))
            l.form = FMHA_FORM_WIDE;
        return l;
    }
    if (balanced_plan(p, batch, causal, cus, plan_xccs(l.order, l.dev), plan_mode(v), nullptr, &need) && need <= bytes)
        l.form = v;
    return l;
}

hipError_t balanced_launch(const FmhaFwdParams* p, int batch, int causal, const Launch& l, void* workspace,
                           hipStream_t stream) {
    FmhaBalancedArgs a;
    const int mode = l.plan_auto ? (int)kPlanAuto : plan_mode(l.form);
    if (!balanced_plan(p, batch, causal, l.dev.cus, plan_xccs(l.order, l.dev), mode, &a, nullptr))
        return hipErrorInvalidValue;
    a.p = *p;
    a.part = (float*)workspace;
    if (a.pair)
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_balanced_pair_msk1, dim3(p->nhead_q, batch, a.n_items),
                           dim3(FMHA_SPLIT_KBLOCK), 0, stream, a);
    else
        hipLaunchKernelGGL(fmha_fwd_d64_bf16_balanced_msk1, dim3(p->nhead_q, batch, a.n_items), dim3(kBlockSize), 0,
                           stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.n_split == 0) return e;
    hipLaunchKernelGGL(fmha_fwd_d64_bf16_balanced_merge, dim3(p->nhead_q, a.n_split, batch), dim3(kBlockSize), 0,
                       stream, a);
    return hipGetLastError();
}

// The M-tile forms and the wide form.
hipError_t grid_launch(const FmhaFwdParams* p, int batch, int causal, const Launch& l, hipStream_t stream) {
    const int variant = l.form;
    const bool varlen = p->seqstart_q != nullptr;
    const bool tile_major = dense_tile_major(p, batch, causal, l.order, l.dev);
    const int m_tiles = (p->seqlen_q + kM0 - 1) / kM0;
    const dim3 grid(p->nhead_q, m_tiles, batch);
    if (variant == FMHA_VARIANT_PAIR_STREAM) {
        // one block per compute unit over the pairs (dense), or one per pair
        // and its mirror (causal)
        const int64_t ny = (m_tiles + 1) / 2;
        const int64_t items = (int64_t)p->nhead_q * ny * batch;
        if (items >= INT32_MAX) return hipErrorInvalidValue;  // item numbers are ints
        const int64_t blocks = causal ? (int64_t)p->nhead_q * ((ny + 1) / 2) * batch
                                      : std::min<int64_t>(items, l.dev.cus);
        FmhaStreamArgs a;
        a.p = *p;
        a.ny = (int)ny;
        a.n_items = (int)items;
        if (causal)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_stream_msk1, dim3((unsigned)blocks), dim3(FMHA_SPLIT_KBLOCK), 0,
                               stream, a);
        else
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_stream_msk0, dim3((unsigned)blocks), dim3(FMHA_SPLIT_KBLOCK), 0,
                               stream, a);
        return hipGetLastError();
    }
    if (variant == FMHA_FORM_WIDE) {
        const int blocks = (m_tiles + 1) / 2;
        if (tile_major)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_wide_msk1_tilemajor, dim3(p->nhead_q, batch, blocks), dim3(kBlockSize),
                               0, stream, *p);
        else if (causal)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_wide_msk1, dim3(p->nhead_q, blocks, batch), dim3(kBlockSize), 0,
                               stream, *p);
        else
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_wide_msk0, dim3(p->nhead_q, blocks, batch), dim3(kBlockSize), 0,
                               stream, *p);
        return hipGetLastError();
    }
    if (variant == FMHA_VARIANT_SHORT) {
        using Entry = void (*)(FmhaFwdParams);
        static const Entry entries[2][2] = {{fmha_fwd_d64_bf16_short_msk0, fmha_fwd_d64_bf16_short_msk0_varlen},
                                            {fmha_fwd_d64_bf16_short_msk1, fmha_fwd_d64_bf16_short_msk1_varlen}};
        hipLaunchKernelGGL(entries[causal ? 1 : 0][varlen ? 1 : 0], grid, dim3(kBlockSize), 0, stream, *p);
        return hipGetLastError();
    }
    if (tile_major) {  // causal, dense, batch > 1
        if (variant == FMHA_VARIANT_PAIR)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_msk1_tilemajor, dim3(p->nhead_q, batch, (m_tiles + 1) / 2),
                               dim3(FMHA_SPLIT_KBLOCK), 0, stream, *p);
        else if (variant == FMHA_VARIANT_SPLITKV)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_splitkv_msk1_tilemajor, dim3(p->nhead_q, batch, m_tiles),
                               dim3(FMHA_SPLIT_KBLOCK), 0, stream, *p);
        else
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk1_tilemajor, dim3(p->nhead_q, batch, m_tiles), dim3(kBlockSize),
                               0, stream, *p);
        return hipGetLastError();
    }
    if (variant == FMHA_VARIANT_PAIR) {
        const dim3 pgrid(p->nhead_q, (m_tiles + 1) / 2, batch);
        const dim3 block(FMHA_SPLIT_KBLOCK);
        if (varlen) {
            if (causal)
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_msk1_varlen, pgrid, block, 0, stream, *p);
            else
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_msk0_varlen, pgrid, block, 0, stream, *p);
        } else {
            if (causal)
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_msk1, pgrid, block, 0, stream, *p);
            else
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_pair_msk0, pgrid, block, 0, stream, *p);
        }
        return hipGetLastError();
    }
    if (variant == FMHA_VARIANT_SPLITKV) {
        const dim3 block(FMHA_SPLIT_KBLOCK);
        if (varlen) {
            if (causal)
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_splitkv_msk1_varlen, grid, block, 0, stream, *p);
            else
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_splitkv_msk0_varlen, grid, block, 0, stream, *p);
        } else {
            if (causal)
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_splitkv_msk1, grid, block, 0, stream, *p);
            else
                hipLaunchKernelGGL(fmha_fwd_d64_bf16_splitkv_msk0, grid, block, 0, stream, *p);
        }
        return hipGetLastError();
    }
    const dim3 block(kBlockSize);
    if (varlen) {
        if (causal)
            switch (varlen_order(p, batch, causal, l.order, l.dev.cus)) {
                case kOrderTileMajor:
                    hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk1_varlen_tilemajor, grid, block, 0, stream, *p);
                    break;
                case kOrderSequence:
                    hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk1_varlen_seqmajor, grid, block, 0, stream, *p);
                    break;
                default:
                    hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk1_varlen, grid, block, 0, stream, *p);
            }
        else
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk0_varlen, grid, block, 0, stream, *p);
    } else {
        if (causal)
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk1, grid, block, 0, stream, *p);
        else
            hipLaunchKernelGGL(fmha_fwd_d64_bf16_msk0, grid, block, 0, stream, *p);
    }
    return hipGetLastError();
}

hipError_t run(const FmhaFwdParams* p, int batch, int causal, const Launch& l, void* workspace, int64_t bytes,
               hipStream_t stream) {
    switch (l.form) {
        case -1: return hipErrorInvalidValue;
        case 0: return hipSuccess;  // nothing to compute
        case FMHA_FORM_DECODE: return decode_run(p, batch, causal, l.dev.cus, workspace, bytes, stream);
        case FMHA_FORM_CHUNK: {
            FmhaChunkArgs c;
            int64_t need = 0;
            if (!chunk_plan(p, batch, causal, l.dev.cus, &c, &need)) return hipErrorInvalidValue;
            c.part = (float*)workspace;
            return chunk_launch(c, batch, causal, stream);
        }
        case FMHA_VARIANT_BALANCED:
        case FMHA_VARIANT_BALANCED_PAIR: return balanced_launch(p, batch, causal, l, workspace, stream);
        default: return grid_launch(p, batch, causal, l, stream);
    }
}

}  // namespace

extern "C" int fmha_fwd_d64_bf16_balanced_plan(const FmhaFwdParams* p, int batch, int causal, int compute_units,
                                               int xccs, int force, unsigned short* items, int capacity,
                                               int* split_from) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess || compute_units < 0 || xccs < 0) return -1;
    if (force < kPlanAuto || force > kPlanPair) return -1;
    FmhaBalancedArgs a;
    if (!balanced_plan(p, batch, causal, compute_units > 0 ? compute_units : device_cus(),
                       xccs > 0 ? xccs : device_shape().xccs, force, &a, nullptr))
        return 0;
    if (items != nullptr)
        for (int i = 0; i < a.n_items && i < capacity; ++i) items[i] = a.item[i];
    if (split_from != nullptr) *split_from = a.split_from;
    return a.n_items;
}

int64_t fmha_balanced_workspace_size(const FmhaFwdParams* p, int batch, int causal, int variant) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess) return -1;
    const int order = order_of(variant);
    if (order < 0) return -1;
    const int mode = plan_mode(variant & ~kOrderFlags);
    if (mode < 0) return 0;
    int64_t bytes = 0;
    // the same plan (and cache entry) as the launch with this variant
    const DeviceShape dev = device_shape();
    if (!balanced_plan(p, batch, causal, dev.cus, plan_xccs(order, dev), mode, nullptr, &bytes)) return 0;
    return bytes;
}

extern "C" int64_t fmha_fwd_d64_bf16_workspace_size(const FmhaFwdParams* p, int batch, int causal, int variant) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess) return -1;
    if (variant == FMHA_VARIANT_AUTO && batch > 0 && p->seqlen_q > 0) {
        const DeviceShape dev = device_shape();
        int64_t bytes = 0;
        if (takes_decode(p, batch, causal, dev, true, true)) return decode_bytes(p, batch, dev.cus);
        if (chunk_plan(p, batch, causal, dev.cus, nullptr, &bytes)) return bytes;
    }
    return fmha_balanced_workspace_size(p, batch, causal, variant);
}

extern "C" int fmha_fwd_d64_bf16_form(const FmhaFwdParams* p, int batch, int causal, int variant,
                                      int64_t workspace_bytes) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess || workspace_bytes < 0) return -1;
    return decide(p, batch, causal, variant, true, workspace_bytes).form;
}

extern "C" hipError_t fmha_fwd_d64_bf16_ws(const FmhaFwdParams* p, int batch, int causal, int variant,
                                           void* workspace, int64_t workspace_bytes, hipStream_t stream) {
    const hipError_t chk = fmha_fwd_d64_bf16_check(p, batch, causal);
    if (chk != hipSuccess) return chk;
    if (plan_mode(variant & ~kOrderFlags) >= 0 &&  // the other variants use no workspace
        (workspace_bytes < 0 || (workspace == nullptr && workspace_bytes != 0) ||
         (reinterpret_cast<uintptr_t>(workspace) & 255u)))
        return hipErrorInvalidValue;
    return run(p, batch, causal, decide(p, batch, causal, variant, true, workspace_bytes), workspace, workspace_bytes,
               stream);
}

extern "C" hipError_t fmha_fwd_d64_bf16_variant(const FmhaFwdParams* p, int batch, int causal, int variant,
                                                hipStream_t stream) {
    const hipError_t chk = fmha_fwd_d64_bf16_check(p, batch, causal);
    if (chk != hipSuccess) return chk;
    return run(p, batch, causal, decide(p, batch, causal, variant, false, 0), nullptr, 0, stream);
}

extern "C" int fmha_fwd_d64_bf16_pick_variant(const FmhaFwdParams* p, int batch, int causal, int compute_units) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess || compute_units < 0) return -1;
    const int64_t cus = compute_units > 0 ? compute_units : device_cus();
    return pick_form(p, batch, causal, cus);
}

extern "C" int fmha_fwd_d64_bf16_tile_major(const FmhaFwdParams* p, int batch, int causal) {
    if (fmha_fwd_d64_bf16_check(p, batch, causal) != hipSuccess) return -1;
    if (p->seqlen_q == 0 || batch == 0) return 0;  // nothing is launched
    const DeviceShape dev = device_shape();
    if (dense_tile_major(p, batch, causal, kOrderAuto, dev)) return 1;
    // varlen: the compact orders, which only the regular form has
    if (pick_form(p, batch, causal, dev.cus) != FMHA_VARIANT_REGULAR) return 0;
    const int o = varlen_order(p, batch, causal, kOrderAuto, dev.cus);
    return o == kOrderTileMajor ? 1 : o == kOrderSequence ? 2 : 0;
}

extern "C" hipError_t fmha_fwd_d64_bf16(const FmhaFwdParams* p, int batch, int causal, hipStream_t stream) {
    return fmha_fwd_d64_bf16_variant(p, batch, causal, FMHA_VARIANT_AUTO, stream);
}

extern "C" void fmha_fwd_d64_bf16_tile_config(int* m0, int* n0, int* block_size, int* head_dim) {
    if (m0) *m0 = kM0;
    if (n0) *n0 = kN0;
    if (block_size) *block_size = kBlockSize;
    if (head_dim) *head_dim = kHeadDim;
}
