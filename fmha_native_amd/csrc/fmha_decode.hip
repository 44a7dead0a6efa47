// fmha_decode.hip — decode form: a few query rows per KV head over a long key
// range (gfx950).  This build's own; the reference has no counterpart (its
// grid gives every query head a 128-row M-tile of its own, however few rows
// are live).
//
// What bounds it: one decode step reads every sequence's K and V once and does
// almost no arithmetic per byte, so the floor is the K/V stream.  The M-tile
// forms miss it three ways: each query head of a GQA group streams its KV
// head's keys for itself, a block's waves compute 128 rows of which one is
// live, and one block walks a sequence's keys alone.  Here:
//  * Rows are packed: the g = nhead_q / nhead_k query heads of a KV head times
//    the new tokens are the rows of one 32-row tile (row r = token * g + head),
//    so K and V are read once per KV head for up to 32 rows.
//  * Every wave of a block walks its own 32-key steps (wave w of W takes steps
//    w, w + W, ...), so the serial chain of a step (K reads, GEMM0, row max,
//    exponentials, GEMM1: ~0.5 us for one wave) runs W-fold in parallel, and
//    its two-stage K/V ring in LDS is its own: the loop has no barrier.
//    W = 8 with one 128 KiB block per CU keeps 64-128 KiB of loads in flight;
//    four stages at W = 4 kept as many but only one wave per SIMD to hide the
//    chain (B1 H8/1 4 x 4096 whole: 26.4 us, W = 8 15.7).
//  * A sequence's keys are split over n_chunks blocks where the (sequence, KV
//    head) pairs alone do not fill the GPU; each block then leaves an fp32
//    partial result (unnormalised O, row max and row sum) in the workspace and
//    a second launch merges them.
// Measured (back to back, before: the M-tile forms): B16 H32/8 1 x 4100, 134 MB
// of K/V: 82.5 -> 28.2 us, 4.8 TB/s (a large device copy reaches 5.1); twelve
// sequences of 500-16,000 keys, H16/2, 51 MB: 119 -> 16.3 us.
// The tile arithmetic is the other forms' (S^T = K.Q^T, O^T = V^T.P^T on
// v_mfma_f32_32x32x16_bf16, exp2 domain, exact running row max).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fmha_device.h"
#include "fmha_fwd.h"
#include "fmha_internal.h"

namespace fmha_gfx950 {
namespace {

constexpr int kDecStages = 2;                          // ring stages per wave
constexpr int kDecStep = 32;                           // keys per wave and step
constexpr int kDecRows = FMHA_DECODE_ROWS;             // packed query rows per block
constexpr int kDecWaveBytes = 2 * kDecStep * kRowBytes;  // one stage of one wave: 4 KiB of K, 4 KiB of V
constexpr int kDecLoads = 8;                           // DMA instructions per step (4 K, 4 V)
static_assert(kDecRows == 32 && FMHA_DECODE_KEY_STEP % (8 * kDecStep) == 0, "launcher and kernel geometry");

// s_waitcnt immediate for vmcnt(n) alone (gfx9 encoding)
constexpr int wait_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

// One sequence: its lengths and packed rows.
struct DecodeSeq {
    int64_t off_q, off_k;  // packed row offsets (varlen)
    int sq, sk;
    int rows;  // live packed rows of the sequence within the launch's bound
    int past;  // varlen: one past the last row a grid of M-tiles would reach (>= rows)
};
template <bool kVarlen>
__device__ __forceinline__ DecodeSeq decode_seq(const FmhaDecodeArgs& a, int b) {
    const FmhaFwdParams& p = a.p;
    DecodeSeq s;
    s.off_q = s.off_k = 0;
    s.sq = p.seqlen_q;
    s.sk = p.seqlen_k;
    if constexpr (kVarlen) {
        s.off_q = p.seqstart_q[b];
        s.off_k = p.seqstart_k[b];
        s.sq = p.seqstart_q[b + 1] - (int)s.off_q;
        s.sk = p.seqstart_k[b + 1] - (int)s.off_k;
    }
    const int g = p.nhead_q / p.nhead_k;
    s.rows = min(s.sq, p.seqlen_q) * g;  // the launch's bound: what the workspace was sized for
    s.past = kVarlen ? min(s.sq, a.grid_rows) * g : s.rows;
    return s;
}
// Keys visible to the last of packed rows row0 .. end - 1 that a 32-row tile
// from row0 holds.
template <bool kCausal>
__device__ __forceinline__ int visible_keys(const DecodeSeq& s, int row0, int end, int g) {
    if constexpr (!kCausal) return s.sk;
    const int last = (min(row0 + kDecRows, end) - 1) / g;  // the tile's last token
    return max(0, min(s.sk, last + (s.sk - s.sq) + 1));
}
// Chunks with keys to walk (at least one: an empty range still has a result).
// The last chunk takes whatever lies past the launch's seqlen_k bound.
__device__ __forceinline__ int live_chunks(const FmhaDecodeArgs& a, int kv_end) {
    return max(1, min(a.n_chunks, (kv_end + a.chunk_keys - 1) / a.chunk_keys));
}

struct DecodeLds {
    lds_char* st[kDecStages];
};

// The block's part of packed rows row0 .. end - 1 (at most 32) of KV head kvh:
// keys k0 .. k1 - 1, into O and LSE or (split) chunk `chunk`'s partial.
template <bool kCausal, bool kVarlen, int kDecWaves>
__device__ __forceinline__ void decode_tile(const FmhaDecodeArgs& a, const DecodeLds& lds, const DecodeSeq& sq, int b,
                                            int kvh, int chunk, int row0, int end, int k0, int k1, bool split) {
    const FmhaFwdParams& p = a.p;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hi = lane >> 5;
    const int g = p.nhead_q / p.nhead_k;

    // this lane's packed row: token qi of head kvh * g + gi
    const int row = row0 + l32;
    const bool live = row < end;
    const int qi = live ? row / g : 0, gi = live ? row - qi * g : 0;
    const int64_t head = (int64_t)kvh * g + gi;
    bf16x8 qop[4];
    {
        const __bf16* q = (const __bf16*)p.q + (kVarlen ? 0 : (int64_t)b * p.batch_stride_q) +
                          head * p.nhead_stride_q + (sq.off_q + qi) * p.stride_q + 8 * hi;
#pragma unroll
        for (int t = 0; t < 4; ++t) qop[t] = *(const bf16x8*)(q + 16 * t);  // a dead row repeats the first, unused
    }

    const char* kbase = (const char*)((const __bf16*)p.k + (kVarlen ? 0 : (int64_t)b * p.batch_stride_k) +
                                      (int64_t)kvh * p.nhead_stride_k + sq.off_k * p.stride_k);
    const char* vbase = (const char*)((const __bf16*)p.v + (kVarlen ? 0 : (int64_t)b * p.batch_stride_v) +
                                      (int64_t)kvh * p.nhead_stride_v + sq.off_k * p.stride_v);

    // DMA of a 32-key step: load j brings rows 8j + lane/8; physical chunk
    // lane%8 of a row holds logical chunk (lane%8) ^ swz(row).
    int k_off[4], v_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 8 * j + (lane >> 3), pc = lane & 7;
        k_off[j] = r * p.stride_k * 2 + ((pc ^ k_swz(r)) << 4);
        v_off[j] = r * p.stride_v * 2 + ((pc ^ v_swz(r)) << 4);
    }
    const int wave_off = wave * kDecWaveBytes;
    // The wave's step i: keys step_key(i) .. +31; steps past the range get an
    // empty descriptor (zero fill, no traffic), so every step issues the same
    // number of loads.
    auto step_key = [&](int i) { return k0 + (i * kDecWaves + wave) * kDecStep; };
    auto issue = [&](int i, auto stage_c) {
        lds_char* dst = lds.st[decltype(stage_c)::value] + wave_off;
        const int key = step_key(i);
        const int n = min(kDecStep, k1 - key);  // live keys
        const uint32_t kb = n > 0 ? (uint32_t)((n - 1) * p.stride_k * 2 + kRowBytes) : 0u;
        const uint32_t vb = n > 0 ? (uint32_t)((n - 1) * p.stride_v * 2 + kRowBytes) : 0u;
        const int64_t at = n > 0 ? key : 0;
        const auto rk = make_rsrc(kbase + at * p.stride_k * 2, kb);
        const auto rv = make_rsrc(vbase + at * p.stride_v * 2, vb);
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_dma_16(rk, dst + j * 1024, k_off[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_dma_16(rv, dst + kDecStep * kRowBytes + j * 1024, v_off[j]);
    };

    // LDS read offsets of the operands, as the other forms'
    uint32_t k_rd[4], v_rd[2];
    {
        const int f = k_swz(l32);
#pragma unroll
        for (int t = 0; t < 4; ++t) k_rd[t] = wave_off + l32 * kRowBytes + (((2 * t + hi) ^ f) << 4);
        const int grp = lane >> 4, i16 = lane & 15;
        const int r = 4 * hi + (i16 >> 2), c = i16 & 3;
#pragma unroll
        for (int db = 0; db < 2; ++db) {
            const int ch = 4 * db + 2 * (grp & 1) + (c >> 1);
            v_rd[db] = wave_off + kDecStep * kRowBytes + r * kRowBytes + ((ch ^ v_swz(r)) << 4) + (c & 1) * 8;
        }
    }

    const float scale = p.scale, scale_v = in_vgpr(scale);
    const float ninf = in_vgpr(-__builtin_inff());
    // last key this lane's row sees within the block's range
    const int lim = kCausal ? min(k1 - 1, qi + (sq.sk - sq.sq)) : k1 - 1;
    float m_ref = kMaxSeed, l_part = 0.0f;
    f32x16 oacc[2] = {f32x16{}, f32x16{}};

    auto step = [&](int i, auto stage_c) {
        constexpr int J = decltype(stage_c)::value;
        // the stage refilled here is the previous step's: its LDS reads have
        // returned (nothing but this wave touches its ring)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(i + kDecStages - 1, std::integral_constant<int, (J + kDecStages - 1) % kDecStages>{});
        // step i has landed; the kDecStages - 1 later ones may fly.  The
        // builtin, so that the compiler's wait placement sees it.
        __builtin_amdgcn_s_waitcnt(wait_vmcnt(kDecLoads * (kDecStages - 1)));
        asm volatile("" ::: "memory");
        const lds_char* st = lds.st[J];
        f32x16 s = {};
#pragma unroll
        for (int t = 0; t < 4; ++t) s = mfma(lds_read_b128(st + k_rd[t]), qop[t], s);
        // element r holds key step_key(i) + 4h + c, c = 8(r/4) + r%4
        const int d = lim - (step_key(i) + 4 * hi);
        if (__builtin_amdgcn_ballot_w64(d < 31)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = (8 * (r >> 2) + (r & 3)) <= d ? s[r] : ninf;
        }
        float mx = ninf;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
        const float m_new = fmaxf(m_ref, wave_max_halves(mx) * scale);
        if (__builtin_amdgcn_ballot_w64(m_new > m_ref)) {
            const float alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
            l_part *= alpha;
            m_ref = m_new;
        }
        const float neg_ms = -m_ref;
        bf16x8 pp[2];
        float ls[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float acc = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * k + e], scale_v, neg_ms));
                acc = e == 0 ? pv : acc + pv;
                pp[k][e] = (__bf16)pv;
            }
            ls[k] = acc;
        }
        l_part += ls[0] + ls[1];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int db = 0; db < 2; ++db)
                oacc[db] = mfma(lds_read_vt(st + v_rd[db] + 16 * k * kRowBytes), pp[k], oacc[db]);
    };

    // this wave's live steps
    const int left = k1 - step_key(0);
    const int n = left > 0 ? (left + kDecWaves * kDecStep - 1) / (kDecWaves * kDecStep) : 0;
    if (n > 0) {
        issue(0, std::integral_constant<int, 0>{});
        for (int i = 0; i < n; i += 2) {  // stage indices are compile-time
            step(i, std::integral_constant<int, 0>{});
            if (i + 1 < n) step(i + 1, std::integral_constant<int, 1>{});
        }
    }
    vmcnt_wait<0>();  // every DMA landed: the ring becomes the exchange area

    // The waves' partial results meet in LDS (each wave's own slices: O^T in
    // stage 0, m and l in stage 1); wave w then reduces elements
    // [w * kPer, (w + 1) * kPer) of every row over the waves.
    typedef __attribute__((address_space(3))) float lds_float;
    constexpr int kPer = 32 / kDecWaves;
    {
        lds_float* xo = (lds_float*)(lds.st[0] + wave_off);
        lds_float* xm = (lds_float*)(lds.st[1] + wave_off);
#pragma unroll
        for (int e = 0; e < 32; ++e) xo[e * 64 + lane] = oacc[e >> 4][e & 15];
        xm[lane] = m_ref;
        xm[64 + lane] = l_part;
    }
    __syncthreads();
    float mw[kDecWaves], m = kMaxSeed, l = 0.0f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
        mw[w] = ((const lds_float*)(lds.st[1] + w * kDecWaveBytes))[lane];
        m = fmaxf(m, mw[w]);
    }
    float out[kPer] = {};
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
        const float al = __builtin_amdgcn_exp2f(mw[w] - m);
        l += al * ((const lds_float*)(lds.st[1] + w * kDecWaveBytes))[64 + lane];
        const lds_float* xo = (const lds_float*)(lds.st[0] + w * kDecWaveBytes) + wave * kPer * 64 + lane;
#pragma unroll
        for (int e = 0; e < kPer; ++e) out[e] = __builtin_fmaf(al, xo[e * 64], out[e]);
    }
    l = wave_sum_halves(l);
    if (!live) return;
    // element e = 16 db + r of the lane is column 32 db + 8 (r / 4) + 4 h + r % 4
    if (split) {
        const int64_t slot = ((int64_t)b * p.nhead_k + kvh) * a.n_chunks + chunk;
        const int64_t at = slot * a.rows + row;
#pragma unroll
        for (int e = 0; e < kPer; e += 4) {
            const int ge = wave * kPer + e;
            const int col = 32 * (ge >> 4) + 8 * ((ge & 15) >> 2) + 4 * hi;
            *(float4*)(a.part + at * FMHA_HEAD_DIM + col) = float4{out[e], out[e + 1], out[e + 2], out[e + 3]};
        }
        if (wave == 0 && hi == 0) *(float2*)(a.ml + 2 * at) = float2{m, l};
        return;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    __bf16* o = (__bf16*)p.o + (kVarlen ? 0 : (int64_t)b * p.batch_stride_o) + head * p.nhead_stride_o +
                (sq.off_q + qi) * p.stride_o;
#pragma unroll
    for (int e = 0; e < kPer; e += 4) {
        const int ge = wave * kPer + e;
        const int col = 32 * (ge >> 4) + 8 * ((ge & 15) >> 2) + 4 * hi;
        bf16x2 x0, x1;
        x0[0] = (__bf16)(out[e] * inv);
        x0[1] = (__bf16)(out[e + 1] * inv);
        x1[0] = (__bf16)(out[e + 2] * inv);
        x1[1] = (__bf16)(out[e + 3] * inv);
        *(i32x2*)(o + col) = i32x2{__builtin_bit_cast(int, x0), __builtin_bit_cast(int, x1)};
    }
    if (p.lse != nullptr && wave == 0 && hi == 0) {
        float* lse = kVarlen ? p.lse + head * (p.nhead_stride_q / p.stride_q) + sq.off_q
                             : p.lse + ((int64_t)b * p.nhead_q + head) * p.seqlen_q;
        lse[qi] = (__builtin_log2f(l) + m) * 0.69314718055994530942f;  // -inf when l == 0
    }
}

template <bool kCausal, bool kVarlen, int kDecWaves>
__device__ __forceinline__ void fwd_decode(const FmhaDecodeArgs& a, const DecodeLds& lds) {
    const int nhead_k = a.p.nhead_k, g = a.p.nhead_q / nhead_k;
    const int kvh = blockIdx.x % nhead_k, chunk = blockIdx.x / nhead_k;
    const int b = blockIdx.z;
    const DecodeSeq sq = decode_seq<kVarlen>(a, b);
    int row0 = blockIdx.y * kDecRows, end = sq.rows;
    int kv_end = 0, k0 = 0, k1 = 0;
    bool split = a.n_chunks > 1, work = row0 < end;
    if (work) {
        kv_end = visible_keys<kCausal>(sq, row0, end, g);
        work = chunk < live_chunks(a, kv_end);  // the merge skips the others too
        k0 = chunk * a.chunk_keys;
        k1 = chunk == a.n_chunks - 1 ? kv_end : min(kv_end, k0 + a.chunk_keys);
    }
    if constexpr (!kVarlen) {
        if (work) decode_tile<kCausal, kVarlen, kDecWaves>(a, lds, sq, b, kvh, chunk, row0, end, k0, k1, split);
    } else {
        // A sequence with more queries than the launch's bound: the rows up to
        // the M-tile grid's, which the forms without packed rows compute, run
        // whole, one tile after the other, on its first block.
        const bool tail = blockIdx.x < nhead_k && blockIdx.y == 0;
        int next = end;
        for (;;) {
            if (work) decode_tile<kCausal, kVarlen, kDecWaves>(a, lds, sq, b, kvh, chunk, row0, end, k0, k1, split);
            if (!tail || next >= sq.past) return;
            __syncthreads();  // the exchange area becomes the ring again
            row0 = next;
            end = sq.past;
            next += kDecRows;
            k0 = 0;
            k1 = visible_keys<kCausal>(sq, row0, end, g);
            split = false;
            work = true;
        }
    }
}

// Merge of a row's chunk partials: one wave per packed row.  Lane c holds
// chunk c's max and sum (n_chunks <= 64), 16 lanes x 4 floats cover a partial
// O row, so a wave reads four chunks' rows per load.
template <bool kCausal, bool kVarlen>
__device__ __forceinline__ void decode_merge(const FmhaDecodeArgs& a) {
    const FmhaFwdParams& p = a.p;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * FMHA_DECODE_MERGE_ROWS + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kvh = blockIdx.y, b = blockIdx.z;
    const DecodeSeq sq = decode_seq<kVarlen>(a, b);
    if (row >= sq.rows) return;
    const int g = p.nhead_q / p.nhead_k;
    const int n = live_chunks(a, visible_keys<kCausal>(sq, row / kDecRows * kDecRows, sq.rows, g));
    const int64_t first = ((int64_t)b * p.nhead_k + kvh) * a.n_chunks;
    float m = kMaxSeed, l = 0.0f;
    if (lane < n) {
        const float2 v = *(const float2*)(a.ml + 2 * ((first + lane) * a.rows + row));
        m = v.x;
        l = v.y;
    }
    float mm = m;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) mm = fmaxf(mm, __shfl_xor(mm, d));
    const float w = lane < n ? __builtin_amdgcn_exp2f(m - mm) : 0.0f;
    float lt = w * l;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) lt += __shfl_xor(lt, d);
    const int sub = lane >> 4, col = 4 * (lane & 15);
    float4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 < n; c0 += 4) {  // loads past the last chunk repeat it, unused
        const int c = c0 + sub;
        const float wc = __shfl(w, c & 63);
        const float4 v = *(const float4*)(a.part + ((first + min(c, n - 1)) * a.rows + row) * FMHA_HEAD_DIM + col);
        acc.x = c < n ? __builtin_fmaf(wc, v.x, acc.x) : acc.x;
        acc.y = c < n ? __builtin_fmaf(wc, v.y, acc.y) : acc.y;
        acc.z = c < n ? __builtin_fmaf(wc, v.z, acc.z) : acc.z;
        acc.w = c < n ? __builtin_fmaf(wc, v.w, acc.w) : acc.w;
    }
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) {
        acc.x += __shfl_xor(acc.x, d);
        acc.y += __shfl_xor(acc.y, d);
        acc.z += __shfl_xor(acc.z, d);
        acc.w += __shfl_xor(acc.w, d);
    }
    if (lane >= 16) return;
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    const int qi = row / g, gi = row - qi * g;
    const int64_t head = (int64_t)kvh * g + gi;
    bf16x2 x0, x1;
    x0[0] = (__bf16)(acc.x * inv);
    x0[1] = (__bf16)(acc.y * inv);
    x1[0] = (__bf16)(acc.z * inv);
    x1[1] = (__bf16)(acc.w * inv);
    __bf16* o = (__bf16*)p.o + (kVarlen ? 0 : (int64_t)b * p.batch_stride_o) + head * p.nhead_stride_o +
                (sq.off_q + qi) * p.stride_o + col;
    *(i32x2*)o = i32x2{__builtin_bit_cast(int, x0), __builtin_bit_cast(int, x1)};
    if (p.lse != nullptr && lane == 0) {
        float* lse = kVarlen ? p.lse + head * (p.nhead_stride_q / p.stride_q) + sq.off_q
                             : p.lse + ((int64_t)b * p.nhead_q + head) * p.seqlen_q;
        lse[qi] = (__builtin_log2f(lt) + mm) * 0.69314718055994530942f;
    }
}

}  // namespace
}  // namespace fmha_gfx950

using namespace fmha_gfx950;

// each stage its own array: a DMA into one does not alias reads of another
#define FMHA_DECODE_ENTRY(name, causal, varlen, waves)                                                        \
    __global__ __launch_bounds__(64 * waves) void name(FmhaDecodeArgs args) {                                 \
        __shared__ __attribute__((aligned(1024))) char s0[waves * kDecWaveBytes], s1[waves * kDecWaveBytes];  \
        const DecodeLds lds{{(lds_char*)s0, (lds_char*)s1}};                                                  \
        fwd_decode<causal, varlen, waves>(args, lds);                                                         \
    }
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode_msk0, false, false, 8)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode_msk1, true, false, 8)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode_msk0_varlen, false, true, 8)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode_msk1_varlen, true, true, 8)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode4_msk0, false, false, 4)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode4_msk1, true, false, 4)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode4_msk0_varlen, false, true, 4)
FMHA_DECODE_ENTRY(fmha_fwd_d64_bf16_decode4_msk1_varlen, true, true, 4)

#define FMHA_DECODE_MERGE(name, causal, varlen)                                                    \
    __global__ __launch_bounds__(64 * FMHA_DECODE_MERGE_ROWS) void name(FmhaDecodeArgs args) {     \
        decode_merge<causal, varlen>(args);                                                        \
    }
FMHA_DECODE_MERGE(fmha_fwd_d64_bf16_decode_merge_msk0, false, false)
FMHA_DECODE_MERGE(fmha_fwd_d64_bf16_decode_merge_msk1, true, false)
FMHA_DECODE_MERGE(fmha_fwd_d64_bf16_decode_merge_msk0_varlen, false, true)
FMHA_DECODE_MERGE(fmha_fwd_d64_bf16_decode_merge_msk1_varlen, true, true)
