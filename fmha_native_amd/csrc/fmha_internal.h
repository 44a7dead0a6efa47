// fmha_internal.h — declarations shared by the kernel and launcher sources
// (not part of the C-ABI in include/).
#pragma once
#include <hip/hip_runtime.h>

#include "fmha_fwd.h"

// Balanced causal form (see fmha_fwd_kernel.hip): the item table of a launch
// and its workspace of partial results.
#define FMHA_BALANCED_MAX_ITEMS 1920                       // items per (batch, head): 3,840 bytes of table
#define FMHA_BALANCED_PART_BYTES (4 * 34 * 64 * 4)         // one partial result: 4 waves x 34 floats x 64 lanes

struct FmhaBalancedArgs {
    FmhaFwdParams p;
    float* part;     // workspace: 2 partial results per split M-tile of every (batch, head)
    int split_from;  // M-tiles >= split_from are split in two key halves
    int n_split;     // split M-tiles per (batch, head): m_tiles - split_from
    int n_items;     // items per (batch, head) (the grid's z)
    int pair;        // items are M-tile pairs (the pair entry, FMHA_SPLIT_KBLOCK threads)
    unsigned short item[FMHA_BALANCED_MAX_ITEMS];  // dispatch order: M-tile (pair) | half << 15
};

__global__ void fmha_fwd_d64_bf16_balanced_msk1(FmhaBalancedArgs args);
__global__ void fmha_fwd_d64_bf16_balanced_pair_msk1(FmhaBalancedArgs args);
__global__ void fmha_fwd_d64_bf16_balanced_merge(FmhaBalancedArgs args);

// Chunk form (see fmha_fwd_kernel.hip): long M-tiles cut into key chunks, on
// dense grids whose M-tiles are too few to fill the GPU.
#define FMHA_CHUNK_TABLE 1920
#define FMHA_CHUNK_MAX_MTILES 1024 // 10 bits of an item
#define FMHA_CHUNK_MAX_CHUNKS 64   // 6 bits
struct FmhaChunkArgs {
    FmhaFwdParams p;
    float* part;     // partial results (FMHA_BALANCED_PART_BYTES each), n_slots per (batch, head)
    int tiles;       // key tiles a chunk may hold
    int max_chunks;  // chunks an M-tile may have
    int n_items;     // items per (batch, head) (the grid's z)
    int n_slots;     // slots per (batch, head)
    // n_items items in dispatch order (M-tile << 6 | chunk), then every M-tile's
    // first slot
    unsigned short tab[FMHA_CHUNK_TABLE];
};
__global__ void fmha_fwd_d64_bf16_chunk_msk0(FmhaChunkArgs args);
__global__ void fmha_fwd_d64_bf16_chunk_msk1(FmhaChunkArgs args);
__global__ void fmha_fwd_d64_bf16_chunk_merge_msk0(FmhaChunkArgs args);
__global__ void fmha_fwd_d64_bf16_chunk_merge_msk1(FmhaChunkArgs args);

// Pair stream form (see fmha_fwd_kernel.hip): one 8-wave pair block per
// compute unit looping over a static list of M-tile pairs.
struct FmhaStreamArgs {
    FmhaFwdParams p;
    int ny;       // pairs per (batch, head): ceil(ceil(seqlen_q / kM0) / 2)
    int n_items;  // pairs of the launch: nhead_q * ny * batch
};
__global__ void fmha_fwd_d64_bf16_pair_stream_msk0(FmhaStreamArgs args);
__global__ void fmha_fwd_d64_bf16_pair_stream_msk1(FmhaStreamArgs args);

// Decode form (see fmha_decode.hip): packed query rows of one KV head over
// key chunks.
#define FMHA_DECODE_ROWS 32                            // packed rows (query heads of a KV head x tokens) per block
#define FMHA_DECODE_KEY_STEP 256                       // keys eight waves take per step; chunks are multiples of it
#define FMHA_DECODE_MAX_CHUNKS 64                      // the merge holds one chunk's weight per lane
#define FMHA_DECODE_MERGE_ROWS 4                       // rows (waves) per merge block
struct FmhaDecodeArgs {
    FmhaFwdParams p;
    float* part;     // [batch][nhead_k][n_chunks][rows][64] unnormalised O (n_chunks > 1)
    float* ml;       // [batch][nhead_k][n_chunks][rows][2] row max (scaled) and row sum
    int n_chunks;    // key chunks per (sequence, KV head)
    int chunk_keys;  // keys per chunk (the last takes the rest)
    int waves;       // waves per block: 8 (decode entries) or 4 (decode4)
    int rows;        // packed rows per (sequence, KV head): nhead_q / nhead_k * seqlen_q
    int grid_rows;   // queries per sequence the M-tile grid would reach (varlen: seqlen_q may lie below it)
};
__global__ void fmha_fwd_d64_bf16_decode_msk0(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_msk1(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_msk0_varlen(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_msk1_varlen(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode4_msk0(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode4_msk1(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode4_msk0_varlen(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode4_msk1_varlen(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_merge_msk0(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_merge_msk1(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_merge_msk0_varlen(FmhaDecodeArgs args);
__global__ void fmha_fwd_d64_bf16_decode_merge_msk1_varlen(FmhaDecodeArgs args);

// fmha_fwd_d64_bf16_workspace_size for the balanced forms alone: what the entry
// point on the static array gives a launch (calls on several streams that need
// no balanced plan must not share it).
int64_t fmha_balanced_workspace_size(const FmhaFwdParams* p, int batch, int causal, int variant);

// Wide form (see fmha_fwd_kernel.hip): 64 query rows per wave.
__global__ void fmha_fwd_d64_bf16_wide_msk0(FmhaFwdParams params);
__global__ void fmha_fwd_d64_bf16_wide_msk1(FmhaFwdParams params);
__global__ void fmha_fwd_d64_bf16_wide_msk1_tilemajor(FmhaFwdParams params);
