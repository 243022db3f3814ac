// kv_attention_route.h -- which attention kernel a call takes and how it is
// split: sizes and alignments in, launch geometry out. It makes no HIP call,
// so that the choice can be checked without a GPU.
#ifndef SGLKV_ATTENTION_ROUTE_H
#define SGLKV_ATTENTION_ROUTE_H

#include "kv_internal.h"

namespace sglkv {

// The kernels, in the order of sgl_rocm_kv_ctx::attention.
enum AttentionBody : int {
    kAttnVector,         // generic, 16-byte pieces
    kAttnElement,        // generic, element by element
    kAttnPipe128,        // pipelined, dims 128
    kAttnPipe,           // pipelined, dims up to 128
    kAttnWide576,        // wide: K up to 576, V up to 512
    kAttnWide128,        // wide, dims up to 128
    kAttnLatent,         // MLA (K 576, V 512), bf16 weights
    kAttnStaged128,      // staged: rows in LDS
    kAttnStaged64,
    kAttnLatentExact,    // MLA, hi + lo weights
    kAttnStaged256,
    kAttnStaged128K,     // staged, K in registers: head-major pages
    kAttnTile128,        // tiles of several queries per request
    kAttnTile64,
    kAttnTile256,
    kAttnBodies
};

// What the choice needs to know of the device: its CUs, a workgroup's LDS
// limit, and how many workgroups of a body a CU holds (0: unknown, an error
// that the query keeps).
struct AttentionDevice {
    uint64_t cus;
    uint64_t max_lds;
    void *context;
    uint32_t (*resident)(void *context, int body, unsigned threads, unsigned lds);
};

struct AttentionRoute {
    int body;
    unsigned threads, lds;
    uint64_t grid;            // workgroups of one split (p->splits of them in y)
    bool half_records;        // scaled fp16 split records (SGLKV_ATTN_HPAD)
    uint64_t record_bytes;    // all split records of the launch (0: one split)
    bool apart;               // the records go to the tiles' own buffer
    bool shortened;           // a ragged batch's splits, shorter than equal ones
    uint64_t combine_grid;
    unsigned combine_threads;
};

// The reference's overflow error.
int32_t attention_overflow();

// Where split records can go: the caller's fixed workspace (its size, 0 if
// there is none), else the buffer that all splitting calls of a context share,
// or, where `apart`, the tiles' own. A ragged batch's splits are made shorter
// than equal ones as far as their records fit `shorter` bytes.
struct AttentionRecords {
    uint64_t workspace_bytes;
    uint64_t shorter;
    bool apart;
};
// The most that shorter splits may take, with the no-allocation entry point's
// workspace as without, so that both split alike; the context's buffer starts
// at this size, so that a call never makes it grow for shorter splits.
constexpr uint64_t kAttentionShorterBytes = SGL_KV_NOALLOC_WORKSPACE_BYTES;
// The size of the tiles' own buffer. A launch of tiles leaves at most
// SGLKV_ATTN_TILE_ROWS records for each workgroup that it splits into, and no
// more of these than stay resident at once: 34 MB at dims 128 and 256 and 26 MB at
// dims 64 on 256 CUs (well inside the no-allocation entry point's workspace, too).
constexpr uint64_t kAttentionTileRecordBytes = 64ull << 20;

// Chooses for `p`, whose pointers, sizes, strides and page_shift are set, and
// sets its launch fields (chunk_tokens, splits, ...).
int32_t attention_route(const AttentionDevice &device, const sgl_kv_attention_plan_config &c, uint64_t max_len,
                        const AttentionRecords &records, sglkv_attn_params *p, AttentionRoute *r);

}  // namespace sglkv

#endif
