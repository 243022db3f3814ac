// kv_attention.cpp -- host side of the paged-attention reader: the plan
// (CudaBf16PagedAttentionPlan::new, crates/sglang-kernel/src/
// cuda_attention.rs:277-430, same validation order and error variants),
// the plan derived from a pool layout (build_plan,
// crates/sglang-srt/src/cuda_attention.rs:505-572) and the launch
// (CudaBf16PagedAttentionKernels::forward, cuda_attention.rs:681-850:
// device and range checks, clear the error word, launch, synchronise, read
// the word).
#include <hip/hip_runtime.h>

#include <mutex>
#include <math.h>
#include <string.h>

#include "kv_attention_route.h"
#include "kv_internal.h"

using namespace sglkv;

namespace {

// The plan flags: EXACT_WEIGHTS (the default, kept for callers that set it)
// and FAST_WEIGHTS exclude each other; other bits are unknown.
int32_t check_flags(uint32_t flags) {
    constexpr uint32_t known = SGL_KV_ATTN_EXACT_WEIGHTS | SGL_KV_ATTN_FAST_WEIGHTS;
    if (flags & ~known)
        return fail(SGL_KV_INVALID_ARGUMENT, "flags", flags, known, 0, "unknown attention plan flags 0x%x", flags);
    if ((flags & known) == known)
        return fail(SGL_KV_INVALID_ARGUMENT, "flags", flags, known, 0,
                    "attention plan flags 0x%x ask for exact and fast weights at once", flags);
    return SGL_KV_OK;
}

int32_t region_end(const char *tensor, uint64_t offset, uint64_t page_bytes, uint64_t stride,
                   uint64_t *end) {
    if (add_ovf(offset, page_bytes, end)) return attention_overflow();
    if (*end > stride)
        return fail(SGL_KV_TENSOR_PAGE_REGION_OUT_OF_BOUNDS, tensor, offset, page_bytes, stride,
                    "CUDA paged attention %s page region [%llu, %llu) exceeds page stride %llu", tensor,
                    (unsigned long long)offset, (unsigned long long)*end, (unsigned long long)stride);
    return SGL_KV_OK;
}

}  // namespace

// Device error word bits of the attention kernels ->
// DeviceMetadataInvalid with the reference's bit values (request 0x1,
// sequence 0x2, slot 0x4; cuda_attention.rs:59-99).
int32_t sglkv::attention_flag_status(uint32_t flag) {
    const uint32_t bad = ((flag & SGLKV_FLAG_ATTN_REQUEST) ? 1u : 0u) |
                         ((flag & SGLKV_FLAG_ATTN_SEQUENCE) ? 2u : 0u) |
                         ((flag & SGLKV_FLAG_ATTN_SLOT) ? 4u : 0u);
    if (bad)
        return fail(SGL_KV_ATTN_DEVICE_METADATA_INVALID, nullptr, bad, 0, 0,
                    "CUDA paged attention rejected device metadata with error flags 0x%x "
                    "(request=0x1, sequence=0x2, slot=0x4)",
                    bad);
    return ok();
}

extern "C" int32_t sgl_kv_attention_plan_new(const sgl_kv_attention_plan_config *c,
                                             sgl_kv_attention_plan *out) {
    if (!c || !out) return fail(SGL_KV_INVALID_ARGUMENT, "config/out", 0, 0, 0, "null argument");
    const sgl_kv_attention_layout &lay = c->layout;
    const struct {
        const char *name;
        uint64_t value;
    } dims[] = {{"query_count", c->query_count},
                {"request_count", c->request_count},
                {"sequence_slot_count", c->sequence_slot_count},
                {"slot_count", c->slot_count},
                {"query_head_count", c->query_head_count},
                {"kv_head_count", c->kv_head_count},
                {"query_key_head_dim", c->query_key_head_dim},
                {"value_head_dim", c->value_head_dim},
                {"page_size", lay.page_size},
                {"page_stride_bytes", lay.page_stride_bytes},
                {"key_row_bytes", lay.key_row_bytes},
                {"value_row_bytes", lay.value_row_bytes}};
    for (const auto &d : dims)
        if (d.value == 0)
            return fail(SGL_KV_ZERO_DIMENSION, d.name, 0, 0, 0,
                        "CUDA paged attention dimension %s must be non-zero", d.name);
    if (!isfinite(c->scale) || c->scale <= 0.0f) {
        uint32_t bits;
        memcpy(&bits, &c->scale, sizeof bits);
        return fail(SGL_KV_ATTN_INVALID_SCALE, nullptr, bits, 0, 0,
                    "CUDA paged attention scale must be finite and positive, got %g", (double)c->scale);
    }
    if (c->query_head_count % c->kv_head_count)
        return fail(SGL_KV_ATTN_QUERY_HEADS_NOT_DIVISIBLE, nullptr, c->query_head_count,
                    c->kv_head_count, 0,
                    "CUDA paged attention query head count %llu is not divisible by KV head count %llu",
                    (unsigned long long)c->query_head_count, (unsigned long long)c->kv_head_count);
    uint64_t want;
    if (mul_ovf(c->kv_head_count, c->query_key_head_dim, &want) || mul_ovf(want, 2, &want))
        return attention_overflow();
    if (lay.key_row_bytes != want)
        return fail(SGL_KV_ATTN_KEY_ROW_BYTES_MISMATCH, nullptr, want, lay.key_row_bytes, 0,
                    "CUDA BF16 paged attention requires %llu bytes per KV row, layout has %llu",
                    (unsigned long long)want, (unsigned long long)lay.key_row_bytes);
    if (mul_ovf(c->kv_head_count, c->value_head_dim, &want) || mul_ovf(want, 2, &want))
        return attention_overflow();
    if (lay.value_row_bytes != want)
        return fail(SGL_KV_ATTN_VALUE_ROW_BYTES_MISMATCH, nullptr, want, lay.value_row_bytes, 0,
                    "CUDA BF16 paged attention requires %llu bytes per value row, layout has %llu",
                    (unsigned long long)want, (unsigned long long)lay.value_row_bytes);
    uint64_t key_page, value_page, key_end, value_end;
    if (mul_ovf(lay.page_size, lay.key_row_bytes, &key_page) ||
        mul_ovf(lay.page_size, lay.value_row_bytes, &value_page))
        return attention_overflow();
    int32_t rc;
    if ((rc = region_end("key", lay.key_in_page_offset, key_page, lay.page_stride_bytes, &key_end)) ||
        (rc = region_end("value", lay.value_in_page_offset, value_page, lay.page_stride_bytes, &value_end)))
        return rc;
    if (lay.key_in_page_offset < value_end && lay.value_in_page_offset < key_end) {
        rc = fail(SGL_KV_ATTN_TENSOR_PAGE_REGIONS_OVERLAP, nullptr, lay.key_in_page_offset,
                  lay.value_in_page_offset, key_page,
                  "CUDA paged attention key/value page regions overlap: key offset %llu (%llu bytes), "
                  "value offset %llu (%llu bytes)",
                  (unsigned long long)lay.key_in_page_offset, (unsigned long long)key_page,
                  (unsigned long long)lay.value_in_page_offset, (unsigned long long)value_page);
        set_detail_d(value_page);
        return rc;
    }
    if (lay.head_layout > SGL_KV_HND)
        return fail(SGL_KV_INVALID_ARGUMENT, "head_layout", lay.head_layout, 0, 0,
                    "unknown head layout %u", lay.head_layout);
    if ((rc = check_flags(c->flags))) return rc;

    sgl_kv_attention_plan p;
    memset(&p, 0, sizeof p);
    p.config = *c;
    uint64_t v;
    if (mul_ovf(c->query_count, c->query_head_count, &v) || mul_ovf(v, c->query_key_head_dim, &v) ||
        mul_ovf(v, 2, &p.query_required_bytes))
        return attention_overflow();
    if (mul_ovf(c->query_count, 4, &p.query_request_indices_required_bytes) ||
        mul_ovf(c->query_count, 8, &p.query_sequence_lengths_required_bytes) ||
        add_ovf(c->request_count, 1, &v) || mul_ovf(v, 8, &p.request_slot_offsets_required_bytes) ||
        mul_ovf(c->sequence_slot_count, 8, &p.sequence_slots_required_bytes))
        return attention_overflow();
    // The pool must reach the last slot's key and value rows (NHD, as the
    // reference computes it) or, for head-major pages, the last page's
    // whole key and value regions.
    const uint64_t last_slot = c->slot_count - 1;
    const uint64_t last_page = last_slot / lay.page_size, last_token = last_slot % lay.page_size;
    uint64_t kend, vend;
    if (lay.head_layout == SGL_KV_HND) {
        kend = key_end;
        vend = value_end;
    } else if (mul_ovf(last_token, lay.key_row_bytes, &kend) ||
               add_ovf(kend, lay.key_in_page_offset, &kend) || add_ovf(kend, lay.key_row_bytes, &kend) ||
               mul_ovf(last_token, lay.value_row_bytes, &vend) ||
               add_ovf(vend, lay.value_in_page_offset, &vend) ||
               add_ovf(vend, lay.value_row_bytes, &vend)) {
        return attention_overflow();
    }
    if (mul_ovf(last_page, lay.page_stride_bytes, &v) ||
        add_ovf(v, kend > vend ? kend : vend, &p.pool_required_bytes))
        return attention_overflow();
    if (mul_ovf(c->query_count, c->query_head_count, &v) || mul_ovf(v, c->value_head_dim, &v) ||
        mul_ovf(v, 2, &p.output_required_bytes))
        return attention_overflow();
    // The reference sizes its block's shared memory as (256 + dv) floats and
    // launches one block per (query, head); keep its limits.
    if (add_ovf(256, c->value_head_dim, &v) || mul_ovf(v, 4, &v) || v > UINT32_MAX) return attention_overflow();
    if (c->query_count > UINT32_MAX)
        return too_large_dim("query_count", c->query_count, UINT32_MAX);
    if (c->query_head_count > UINT32_MAX)
        return too_large_dim("query_head_count", c->query_head_count, UINT32_MAX);
    *out = p;
    return ok();
}

// build_plan (crates/sglang-srt/src/cuda_attention.rs:505-572): the
// attention geometry of one layer of a bf16 pool.
extern "C" int32_t sgl_kv_attention_plan_for_layer(const sgl_kv_paged_layout *layout, uint64_t layer,
                                                   uint64_t query_count, uint64_t request_count,
                                                   uint64_t sequence_slot_count,
                                                   uint64_t query_head_count, float scale,
                                                   uint32_t head_layout, sgl_kv_attention_plan *out) {
    if (!layout || !out) return fail(SGL_KV_INVALID_ARGUMENT, "layout/out", 0, 0, 0, "null argument");
    const sgl_kv_runtime_layout &rt = layout->runtime;
    if (rt.dtype != SGL_KV_DTYPE_BFLOAT16) {
        static const char *const names[] = {"Auto", "Float32", "Bfloat16", "Fp8E4M3", "Fp8E5M2", "Fp4E2M1"};
        const char *name = rt.dtype >= 0 && rt.dtype <= 5 ? names[rt.dtype] : "unknown";
        return fail(SGL_KV_ATTN_UNSUPPORTED_KV_DTYPE, nullptr, (uint64_t)(int64_t)rt.dtype,
                    SGL_KV_DTYPE_BFLOAT16, 0,
                    "CUDA paged attention requires KV cache dtype Bfloat16, found %s", name);
    }
    uint64_t start, end, key_row, value_row;
    int32_t rc;
    if ((rc = sgl_kv_paged_layout_tensor_token_byte_range(layout, 0, layer, 0, 0, &start, &end)))
        return rc;
    key_row = end - start;
    const uint64_t key_offset = start;
    if ((rc = sgl_kv_paged_layout_tensor_token_byte_range(layout, 0, layer, 1, 0, &start, &end)))
        return rc;
    value_row = end - start;
    const uint64_t value_offset = start;
    uint64_t denom;
    if (mul_ovf(rt.kv_heads, 2, &denom) || key_row % denom)
        return fail(SGL_KV_ATTN_TENSOR_ROW_GEOMETRY_MISMATCH, "key", key_row, rt.kv_heads, 2,
                    "CUDA paged attention key row has %llu bytes, which cannot be divided across %llu "
                    "heads of 2-byte elements",
                    (unsigned long long)key_row, (unsigned long long)rt.kv_heads);
    if (value_row % denom)
        return fail(SGL_KV_ATTN_TENSOR_ROW_GEOMETRY_MISMATCH, "value", value_row, rt.kv_heads, 2,
                    "CUDA paged attention value row has %llu bytes, which cannot be divided across %llu "
                    "heads of 2-byte elements",
                    (unsigned long long)value_row, (unsigned long long)rt.kv_heads);
    sgl_kv_attention_plan_config c;
    memset(&c, 0, sizeof c);
    c.query_count = query_count;
    c.request_count = request_count;
    c.sequence_slot_count = sequence_slot_count;
    c.slot_count = layout->slot_count;
    c.query_head_count = query_head_count;
    c.kv_head_count = rt.kv_heads;
    c.query_key_head_dim = key_row / denom;
    c.value_head_dim = value_row / denom;
    c.scale = scale;
    c.layout.page_size = rt.page_size;
    c.layout.page_stride_bytes = rt.page_size_bytes;
    c.layout.key_in_page_offset = key_offset;
    c.layout.value_in_page_offset = value_offset;
    c.layout.key_row_bytes = key_row;
    c.layout.value_row_bytes = value_row;
    c.layout.head_layout = head_layout;
    return sgl_kv_attention_plan_new(&c, out);
}

namespace {

int32_t attn_ptr(const char *name, const sgl_kv_device_buffer &b, uint64_t offset, uint64_t need,
                 uint64_t *addr) {
    if (!b.ptr) return fail(SGL_KV_INVALID_ARGUMENT, name, 0, 0, 0, "null buffer %s", name);
    uint64_t end;
    if (add_ovf(offset, need, &end) || end > b.byte_len)
        return fail(SGL_KV_ALLOCATION_OUT_OF_BOUNDS, name, offset, need, b.byte_len,
                    "allocation %s range [%llu, +%llu) exceeds its %llu bytes", name,
                    (unsigned long long)offset, (unsigned long long)need,
                    (unsigned long long)b.byte_len);
    *addr = (uint64_t)(uintptr_t)b.ptr + offset;
    return SGL_KV_OK;
}

uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// The tiles of a launch with several queries per request, and whether they
// are the faster way.
struct TileShape {
    uint64_t queries, per_request, live, max_len, dims, mean;

    TileShape(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p, uint64_t longest)
        : queries(p.group && p.group <= SGLKV_ATTN_TILE_ROWS(p.dk) ? SGLKV_ATTN_TILE_ROWS(p.dk) / p.group : 1),
          // (the queries shared evenly among the requests)
          per_request(ceil_div(ceil_div(c.query_count, c.request_count), queries)),
          live(per_request * c.request_count * p.kv_heads), max_len(longest), dims(p.dk),
          mean(ceil_div(c.sequence_slot_count, c.request_count)) {}

    // Splits that fill `target` resident workgroups: of 256 tokens or more,
    // or of 128 where a request is one tile (few queries, so the records that
    // the splits leave are few). They are counted for the longest sequence
    // also where most are shorter: with as many more as the average leaves
    // room for, 24 requests of 200..3,000 tokens (dims 256) took 49 us, not 38.
    uint64_t splits(uint64_t target) const {
        const uint64_t want = live >= target ? 1 : target / live, least = per_request > 1 ? 256 : 128;
        return want < max_len / least ? want : (max_len >= 2 * least ? max_len / least : 1);
    }

    // Whether the tiles are estimated to take less time than the staged
    // bodies, whose work items are one query's. Times in units of 50 ns, from
    // measurements on MI355X: the staged bodies take about 8 us, 6 more once
    // they split (and merge: where twice the work items fit the resident slots,
    // or a sequence is longer than a slot table), and 50 ns for each token that a resident
    // workgroup's share comes to (100 past 128; half of that at dims 64, whose
    // workgroups are twice as many); a tile takes about 11 us to its first
    // block, 5 more if split, and per block 0.8, 1.5 or 1.0 us (dims 64, 128;
    // 256, whose blocks are half as long) where other tiles of the request
    // have brought the rows into L2, 2.2 us where it reads them first. Tiles
    // and staged measured: 64 queries of one prompt (dims 128) 13.9 and 12.0
    // us, 4 x 64 12.8 and 17.9, 160 15.2 and 19.1, 4 x 160 16 and 51; 4 x 2
    // queries of up to 1,000 tokens 22 and 15, 20 x 5 30 and 57 (over 8 KV
    // heads; over one 27 and 18).
    bool pays(int cu_count, uint64_t items) const {
        const uint64_t cus = cu_count > 0 ? (uint64_t)cu_count : 256, lds = 160u * 1024u;
        const uint64_t staged_slots = cus * (lds / SGLKV_ATTN_STAGED_LDS_BYTES(dims));
        uint64_t share;  // tokens per resident workgroup
        if (mul_ovf(items, mean, &share)) return true;
        share = share / staged_slots / (dims == 64 ? 2 : 1);
        const bool cuts = (max_len > 64 && items <= staged_slots / 2) || max_len > SGLKV_ATTN_STAGED_SLOTS;
        const uint64_t staged = 160 + (cuts ? 120 : 0) + share + (share > 128 ? share - 128 : 0);
        const uint64_t cut = splits(cus * (lds / SGLKV_ATTN_TILE_LDS_BYTES(dims)));
        const uint64_t blocks = ceil_div(ceil_div(max_len, cut), SGLKV_ATTN_TILE_BLOCK(dims));
        const uint64_t block = per_request == 1 ? 44 : dims == 64 ? 16 : dims == 128 ? 30 : 20;
        return 220 + blocks * block + (cut > 1 ? 100 : 0) < staged;
    }
};

// Checks a call and sets the kernels' parameters that do not depend on how it
// is launched.
int32_t attention_params(sgl_rocm_kv_ctx *ctx, const sgl_kv_attention_plan *plan, const sgl_kv_attention_buffers *b,
                         uint32_t *flag_word, sglkv_attn_params *params) {
    if (!ctx || !plan || !b)
        return fail(SGL_KV_INVALID_ARGUMENT, "ctx/plan/buffers", 0, 0, 0, "null argument");
    const sgl_kv_attention_plan_config &c = plan->config;
    const sgl_kv_attention_layout &lay = c.layout;
    const struct {
        const char *name;
        const sgl_kv_device_buffer *buf;
    } all[] = {{"queries", &b->queries},
               {"query_request_indices", &b->query_request_indices},
               {"query_sequence_lengths", &b->query_sequence_lengths},
               {"request_slot_offsets", &b->request_slot_offsets},
               {"sequence_slots", &b->sequence_slots},
               {"pool", &b->pool},
               {"output", &b->output}};
    int32_t rc;
    for (const auto &a : all)
        if ((rc = check_device(ctx, a.name, *a.buf))) return rc;
    // A plan is a plain struct the caller may have edited since plan_new.
    if ((rc = check_flags(c.flags))) return rc;
    uint64_t qp, rip, slp, rop, ssp, poolp, outp;
    if ((rc = attn_ptr("queries", b->queries, b->queries_offset, plan->query_required_bytes, &qp)) ||
        (rc = attn_ptr("query_request_indices", b->query_request_indices, b->query_request_indices_offset,
                       plan->query_request_indices_required_bytes, &rip)) ||
        (rc = attn_ptr("query_sequence_lengths", b->query_sequence_lengths,
                       b->query_sequence_lengths_offset, plan->query_sequence_lengths_required_bytes,
                       &slp)) ||
        (rc = attn_ptr("request_slot_offsets", b->request_slot_offsets, b->request_slot_offsets_offset,
                       plan->request_slot_offsets_required_bytes, &rop)) ||
        (rc = attn_ptr("sequence_slots", b->sequence_slots, b->sequence_slots_offset,
                       plan->sequence_slots_required_bytes, &ssp)) ||
        (rc = attn_ptr("pool", b->pool, b->pool_offset, plan->pool_required_bytes, &poolp)) ||
        (rc = attn_ptr("output", b->output, b->output_offset, plan->output_required_bytes, &outp)))
        return rc;
    if (c.query_key_head_dim > SGLKV_ATTN_MAX_DK)
        return too_large_dim("query_key_head_dim", c.query_key_head_dim, SGLKV_ATTN_MAX_DK);
    // Every element access is naturally aligned.
    const bool aligned = qp % 2 == 0 && outp % 2 == 0 && rip % 4 == 0 && slp % 8 == 0 && rop % 8 == 0 &&
                         ssp % 8 == 0 &&
                         ((poolp | lay.key_in_page_offset | lay.value_in_page_offset |
                           lay.page_stride_bytes | lay.key_row_bytes | lay.value_row_bytes) & 1) == 0;
    if (!aligned)
        return fail(SGL_KV_INVALID_ARGUMENT, "alignment", 0, 0, 0,
                    "paged attention buffers must be aligned to their element sizes");

    sglkv_attn_params &p = *params;
    memset(&p, 0, sizeof p);
    p.queries = reinterpret_cast<const uint16_t *>(qp);
    p.query_request_indices = reinterpret_cast<const uint32_t *>(rip);
    p.query_sequence_lengths = reinterpret_cast<const uint64_t *>(slp);
    p.request_slot_offsets = reinterpret_cast<const uint64_t *>(rop);
    p.sequence_slots = reinterpret_cast<const uint64_t *>(ssp);
    p.pool = reinterpret_cast<const uint8_t *>(poolp);
    p.output = reinterpret_cast<uint16_t *>(outp);
    p.flag = flag_word;
    p.query_count = c.query_count;
    p.request_count = c.request_count;
    p.sequence_slot_count = c.sequence_slot_count;
    p.slot_count = c.slot_count;
    p.page_size = lay.page_size;
    p.page_stride = lay.page_stride_bytes;
    p.key_offset = lay.key_in_page_offset;
    p.value_offset = lay.value_in_page_offset;
    const uint64_t kh = c.query_key_head_dim * 2, vh = c.value_head_dim * 2;
    if (lay.head_layout == SGL_KV_HND) {
        p.key_head_stride = lay.page_size * kh;
        p.key_token_stride = kh;
        p.value_head_stride = lay.page_size * vh;
        p.value_token_stride = vh;
    } else {
        p.key_head_stride = kh;
        p.key_token_stride = lay.key_row_bytes;
        p.value_head_stride = vh;
        p.value_token_stride = lay.value_row_bytes;
    }
    p.query_heads = (uint32_t)c.query_head_count;
    p.kv_heads = (uint32_t)c.kv_head_count;
    p.group = (uint32_t)(c.query_head_count / c.kv_head_count);
    p.head_groups = (uint32_t)(((uint64_t)p.group + SGLKV_ATTN_HEADS - 1) / SGLKV_ATTN_HEADS);
    p.dk = (uint32_t)c.query_key_head_dim;
    p.dk_pad = (p.dk + 31) / 32 * 32;
    p.dv = (uint32_t)c.value_head_dim;
    p.dv_blocks = (p.dv + SGLKV_ATTN_DV - 1) / SGLKV_ATTN_DV;
    p.scale_log2 = c.scale * 1.4426950408889634f;
    p.page_shift = 32;
    if ((lay.page_size & (lay.page_size - 1)) == 0) {
        p.page_shift = 0;
        while ((1ull << p.page_shift) < lay.page_size) ++p.page_shift;
    }
    p.zero_row = ctx->zero_row;
    return SGL_KV_OK;
}

// Workgroups of `body` that a CU holds, asked of the device once per LDS size.
uint32_t attention_resident(void *context, int body, unsigned threads, unsigned lds) {
    sgl_rocm_kv_ctx *ctx = static_cast<sgl_rocm_kv_ctx *>(context);
    if (ctx->attention_occupancy_lds[body] != lds) {
        int per_cu = 0;
        const hipError_t err =
            hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ctx->attention[body], (int)threads, lds);
        if (err != hipSuccess) {
            (void)hip_fail(err, "hipModuleOccupancyMaxActiveBlocksPerMultiprocessor");
            return 0;
        }
        ctx->attention_occupancy[body] = per_cu > 0 ? (uint32_t)per_cu : 1;
        ctx->attention_occupancy_lds[body] = lds;
    }
    return ctx->attention_occupancy[body];
}

AttentionDevice attention_device(sgl_rocm_kv_ctx *ctx) {
    return {ctx->cu_count > 0 ? (uint64_t)ctx->cu_count : 256, (uint64_t)(unsigned)ctx->max_lds_per_block, ctx,
            attention_resident};
}

// The tiles' own record buffer and the event that orders the calls that use
// it, made at the first such call. False where there is no memory for them.
// Only kernels of this device touch the records, each of which makes its
// writes visible to the device at its end: the event needs no system fence
// (with one a call took 3 us longer than without any order, so 1).
bool attention_tile_records(sgl_rocm_kv_ctx *ctx) {
    if (ctx->tile_records) return true;
    if (!ctx->tile_order && hipEventCreateWithFlags(&ctx->tile_order, hipEventDisableTiming | hipEventDisableSystemFence) !=
                                hipSuccess)
        ctx->tile_order = nullptr;
    if (!ctx->tile_order || hipMalloc(&ctx->tile_records, kAttentionTileRecordBytes) != hipSuccess) {
        ctx->tile_records = nullptr;
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// Where a call's records can go.
AttentionRecords attention_records(const sgl_rocm_kv_ctx *ctx, uint64_t workspace_bytes) {
    const uint64_t held = workspace_bytes ? workspace_bytes : ctx->attention_partial_bytes;
    return {workspace_bytes, held && held < kAttentionShorterBytes ? held : kAttentionShorterBytes, true};
}

// Makes the context's record buffer hold `bytes`; a new one holds
// kAttentionShorterBytes, or `bytes` alone where memory is short.
hipError_t attention_grow(sgl_rocm_kv_ctx *ctx, uint64_t bytes) {
    if (ctx->attention_partial) {
        hipError_t err = hipDeviceSynchronize();
        if (err == hipSuccess) err = hipFree(ctx->attention_partial);
        if (err != hipSuccess) return err;
        ctx->attention_partial = nullptr;
        ctx->attention_partial_bytes = 0;
    }
    uint64_t size = bytes < kAttentionShorterBytes ? kAttentionShorterBytes : bytes;
    hipError_t err = hipMalloc(&ctx->attention_partial, size);
    if (err == hipErrorOutOfMemory && size > bytes) {
        (void)hipGetLastError();
        size = bytes;
        err = hipMalloc(&ctx->attention_partial, size);
    }
    if (err == hipSuccess)
        ctx->attention_partial_bytes = size;
    else
        ctx->attention_partial = nullptr;
    return err;
}

// Validates, sizes the split and launches the attention (and, with
// several splits, the combine pass) on `stream`; nothing waits. Metadata
// errors raise `flag_word`. `workspace` (fixed, `workspace_bytes` long)
// holds the split records when given; otherwise the context's buffers.
int32_t attention_enqueue(sgl_rocm_kv_ctx *ctx, const sgl_kv_attention_plan *plan,
                          const sgl_kv_attention_buffers *b, uint64_t max_sequence_length,
                          hipStream_t s, uint32_t *flag_word, void *workspace = nullptr,
                          uint64_t workspace_bytes = 0) {
    sglkv_attn_params p;
    AttentionRoute r;
    int32_t rc = attention_params(ctx, plan, b, flag_word, &p);
    if (rc) return rc;
    DeviceScope scope(ctx->device);
    if (scope.status() != hipSuccess) return hip_fail(scope.status(), "hipSetDevice");
    const sglkv_attn_params unrouted = p;
    AttentionRecords records = attention_records(ctx, workspace_bytes);
    auto route = [&] {
        p = unrouted;
        return attention_route(attention_device(ctx), plan->config, max_sequence_length, records, &p, &r);
    };
    if ((rc = route())) return rc;
    const bool grows = !workspace && !r.apart && r.record_bytes > ctx->attention_partial_bytes;
    if (r.apart || (grows && r.shortened)) {
        // A capture can neither allocate nor wait for an event recorded
        // outside it.
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        SGLKV_CHECK_HIP(hipStreamIsCapturing(s, &capture));
        const bool captures = capture != hipStreamCaptureStatusNone;
        if (r.apart) records.apart = !captures && attention_tile_records(ctx);
        if (r.shortened && captures) records.shorter = 0;
        if ((!records.apart || !records.shorter) && (rc = route())) return rc;
    }
    if (workspace) {
        if (r.record_bytes > workspace_bytes)
            return fail(SGL_KV_DIMENSION_TOO_LARGE, "workspace", r.record_bytes, workspace_bytes, 0,
                        "paged attention needs %llu bytes of split records, more than the "
                        "%llu-byte workspace",
                        (unsigned long long)r.record_bytes, (unsigned long long)workspace_bytes);
    } else if (!r.apart && r.record_bytes > ctx->attention_partial_bytes) {
        hipError_t err = attention_grow(ctx, r.record_bytes);
        if (err == hipErrorOutOfMemory && r.shortened) {
            (void)hipGetLastError();
            records.shorter = 0;
            if ((rc = route())) return rc;
            err = attention_grow(ctx, r.record_bytes);
        }
        if (err != hipSuccess) return hip_fail(err, "hipMalloc");
    }
    if (p.splits > 1)
        p.partial = static_cast<float *>(workspace ? workspace : r.apart ? ctx->tile_records : ctx->attention_partial);
    if (r.apart) SGLKV_CHECK_HIP(hipStreamWaitEvent(s, ctx->tile_order, 0));
    void *args[] = {&p};
    hipError_t err = hipModuleLaunchKernel(p.compact ? ctx->attention_live[r.body] : ctx->attention[r.body],
                                           (unsigned)r.grid, p.splits, 1, r.threads, 1, 1, r.lds, s, args, nullptr);
    if (err == hipSuccess && p.splits > 1)
        err = hipModuleLaunchKernel(r.half_records ? ctx->attention_combine_h : ctx->attention_combine,
                                    (unsigned)r.combine_grid, 1, 1, r.combine_threads, 1, 1, 0, s, args, nullptr);
    // Recorded also after a failure: a first launch may have been made.
    if (r.apart) {
        const hipError_t rec = hipEventRecord(ctx->tile_order, s);
        if (err == hipSuccess) err = rec;
    }
    return err == hipSuccess ? SGL_KV_OK : hip_fail(err, "paged attention launch");
}

}  // namespace

extern "C" int32_t sgl_rocm_kv_paged_attention(sgl_rocm_kv_ctx *ctx, const sgl_kv_attention_plan *plan,
                                               const sgl_kv_attention_buffers *b,
                                               uint64_t max_sequence_length, void *stream) {
    if (!ctx) return fail(SGL_KV_INVALID_ARGUMENT, "ctx", 0, 0, 0, "null argument");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // The synchronous forward has an error word of its own, as the
    // reference's kernels object has its flag (cuda_attention.rs:667,
    // 706-707): asynchronous launches still running on other streams raise
    // the asynchronous word, so nothing here can take or clear their bits.
    // Calls on one context do not overlap, so the word is clean on entry:
    // every synchronous call leaves it zero.
    int32_t rc = attention_enqueue(ctx, plan, b, max_sequence_length, s, ctx->sync_attn_flag);
    if (rc) return rc;
    DeviceScope scope(ctx->device);
    if (scope.status() != hipSuccess) return hip_fail(scope.status(), "hipSetDevice");
    // The word is read and cleared on the stream, into a pinned host word (a
    // blocking copy after the wait costs more than the launch).
    uint32_t *out = ctx->host_attn(), *word = ctx->sync_attn_flag;
    void *args[] = {&word, &word, &out};
    SGLKV_CHECK_HIP(hipModuleLaunchKernel(ctx->take_flags, 1, 1, 1, 64, 1, 1, 0, s, args, nullptr));
    SGLKV_CHECK_HIP(hipStreamSynchronize(s));
    return attention_flag_status(__atomic_load_n(out, __ATOMIC_ACQUIRE) | __atomic_load_n(out + 1, __ATOMIC_ACQUIRE));
}

extern "C" int32_t sgl_rocm_kv_attention_route(sgl_rocm_kv_ctx *ctx, const sgl_kv_attention_plan *plan,
                                               const sgl_kv_attention_buffers *b, uint64_t max_sequence_length,
                                               sgl_kv_attention_route *out) {
    if (!out) return fail(SGL_KV_INVALID_ARGUMENT, "out", 0, 0, 0, "null argument");
    sglkv_attn_params p;
    AttentionRoute r;
    int32_t rc = attention_params(ctx, plan, b, nullptr, &p);
    if (rc) return rc;
    DeviceScope scope(ctx->device);
    if (scope.status() != hipSuccess) return hip_fail(scope.status(), "hipSetDevice");
    if ((rc = attention_route(attention_device(ctx), plan->config, max_sequence_length,
                              attention_records(ctx, 0), &p, &r)))
        return rc;
    memset(out, 0, sizeof *out);
    out->body = (uint32_t)r.body;
    out->live_splits_first = p.compact != 0;
    out->splits = p.splits;
    out->chunk_tokens = p.chunk_tokens;
    out->workgroups = r.grid * p.splits;
    out->record_bytes = r.record_bytes;
    out->records_apart = r.apart;
    return ok();
}

extern "C" int32_t sgl_rocm_kv_paged_attention_async(sgl_rocm_kv_ctx *ctx,
                                                     const sgl_kv_attention_plan *plan,
                                                     const sgl_kv_attention_buffers *b,
                                                     uint64_t max_sequence_length, void *stream) {
    if (!ctx) return fail(SGL_KV_INVALID_ARGUMENT, "ctx", 0, 0, 0, "null argument");
    const int32_t rc =
        attention_enqueue(ctx, plan, b, max_sequence_length, static_cast<hipStream_t>(stream), ctx->attn_flag);
    return rc ? rc : ok();
}

extern "C" int32_t sgl_rocm_kv_paged_attention_async_noalloc(sgl_rocm_kv_ctx *ctx,
                                                             const sgl_kv_attention_plan *plan,
                                                             const sgl_kv_attention_buffers *b,
                                                             uint64_t max_sequence_length, void *stream) {
    if (!ctx) return fail(SGL_KV_INVALID_ARGUMENT, "ctx", 0, 0, 0, "null argument");
    if (!ctx->noalloc_workspace || !ctx->noalloc_order)
        return fail(SGL_KV_MODULE, "workspace", 0, 0, 0, "the context has no workspace address");
    hipStream_t s = static_cast<hipStream_t>(stream);
    DeviceScope scope(ctx->device);
    if (scope.status() != hipSuccess) return hip_fail(scope.status(), "hipSetDevice");
    // Every call on this device shares the workspace. The device's event
    // marks the end of the last call that used it: this call's launches
    // wait for it on `s`, and the event then moves past this call's
    // combine. The lock makes wait, launch and record one step for all
    // host threads and contexts, so calls on any streams run in the order
    // they were made. Under stream capture the graph's own dependencies
    // order its launches (an event recorded outside the capture cannot be
    // waited on there), so the event is left alone.
    NoallocOrder *order = ctx->noalloc_order;
    std::lock_guard<std::mutex> guard(order->lock);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    SGLKV_CHECK_HIP(hipStreamIsCapturing(s, &capture));
    const bool ordered = capture == hipStreamCaptureStatusNone;
    if (ordered) SGLKV_CHECK_HIP(hipStreamWaitEvent(s, order->last, 0));
    const int32_t rc = attention_enqueue(ctx, plan, b, max_sequence_length, s, ctx->attn_flag,
                                         ctx->noalloc_workspace, SGL_KV_NOALLOC_WORKSPACE_BYTES);
    // Recorded whatever the enqueue returned: a failure after its first
    // launch still leaves work on `s` that uses the workspace.
    const hipError_t rec = ordered ? hipEventRecord(order->last, s) : hipSuccess;
    if (rc) return rc;
    if (rec != hipSuccess) return hip_fail(rec, "hipEventRecord");
    return ok();
}
