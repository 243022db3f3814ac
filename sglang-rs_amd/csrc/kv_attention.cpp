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

int32_t attn_overflow() {
    return fail(SGL_KV_SHAPE_OVERFLOW, nullptr, 0, 0, 0, "CUDA paged attention shape overflowed");
}

int32_t region_end(const char *tensor, uint64_t offset, uint64_t page_bytes, uint64_t stride,
                   uint64_t *end) {
    if (add_ovf(offset, page_bytes, end)) return attn_overflow();
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
        return attn_overflow();
    if (lay.key_row_bytes != want)
        return fail(SGL_KV_ATTN_KEY_ROW_BYTES_MISMATCH, nullptr, want, lay.key_row_bytes, 0,
                    "CUDA BF16 paged attention requires %llu bytes per KV row, layout has %llu",
                    (unsigned long long)want, (unsigned long long)lay.key_row_bytes);
    if (mul_ovf(c->kv_head_count, c->value_head_dim, &want) || mul_ovf(want, 2, &want))
        return attn_overflow();
    if (lay.value_row_bytes != want)
        return fail(SGL_KV_ATTN_VALUE_ROW_BYTES_MISMATCH, nullptr, want, lay.value_row_bytes, 0,
                    "CUDA BF16 paged attention requires %llu bytes per value row, layout has %llu",
                    (unsigned long long)want, (unsigned long long)lay.value_row_bytes);
    uint64_t key_page, value_page, key_end, value_end;
    if (mul_ovf(lay.page_size, lay.key_row_bytes, &key_page) ||
        mul_ovf(lay.page_size, lay.value_row_bytes, &value_page))
        return attn_overflow();
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
        return attn_overflow();
    if (mul_ovf(c->query_count, 4, &p.query_request_indices_required_bytes) ||
        mul_ovf(c->query_count, 8, &p.query_sequence_lengths_required_bytes) ||
        add_ovf(c->request_count, 1, &v) || mul_ovf(v, 8, &p.request_slot_offsets_required_bytes) ||
        mul_ovf(c->sequence_slot_count, 8, &p.sequence_slots_required_bytes))
        return attn_overflow();
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
        return attn_overflow();
    }
    if (mul_ovf(last_page, lay.page_stride_bytes, &v) ||
        add_ovf(v, kend > vend ? kend : vend, &p.pool_required_bytes))
        return attn_overflow();
    if (mul_ovf(c->query_count, c->query_head_count, &v) || mul_ovf(v, c->value_head_dim, &v) ||
        mul_ovf(v, 2, &p.output_required_bytes))
        return attn_overflow();
    // The reference sizes its block's shared memory as (256 + dv) floats and
    // launches one block per (query, head); keep its limits.
    if (add_ovf(256, c->value_head_dim, &v) || mul_ovf(v, 4, &v) || v > UINT32_MAX) return attn_overflow();
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

// Validates, sizes the split and launches the attention (and, with
// several splits, the combine pass) on `stream`; nothing waits. Metadata
// errors raise `flag_word`. `workspace` (fixed, `workspace_bytes` long)
// holds the split records when given; otherwise the context's buffer,
// grown on demand.
int32_t attention_enqueue(sgl_rocm_kv_ctx *ctx, const sgl_kv_attention_plan *plan,
                          const sgl_kv_attention_buffers *b, uint64_t max_sequence_length,
                          hipStream_t s, uint32_t *flag_word, void *workspace = nullptr,
                          uint64_t workspace_bytes = 0) {
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

    sglkv_attn_params p;
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
    p.head_groups = (uint32_t)ceil_div(p.group, SGLKV_ATTN_HEADS);
    p.dk = (uint32_t)c.query_key_head_dim;
    p.dk_pad = (uint32_t)ceil_div(p.dk, 32) * 32;
    p.dv = (uint32_t)c.value_head_dim;
    p.dv_blocks = (uint32_t)ceil_div(p.dv, SGLKV_ATTN_DV);
    p.scale_log2 = c.scale * 1.4426950408889634f;
    p.page_shift = 32;
    if ((lay.page_size & (lay.page_size - 1)) == 0) {
        p.page_shift = 0;
        while ((1ull << p.page_shift) < lay.page_size) ++p.page_shift;
    }

    const bool vec = (p.dk % 8 == 0) && (p.dv % 8 == 0) &&
                     ((poolp + lay.key_in_page_offset) % 16 == 0) &&
                     ((poolp + lay.value_in_page_offset) % 16 == 0) &&
                     ((lay.page_stride_bytes | p.key_head_stride | p.key_token_stride | p.value_head_stride |
                       p.value_token_stride) % 16 == 0);
    // 16-byte rows, power-of-two pages and strides that fit 32 bits admit
    // the pipelined and wide bodies (32-bit slots, shift-and-mask pages);
    // head dims up to 128 take the software-pipelined body.
    const bool fast = vec && p.page_shift < 32 && c.slot_count < (1ull << 32) &&
                      lay.page_stride_bytes <= UINT32_MAX && p.key_token_stride <= UINT32_MAX &&
                      p.value_token_stride <= UINT32_MAX;
    const bool pipe = fast && p.dk_pad <= 128 && p.dv <= SGLKV_ATTN_DV;
    int which = !vec ? 1 : !pipe ? 0 : (p.dk == 128 && p.dv == 128) ? 2 : 3;
    // Many query heads per KV head (more than one 16-head group) or wide
    // values: the wide bodies share each K/V block among 4 head groups
    // instead of every group and value block reading it again. They hold
    // the queries in registers as 16-byte vectors.
    unsigned threads = 64;
    unsigned lds = (unsigned)((SGLKV_ATTN_HEADS * (p.dk_pad + 8) + SGLKV_ATTN_DV * SGLKV_ATTN_VT_STRIDE) *
                              sizeof(uint16_t));
    uint64_t max_len = max_sequence_length ? max_sequence_length : c.sequence_slot_count;
    if (max_len > c.sequence_slot_count) max_len = c.sequence_slot_count;
    // (Their chunks fit the slot table, so the grid's 65535 splits bound
    // the length they take.)
    if (fast && qp % 16 == 0 && (p.head_groups > 1 || p.dv > SGLKV_ATTN_DV) &&
        max_len <= 65535ull * SGLKV_ATTN_WIDE_SLOTS) {
        const unsigned narrow = SGLKV_ATTN_WIDE_LDS_BYTES(4u, 8u), wide = SGLKV_ATTN_WIDE_LDS_BYTES(18u, 32u);
        if (p.dk_pad <= 128 && p.dv <= 128 && narrow <= (unsigned)ctx->max_lds_per_block) {
            which = 5;
            lds = narrow;
            threads = 64 * SGLKV_ATTN_WIDE_WAVES;
        } else if (p.dk > 512 && p.dk <= 576 && p.dv == 512 &&
                   SGLKV_ATTN_LATENT_LDS_BYTES <= (unsigned)ctx->max_lds_per_block) {
            // MLA's latent rows (K 576 = 512 + 64 rope dims, V 512): 32 heads
            // per wave, rows loaded straight into LDS.
            which = 6;
            lds = SGLKV_ATTN_LATENT_LDS_BYTES;
            threads = 64 * SGLKV_ATTN_LATENT_WAVES;
        } else if (p.dk_pad <= 576 && p.dv <= 512 && wide <= (unsigned)ctx->max_lds_per_block) {
            which = 4;
            lds = wide;
            threads = 64 * SGLKV_ATTN_WIDE_WAVES;
        }
    }
    // Dims 128 or 64 with one head group per KV head (the Llama/Qwen GQA
    // decodes): the staged bodies, rows loaded straight into LDS. They
    // share one in-page offset between a token's K and V rows and form it
    // with a 24-bit multiply.
    // Dims 256 (Qwen3.5's full-attention layers) take the staged body too,
    // one wave covering all 256 value dims.
    const bool d64 = which == 3 && p.dk == 64 && p.dv == 64;
    const bool d256 = fast && p.dk == 256 && p.dv == 256;
    if ((which == 2 || d64 || d256) && qp % 16 == 0 && p.head_groups == 1 &&
        p.key_token_stride == p.value_token_stride && p.key_token_stride < (1u << 24) &&
        lay.page_size <= (1u << 24) &&
        max_len <= 65535ull * SGLKV_ATTN_STAGED_SLOTS &&
        SGLKV_ATTN_STAGED_LDS_BYTES(p.dk) <= (unsigned)ctx->max_lds_per_block) {
        which = d64 ? 8 : d256 ? 10 : 7;
        lds = SGLKV_ATTN_STAGED_LDS_BYTES(p.dk);
        // Head-major pages at dims 128: K in registers, V alone in LDS.
        // (Dims 64 keep K in LDS: the same body with K in registers,
        // 125 VGPRs, measured no faster on head-major pages.)
        if (which == 7 && lay.head_layout == SGL_KV_HND) {
            which = 11;
            lds = SGLKV_ATTN_KREG_LDS_BYTES(p.dk);
        }
        threads = 64;
        p.dv_blocks = 1;
    }
    // Several queries per request on average (prefill, chunked prefill,
    // drafted tokens): the tile bodies, which read a K/V row once per tile of
    // queries instead of once per query. They take the staged bodies' shapes
    // and any group of up to 64 query heads, 32 at dims 256 (a tile then holds
    // at least two queries), count tokens in 32 bits and write 8-byte pieces.
    const bool tileable = fast && p.dk == p.dv && (p.dk == 64 || p.dk == 128 || p.dk == 256) && qp % 16 == 0 &&
                          outp % 8 == 0 && p.group <= SGLKV_ATTN_TILE_ROWS(p.dk) / 2 &&
                          p.key_token_stride == p.value_token_stride && p.key_token_stride < (1u << 24) &&
                          lay.page_size <= (1u << 24) && c.query_count / 2 >= c.request_count &&
                          c.query_count <= SGLKV_ATTN_TILE_QUERIES_MAX &&
                          c.query_count <= UINT32_MAX / 512 / p.kv_heads && max_len <= (1u << 30) &&
                          SGLKV_ATTN_TILE_LDS_BYTES(p.dk) <= (unsigned)ctx->max_lds_per_block;
    const TileShape shape(c, p, tileable ? max_len : 1);
    const bool tile = tileable && (which < 7 || shape.pays(ctx->cu_count, c.query_count * p.kv_heads));
    if (tile) {
        which = p.dk == 128 ? 12 : p.dk == 64 ? 13 : 14;
        lds = SGLKV_ATTN_TILE_LDS_BYTES(p.dk);
        threads = 256;
        p.tile_queries = (uint32_t)shape.queries;
        p.tile_recip = UINT32_MAX / p.tile_queries + 1;
        // Queries that come request by request make at most this many tiles.
        const uint64_t most = c.query_count / p.tile_queries + c.request_count;
        p.tile_slots = (uint32_t)(most < c.query_count ? most : c.query_count);
        // Later tiles of a causal prompt attend more tokens: they start
        // first, except where each request is one tile. (Several prompts'
        // last tiles in turn were no faster: 4 of 2,048 tokens 266 us against
        // 259, 4 of 300..2,048 189 against 143.)
        p.tile_backward = shape.per_request > 1;
    }
    p.zero_row = ctx->zero_row;
    p.page_stride32 = (uint32_t)lay.page_stride_bytes;
    p.key_token_stride32 = (uint32_t)p.key_token_stride;
    p.value_token_stride32 = (uint32_t)p.value_token_stride;
    DeviceScope scope(ctx->device);
    if (scope.status() != hipSuccess) return hip_fail(scope.status(), "hipSetDevice");

    // Workgroups before splitting; split each query's sequence so that the
    // launch fills every CU with as many workgroups as stay resident at
    // once (the kernel's occupancy at this LDS size), in one round.
    const bool wide = which >= 4 && which <= 6;  // the wide and latent bodies (7, 8, 10, 11: staged)
    const uint64_t hblocks = which == 6 ? ceil_div(p.group, SGLKV_ATTN_LATENT_HEADS)
                                        : (p.head_groups + SGLKV_ATTN_WIDE_GROUPS - 1) / SGLKV_ATTN_WIDE_GROUPS;
    uint64_t base = tile ? p.tile_slots : c.query_count;
    if (mul_ovf(base, p.kv_heads, &base) || (wide && mul_ovf(base, hblocks, &base)) ||
        (!wide && !tile && (mul_ovf(base, p.head_groups, &base) || mul_ovf(base, p.dv_blocks, &base))) ||
        base > UINT32_MAX / threads)  // a dispatch counts its work-items in 32 bits
        return too_large_dim("workgroups", base, UINT32_MAX / threads);
    // The latent body has two functions: hi + lo weights (the default, as
    // precise as the other bodies) and, on request, bf16 weights.
    const int fn = which == 6 && !(c.flags & SGL_KV_ATTN_FAST_WEIGHTS) ? 9 : which;
    if (ctx->attention_occupancy_lds[fn] != lds) {
        int per_cu = 0;
        SGLKV_CHECK_HIP(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ctx->attention[fn],
                                                                           (int)threads, lds));
        ctx->attention_occupancy[fn] = per_cu > 0 ? (uint32_t)per_cu : 1;
        ctx->attention_occupancy_lds[fn] = lds;
    }
    const uint64_t target =
        (uint64_t)ctx->attention_occupancy[fn] * (uint64_t)(ctx->cu_count > 0 ? ctx->cu_count : 256);
    // A launch of whole tiles that fits the chip in one round starts one
    // workgroup on each CU and then a second: in that order the first CUs
    // would get two long tiles, so the second ones come from the other end (a
    // prompt of 1,500 tokens, dims 128, 55 -> 51 us, of 2,048 77 -> 74).
    if (tile && p.tile_backward && base <= target && ctx->cu_count > 0 && base > (uint64_t)ctx->cu_count &&
        shape.splits(target) == 1)
        p.tile_fold = (uint32_t)ctx->cu_count / p.kv_heads;
    uint64_t want = tile ? shape.splits(target) : base >= target ? 1 : target / base;
    if (tile && workspace) {
        // Never more split records than the fixed workspace holds: fewer,
        // longer splits instead (the tile bodies take chunks of any length).
        const uint64_t record = 4ull * (SGLKV_ATTN_OPAD(p.dv) + 2);
        const uint64_t room = workspace_bytes / record / (c.query_count * c.query_head_count);
        if (want > room) want = room ? room : 1;
    }
    uint64_t chunk = ceil_div(max_len, want);
    // The shortest chunk a split takes. Small batches split further when
    // the combine merges many splits per memory round (both combines spread
    // a query's split groups over several waves or thread sets), which puts
    // more CUs to work. Measured:
    //  - staged bodies (GQA dims 128 / 64, 32 heads over 8 KV heads, 4,096
    //    tokens): 1 query 23.3 -> 15.5 us / 16.7 -> 11.8 us at 64 tokens
    //    against 256, 2 queries 24.6 -> 17.8 / 17.5 -> 12.2, 4 queries 26.4
    //    -> 23.3 / 18.8 -> 15.9; from 16 queries on the split count is set
    //    by the occupancy target, not by this minimum. The dims-128 body
    //    with K in registers (eight waves per CU) takes 128: at 64, 4
    //    queries took 22.4 us against 20.6;
    //  - latent body (MLA over 8,192 tokens): 64 tokens for one workgroup
    //    before splitting, 128 for two or three (1 query 40.0 -> 33.2 us,
    //    2 queries 41.0 -> 35.2 us), 256 from four on (best there);
    //  - the other bodies keep 256 (not measured otherwise).
    const uint64_t min_chunk = tile                        ? 0
                               : which == 11               ? 128
                               : which >= 7                ? 64
                               : which == 6 && base < 4    ? (base <= 1 ? 64 : 128)
                                                           : 256;
    const uint64_t block = tile ? SGLKV_ATTN_TILE_BLOCK(p.dk) : SGLKV_ATTN_TOKENS;  // splits are whole blocks
    chunk = ceil_div(chunk < min_chunk ? min_chunk : chunk, block) * block;
    uint64_t splits = ceil_div(max_len, chunk);
    const uint64_t table = tile ? 0 : wide ? SGLKV_ATTN_WIDE_SLOTS : which >= 7 ? SGLKV_ATTN_STAGED_SLOTS : 0;
    if (table && chunk > table) {  // the slot table of the wide, latent and staged bodies
        chunk = table;
        splits = ceil_div(max_len, chunk);
    }
    // Ragged batches (the average request below two thirds of the longest):
    // the split above is sized for equal lengths, so most queries leave their
    // last splits empty and the chip part idle. With enough work (128 tokens a
    // resident slot, 96 of the shorter dims-64 ones: 24 queries of 62..999 at
    // dims 128, 100 a slot, took 21.1 us so and 20.5 without) the launch numbers the splits that have tokens first (compact).
    // Its chunk is the shortest whose live workgroups, at most total / chunk +
    // queries of each query's, fit the resident slots in one round (seventeen
    // twentieths of the staged bodies'): at least 64 tokens (128 for long
    // sequences, whose merge grows) and at most the equal-length chunk for
    // the latent body, between 192 and 512 for the staged ones, whose larger
    // batches take several rounds anyway (past 32,768 tokens up to the
    // equal-length chunk: 64 splits of the longest are enough, and more only
    // add workgroups without tokens: one of 131,072 tokens among 63 of 1,000
    // 248 us at 512 a split, 181 so; dims 64, one of 65,536, 81 and 67).
    // Measured on MI355X, per layer, before -> after:
    //  - latent, 32 queries of 1,000..8,192 tokens (1,024 -> 672 a split) 125
    //    -> 102 us, 23 of 955..7,643 93 -> 78, 7 of 100..900 (256 -> 64) 43 ->
    //    30, 30 of 80..300 46 -> 33;
    //  - dims 128, 64 queries of 100..4,096 (1,024 -> 512) 132 -> 115, 40 of
    //    300..4,096 111 -> 83, 8 of 500..4,000 29 -> 26; head-major 140 -> 116;
    //    one of 131,072 among 63 of 1,000 1,683 -> 181, of 32,768 453 -> 96;
    //  - dims 64, 64 of 100..4,096 73 -> 63; dims 256, 32 of 500..4,000 45 -> 40.
    // The latent body's live splits are always numbered first where they are
    // sized to one round: one workgroup a CU, an uneven share of the XCDs is a
    // second round (15 queries of 454..3,638 tokens 72 us a layer in grid
    // order, 48 so; 9 of 739..5,919 69 and 47).
    // Batches nearer one length keep the split above (33 queries of 500..1,300:
    // 33 us either way, 34 with this one; 128 of 2,000..3,000: 239, 250).
    const uint64_t mean = ceil_div(c.sequence_slot_count, c.request_count);
    uint64_t total;  // tokens times the workgroups that share them
    if (splits > 1 && (which == 6 || which == 7 || which == 8 || which == 10 || which == 11) &&
        c.query_count <= SGLKV_ATTN_COMPACT_QUERIES && mean < max_len - max_len / 3 && !mul_ovf(mean, base, &total)) {
        const bool worth = total / target >= (which == 8 ? 96 : 128);
        const uint64_t room = which == 6 ? target : target / 20 * 17;
        uint64_t balanced = room > base ? ceil_div(total, room - base) : chunk;
        const uint64_t least = which == 6 ? (max_len > 4096 ? 128 : 64) : (chunk < 192 ? chunk : 192);
        const uint64_t most = which == 6 || max_len > 32768 ? chunk : 512;
        balanced = balanced < least ? least : (balanced > most ? most : balanced);
        balanced = ceil_div(balanced, block) * block;
        // (Never more records than the fixed workspace holds.)
        uint64_t bytes;
        const bool fits = !workspace ||
                          (!mul_ovf(c.query_count * c.query_head_count, ceil_div(max_len, balanced), &bytes) &&
                           !mul_ovf(bytes, which == 6 ? 2ull * SGLKV_ATTN_HPAD(p.dv) + 16 : 4ull * (SGLKV_ATTN_OPAD(p.dv) + 2),
                                    &bytes) &&
                           bytes <= workspace_bytes);
        if (balanced < chunk && fits && (worth || which == 6)) {
            chunk = balanced;
            splits = ceil_div(max_len, chunk);
        }
        if ((worth || (which == 6 && chunk == balanced)) && max_len <= (1u << 30) && base * splits <= UINT32_MAX)
            p.compact = lay.head_layout == SGL_KV_HND || base == c.query_count ? SGLKV_ATTN_COMPACT_HEADS_FIRST
                                                                               : SGLKV_ATTN_COMPACT_QUERY_FIRST;
    }
    if (splits > 65535) {  // grid y limit
        p.compact = 0;
        chunk = ceil_div(ceil_div(max_len, 65535), block) * block;
        splits = ceil_div(max_len, chunk);
    }
    p.chunk_tokens = chunk;
    p.splits = (uint32_t)splits;

    // The latent body writes scaled fp16 records (SGLKV_ATTN_HPAD), the
    // others fp32 ones (SGLKV_ATTN_OPAD).
    const bool half_records = which == 6;
    // The fp16 records and their combine are laid out for the latent body's
    // 512-wide values (SGLKV_ATTN_HPAD); nothing else selects that body.
    if (half_records && p.dv != 512)
        return fail(SGL_KV_INVALID_ARGUMENT, "value_head_dim", p.dv, 512, 0,
                    "the latent body's fp16 split records need 512-wide values, not %u", (unsigned)p.dv);
    if (splits > 1) {
        uint64_t bytes;
        const uint64_t per_record = half_records ? 2ull * SGLKV_ATTN_HPAD(p.dv) + 16 : 4ull * (SGLKV_ATTN_OPAD(p.dv) + 2);
        if (mul_ovf(c.query_count * c.query_head_count, splits, &bytes) || mul_ovf(bytes, per_record, &bytes))
            return attn_overflow();
        if (workspace) {
            if (bytes > workspace_bytes)
                return fail(SGL_KV_DIMENSION_TOO_LARGE, "workspace", bytes, workspace_bytes, 0,
                            "paged attention needs %llu bytes of split records, more than the "
                            "%llu-byte workspace",
                            (unsigned long long)bytes, (unsigned long long)workspace_bytes);
        } else if (bytes > ctx->attention_partial_bytes) {
            if (ctx->attention_partial) {
                SGLKV_CHECK_HIP(hipDeviceSynchronize());
                SGLKV_CHECK_HIP(hipFree(ctx->attention_partial));
                ctx->attention_partial = nullptr;
                ctx->attention_partial_bytes = 0;
            }
            SGLKV_CHECK_HIP(hipMalloc(&ctx->attention_partial, bytes));
            ctx->attention_partial_bytes = bytes;
        }
        p.partial = static_cast<float *>(workspace ? workspace : ctx->attention_partial);
    }
    // The combine pass: the workgroup's sets of threads, SGLKV_ATTN_COMBINE_PER
    // to a (query, head); the fp16 one in blocks of 64 per 8 groups of 8 heads
    // (its XCD map), padded.
    uint64_t combine_grid = 0;
    if (splits > 1) {
        uint64_t heads;
        if (mul_ovf(c.query_count, c.query_head_count, &heads)) return attn_overflow();
        combine_grid = half_records ? 64 * ceil_div(c.query_count * ceil_div(c.query_head_count, 8), 8)
                                    : ceil_div(heads, SGLKV_ATTN_COMBINE_SETS(p.dv) / SGLKV_ATTN_COMBINE_PER(p.dv, p.splits));
        const uint64_t limit = UINT32_MAX / (half_records ? 256 : 128);  // work-items in 32 bits
        if (heads > limit / 2 || combine_grid > limit)
            return too_large_dim("combine workgroups", heads, limit / 2);
    }
    void *args[] = {&p};
    SGLKV_CHECK_HIP(hipModuleLaunchKernel(ctx->attention[fn], (unsigned)base, (unsigned)splits, 1, threads,
                                          1, 1, lds, s, args, nullptr));
    // The fp16 combine: one wave per group of eight splits, up to four.
    const unsigned combine_threads = half_records ? 64 * (unsigned)(splits > 24 ? 4 : ceil_div(splits, 8)) : SGLKV_ATTN_COMBINE_THREADS;
    if (splits > 1)
        SGLKV_CHECK_HIP(hipModuleLaunchKernel(half_records ? ctx->attention_combine_h : ctx->attention_combine,
                                              (unsigned)combine_grid, 1, 1, combine_threads, 1, 1, 0, s, args,
                                              nullptr));
    return SGL_KV_OK;
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
