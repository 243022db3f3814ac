// The choice of attention kernel and splits (kv_attention_route.cpp) over
// random calls, for a device of 256 CUs: what every launch must satisfy for
// its kernel to be in bounds, and the calls whose route is pinned.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "kv_attention_route.h"

using namespace sglkv;

namespace {

// Workgroups of a body that a CU holds: as many as its LDS admits, at most
// what its registers do.
uint32_t resident(void *, int body, unsigned threads, unsigned lds) {
    uint32_t most = body == kAttnTile64 ? 3 : threads == 64 ? 8 : 2;
    if (body == kAttnLatent || body == kAttnLatentExact) most = 1;
    const uint32_t fit = lds ? 160 * 1024 / lds : most;
    return fit < most ? fit : most;
}

const AttentionDevice kDevice = {256, 160 * 1024, nullptr, resident};

struct Call {
    uint64_t queries, requests, slots, max_len;
    uint32_t qheads, heads, dk, dv;
    bool hnd;
    uint64_t page = 64;
};

struct Routed {
    int32_t rc;
    sglkv_attn_params p;
    AttentionRoute r;
};

Routed route(const Call &x, const AttentionRecords &records = {0, kAttentionShorterBytes, true}) {
    Routed o;
    memset(&o, 0, sizeof o);
    sgl_kv_attention_plan_config c;
    memset(&c, 0, sizeof c);
    c.query_count = x.queries;
    c.request_count = x.requests;
    c.sequence_slot_count = x.slots;
    c.slot_count = x.slots + 64;
    c.query_head_count = x.qheads;
    c.kv_head_count = x.heads;
    c.query_key_head_dim = x.dk;
    c.value_head_dim = x.dv;
    c.scale = 0.1f;
    c.layout.page_size = x.page;
    c.layout.key_row_bytes = 2ull * x.heads * x.dk;
    c.layout.value_row_bytes = 2ull * x.heads * x.dv;
    c.layout.value_in_page_offset = x.page * c.layout.key_row_bytes;
    c.layout.page_stride_bytes = x.page * (c.layout.key_row_bytes + c.layout.value_row_bytes);
    c.layout.head_layout = x.hnd ? SGL_KV_HND : SGL_KV_NHD;
    sglkv_attn_params &p = o.p;
    p.queries = reinterpret_cast<const uint16_t *>(0x10000);
    p.output = reinterpret_cast<uint16_t *>(0x20000);
    p.pool = reinterpret_cast<const uint8_t *>(0x30000);
    p.query_count = c.query_count;
    p.request_count = c.request_count;
    p.key_head_stride = x.hnd ? x.page * 2 * x.dk : 2 * x.dk;
    p.key_token_stride = x.hnd ? 2 * x.dk : c.layout.key_row_bytes;
    p.value_head_stride = x.hnd ? x.page * 2 * x.dv : 2 * x.dv;
    p.value_token_stride = x.hnd ? 2 * x.dv : c.layout.value_row_bytes;
    p.query_heads = x.qheads;
    p.kv_heads = x.heads;
    p.group = x.qheads / x.heads;
    p.head_groups = (p.group + SGLKV_ATTN_HEADS - 1) / SGLKV_ATTN_HEADS;
    p.dk = x.dk;
    p.dk_pad = (x.dk + 31) / 32 * 32;
    p.dv = x.dv;
    p.dv_blocks = (x.dv + SGLKV_ATTN_DV - 1) / SGLKV_ATTN_DV;
    p.page_shift = 6;
    o.rc = attention_route(kDevice, c, x.max_len, records, &p, &o.r);
    return o;
}

bool is_tile(int body) { return body >= kAttnTile128 && body <= kAttnTile256; }
bool is_staged(int body) {
    return body == kAttnStaged128 || body == kAttnStaged64 || body == kAttnStaged256 || body == kAttnStaged128K;
}
bool is_wide(int body) {
    return body == kAttnWide576 || body == kAttnWide128 || body == kAttnLatent || body == kAttnLatentExact;
}

[[noreturn]] void fail_call(const char *what, const Call &x, const Routed &o) {
    std::fprintf(stderr,
                 "%s: %llu queries of %llu requests, %llu slots, longest %llu, %u heads over %u, dims %u/%u hnd %d: rc %d "
                 "body %d grid %llu splits %u chunk %llu live first %u records %llu\n",
                 what, (unsigned long long)x.queries, (unsigned long long)x.requests, (unsigned long long)x.slots,
                 (unsigned long long)x.max_len, x.qheads, x.heads, x.dk, x.dv, x.hnd, o.rc, o.r.body,
                 (unsigned long long)o.r.grid, o.p.splits, (unsigned long long)o.p.chunk_tokens, o.p.compact,
                 (unsigned long long)o.r.record_bytes);
    std::exit(1);
}

void check(const Call &x, const Routed &o) {
    if (o.rc == SGL_KV_DIMENSION_TOO_LARGE && x.queries * x.qheads > 1u << 22) return;
    if (o.rc) fail_call("refused", x, o);
    const uint64_t max_len = x.max_len && x.max_len < x.slots ? x.max_len : x.slots, chunk = o.p.chunk_tokens,
                   splits = o.p.splits;
    if (!splits || !chunk || chunk * splits < max_len || (splits > 1 && chunk * (splits - 1) >= max_len))
        fail_call("the splits do not cover the longest sequence once", x, o);
    if (splits > 65535 || o.r.grid == 0 || o.r.grid > UINT32_MAX / o.r.threads) fail_call("grid", x, o);
    const uint64_t block = is_tile(o.r.body) ? SGLKV_ATTN_TILE_BLOCK(x.dk) : SGLKV_ATTN_TOKENS;
    if (splits > 1 && chunk % block) fail_call("a split of part of a block", x, o);
    if (is_staged(o.r.body) && chunk > SGLKV_ATTN_STAGED_SLOTS) fail_call("a split longer than the slot table", x, o);
    if (is_wide(o.r.body) && chunk > SGLKV_ATTN_WIDE_SLOTS) fail_call("a split longer than the slot table", x, o);
    if (o.p.compact) {
        if (!is_staged(o.r.body) && o.r.body != kAttnLatent && o.r.body != kAttnLatentExact)
            fail_call("a body that does not number its splits", x, o);
        if (x.queries > SGLKV_ATTN_COMPACT_QUERIES || splits < 2 || chunk * splits >= 1ull << 31 ||
            o.r.grid * splits > UINT32_MAX)
            fail_call("numbered splits past their bounds", x, o);
    }
    if (is_tile(o.r.body)) {
        const uint64_t rows = SGLKV_ATTN_TILE_ROWS(x.dk);
        if (o.p.tile_queries < 2 || o.p.tile_queries * o.p.group > rows || chunk * splits >= 1ull << 31 ||
            o.p.tile_fold >= o.p.tile_slots || o.r.grid != (uint64_t)o.p.tile_slots * x.heads)
            fail_call("tile shape", x, o);
    }
    const uint64_t record = o.r.half_records ? 2 * SGLKV_ATTN_HPAD(x.dv) + 16 : 4 * (SGLKV_ATTN_OPAD(x.dv) + 2);
    if (o.r.record_bytes != (splits > 1 ? x.queries * x.qheads * splits * record : 0)) fail_call("records", x, o);
}

int shortened = 0;

// Records go to the buffer that all splitting calls share only where the
// queries one by one (as many requests, so no tiles) would be split too.
void check_apart(const Call &x, const Routed &o) {
    if (!is_tile(o.r.body)) {
        if (o.r.apart) fail_call("no tiles, but records apart", x, o);
        return;
    }
    Call single = x;
    single.requests = x.queries;
    const Routed alone = route(single);
    const bool splits = alone.rc == SGL_KV_OK && alone.p.splits > 1;
    if (o.r.apart != (o.p.splits > 1 && !splits)) fail_call("records in the wrong buffer", x, o);
    if (o.r.record_bytes > kAttentionTileRecordBytes) fail_call("more records than the tiles' buffer holds", x, o);
    const Routed fixed = route(x, {SGL_KV_NOALLOC_WORKSPACE_BYTES, kAttentionShorterBytes, true});
    check(x, fixed);
    if (fixed.r.record_bytes > kAttentionTileRecordBytes) fail_call("more tile records than a workspace takes", x, fixed);
    // Without that buffer the call is made all the same, in whole tiles.
    const Routed without = route(x, {0, kAttentionShorterBytes, false});
    check(x, without);
    if (without.r.apart || (!splits && without.p.splits != 1)) fail_call("records without a buffer", x, without);
}

// A ragged batch's splits take no more than the bytes they may, nor more than
// the equal splits where these bytes are few, and the same with a workspace.
void check_ragged(const Call &x, const Routed &o) {
    const Routed equal = route(x, {0, 0, true});
    check(x, equal);
    if (equal.r.shortened || o.r.record_bytes < equal.r.record_bytes) fail_call("longer than equal splits", x, o);
    if (o.r.shortened ? o.r.record_bytes > kAttentionShorterBytes : o.r.record_bytes != equal.r.record_bytes)
        fail_call("records past their bound", x, o);
    const Routed fixed = route(x, {SGL_KV_NOALLOC_WORKSPACE_BYTES, kAttentionShorterBytes, true});
    if (fixed.p.chunk_tokens != o.p.chunk_tokens || fixed.p.splits != o.p.splits || fixed.p.compact != o.p.compact ||
        fixed.r.body != o.r.body)
        fail_call("another split with a workspace", x, o);
    if (o.r.shortened) ++shortened;
}

struct Shape {
    uint32_t qheads, heads, dk, dv;
};
const Shape kShapes[] = {{32, 8, 128, 128}, {8, 1, 128, 128}, {14, 2, 64, 64},  {32, 8, 64, 64},   {8, 2, 256, 256},
                         {128, 1, 576, 512}, {64, 1, 128, 128}, {48, 2, 64, 64}, {32, 1, 256, 256}, {16, 4, 112, 112},
                         {4, 4, 64, 64},     {16, 2, 192, 128}, {8, 8, 100, 100}};

void random_calls() {
    std::mt19937_64 rng(11);
    auto log = [&](double low, double high) {
        return (uint64_t)std::exp(std::uniform_real_distribution<double>(std::log(low), std::log(high))(rng));
    };
    for (int i = 0; i < 200000; ++i) {
        const Shape &s = kShapes[rng() % (sizeof kShapes / sizeof *kShapes)];
        Call x = {0, 0, 0, 0, s.qheads, s.heads, s.dk, s.dv, rng() % 3 == 0};
        x.requests = log(1, 3000);
        x.queries = rng() % 2 ? x.requests : x.requests * log(1, 600);
        x.max_len = log(1, 300000);
        const uint64_t mean = rng() % 2 ? x.max_len : log(1, (double)x.max_len + 1);
        x.slots = mean * x.requests;
        if (x.slots < x.max_len) x.slots = x.max_len;
        if (rng() % 8 == 0) x.max_len = 0;
        const Routed o = route(x);
        check(x, o);
        if (o.rc != SGL_KV_OK) continue;
        check_apart(x, o);
        check_ragged(x, o);
    }
}

// A plan is a plain struct: one whose request_count was set to 0 after it was
// made still launches, and its queries are refused on the device.
void no_requests() {
    for (const Shape &s : kShapes)
        for (uint64_t queries : {1, 7, 500}) {
            const Call x = {queries, 0, 1000, 1000, s.qheads, s.heads, s.dk, s.dv, false};
            const Routed o = route(x);
            check(x, o);
            if (is_tile(o.r.body)) fail_call("a tile of no request", x, o);
        }
}

}  // namespace

int main() {
    no_requests();
    random_calls();
    if (shortened < 1000) {
        std::fprintf(stderr, "only %d ragged batches\n", shortened);
        return 1;
    }
    std::puts("attention route ok");
    return 0;
}
