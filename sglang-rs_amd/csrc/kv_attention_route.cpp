// kv_attention_route.cpp -- the choice of the attention kernel and of its
// splits (kv_attention_route.h).
#include <string.h>

#include "kv_attention_route.h"

using namespace sglkv;

namespace {

uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

}  // namespace

int32_t sglkv::attention_overflow() {
    return fail(SGL_KV_SHAPE_OVERFLOW, nullptr, 0, 0, 0, "CUDA paged attention shape overflowed");
}

namespace {

uint64_t whole_blocks(uint64_t tokens, uint64_t block) { return ceil_div(tokens, block) * block; }

// Rows of K and V that 16-byte accesses read.
bool rows16(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p) {
    const sgl_kv_attention_layout &lay = c.layout;
    const uint64_t poolp = reinterpret_cast<uint64_t>(p.pool);
    return (p.dk % 8 == 0) && (p.dv % 8 == 0) && ((poolp + lay.key_in_page_offset) % 16 == 0) &&
           ((poolp + lay.value_in_page_offset) % 16 == 0) &&
           ((lay.page_stride_bytes | p.key_head_stride | p.key_token_stride | p.value_head_stride |
             p.value_token_stride) % 16 == 0);
}

// 16-byte rows, power-of-two pages and strides that fit 32 bits admit the
// pipelined, wide, staged and tile bodies (32-bit slots, shift-and-mask pages).
bool fast_rows(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p) {
    return rows16(c, p) && p.page_shift < 32 && c.slot_count < (1ull << 32) &&
           c.layout.page_stride_bytes <= UINT32_MAX && p.key_token_stride <= UINT32_MAX &&
           p.value_token_stride <= UINT32_MAX;
}

struct Body {
    int which;
    unsigned threads, lds;
    // The latent body has two functions: hi + lo weights (the default, as
    // precise as the other bodies) and, on request, bf16 weights.
    int function(const sgl_kv_attention_plan_config &c) const {
        return which == kAttnLatent && !(c.flags & SGL_KV_ATTN_FAST_WEIGHTS) ? kAttnLatentExact : which;
    }
};

// (A plan edited after it was made may have no request: its queries are
// refused one by one on the device.)
uint64_t requests(const sgl_kv_attention_plan_config &c) { return c.request_count ? c.request_count : 1; }

// The body that takes each query by itself.
Body query_body(const AttentionDevice &device, const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p,
                uint64_t max_len) {
    const sgl_kv_attention_layout &lay = c.layout;
    const uint64_t qp = reinterpret_cast<uint64_t>(p.queries);
    const bool vec = rows16(c, p), fast = fast_rows(c, p);
    const bool pipe = fast && p.dk_pad <= 128 && p.dv <= SGLKV_ATTN_DV;
    int which = !vec ? 1 : !pipe ? 0 : (p.dk == 128 && p.dv == 128) ? 2 : 3;
    // Many query heads per KV head (more than one 16-head group) or wide
    // values: the wide bodies share each K/V block among 4 head groups
    // instead of every group and value block reading it again. They hold
    // the queries in registers as 16-byte vectors.
    unsigned threads = 64;
    unsigned lds = (unsigned)((SGLKV_ATTN_HEADS * (p.dk_pad + 8) + SGLKV_ATTN_DV * SGLKV_ATTN_VT_STRIDE) *
                              sizeof(uint16_t));
    // (Their chunks fit the slot table, so the grid's 65535 splits bound
    // the length they take.)
    if (fast && qp % 16 == 0 && (p.head_groups > 1 || p.dv > SGLKV_ATTN_DV) &&
        max_len <= 65535ull * SGLKV_ATTN_WIDE_SLOTS) {
        const unsigned narrow = SGLKV_ATTN_WIDE_LDS_BYTES(4u, 8u), wide = SGLKV_ATTN_WIDE_LDS_BYTES(18u, 32u);
        if (p.dk_pad <= 128 && p.dv <= 128 && narrow <= device.max_lds) {
            which = 5;
            lds = narrow;
            threads = 64 * SGLKV_ATTN_WIDE_WAVES;
        } else if (p.dk > 512 && p.dk <= 576 && p.dv == 512 &&
                   SGLKV_ATTN_LATENT_LDS_BYTES <= device.max_lds) {
            // MLA's latent rows (K 576 = 512 + 64 rope dims, V 512): 32 heads
            // per wave, rows loaded straight into LDS.
            which = 6;
            lds = SGLKV_ATTN_LATENT_LDS_BYTES;
            threads = 64 * SGLKV_ATTN_LATENT_WAVES;
        } else if (p.dk_pad <= 576 && p.dv <= 512 && wide <= device.max_lds) {
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
        SGLKV_ATTN_STAGED_LDS_BYTES(p.dk) <= device.max_lds) {
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
    }
    return {which, threads, lds};
}

// A launch's workgroups of one split, how many stay resident at once, and the
// equal splits of its longest sequence.
struct Split {
    uint64_t base, target, chunk, splits;
};

// Splits each query's sequence so that a per-query body's launch fills every
// CU with as many workgroups as stay resident at once (the kernel's occupancy
// at this LDS size), in one round.
int32_t split_queries(const AttentionDevice &device, const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p,
                      const Body &body, uint64_t max_len, Split *s) {
    const int which = body.which;
    const bool wide = which >= kAttnWide576 && which <= kAttnLatent;  // the wide and latent bodies (7, 8, 10, 11: staged)
    const uint64_t hblocks = which == 6 ? ceil_div(p.group, SGLKV_ATTN_LATENT_HEADS)
                                        : (p.head_groups + SGLKV_ATTN_WIDE_GROUPS - 1) / SGLKV_ATTN_WIDE_GROUPS;
    uint64_t base = c.query_count;
    if (mul_ovf(base, p.kv_heads, &base) || (wide && mul_ovf(base, hblocks, &base)) ||
        (!wide && (mul_ovf(base, p.head_groups, &base) || mul_ovf(base, p.dv_blocks, &base))) ||
        base > UINT32_MAX / body.threads)  // a dispatch counts its work-items in 32 bits
        return too_large_dim("workgroups", base, UINT32_MAX / body.threads);
    s->base = base;
    s->target = device.resident(device.context, body.function(c), body.threads, body.lds) * device.cus;
    if (!s->target) return SGL_KV_MODULE;
    uint64_t chunk = ceil_div(max_len, base >= s->target ? 1 : s->target / base);
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
    const uint64_t min_chunk = which == 11               ? 128
                               : which >= 7              ? 64
                               : which == 6 && base < 4  ? (base <= 1 ? 64 : 128)
                                                         : 256;
    chunk = whole_blocks(chunk < min_chunk ? min_chunk : chunk, SGLKV_ATTN_TOKENS);
    const uint64_t table = wide ? SGLKV_ATTN_WIDE_SLOTS : which >= 7 ? SGLKV_ATTN_STAGED_SLOTS : 0;
    if (table && chunk > table) chunk = table;  // the slot table of the wide, latent and staged bodies
    s->chunk = chunk;
    s->splits = ceil_div(max_len, chunk);
    return SGL_KV_OK;
}

// Split records of a launch; false where their bytes pass 64 bits.
bool record_bytes(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p, bool half_records, uint64_t splits,
                  uint64_t *bytes) {
    const uint64_t record = half_records ? 2ull * SGLKV_ATTN_HPAD(p.dv) + 16 : 4ull * (SGLKV_ATTN_OPAD(p.dv) + 2);
    return !mul_ovf(c.query_count, c.query_head_count, bytes) && !mul_ovf(*bytes, splits, bytes) &&
           !mul_ovf(*bytes, record, bytes);
}

// Ragged batches (the average request below two thirds of the longest):
// the split above is sized for equal lengths, so most queries leave their
// last splits empty and the chip part idle. With enough work (128 tokens a
// resident slot, 96 of the shorter dims-64 ones: 24 queries of 62..999 at
// dims 128, 100 a slot, took 21.1 us so and 20.5 without) the launch numbers
// the splits that have tokens first (compact).
// Its chunk is the shortest whose live workgroups, at most total / chunk +
// queries of each query's, fit the resident slots in one round (seventeen
// twentieths of the staged bodies'): at least 64 tokens (128 for long
// sequences, whose merge grows) and at most the equal-length chunk for
// the latent body, between 192 and 512 for the staged ones, whose larger
// batches take several rounds anyway (where the equal chunk takes one, that;
// past 32,768 tokens up to the equal-length chunk: 64 splits of the longest
// are enough, and more only add workgroups without tokens: one of 131,072
// tokens among 63 of 1,000 248 us at 512 a split, 181 so; dims 64, one of
// 65,536, 81 and 67).
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
// Their records, up to 9 times those of equal splits (one MLA query of 65,536
// tokens among 31 of 1,000: 626 MB against 68), stay within `shorter` bytes,
// 128 MiB; the chunk is then the shortest that does. That is slower where one
// MLA sequence is far the longest: 64 queries, one of 30,000 among 1,000s, 195
// us a layer so, 88 with records of any size (357 with equal splits); 16, one
// of 20,000, 54 and 44 (126).
// Returns whether the splits were made shorter.
bool split_ragged(const sgl_kv_attention_plan_config &c, const Body &body, uint64_t max_len, uint64_t shorter,
                  sglkv_attn_params *params, Split *s) {
    sglkv_attn_params &p = *params;
    const int which = body.which;
    if (s->splits < 2 || (which != kAttnLatent && which < kAttnStaged128) ||
        c.query_count > SGLKV_ATTN_COMPACT_QUERIES)
        return false;
    const uint64_t mean = ceil_div(c.sequence_slot_count, requests(c)), base = s->base, target = s->target;
    uint64_t total;  // tokens times the workgroups that share them
    if (mean >= max_len - max_len / 3 || mul_ovf(mean, base, &total)) return false;
    const bool worth = total / target >= (which == kAttnStaged64 ? 96 : 128);
    const uint64_t room = which == kAttnLatent ? target : target / 20 * 17;
    uint64_t balanced = room > base ? ceil_div(total, room - base) : s->chunk;
    const uint64_t least = which == kAttnLatent ? (max_len > 4096 ? 128 : 64) : (s->chunk < 192 ? s->chunk : 192);
    // Workgroups with tokens at a chunk of k, each sequence's last one half full.
    auto live = [&](uint64_t k) { return mean < k / 2 ? base : base * (mean + k / 2) / k; };
    // Shorter than 512 helps no more where that takes a second round and the
    // equal chunk does not: 57 queries of 650 or 6,566 tokens (dims 256) 84.7 us a
    // layer at 512, 74.9 at 1,024; 42 of up to 14,923 90.4 and 75.7; 84 of up to
    // 5,813 (dims 128, head-major) 155.7 and 147.2; 54 of up to 3,838 spread evenly
    // (dims 256) 78.1 and 69.7. (Just past one round batches of two lengths would
    // still gain, 238 of 126 or 1,262 tokens 98 and 113, of 118 without numbers.)
    const bool capped = which != kAttnLatent && max_len <= 32768;
    const bool second = capped && live(512) > target && live(s->chunk) <= target;
    const uint64_t most = capped && !second ? 512 : s->chunk;
    balanced = second ? most : balanced < least ? least : (balanced > most ? most : balanced);
    uint64_t bytes;
    if (!record_bytes(c, p, which == kAttnLatent, 1, &bytes)) return false;
    const uint64_t fit = ceil_div(max_len, shorter / bytes ? shorter / bytes : 1);
    balanced = whole_blocks(balanced < fit ? fit : balanced, SGLKV_ATTN_TOKENS);
    const bool shortened = balanced < s->chunk && (worth || which == kAttnLatent);
    if (shortened) {
        s->chunk = balanced;
        s->splits = ceil_div(max_len, s->chunk);
    }
    if ((worth || (which == kAttnLatent && s->chunk == balanced)) && max_len <= (1u << 30) &&
        base * s->splits <= UINT32_MAX)
        p.compact = c.layout.head_layout == SGL_KV_HND || base == c.query_count ? SGLKV_ATTN_COMPACT_HEADS_FIRST
                                                                                : SGLKV_ATTN_COMPACT_QUERY_FIRST;
    return shortened;
}

// The tiles of a launch with several queries per request.
struct TileShape {
    uint64_t queries, per_request, slots, step_slots, live, max_len;

    TileShape(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p, uint64_t longest)
        : queries(p.group && p.group <= SGLKV_ATTN_TILE_ROWS(p.dk) ? SGLKV_ATTN_TILE_ROWS(p.dk) / p.group : 1),
          // (the queries shared evenly among the requests)
          per_request(ceil_div(ceil_div(c.query_count, requests(c)), queries)), max_len(longest) {
        // Queries that come request by request make at most this many tiles. Past
        // one step of the search each step has its workgroups, for its share
        // of the requests.
        step_slots = 0;
        const uint64_t steps = (c.query_count - 1) / SGLKV_ATTN_TILE_STEP + 1;
        auto most = [&](uint64_t count, uint64_t runs) {
            const uint64_t n = count / queries + runs;
            return n < count ? n : count;
        };
        if (requests(c) == 1 || steps == 1) {
            slots = most(c.query_count, requests(c));
        } else {
            const uint64_t runs = ceil_div(requests(c), steps) + 1;
            step_slots = most(SGLKV_ATTN_TILE_STEP, runs);
            slots = (steps - 1) * step_slots + most(c.query_count - (steps - 1) * SGLKV_ATTN_TILE_STEP, runs);
        }
        // Workgroups with tokens: as many as even shares make if the requests
        // have as many queries each, nearly all where one has most of them (a
        // prompt among decodes). Half way between, since the host cannot tell:
        // sized for even shares, the mixed batches of 20 took a second round
        // and 10 % longer (7 queries a KV head, dims 64: 512 queries of a
        // prompt and 63 decodes over 2,000 tokens 72.7 us, so 55.4), while
        // the 50 even ones are as fast (0.95 to 1.11 of it).
        live = per_request * requests(c) * p.kv_heads;
        if (requests(c) > 1) live = (live + slots * p.kv_heads) / 2;
    }

    // Splits that fill `target` resident workgroups: of 256 tokens or more,
    // or of 128 where a request is one tile (few queries, so the records that
    // the splits leave are few). They are counted for the longest sequence
    // also where most are shorter: with as many more as the average leaves
    // room for, 24 requests of 200..3,000 tokens (dims 256) took 49 us, not 38.
    uint64_t splits(uint64_t target) const {
        const uint64_t want = live >= target ? 1 : target / live, least = per_request > 1 ? 256 : 128;
        return want < max_len / least ? want : (max_len >= 2 * least ? max_len / least : 1);
    }
};

// Whether the tile bodies can take the call: several queries per request on
// average (prefill, chunked prefill, drafted tokens). They read a K/V row once
// per tile of queries instead of once per query, take the staged bodies' shapes
// and any group of up to 64 query heads, 32 at dims 256 (a tile then holds
// at least two queries), count tokens in 32 bits and write 8-byte pieces.
bool tiles_take(const AttentionDevice &device, const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p,
                uint64_t max_len) {
    return fast_rows(c, p) && p.dk == p.dv && (p.dk == 64 || p.dk == 128 || p.dk == 256) &&
           reinterpret_cast<uint64_t>(p.queries) % 16 == 0 && reinterpret_cast<uint64_t>(p.output) % 8 == 0 &&
           p.group <= SGLKV_ATTN_TILE_ROWS(p.dk) / 2 && p.key_token_stride == p.value_token_stride &&
           p.key_token_stride < (1u << 24) && c.layout.page_size <= (1u << 24) && c.request_count > 0 &&
           c.query_count / 2 >= c.request_count && c.query_count <= SGLKV_ATTN_TILE_QUERIES_MAX &&
           c.query_count <= UINT32_MAX / 512 / p.kv_heads && max_len <= (1u << 30) &&
           SGLKV_ATTN_TILE_LDS_BYTES(p.dk) <= device.max_lds;
}

// Whether the tiles are estimated to take less time than `body`, whose work
// items are one query's, by a tenth. Both estimates are straight lines through
// 420 random calls on MI355X (1 to 48 requests: prompts, chunks of prompts
// over a cached prefix, drafts; 14 shapes of heads), each run both ways; their
// coefficients are us.
//  - A per-query body: its start; a merge, if split; each 32-token block of a
//    workgroup's chain; the blocks that a resident workgroup has beyond its
//    first chain; each round of work items past the first. Never less than
//    the rows that all queries read, at 4.9 TB/s (64 x 4 queries over 1,100
//    tokens, dims 64: 114 us, tiles 52).
//  - Tiles: their start; with several requests the search, by the runs that a
//    stretch of 64 queries holds; a merge, if split; each block of a chain; the
//    blocks beyond it; start and search again for each round past the first.
//    Never less than each row read once.
// Queries attend the average request's tokens, less half its queries. Over
// these calls and 420 others the way chosen takes 0.72 of the per-query
// bodies' time (geometric mean) and 2 % more than the faster of both; 13 of
// the 840 take over a tenth longer than one query at a time, at most 28 %. A
// batch of one prompt and many decodes, which looks like one of drafts, is
// beyond what the counts tell.
bool tiles_pay(const sgl_kv_attention_plan_config &c, const sglkv_attn_params &p, const TileShape &shape,
               const Body &body, const Split &single, uint64_t tile_target) {
    const struct {
        double start, merge, block, beyond, round;
    } staged[] = {{8.1, 1.7, 1.05, 1.3, 4.6}, {7.2, 1.4, 1.65, 1.9, 6.5}, {8.7, 3.1, 2.0, 2.8, 9.3}},
      wide[] = {{7.4, 2.4, 1.35, 1.8, 7.6}, {7.1, 3.3, 1.3, 1.1, 15.2}, {8.8, 2.3, 2.6, 3.8, 8.7}};
    const struct {
        double start, search, run, merge, block, beyond;
    } tile[] = {{4.0, 3.5, 0.33, 4.0, 1.6, 2.5}, {6.0, 2.8, 0.28, 4.0, 2.05, 3.0}, {6.5, 3.3, 0.34, 4.0, 1.5, 3.0}};
    const int d = p.dk == 64 ? 0 : p.dk == 128 ? 1 : 2;
    const double per = (double)c.query_count / c.request_count, mean = (double)c.sequence_slot_count / c.request_count,
                 attended = mean - (mean < per ? mean : per) / 2;
    auto past = [](double x, double y) { return x > y ? x - y : 0.0; };

    const auto &q = body.which < kAttnStaged128 ? wide[d] : staged[d];
    const double rounds = (double)single.base / single.target,
                 chain = (double)(single.chunk < shape.max_len ? single.chunk : shape.max_len) / SGLKV_ATTN_TOKENS;
    const double row = 2.0 * (p.dk + p.dv) / 4.9e6;  // us to read a token's K and V of one head
    double alone = q.start + (single.splits > 1 ? q.merge : 0) + q.block * chain +
                   q.beyond * past(rounds * attended / SGLKV_ATTN_TOKENS, chain) + q.round * past(rounds, 1);
    alone = alone > single.base * attended * row ? alone : single.base * attended * row;

    const auto &t = tile[d];
    const double size = SGLKV_ATTN_TILE_BLOCK(p.dk), requests = (double)c.request_count;
    double runs = c.query_count > 64 ? 64 / per : requests;  // of a stretch
    runs = runs < 1 ? 1 : runs > requests ? requests : runs;
    const uint64_t splits = shape.splits(tile_target);
    const double blocks = (double)ceil_div(ceil_div(shape.max_len, splits), (uint64_t)size);
    const double start = t.start + (c.request_count > 1 ? t.search + t.run * runs : 0),
                 tile_rounds = (double)shape.live / tile_target;
    double tiled = start * (1 + past(tile_rounds, 1)) + (splits > 1 ? t.merge : 0) + t.block * blocks +
                   t.beyond * past(tile_rounds * attended / size, blocks);
    const double once = c.sequence_slot_count * (double)p.kv_heads * row;
    tiled = tiled > once ? tiled : once;
    return 1.1 * tiled < alone;
}

// Splits for a launch of tiles.
int32_t split_tiles(const AttentionDevice &device, const TileShape &shape, const Body &body, uint64_t max_len,
                    sglkv_attn_params *params, Split *s) {
    sglkv_attn_params &p = *params;
    p.tile_queries = (uint32_t)shape.queries;
    p.tile_recip = UINT32_MAX / p.tile_queries + 1;
    p.tile_slots = (uint32_t)shape.slots;
    p.tile_step_slots = (uint32_t)shape.step_slots;
    // Later tiles of a causal prompt attend more tokens: they start
    // first, except where each request is one tile. (Several prompts'
    // last tiles in turn were no faster: 4 of 2,048 tokens 266 us against
    // 259, 4 of 300..2,048 189 against 143.)
    p.tile_backward = shape.per_request > 1;
    const uint64_t base = s->base = (uint64_t)p.tile_slots * p.kv_heads;
    if (base > UINT32_MAX / body.threads)  // a dispatch counts its work-items in 32 bits
        return too_large_dim("workgroups", base, UINT32_MAX / body.threads);
    const uint64_t target = s->target =
        device.resident(device.context, body.which, body.threads, body.lds) * device.cus;
    if (!target) return SGL_KV_MODULE;
    // A launch of whole tiles that fits the chip in one round starts one
    // workgroup on each CU and then a second: in that order the first CUs
    // would get two long tiles, so the second ones come from the other end (a
    // prompt of 1,500 tokens, dims 128, 55 -> 51 us, of 2,048 77 -> 74).
    if (p.tile_backward && base <= target && base > device.cus && shape.splits(target) == 1)
        p.tile_fold = (uint32_t)device.cus / p.kv_heads;
    s->chunk = whole_blocks(ceil_div(max_len, shape.splits(target)), SGLKV_ATTN_TILE_BLOCK(p.dk));
    s->splits = ceil_div(max_len, s->chunk);
    return SGL_KV_OK;
}

}  // namespace

int32_t sglkv::attention_route(const AttentionDevice &device, const sgl_kv_attention_plan_config &c, uint64_t max_len,
                               const AttentionRecords &records, sglkv_attn_params *params, AttentionRoute *route) {
    sglkv_attn_params &p = *params;
    if (!max_len || max_len > c.sequence_slot_count) max_len = c.sequence_slot_count;
    p.page_stride32 = (uint32_t)c.layout.page_stride_bytes;
    p.key_token_stride32 = (uint32_t)p.key_token_stride;
    p.value_token_stride32 = (uint32_t)p.value_token_stride;
    Body body = query_body(device, c, p, max_len);
    if (body.which >= kAttnStaged128) p.dv_blocks = 1;
    Split s = {0, 0, 0, 0};
    uint64_t block = SGLKV_ATTN_TOKENS;
    route->apart = route->shortened = false;
    const Body tile = {p.dk == 128 ? kAttnTile128 : p.dk == 64 ? kAttnTile64 : kAttnTile256, 256,
                       SGLKV_ATTN_TILE_LDS_BYTES(p.dk)};
    const TileShape shape(c, p, max_len);
    bool tiles = tiles_take(device, c, p, max_len);
    int32_t rc = split_queries(device, c, p, body, max_len, &s);
    if (tiles && rc == SGL_KV_OK) {
        const uint64_t target = device.resident(device.context, tile.which, tile.threads, tile.lds) * device.cus;
        if (!target) return SGL_KV_MODULE;
        tiles = tiles_pay(c, p, shape, body, s, target);
    }
    if (tiles) {
        const bool splits_alone = rc == SGL_KV_OK && s.splits > 1;
        body = tile;
        block = SGLKV_ATTN_TILE_BLOCK(p.dk);
        if ((rc = split_tiles(device, shape, body, max_len, &p, &s))) return rc;
        // The calls of a context that split share one buffer, so a caller
        // issues them on one stream. Where the per-query body would not split,
        // the caller need not: those records go to the tiles' own buffer,
        // whose calls the library orders itself, or the tiles stay whole
        // (where there is no such buffer, and under graph capture).
        if (s.splits > 1 && !records.workspace_bytes && !splits_alone) {
            uint64_t bytes;
            route->apart = records.apart && record_bytes(c, p, false, s.splits, &bytes) &&
                           bytes <= kAttentionTileRecordBytes;
            if (!route->apart) {
                s.chunk = whole_blocks(max_len, block);
                s.splits = 1;
            }
        }
    } else {
        if (rc) return rc;
        route->shortened = split_ragged(c, body, max_len, records.shorter, &p, &s);
    }
    if (s.splits > 65535) {  // grid y limit
        p.compact = 0;
        s.chunk = whole_blocks(ceil_div(max_len, 65535), block);
        s.splits = ceil_div(max_len, s.chunk);
    }
    const uint64_t splits = s.splits;
    p.chunk_tokens = s.chunk;
    p.splits = (uint32_t)splits;

    // The latent body writes scaled fp16 records (SGLKV_ATTN_HPAD), the
    // others fp32 ones (SGLKV_ATTN_OPAD).
    const bool half_records = body.which == kAttnLatent;
    // The fp16 records and their combine are laid out for the latent body's
    // 512-wide values (SGLKV_ATTN_HPAD); nothing else selects that body.
    if (half_records && p.dv != 512)
        return fail(SGL_KV_INVALID_ARGUMENT, "value_head_dim", p.dv, 512, 0,
                    "the latent body's fp16 split records need 512-wide values, not %u", (unsigned)p.dv);
    route->body = body.function(c);
    route->threads = body.threads;
    route->lds = body.lds;
    route->grid = s.base;
    route->half_records = half_records;
    route->record_bytes = 0;
    route->combine_grid = 0;
    route->combine_threads = 0;
    if (splits == 1) return SGL_KV_OK;
    uint64_t heads;
    if (mul_ovf(c.query_count, c.query_head_count, &heads) ||
        !record_bytes(c, p, half_records, splits, &route->record_bytes))
        return attention_overflow();
    // The combine pass: the workgroup's sets of threads, SGLKV_ATTN_COMBINE_PER
    // to a (query, head); the fp16 one in blocks of 64 per 8 groups of 8 heads
    // (its XCD map), padded, one wave per group of eight splits up to four.
    route->combine_grid = half_records ? 64 * ceil_div(c.query_count * ceil_div(c.query_head_count, 8), 8)
                                       : ceil_div(heads, SGLKV_ATTN_COMBINE_SETS(p.dv) / SGLKV_ATTN_COMBINE_PER(p.dv, p.splits));
    route->combine_threads = half_records ? 64 * (unsigned)(splits > 24 ? 4 : ceil_div(splits, 8)) : SGLKV_ATTN_COMBINE_THREADS;
    const uint64_t limit = UINT32_MAX / (half_records ? 256 : 128);  // work-items in 32 bits
    if (heads > limit / 2 || route->combine_grid > limit)
        return too_large_dim("combine workgroups", heads, limit / 2);
    return SGL_KV_OK;
}
