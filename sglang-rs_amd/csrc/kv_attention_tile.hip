// kv_attention_tile.hip -- paged attention for launches with several queries
// per request: prefill (one query per prompt token, as the reference's
// scheduler metadata has it), chunked prefill, verification of drafted tokens.
//
// The per-query bodies of kv_attention.hip give every (query, KV head) a wave
// of its own, so each query of a prompt reads the prompt's K and V again and
// fills only `group` of the 16 columns of its matrix products. Here a
// workgroup of four waves owns a tile: up to tile_queries consecutive queries
// of one request, whose query heads of one KV head are the tile's rows
// (row = query * group + head, at most 128, 32 per wave; at dims 256, whose
// outputs of 32 rows are too many registers for one wave, 64 rows, 32 per pair
// of waves: both compute the scores, each has half the value dims). Every K and
// V row is staged in LDS once per tile.
//  - Tiles. The queries are taken in steps of 2,048, each with its own
//    workgroups (tile_step_slots; the rest of tile_slots for the last step). A
//    run is a maximal stretch of consecutive queries of one request within a
//    step; it is cut into tiles of tile_queries from its start, and a step's
//    tiles are numbered over its runs. Which queries tile t holds is found from
//    query_request_indices by the workgroup itself (attn_tile_find), so queries
//    of different requests never share a tile whatever their order, and no
//    planning launch or device list is needed. Where the queries of a step do
//    not come request by request, its tiles gather those of a request. The host
//    launches enough workgroups for queries that come request by request; those
//    of a step go on by their number, so any other order is covered too. Later
//    tiles of a causal prompt attend more tokens, so the tiles are taken from
//    the last to the first.
//  - q.k: S[token][row] = K (A operand) x Q^T (B operand) with
//    v_mfma_f32_32x32x16_bf16, the queries in registers. Lane l holds row
//    l % 32's scores of tokens 8(i/4) + 4(l/32) + i%4, i < 16, of each
//    32-token tile, so a row's softmax state is one value per lane.
//  - p.v: O^T[dim][row] = V^T (A operand, two transposing LDS reads per
//    32-dim tile and 16-token step) x P^T (B operand). P's lane order is the
//    one S came out in, and O^T keeps a row's outputs in its own two lanes:
//    rescaling and normalising need no lane exchange.
//  - Softmax as in the staged bodies: fp32, lazy rescaling (the reference
//    maximum moves only when passed by more than 8 log2 units), weights as
//    hi + lo bf16 pairs, the normaliser from the unrounded weights. Each row
//    masks by its own query's length, in the blocks that pass the shortest
//    length of the wave's rows; a wave whose rows all end before a block only
//    loads for the others.
//  - Rows go straight into LDS (global_load_lds_dwordx4), two stages: block
//    k+1 loads while block k is computed, one barrier per block. A piece
//    (16 bytes) pc of token t's K row sits at pc ^ kswz(t), of its V row at
//    pc ^ vswz(t), chosen so that the 16 tokens of a q.k read, and the four
//    tokens of a half-wave's transposing read, land in distinct banks.
// What bounds it, by SQ counters, on two waves per SIMD (dims 64: three):
//  - long causal prompts, dims 128: a wave's products (48 per 64-token block, 32
//    of them p.v's, hi and lo) and its softmax follow each other, so neither
//    pipe is full: matrix cores busy 39 % of the SIMD cycles, vector issue 48 %;
//    a quarter of a wave's time at the block barrier, no LDS bank conflicts;
//  - a chunk over a long prefix, dims 64: 26 % and 52 %, a third of the time
//    waiting for rows;
//  - a few queries a request, dims 256: waiting for rows, 56 % of a wave's time
//    (one block in flight, and waves without a row only load).
// Short calls take the chain of loads before the first block: 4.0 to 6.5 us
// (fitted, by dims) and 3 us of search where there are several requests.
// Measured on MI355X, per layer, against the per-query bodies:
//   causal prompts of 300..2,048 tokens (5,206 queries, 32 heads over 8, dims
//   128): 1,755 -> 125 us (532 TFLOP/s of q.k and p.v; 688 where 2,048 queries
//   each attend 6,144..8,192 tokens);
//   384 queries over 6,144 tokens (14 heads over 2, dims 64): 112 -> 33 us;
//   5 queries of each of 24 requests of 200..3,000 tokens (8 heads over 2, dims
//   256): 110 -> 38 us.
// Of these, the search for the tile's queries in steps of 2,048 (not 128
// at a time) took the prompts from 185 to 135 us, and products at raised wave
// priority with the next step's weights scheduled between them 388 -> 350 us on
// the 8,192-token shape.

namespace {

constexpr uint32_t kTileRaw = 1;    // slots per thread that are loaded ahead of the row lengths

template <uint32_t D>
struct attn_tl {
    static constexpr uint32_t ROW = 2 * D;                // bytes of one token's head slice
    static constexpr uint32_t PIECES = D / 8;             // 16-byte pieces per row
    static constexpr uint32_t TPL = 1024 / ROW;           // tokens per load
    static constexpr uint32_t B = SGLKV_ATTN_TILE_BLOCK(D);  // tokens per block
    static constexpr uint32_t LPW = B / TPL / 4;          // K loads (and V loads) of a wave per block
    static constexpr uint32_t V = B * ROW;                // V rows' offset in a stage
    static constexpr uint32_t STAGE = 2 * V;
    static constexpr uint32_t TABLE = SGLKV_ATTN_TILE_SLOTS(D);  // slot table entries (whole blocks)
    static constexpr uint32_t KC = D / 16;                // q.k steps
    static constexpr uint32_t ROWS = SGLKV_ATTN_TILE_ROWS(D);  // (query, head) rows per tile
    static constexpr uint32_t SHARE = 4 * 32 / ROWS;      // waves that share 32 rows, each with D / SHARE outputs
    static constexpr uint32_t NT = D / SHARE / 32;        // 32-dim output tiles of a wave
    static constexpr uint32_t TB = B / 32;                // 32-token score tiles
    static constexpr uint32_t AHEAD = 4;                  // products that the K reads run ahead
    static_assert(D == 64 || D == 128 || D == 256, "head dims");
    static_assert(2 * STAGE + 4 * TABLE == SGLKV_ATTN_TILE_LDS_BYTES(D), "the host sizes the same LDS");
    static_assert(LPW * TPL * 4 == B && TABLE % B == 0, "whole loads and blocks");
    // K: 256- and 512-byte rows start on a bank period, so 16 tokens need 16
    // positions; 128-byte rows leave t & 1 apart already.
    static __device__ __forceinline__ uint32_t kswz(uint32_t t) { return D >= 128 ? t & 15 : (t >> 1) & 7; }
    // V: four tokens' 64-byte spans in the four quarters of a bank period.
    static __device__ __forceinline__ uint32_t vswz(uint32_t t) { return D >= 128 ? (t & 3) << 2 : (t & 2) << 1; }
};

// The kernel's parameters, read again by whoever asks: the address passes
// through an empty asm, so what one part of the kernel needs (the search, a
// tile's set-up, its loop, its stores) is not held in scalar registers by all
// of them.
__device__ __forceinline__ const sglkv_attn_params &attn_tile_params() {
    typedef const __attribute__((address_space(4))) sglkv_attn_params kernarg;
    kernarg *k = (kernarg *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const sglkv_attn_params *)k;
}

// Most runs of a stretch of 64 queries that a lane walks one after another,
// which takes 0.3 us a run; the other way 1 to 2 us whatever the runs. Measured
// on MI355X with every stretch walked and with this: 512 queries of a prompt and
// 63 decodes over 2,000 tokens (7 queries a KV head, dims 64) 55.6 -> 27.4 us a layer;
// with none walked, 16 prompts of 64 tokens (dims 64) 10.5 -> 11.9 us.
constexpr uint32_t kTileWalk = 6;

constexpr uint32_t kTileGathered = 0xFFFFFFFFu;  // q0 of a tile whose queries are listed

// The nq queries of tile `want` of the step of queries from `base` on, or false
// if it has fewer tiles (uniform over the workgroup): queries [q0, q0 + nq), or
// those listed where q0 is kTileGathered. `masks`: 512 bytes of LDS, the list
// (128 words) behind the first 256; `seen_requests`: 17 KiB, first the step's
// request indices, from which the tile's own request and end are read without
// another memory latency.
// The SGLKV_ATTN_TILE_STEP queries of a step have tiles numbered by themselves
// (numbered over all steps, each workgroup looked through those before its own:
// 1,024 queries of each of 128 prompts, 7 a KV head of dims 64, 3,310 us, so
// 574; 200 of each of 5,000 190 ms, so 2.2). Each wave ballots where runs start
// in 8 stretches of 64 queries (its loads all in flight at once: stepping
// through 128 queries at a time by one wave, each step a memory latency, took
// most of a short tile's time), then lane l of every wave takes the tiles that
// start in stretch l and sums over the lanes. A run ends with its step.
// A step with more runs than there are requests holds queries of one request
// apart from each other. Its tiles gather the queries of one request wherever
// they are in the step: with a tile for each run, 200 queries of each of four
// prompts in turn were 800 tiles of one query and took 495 us (dims 64), so 14.
__device__ __forceinline__ bool attn_tile_find(const sglkv_attn_params &p, uint32_t base, uint32_t want, uint32_t w,
                                               uint32_t lane, uint64_t *masks, uint32_t *seen_requests, uint32_t *q0, uint32_t *nq,
                                               uint32_t *request) {
    asm volatile("" : "+v"(lane));  // (what it computes from the lane is not held across tiles)
    constexpr uint32_t U = 8, STEP = SGLKV_ATTN_TILE_STEP;
    static_assert(STEP == 4 * U * 64, "a stretch of 64 queries per load");
    const uint32_t count = static_cast<uint32_t>(p.query_count);  // host: at most SGLKV_ATTN_TILE_QUERIES_MAX
    const uint32_t *req = p.query_request_indices;
    // ceil(x / tile_queries) for x up to 2^24 (the host's reciprocal is exact there)
    auto tiles_to = [&](uint32_t x) { return __umulhi(x + p.tile_queries - 1, p.tile_recip); };
    // Walks the runs of one stretch: queries [from, from + n), `starts` its
    // run starts, `run` the start of the run that it begins in. Counts the
    // tiles that start there; the k-th (from 0) starts at *at.
    auto walk = [&](uint32_t from, uint32_t n, uint64_t starts, uint32_t run, uint32_t k, uint32_t *at) {
        uint32_t tiles = 0;
        for (uint32_t pos = 0; pos < n;) {
            if ((starts >> pos) & 1) run = from + pos;
            const uint64_t rest = starts & ~((2ull << pos) - 1);
            const uint32_t next = rest ? static_cast<uint32_t>(__builtin_ctzll(rest)) : n;
            const uint32_t a = tiles_to(from + pos - run), b = tiles_to(from + next - run);
            if (k - tiles < b - a) *at = run + (a + k - tiles) * p.tile_queries;
            tiles += b - a;
            pos = next;
        }
        return tiles;
    };
    uint32_t cur[U], before[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        // (Past the last query both are that query: no start.)
        const uint32_t i = base + 64 * (U * w + u) + lane, at = i < count ? i : count;
        cur[u] = req[i < count - 1 ? i : count - 1];
        before[u] = req[(at > 1 ? at : 1) - 1];
    }
    __syncthreads();  // the table and stage that the masks and indices overlay are no longer read
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint64_t starts = __ballot(cur[u] != before[u]) | (w + u == 0 ? 1 : 0);
        seen_requests[64 * (U * w + u) + lane] = cur[u];
        if (lane == 0) masks[U * w + u] = starts;
    }
    __syncthreads();
    const uint64_t starts = lane < 4 * U ? masks[lane] : 0;
    const uint32_t from = base + 64 * lane;
    uint32_t runs = __popcll(starts);
#pragma unroll
    for (uint32_t d = 1; d < 32; d <<= 1) runs += __shfl_xor(runs, d);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(runs) > p.request_count, 0)) {
        // The step's queries of each request (below 2,048 of them; bad
        // indices count as one more), the tiles that they make, in the
        // requests' order, and the tile's own queries in theirs.
        uint32_t *const counts = seen_requests + STEP, bad = p.request_count;
        for (uint32_t i = 64 * w + lane; i <= bad; i += 256) counts[i] = 0;
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (base + 64 * (U * w + u) + lane < count) atomicAdd(&counts[cur[u] < bad ? cur[u] : bad], 1u);
        __syncthreads();
        uint32_t seen = 0;
        for (uint32_t r0 = 0; r0 <= bad; r0 += 64) {
            const uint32_t r = r0 + lane, own = r <= bad ? counts[r] : 0, t = tiles_to(own);
            uint32_t sum = t;
#pragma unroll
            for (uint32_t d = 1; d < 64; d <<= 1) {
                const uint32_t x = __shfl_up(sum, d);
                sum += lane >= d ? x : 0u;
            }
            const uint64_t here = __ballot(want - seen < sum);  // (want >= seen)
            if (here) {
                const int l = __builtin_ctzll(here);
                const uint32_t skip = (want - seen - __shfl(sum - t, l)) * p.tile_queries;
                const uint32_t left = __shfl(own, l) - skip;
                uint32_t *const members = reinterpret_cast<uint32_t *>(masks + 4 * U);
                uint32_t rank = 0;
                // (Every wave writes the whole list.)
                for (uint32_t i = lane; base + i - lane < count && i < STEP; i += 64) {
                    const uint32_t x = seen_requests[i];
                    const bool is = base + i < count && (x < bad ? x : bad) == r0 + l;
                    const uint64_t m = __ballot(is);
                    const uint32_t k = rank - skip +
                                       __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0));
                    if (is && k < p.tile_queries) members[k] = base + i;
                    rank += __popcll(m);
                }
                *q0 = kTileGathered;
                *nq = __builtin_amdgcn_readfirstlane(left < p.tile_queries ? left : p.tile_queries);
                *request = r0 + l;
                return true;
            }
            seen += __builtin_amdgcn_readfirstlane(__shfl(sum, 63));
        }
        return false;
    }
    // Start of the last run at or before the stretch's end: a running
    // maximum over the lanes.
    uint32_t last = starts ? from + 63 - static_cast<uint32_t>(__builtin_clzll(starts)) : 0;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t x = __shfl_up(last, d);
        last = lane >= d && x > last ? x : last;
    }
    const uint32_t in = __shfl_up(last, 1);  // (lane 0's stretch begins with a start)
    const uint32_t n = lane >= 4 * U || from >= count ? 0 : (count - from < 64 ? count - from : 64);
    // Few runs a stretch (prompts, chunks): lane l walks the runs of
    // stretch l. Many (drafts, decodes): all 64 queries of a stretch at
    // once, a tile starting at each multiple of tile_queries from its
    // run's start; wave w takes stretches w, w + 4, ....
    const bool dense = __ballot(__popcll(starts) > kTileWalk) != 0;
    uint64_t tiles = 0;
    uint32_t mine, unused;
    if (dense) {
        for (uint32_t x = w; x < 4 * U && base + 64 * x < count; x += 4) {
            const uint32_t i = base + 64 * x + lane;
            const uint32_t high = __builtin_amdgcn_readlane(static_cast<uint32_t>(starts >> 32), x),
                           low = __builtin_amdgcn_readlane(static_cast<uint32_t>(starts), x);  // (readlane is signed)
            const uint64_t m = static_cast<uint64_t>(high) << 32 | low;
            const uint32_t carried = __builtin_amdgcn_readlane(in, x);
            const uint64_t upto = m & ((2ull << lane) - 1);
            const uint32_t run = upto ? base + 64 * x + 63 - static_cast<uint32_t>(__builtin_clzll(upto)) : carried;
            const uint64_t t = __ballot(i < count && tiles_to(i - run) * p.tile_queries == i - run);
            if (lane == 0) masks[4 * U + x] = t;
        }
        __syncthreads();
        tiles = n ? masks[4 * U + lane] : 0;
        mine = __popcll(tiles);
    } else {
        mine = walk(from, n, starts, in, 0xFFFFFFFFu, &unused);
    }
    uint32_t sum = mine;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t x = __shfl_up(sum, d);
        sum += lane >= d ? x : 0u;
    }
    const uint64_t here = __ballot(want < sum);
    if (!here) return false;
    const int l = __builtin_ctzll(here);
    const uint32_t k = want - __shfl(sum - mine, l);
    const uint64_t from_l = dense ? tiles : starts;
    const uint64_t bits = static_cast<uint64_t>(__shfl(static_cast<uint32_t>(from_l >> 32), l)) << 32 |
                          __shfl(static_cast<uint32_t>(from_l), l);
    uint32_t first = 0;
    if (dense) {
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(bits >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bits), 0));
        first = base + 64 * l + __builtin_ctzll(__ballot(below == k && ((bits >> lane) & 1)));
    } else {
        walk(base + 64 * l, __shfl(n, l), bits, __shfl(in, l), k, &first);
    }
    first = __builtin_amdgcn_readfirstlane(first);
    // The tile ends with its run, its step or after tile_queries (at most
    // 128): how many of the step's queries from `first` on are of its
    // request.
    const uint32_t end = count - base < STEP ? count - base : STEP, i = first - base + lane, j = i + 64;
    const uint32_t ri = seen_requests[i < end ? i : end - 1], rj = seen_requests[j < end ? j : end - 1];
    const uint32_t own = __builtin_amdgcn_readfirstlane(ri);
    const uint64_t oi = ~__ballot(i < end && ri == own), oj = ~__ballot(j < end && rj == own);
    const uint32_t len = oi ? static_cast<uint32_t>(__builtin_ctzll(oi))
                            : 64 + (oj ? static_cast<uint32_t>(__builtin_ctzll(oj)) : 64u);
    *q0 = first;
    *nq = len < p.tile_queries ? len : p.tile_queries;
    *request = own;
    return true;
}

// Four loads: lane l's 16 bytes of load i from a[i] to LDS at at + 1024 i +
// 16 l. Unlike the per-query bodies' they are cached (no nt): the request's
// other tiles read the same rows.
__device__ __forceinline__ void attn_tile_load4(const uint64_t *a, uint32_t at) {
    uint32_t save;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\t"
        "s_add_u32 m0, %1, 1024\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, off\n\t"
        "s_add_u32 m0, %1, 2048\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, off\n\t"
        "s_add_u32 m0, %1, 3072\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(save)
        : "s"(at), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
        : "scc", "memory");
}
__device__ __forceinline__ void attn_tile_load2(const uint64_t *a, uint32_t at) {
    uint32_t save;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\t"
        "s_add_u32 m0, %1, 1024\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(save)
        : "s"(at), "v"(a[0]), "v"(a[1])
        : "scc", "memory");
}

// Wave w's share of a block's rows (table entries at tb) into a stage:
// tokens (B/4) w .. +B/4 of K, then of V. A slot marked invalid (past the
// chunk, or outside the pool) reads the zero row.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_issue(const sglkv_attn_params &p, uint64_t kbase, uint64_t vbase,
                                                const uint32_t *tb, uint32_t w, uint32_t lane, uint32_t stage_at) {
    typedef attn_tl<D> T;
    const uint32_t c = lane / T::PIECES, pos = lane % T::PIECES, t0 = (T::B / 4) * w + c;
    const uint64_t zero = reinterpret_cast<uint64_t>(p.zero_row) + 16 * pos;
    const uint32_t mask = (1u << p.page_shift) - 1;
    uint64_t ka[T::LPW], va[T::LPW];
#pragma unroll
    for (uint32_t j = 0; j < T::LPW; ++j) {
        const uint32_t t = t0 + T::TPL * j;
        const uint32_t s = tb[t];
        const bool ok = s != kAttnInvalidSlot;
        const uint32_t sj = ok ? s : 0u;
        // K and V share the token's offset (equal token strides below 2^24,
        // page_size at most 2^24: the host's rule).
        const uint64_t off = static_cast<uint64_t>(sj >> p.page_shift) * p.page_stride32 +
                             __umul24(sj & mask, p.key_token_stride32);
        attn_sel64x2(ok, kbase + off + 16 * (pos ^ T::kswz(t)), vbase + off + 16 * (pos ^ T::vswz(t)), zero, ka[j],
                     va[j]);
    }
    const uint32_t at = stage_at + 1024 * T::LPW * w;
    if constexpr (T::LPW == 4) {
        attn_tile_load4(ka, at);
        attn_tile_load4(va, at + T::V);
    } else {
        static_assert(T::LPW == 2, "two or four loads");
        attn_tile_load2(ka, at);
        attn_tile_load2(va, at + T::V);
    }
}

// Two floats rounded to bf16 (to nearest even), the first in the low half:
// one instruction for what element by element takes two and a pack.
__device__ __forceinline__ uint32_t attn_pack_bf16(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

__device__ __forceinline__ float attn_max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

template <uint32_t D>
struct attn_tile_state {
    float m_run, l_part;              // row l % 32 (both half-waves hold the same m; l is this half's share)
    sglkv_f32x16 o[attn_tl<D>::NT];   // o[n][i]: dim 32n + 8(i/4) + 4(l/32) + i%4 of the wave's dims of the row
};

// One block from its stage: scores, softmax, o += p.v. `left`: the row's
// tokens from the block's first on (signed); masked: some row of the wave
// ends inside the block. part: which of the SHARE waves of these rows.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_block(const sglkv_attn_params &p, const uint8_t *st_lds,
                                                const sglkv_u16x8 (&qf)[attn_tl<D>::KC], int32_t left, bool masked,
                                                uint32_t lane, uint32_t part, attn_tile_state<D> &st) {
    typedef attn_tl<D> T;
    const uint32_t t = lane & 31, h = lane >> 5;
    sglkv_f32x16 s[T::TB];
#pragma unroll
    for (uint32_t b = 0; b < T::TB; ++b) s[b] = sglkv_f32x16{};
    // The K reads run AHEAD products ahead (sched_barrier keeps the
    // order: the scheduler would sink each read next to its product, which
    // then waits for the LDS).
    auto kread = [&](uint32_t i) {
        return *reinterpret_cast<const sglkv_u16x8 *>(st_lds + T::ROW * (32 * (i % T::TB) + t) +
                                                      16 * ((2 * (i / T::TB) + h) ^ T::kswz(t)));
    };
    // Products run at raised wave priority, the softmax between them at the
    // normal one: otherwise the older of a SIMD's two waves, in its softmax,
    // takes every issue slot and the matrix cores of the other wait.
    __builtin_amdgcn_s_setprio(1);
    sglkv_u16x8 kf[T::AHEAD];
#pragma unroll
    for (uint32_t i = 0; i < T::AHEAD; ++i) kf[i] = kread(i);
#pragma unroll
    for (uint32_t i = 0; i < T::KC * T::TB; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        const sglkv_u16x8 a = kf[i % T::AHEAD];
        s[i % T::TB] = attn_mfma32(a, qf[i / T::TB], s[i % T::TB]);
        if (i + T::AHEAD < T::KC * T::TB) kf[i % T::AHEAD] = kread(i + T::AHEAD);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    if (masked) {
        // Bitwise selects (all ones where the token is below `left`): a
        // compare per element would hold 32 lane masks in scalar registers.
        const int32_t own = left - 4 * static_cast<int32_t>(h);
#pragma unroll
        for (uint32_t b = 0; b < T::TB; ++b)
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) {
                const uint32_t keep = static_cast<uint32_t>((static_cast<int32_t>(32 * b + 8 * (i >> 2) + (i & 3)) - own) >> 31);
                s[b][i] = __uint_as_float((__float_as_uint(s[b][i]) & keep) | (0xFF800000u & ~keep));
            }
    }
    float mx = s[0][0];
#pragma unroll
    for (uint32_t b = 0; b < T::TB; ++b)
#pragma unroll
        for (uint32_t i = 0; i < 16; i += 2) mx = attn_max3(mx, s[b][i], s[b][i + 1]);
    mx = fmaxf(mx, attn_xor32(mx)) * p.scale_log2;
    if (__builtin_amdgcn_readfirstlane(__ballot(mx > st.m_run + 8.0f) != 0 ? 1u : 0u)) {
        const float m_new = fmaxf(st.m_run, mx);
        const float alpha = exp2f(st.m_run - m_new);
        st.l_part *= alpha;
        st.m_run = m_new;
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n)
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) st.o[n][i] *= alpha;
    }
    // V^T operand of 32-dim tile n, 16-token step `step`: tokens 16 step +
    // 4h + L/4 and + 8 (the same vswz), dims 32n + 16c + 4(L%4).
    const uint32_t L = lane & 15, c = (lane >> 4) & 1, t0 = 4 * h + (L >> 2);
    auto vread = [&](uint32_t n, uint32_t step) {
        const uint32_t pc = (4 * (T::NT * part + n) + 2 * c + ((L & 3) >> 1)) ^ T::vswz(t0);
        const uint8_t *at = st_lds + T::V + T::ROW * (16 * step + t0) + 16 * pc + 8 * (L & 1);
        const attn_i16x4 lo = attn_lat_vtr(at), hi = attn_lat_vtr(at + 8 * T::ROW);
        return sglkv_u16x8{(uint16_t)lo[0], (uint16_t)lo[1], (uint16_t)lo[2], (uint16_t)lo[3],
                           (uint16_t)hi[0], (uint16_t)hi[1], (uint16_t)hi[2], (uint16_t)hi[3]};
    };
    // Step `step`'s weights, hi and lo.
    float psum = 0.0f;
    auto weights = [&](uint32_t step, sglkv_u16x8 &phi, sglkv_u16x8 &plo) {
        attn_u32x4 hi, lo;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t e = 8 * (step & 1) + 2 * i;
            const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[step >> 1][e], p.scale_log2, -st.m_run));
            const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(s[step >> 1][e + 1], p.scale_log2, -st.m_run));
            psum += a;
            psum += b;
            hi[i] = attn_pack_bf16(a, b);
            lo[i] = attn_pack_bf16(a - __uint_as_float(hi[i] << 16), b - __uint_as_float(hi[i] & 0xFFFF0000u));
        }
        phi = __builtin_bit_cast(sglkv_u16x8, hi);
        plo = __builtin_bit_cast(sglkv_u16x8, lo);
    };
    // (Dims 256 have no registers for two steps' values.)
    constexpr uint32_t VBUF = D > 128 ? 1 : 2;
    sglkv_u16x8 phi[2], plo[2], v[VBUF][T::NT];
    if (VBUF == 2) {
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n) v[0][n] = vread(n, 0);
    }
    weights(0, phi[0], plo[0]);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (uint32_t step = 0; step < 2 * T::TB; ++step) {
        // A step's products, with the next step's value reads and weights
        // scheduled between them (one read and a share of the vector
        // instructions behind each product).
        const uint32_t x = step & 1;
        __builtin_amdgcn_sched_barrier(0);
        if (VBUF == 1 || step + 1 < 2 * T::TB) {
#pragma unroll
            for (uint32_t n = 0; n < T::NT; ++n) v[(x + 1) % VBUF][n] = vread(n, VBUF == 2 ? step + 1 : step);
        }
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n) st.o[n] = attn_mfma32(v[x % VBUF][n], phi[x], st.o[n]);
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n) st.o[n] = attn_mfma32(v[x % VBUF][n], plo[x], st.o[n]);
        if (step + 1 < 2 * T::TB) {
            weights(step + 1, phi[x ^ 1], plo[x ^ 1]);
#pragma unroll
            for (uint32_t n = 0; n < 2 * T::NT; ++n) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                      // a product
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      // an LDS read
                __builtin_amdgcn_sched_group_barrier(0x402, T::NT == 4 ? 8 : 16, 0);  // vector and exp instructions
            }
        }
    }
    __builtin_amdgcn_s_setprio(0);
    st.l_part += psum;
}

// The slot table from token `from` on, up to the end of the split's last
// block, each slot checked once; the first kTileRaw per thread from raw, if
// the caller has them.
template <uint32_t D, uint32_t N = 0>
__device__ __forceinline__ void attn_tile_slots(const sglkv_attn_params &p, uint64_t start, uint32_t t0, uint32_t t1,
                                                uint32_t from, uint32_t tid, uint32_t *table, const uint64_t *raw) {
    typedef attn_tl<D> T;
    asm volatile("" : "+v"(tid));  // (its table addresses are not held across the loop)
    const uint32_t left = t0 + (t1 - t0 + T::B - 1) / T::B * T::B - from, n = left < T::TABLE ? left : T::TABLE;
#pragma unroll
    for (uint32_t j = 0; j < N; ++j) {
        const uint32_t i = tid + 256 * j;
        if (i < n) table[i] = attn_wide_slot(p, raw[j], from + i, t1);
    }
    for (uint32_t i = tid + 256 * N; i < n; i += 256) {
        const uint32_t tok = from + i;
        table[i] = attn_wide_slot(p, tok < t1 ? p.sequence_slots[start + tok] : 0, tok, t1);
    }
}
template <uint32_t D>
__device__ __forceinline__ void attn_tile_fill(const sglkv_attn_params &p, uint64_t start, uint32_t t0, uint32_t t1,
                                               uint32_t from, uint32_t tid, uint32_t *table) {
    attn_tile_slots<D>(p, start, t0, t1, from, tid, table, nullptr);
}
template <uint32_t D>
__device__ __forceinline__ void attn_tile_fill(const sglkv_attn_params &p, uint64_t start, uint32_t t0, uint32_t t1,
                                               uint32_t from, uint32_t tid, uint32_t *table,
                                               const uint64_t (&raw)[kTileRaw]) {
    attn_tile_slots<D, kTileRaw>(p, start, t0, t1, from, tid, table, raw);
}

// Tokens [t0, t1) of the tile's request for the wave's 32 rows, the first
// blocks' slots in the table.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_pass(const sglkv_attn_params &p, uint64_t start, uint32_t t0, uint32_t t1,
                                               uint64_t kbase, uint64_t vbase, uint32_t w, uint32_t tid,
                                               uint32_t lane, uint32_t lds_at, uint32_t len, uint32_t wave_min,
                                               uint32_t wave_max, const sglkv_u16x8 (&qf)[attn_tl<D>::KC],
                                               attn_tile_state<D> &st) {
    typedef attn_tl<D> T;
    extern __shared__ __attribute__((aligned(16))) uint8_t attn_tile_lds[];
    uint32_t *table = reinterpret_cast<uint32_t *>(attn_tile_lds + 2 * T::STAGE);
    constexpr uint32_t TBLOCKS = T::TABLE / T::B;
    const uint32_t nb = (t1 - t0 + T::B - 1) / T::B;
    __syncthreads();
    // The queries' loads are complete here, so that the compiler puts no wait
    // for them (which would be one for the rows in flight) into the loop.
    __builtin_amdgcn_s_waitcnt(0x0F70);
    attn_tile_issue<D>(p, kbase, vbase, table, w, lane, lds_at);
    st.m_run = -3.402823466e+38f;
    st.l_part = 0.0f;
#pragma unroll
    for (uint32_t n = 0; n < T::NT; ++n) st.o[n] = sglkv_f32x16{};
    // Block k's rows have landed (every wave waits for its own, then meets
    // the others), and nobody reads block k-1's stage any more: block k+1's
    // rows go there.
    auto next = [&](uint32_t k) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (k + 1 >= nb) return;
        if ((k + 1) % TBLOCKS == 0) {
            attn_tile_fill<D>(p, start, t0, t1, t0 + (k + 1) * T::B, tid, table);
            __syncthreads();
        }
        attn_tile_issue<D>(p, kbase, vbase, table + ((k + 1) % TBLOCKS) * T::B, w, lane,
                           lds_at + ((k + 1) & 1) * T::STAGE);
    };
    // The blocks that the wave's rows attend, then those it only loads for
    // the others (a branch around the block instead would have the compiler
    // copy the outputs every block).
    const uint32_t mine = wave_max <= t0 ? 0 : (wave_max < t1 ? wave_max - t0 + T::B - 1 : nb * T::B) / T::B;
    for (uint32_t k = 0; k < mine; ++k) {
        next(k);
        const uint32_t tb = t0 + k * T::B;
        attn_tile_block<D>(p, attn_tile_lds + (k & 1) * T::STAGE, qf, static_cast<int32_t>(len - tb),
                           tb + T::B > wave_min, lane, w % T::SHARE, st);
    }
    for (uint32_t k = mine; k < nb; ++k) next(k);
}

// The lane's row of a tile: query and head within the group. Worked out anew
// (the lane passes through an empty asm) where it is needed, rather than held
// across the loop.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_row(const sglkv_attn_params &p, uint32_t w, uint32_t lane, uint32_t *query,
                                              uint32_t *head) {
    asm volatile("" : "+v"(lane));
    const uint32_t row = 32 * (w / attn_tl<D>::SHARE) + (lane & 31);
    *query = row / p.group;
    *head = row - *query * p.group;
}

// The output of the row of query `query` (one split), or its split record (rows of the combine
// kernel's layout). Lanes l and l + 32 hold the row's dims 8i + 4h .. +3.
// Plain stores: the two lanes' pieces of a line meet in L2.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_write(const sglkv_attn_params &p, uint32_t query, uint32_t kvh, uint32_t split, uint32_t w,
                                                uint32_t lane, const attn_tile_state<D> &st) {
    typedef attn_tl<D> T;
    uint32_t rq, rh;
    attn_tile_row<D>(p, w, lane, &rq, &rh);
    const uint64_t qrow = static_cast<uint64_t>(query) * p.query_heads + kvh * p.group + rh;
    const uint32_t part = w % T::SHARE, h = lane >> 5;
    const float l_tot = st.l_part + __shfl_xor(st.l_part, 32);
    if (p.splits == 1) {
        const float linv = 1.0f / l_tot;
        uint16_t *out = p.output + qrow * D + D / T::SHARE * part + 4 * h;
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n)
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                sglkv_u16x4 v;
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e) v[e] = attn_to_bf16(st.o[n][4 * i + e] * linv);
                *reinterpret_cast<sglkv_u16x4 *>(out + 32 * n + 8 * i) = v;  // (host: 8-byte aligned output)
            }
        return;
    }
    const uint64_t rec = qrow * p.splits + split;
    if (h == 0 && part == 0) {
        float *pr = attn_rec_ml(p, rec);
        pr[0] = st.m_run;
        pr[1] = l_tot;
    }
    float *out = attn_rec_o(p, rec) + D / T::SHARE * part + 4 * h;
#pragma unroll
    for (uint32_t n = 0; n < T::NT; ++n)
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const sglkv_f32x4 v = {st.o[n][4 * i], st.o[n][4 * i + 1], st.o[n][4 * i + 2], st.o[n][4 * i + 3]};
            *reinterpret_cast<sglkv_f32x4 *>(out + 32 * n + 8 * i) = v;
        }
}

// The first tile of the x-th workgroup of a KV head and split (the host's
// rule).
__device__ __forceinline__ uint32_t attn_tile_order(const sglkv_attn_params &p, uint32_t x) {
    if (p.tile_fold && x >= p.tile_fold) x = p.tile_slots - 1 - (x - p.tile_fold);
    return p.tile_backward ? p.tile_slots - 1 - x : x;
}

template <uint32_t D>
__device__ __forceinline__ void attn_tile_body() {
    typedef attn_tl<D> T;
    const sglkv_attn_params &p = attn_tile_params();
    extern __shared__ __attribute__((aligned(16))) uint8_t attn_tile_lds[];
    uint32_t *table = reinterpret_cast<uint32_t *>(attn_tile_lds + 2 * T::STAGE);
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kvh = blockIdx.x % p.kv_heads, split = blockIdx.y;
    const uint64_t pool = reinterpret_cast<uint64_t>(p.pool);
    const uint64_t kbase = pool + p.key_offset + kvh * p.key_head_stride;
    const uint64_t vbase = pool + p.value_offset + kvh * p.value_head_stride;
    const uint32_t lds_at = attn_lat_lds_at(attn_tile_lds);
    // Plans of one request take their queries in tiles as they come (a query
    // of any other index is refused row by row): no search. Otherwise the
    // tiles of each request's run.
    const uint32_t count = static_cast<uint32_t>(p.query_count);
    auto find = [&](uint32_t base, uint32_t tile, uint32_t *q0, uint32_t *nq, uint32_t *req) {
        const sglkv_attn_params &p = attn_tile_params();
        if (p.request_count > 1)
            return attn_tile_find(p, base, tile, w, lane, reinterpret_cast<uint64_t *>(table),
                                  reinterpret_cast<uint32_t *>(attn_tile_lds), q0, nq, req);
        *q0 = tile * p.tile_queries;
        *nq = *q0 < count && count - *q0 < p.tile_queries ? count - *q0 : p.tile_queries;
        *req = 0;
        return *q0 < count;
    };
    // The workgroup's step (the first ones have tile_step_slots workgroups each,
    // the last one the rest) and its tiles there.
    uint32_t q0, nq, req, tile = attn_tile_order(p, blockIdx.x / p.kv_heads), base = 0, stride = p.tile_slots;
    if (p.tile_step_slots) {
        const uint32_t last = (count - 1) / SGLKV_ATTN_TILE_STEP,
                       own = __builtin_amdgcn_readfirstlane(tile / p.tile_step_slots), step = own < last ? own : last;
        tile -= step * p.tile_step_slots;
        stride = step < last ? p.tile_step_slots : p.tile_slots - last * p.tile_step_slots;
        base = step * SGLKV_ATTN_TILE_STEP;
    }
    for (; find(base, tile, &q0, &nq, &req); tile += stride) {
        const sglkv_attn_params &p = attn_tile_params();
        uint32_t rq, rh;
        attn_tile_row<D>(p, w, lane, &rq, &rh);
        // The tile's request (uniform) and the lane's query: everything that
        // depends on the tile alone is loaded at once (from request 0 and
        // the tile's first query where the lane or the request has none).
        const bool mine = rq < nq;
        // (A listed query is read here, before the list's LDS is used again.)
        const uint32_t member = mine ? rq : 0;
        const uint32_t query = q0 == kTileGathered ? reinterpret_cast<const uint32_t *>(table)[64 + member] : q0 + member;
        const uint64_t qrow = static_cast<uint64_t>(query) * p.query_heads + kvh * p.group + rh;
        const uint32_t known = req < p.request_count ? req : 0;
        const uint64_t start = p.request_slot_offsets[known], end = p.request_slot_offsets[known + 1];
        const uint64_t n = p.query_sequence_lengths[query];
        const uint32_t own_req = p.query_request_indices[query];
        // Queries (B operand of q.k): row l % 32, dims 16c + 8(l/32).
        sglkv_u16x8 qf[T::KC];
#pragma unroll
        for (uint32_t c = 0; c < T::KC; ++c)
            qf[c] = *reinterpret_cast<const sglkv_u16x8 *>(p.queries + qrow * D + 16 * c + 8 * (lane >> 5));
        // The reference's checks; one workgroup per tile reports.
        const uint32_t quiet = split | kvh, chunk = static_cast<uint32_t>(p.chunk_tokens), t0 = split * chunk;
        uint32_t bad = 0;
        if (own_req >= p.request_count)
            bad = SGLKV_FLAG_ATTN_REQUEST;
        else if (start > end || end > p.sequence_slot_count || n == 0 || n > end - start || n > chunk * p.splits)
            bad = SGLKV_FLAG_ATTN_SEQUENCE;  // (host: chunk * splits below 2^31)
        if (mine && bad && quiet == 0) atomicOr(p.flag, bad);
        // The row's tokens (0: no row, or a query that fails its checks).
        const uint32_t len = mine && !bad ? static_cast<uint32_t>(n) : 0;
        // The split's first slots, ahead of the rows' lengths (which tokens
        // are attended, and so checked, is decided at use).
        uint64_t raw[kTileRaw];
        const bool ranged = start < end && end <= p.sequence_slot_count;
#pragma unroll
        for (uint32_t j = 0; j < kTileRaw; ++j) {
            const uint64_t tok = start + t0 + tid + 256 * j;
            raw[j] = ranged ? p.sequence_slots[tok < end ? tok : end - 1] : 0;
        }
        // One round with every row; the tile is done unless its values are
        // not finite. A token that one row attends and another does not has
        // weight 0 in the other's product, and 0 times an infinite or NaN
        // value is NaN, while a query must not see values past its own
        // length. So when a wave whose rows end apart holds an output that is
        // not finite, the rows are done again, one length a round from the
        // longest down: no row then meets a token that it does not attend.
        // That costs a pass per length: up to tile_queries (at most 128) passes
        // more for a tile of a causal prompt that reaches such a value.
        auto wave_reduce = [&](uint32_t v, bool most) {
#pragma unroll
            for (uint32_t d = 1; d < 32; d <<= 1) {
                const uint32_t x = __shfl_xor(v, d);
                v = (x > v) == most ? x : v;
            }
            return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(v));
        };
        // The longest of the tile's rows that are shorter than `below`
        // (through the slot table's first words).
        auto tile_longest = [&](uint32_t below) {
            const uint32_t most = wave_reduce(len < below ? len : 0, true);
            __syncthreads();  // the table and stages are no longer read
            if (lane == 0) table[w] = most;
            __syncthreads();
            uint32_t x = table[0];
#pragma unroll
            for (uint32_t i = 1; i < 4; ++i) x = table[i] > x ? table[i] : x;
            __syncthreads();
            return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(x));
        };
        uint32_t longest = tile_longest(0xFFFFFFFFu);
        if (t0 >= longest) continue;
        uint32_t t1 = longest - t0 < chunk ? longest : t0 + chunk;
        attn_tile_fill<D>(p, start, t0, t1, t0, tid, table, raw);
        bool apart = false;
        for (;;) {
            const uint32_t own = apart && len != longest ? 0 : len;
            const uint32_t wave_max = wave_reduce(own, true);
            const uint32_t wave_min = wave_reduce(own ? own : 0xFFFFFFFFu, false);
            attn_tile_state<D> st;
            attn_tile_pass<D>(attn_tile_params(), start, t0, t1, kbase, vbase, w, tid, lane, lds_at, own, wave_min, wave_max, qf, st);
            if (!apart) {
                float odd = 0.0f;
#pragma unroll
                for (uint32_t n = 0; n < T::NT; ++n)
#pragma unroll
                    for (uint32_t i = 0; i < 16; ++i) odd = __builtin_fmaf(st.o[n][i], 0.0f, odd);
                const bool redo = __ballot(odd != 0.0f && len > t0) != 0 && t1 > wave_min;  // (NaN != 0)
                if (lane == 0) table[w] = redo ? 1u : 0u;  // (the table is not read past the last block's issue)
                __syncthreads();
                apart = __builtin_amdgcn_readfirstlane(table[0] | table[1] | table[2] | table[3]) != 0;
                if (!apart) {
                    if (own > t0) attn_tile_write<D>(attn_tile_params(), query, kvh, split, w, lane, st);
                    break;
                }
                longest = 0xFFFFFFFFu;
            } else if (own > t0) {
                attn_tile_write<D>(attn_tile_params(), query, kvh, split, w, lane, st);
            }
            longest = tile_longest(longest);
            if (t0 >= longest) break;
            t1 = longest - t0 < chunk ? longest : t0 + chunk;
            attn_tile_fill<D>(p, start, t0, t1, t0, tid, table);
        }
    }
}

}  // namespace

extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
sglkv_paged_attention_tile128(sglkv_attn_params) {
    attn_tile_body<128>();
}

extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void
sglkv_paged_attention_tile64(sglkv_attn_params) {
    attn_tile_body<64>();
}

extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
sglkv_paged_attention_tile256(sglkv_attn_params) {
    attn_tile_body<256>();
}
