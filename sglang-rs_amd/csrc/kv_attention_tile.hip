// kv_attention_tile.hip -- paged attention for launches with several queries
// per request: prefill (one query per prompt token, as the reference's
// scheduler metadata has it), chunked prefill, verification of drafted tokens.
//
// The per-query bodies of kv_attention.hip give every (query, KV head) a wave
// of its own, so each query of a prompt reads the prompt's K and V again and
// fills only `group` of the 16 columns of its matrix products. Here a
// workgroup of four waves owns a tile: up to tile_queries consecutive queries
// of one request, whose query heads of one KV head are the tile's rows
// (row = query * group + head, at most 128, 32 per wave). Every K and V row is
// staged in LDS once per tile.
//  - Tiles. A run is a maximal stretch of consecutive queries of one request;
//    it is cut into tiles of tile_queries from its start, and tiles are
//    numbered over all runs. Which queries tile t holds is found from
//    query_request_indices by every wave on its own (64 queries a step,
//    ballots and scalar arithmetic), so queries of different requests never
//    share a tile whatever their order, and no planning launch or device list
//    is needed. The host launches tile_slots tiles per KV head, enough for
//    queries that come request by request; workgroups step by tile_slots, so
//    any other order is covered too. Later tiles of a causal prompt attend
//    more tokens, so the tiles are taken from the last to the first.
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
// What bounds it: the matrix products (48 per 64-token block and wave at dims
// 128, 32 of them p.v's, hi and lo) and the softmax between them, on two waves
// per SIMD. Measured on MI355X, per layer: causal prompts of 300..2,048 tokens
// (5,206 queries, 32 heads over 8, dims 128) 1,744 -> 206 us, 322 TFLOP/s of
// q.k and p.v; 384 queries over 6,144 tokens (14 heads over 2, dims 64)
// 112 -> 41 us.

namespace {

template <uint32_t D>
struct attn_tl {
    static constexpr uint32_t ROW = 2 * D;                // bytes of one token's head slice
    static constexpr uint32_t PIECES = D / 8;             // 16-byte pieces per row
    static constexpr uint32_t TPL = 1024 / ROW;           // tokens per load
    static constexpr uint32_t B = SGLKV_ATTN_TILE_BLOCK;  // tokens per block
    static constexpr uint32_t LPW = B / TPL / 4;          // K loads (and V loads) of a wave per block
    static constexpr uint32_t V = B * ROW;                // V rows' offset in a stage
    static constexpr uint32_t STAGE = 2 * V;
    static constexpr uint32_t TABLE = SGLKV_ATTN_TILE_SLOTS(D);  // slot table entries (whole blocks)
    static constexpr uint32_t KC = D / 16;                // q.k steps
    static constexpr uint32_t NT = D / 32;                // 32-dim output tiles
    static constexpr uint32_t TB = B / 32;                // 32-token score tiles
    static_assert(D == 64 || D == 128, "head dims");
    static_assert(2 * STAGE + 4 * TABLE == SGLKV_ATTN_TILE_LDS_BYTES(D), "the host sizes the same LDS");
    static_assert(LPW * TPL * 4 == B && TABLE % B == 0, "whole loads and blocks");
    // K: 256-byte rows start on a bank period, so 16 tokens need 16
    // positions; 128-byte rows leave t & 1 apart already.
    static __device__ __forceinline__ uint32_t kswz(uint32_t t) { return D == 128 ? t & 15 : (t >> 1) & 7; }
    // V: four tokens' 64-byte spans in the four quarters of a bank period.
    static __device__ __forceinline__ uint32_t vswz(uint32_t t) { return D == 128 ? (t & 3) << 2 : (t & 2) << 1; }
};

// Queries [q0, q0 + nq) of tile `want`, or false if there are fewer tiles.
// Uniform over the wave; every wave of a workgroup finds the same answer.
__device__ __forceinline__ bool attn_tile_find(const sglkv_attn_params &p, uint32_t want, uint32_t lane,
                                               uint32_t *q0, uint32_t *nq) {
    constexpr uint32_t U = 2;  // 64-query steps whose loads are issued together
    const uint32_t count = static_cast<uint32_t>(p.query_count);  // host: at most SGLKV_ATTN_TILE_QUERIES_MAX
    const uint32_t *req = p.query_request_indices;
    // ceil(x / tile_queries) for x below 2^24 (the host's reciprocal is exact there)
    auto tiles_to = [&](uint32_t x) { return __umulhi(x + p.tile_queries - 1, p.tile_recip); };
    uint32_t seen = 0, run = 0;
    bool found = false;
    uint32_t first = 0;
    for (uint32_t base = 0; base < count && !found; base += 64 * U) {
        uint32_t cur[U], before[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = base + 64 * u + lane, at = i < count ? i : count - 1;
            cur[u] = req[at];
            before[u] = req[at ? at - 1 : 0];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t c0 = base + 64 * u;
            if (c0 >= count || found) break;
            const uint32_t n = count - c0 < 64 ? count - c0 : 64;
            uint64_t starts = __ballot(lane < n && (c0 + lane == 0 || cur[u] != before[u]));
            for (uint32_t pos = 0; pos < n;) {
                if ((starts >> pos) & 1) run = c0 + pos;
                starts &= ~(1ull << pos);
                const uint32_t next = starts ? static_cast<uint32_t>(__builtin_ctzll(starts)) : n;
                const uint32_t a = tiles_to(c0 + pos - run), b = tiles_to(c0 + next - run);
                if (want - seen < b - a) {
                    first = run + (a + want - seen) * p.tile_queries;
                    found = true;
                    break;
                }
                seen += b - a;
                pos = next;
            }
        }
    }
    if (!found) return false;
    first = __builtin_amdgcn_readfirstlane(first);
    // The tile ends with its run or after tile_queries (at most 128).
    const uint32_t own = req[first];
    auto leading = [&](uint32_t from) {  // queries from `from` on that are own's, up to 64
        const uint32_t i = from + lane;
        const uint64_t other = ~__ballot(i < count && req[i < count ? i : count - 1] == own);
        return other ? static_cast<uint32_t>(__builtin_ctzll(other)) : 64u;
    };
    uint32_t len = leading(first);
    if (len == 64 && p.tile_queries > 64) len += leading(first + 64);
    *q0 = first;
    *nq = len < p.tile_queries ? len : p.tile_queries;
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

template <uint32_t D>
struct attn_tile_state {
    float m_run, l_part;              // row l % 32 (both half-waves hold the same m; l is this half's share)
    sglkv_f32x16 o[attn_tl<D>::NT];   // o[n][i]: dim 32n + 8(i/4) + 4(l/32) + i%4 of the row
};

// One block from its stage: scores, softmax, o += p.v. `left`: the row's
// tokens from the block's first on (signed); masked: some row of the wave
// ends inside the block.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_block(const sglkv_attn_params &p, const uint8_t *st_lds,
                                                const sglkv_u16x8 (&qf)[attn_tl<D>::KC], int32_t left, bool masked,
                                                uint32_t lane, attn_tile_state<D> &st) {
    typedef attn_tl<D> T;
    const uint32_t t = lane & 31, h = lane >> 5;
    sglkv_f32x16 s[T::TB];
#pragma unroll
    for (uint32_t b = 0; b < T::TB; ++b) s[b] = sglkv_f32x16{};
#pragma unroll
    for (uint32_t c = 0; c < T::KC; ++c)
#pragma unroll
        for (uint32_t b = 0; b < T::TB; ++b) {
            const sglkv_u16x8 kf = *reinterpret_cast<const sglkv_u16x8 *>(
                st_lds + T::ROW * (32 * b + t) + 16 * ((2 * c + h) ^ T::kswz(t)));
            s[b] = attn_mfma32(kf, qf[c], s[b]);
        }
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
        for (uint32_t i = 0; i < 16; ++i) mx = fmaxf(mx, s[b][i]);
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
        const uint32_t pc = (4 * n + 2 * c + ((L & 3) >> 1)) ^ T::vswz(t0);
        const uint8_t *at = st_lds + T::V + T::ROW * (16 * step + t0) + 16 * pc + 8 * (L & 1);
        const attn_i16x4 lo = attn_lat_vtr(at), hi = attn_lat_vtr(at + 8 * T::ROW);
        return sglkv_u16x8{(uint16_t)lo[0], (uint16_t)lo[1], (uint16_t)lo[2], (uint16_t)lo[3],
                           (uint16_t)hi[0], (uint16_t)hi[1], (uint16_t)hi[2], (uint16_t)hi[3]};
    };
    float psum = 0.0f;
#pragma unroll
    for (uint32_t step = 0; step < 2 * T::TB; ++step) {
        sglkv_u16x8 phi, plo;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            const float pr =
                __builtin_amdgcn_exp2f(__builtin_fmaf(s[step >> 1][8 * (step & 1) + i], p.scale_log2, -st.m_run));
            psum += pr;
            attn_split_bf16(pr, phi, plo, i);
        }
#pragma unroll
        for (uint32_t n = 0; n < T::NT; ++n) {
            const sglkv_u16x8 v = vread(n, step);
            st.o[n] = attn_mfma32(v, phi, st.o[n]);
            st.o[n] = attn_mfma32(v, plo, st.o[n]);
        }
    }
    st.l_part += psum;
}

// Tokens [t0, t1) of the tile's request for the wave's 32 rows.
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
    // The slots of blocks [b, b + TBLOCKS), checked once.
    auto fill = [&](uint32_t b) {
        const uint32_t from = t0 + b * T::B;
        const uint32_t left = (nb - b) * T::B, n = left < T::TABLE ? left : T::TABLE;
        for (uint32_t i = tid; i < n; i += 256) {
            const uint32_t tok = from + i;
            table[i] = attn_wide_slot(p, tok < t1 ? p.sequence_slots[start + tok] : 0, tok, t1);
        }
    };
    fill(0);
    __syncthreads();
    attn_tile_issue<D>(p, kbase, vbase, table, w, lane, lds_at);
    st.m_run = -3.402823466e+38f;
    st.l_part = 0.0f;
#pragma unroll
    for (uint32_t n = 0; n < T::NT; ++n) st.o[n] = sglkv_f32x16{};
    for (uint32_t k = 0; k < nb; ++k) {
        // Block k's rows have landed (every wave waits for its own, then
        // meets the others), and nobody reads block k-1's stage any more.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (k + 1 < nb) {
            if ((k + 1) % TBLOCKS == 0) {
                fill(k + 1);
                __syncthreads();
            }
            attn_tile_issue<D>(p, kbase, vbase, table + ((k + 1) % TBLOCKS) * T::B, w, lane,
                               lds_at + ((k + 1) & 1) * T::STAGE);
        }
        const uint32_t tb = t0 + k * T::B;
        if (tb < wave_max)
            attn_tile_block<D>(p, attn_tile_lds + (k & 1) * T::STAGE, qf, static_cast<int32_t>(len - tb),
                                        tb + T::B > wave_min, lane, st);
    }
}

// The row's output (one split), or its split record (rows of the combine
// kernel's layout). Lanes l and l + 32 hold the row's dims 8i + 4h .. +3.
// Plain stores: the two lanes' pieces of a line meet in L2.
template <uint32_t D>
__device__ __forceinline__ void attn_tile_write(const sglkv_attn_params &p, uint64_t qrow, uint32_t split, uint32_t h,
                                                const attn_tile_state<D> &st) {
    typedef attn_tl<D> T;
    const float l_tot = st.l_part + __shfl_xor(st.l_part, 32);
    if (p.splits == 1) {
        const float linv = 1.0f / l_tot;
        uint16_t *out = p.output + qrow * D + 4 * h;
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
    if (h == 0) {
        float *pr = attn_rec_ml(p, rec);
        pr[0] = st.m_run;
        pr[1] = l_tot;
    }
    float *out = attn_rec_o(p, rec) + 4 * h;
#pragma unroll
    for (uint32_t n = 0; n < T::NT; ++n)
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const sglkv_f32x4 v = {st.o[n][4 * i], st.o[n][4 * i + 1], st.o[n][4 * i + 2], st.o[n][4 * i + 3]};
            *reinterpret_cast<sglkv_f32x4 *>(out + 32 * n + 8 * i) = v;
        }
}

template <uint32_t D>
__device__ __forceinline__ void attn_tile_body(const sglkv_attn_params &p) {
    typedef attn_tl<D> T;
    extern __shared__ __attribute__((aligned(16))) uint8_t attn_tile_lds[];
    uint32_t *table = reinterpret_cast<uint32_t *>(attn_tile_lds + 2 * T::STAGE);
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kvh = blockIdx.x % p.kv_heads, split = blockIdx.y;
    const uint64_t pool = reinterpret_cast<uint64_t>(p.pool);
    const uint64_t kbase = pool + p.key_offset + kvh * p.key_head_stride;
    const uint64_t vbase = pool + p.value_offset + kvh * p.value_head_stride;
    const uint32_t lds_at = attn_lat_lds_at(attn_tile_lds);
    // The lane's row of a tile.
    const uint32_t row = 32 * w + (lane & 31), rq = row / p.group, rh = row - rq * p.group;

    uint32_t q0, nq;
    for (uint32_t tile = p.tile_slots - 1 - blockIdx.x / p.kv_heads; attn_tile_find(p, tile, lane, &q0, &nq);
         tile += p.tile_slots) {
        // Metadata of the tile's request (uniform), then of the lane's query.
        const bool report = split == 0 && kvh == 0;
        const uint32_t req = p.query_request_indices[q0];
        if (req >= p.request_count) {
            if (report && tid == 0) atomicOr(p.flag, SGLKV_FLAG_ATTN_REQUEST);
            continue;
        }
        const uint64_t start = p.request_slot_offsets[req], end = p.request_slot_offsets[req + 1];
        if (start > end || end > p.sequence_slot_count) {
            if (report && tid == 0) atomicOr(p.flag, SGLKV_FLAG_ATTN_SEQUENCE);
            continue;
        }
        const bool mine = rq < nq;
        uint32_t len = 0;  // the row's tokens (0: no row, or a query that fails its checks)
        if (mine) {
            const uint64_t n = p.query_sequence_lengths[q0 + rq];
            if (n == 0 || n > end - start || n > p.chunk_tokens * static_cast<uint64_t>(p.splits)) {
                if (report) atomicOr(p.flag, SGLKV_FLAG_ATTN_SEQUENCE);
            } else {
                len = static_cast<uint32_t>(n);  // host: chunk_tokens * splits < 2^31
            }
        }
        const uint32_t chunk = static_cast<uint32_t>(p.chunk_tokens), t0 = split * chunk;
        // Queries (B operand of q.k): row l % 32, dims 16c + 8(l/32).
        const uint64_t qrow = (static_cast<uint64_t>(q0) + rq) * p.query_heads + kvh * p.group + rh;
        sglkv_u16x8 qf[T::KC];
#pragma unroll
        for (uint32_t c = 0; c < T::KC; ++c) {
            qf[c] = sglkv_u16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (mine) qf[c] = *reinterpret_cast<const sglkv_u16x8 *>(p.queries + qrow * D + 16 * c + 8 * (lane >> 5));
        }
        // One round with every row; the tile is done unless its values are
        // not finite. A token that one row attends and another does not has
        // weight 0 in the other's product, and 0 times an infinite or NaN
        // value is NaN, while a query must not see values past its own
        // length. So when a wave whose rows end apart holds an output that is
        // not finite, the rows are done again, one length a round from the
        // longest down: no row then meets a token that it does not attend.
        bool apart = false;
        for (uint32_t below = 0xFFFFFFFFu;;) {
            // The round's longest row over the tile (through the slot
            // table's first words), and the wave's longest and shortest.
            auto wave_reduce = [&](uint32_t v, bool most) {
#pragma unroll
                for (uint32_t d = 1; d < 32; d <<= 1) {
                    const uint32_t x = __shfl_xor(v, d);
                    v = (x > v) == most ? x : v;
                }
                return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(v));
            };
            uint32_t wave_max = wave_reduce(len < below ? len : 0, true);
            __syncthreads();  // the previous round's table and stages are no longer read
            if (lane == 0) table[w] = wave_max;
            __syncthreads();
            uint32_t longest = table[0];
#pragma unroll
            for (uint32_t i = 1; i < 4; ++i) longest = table[i] > longest ? table[i] : longest;
            longest = __builtin_amdgcn_readfirstlane(longest);
            __syncthreads();
            if (t0 >= longest) break;
            below = longest;
            const uint32_t own = apart && len != longest ? 0 : len;
            if (apart) wave_max = wave_reduce(own, true);
            const uint32_t wave_min = wave_reduce(own ? own : 0xFFFFFFFFu, false);
            const uint32_t t1 = longest - t0 < chunk ? longest : t0 + chunk;
            attn_tile_state<D> st;
            attn_tile_pass<D>(p, start, t0, t1, kbase, vbase, w, tid, lane, lds_at, own, wave_min, wave_max, qf, st);
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
                if (apart) {
                    below = 0xFFFFFFFFu;
                    continue;
                }
            }
            if (own > t0) attn_tile_write<D>(p, qrow, split, lane >> 5, st);
            if (!apart) break;
        }
    }
}

}  // namespace

extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
sglkv_paged_attention_tile128(sglkv_attn_params p) {
    attn_tile_body<128>(p);
}

extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
sglkv_paged_attention_tile64(sglkv_attn_params p) {
    attn_tile_body<64>(p);
}
