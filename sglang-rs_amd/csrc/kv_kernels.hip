// kv_kernels.hip -- gfx950 kernels of the KV-cache transfer path.
//
// Built ahead of time into a code object (sgl_rocm_kv_gfx950.co) and loaded
// with hipModuleLoad by kv_runtime.cpp; every entry point is extern "C" so
// the launcher resolves it by its plain name.
//
// The work is pure byte movement (no arithmetic on the payload), so the
// design goal is HBM bandwidth:
//  - A workgroup owns a tile of consecutive transfer rows. Before copying,
//    it resolves each tile row's physical slot into a byte offset once
//    (slot -> page, position -> offset) and stages the offsets in LDS, so
//    the per-vector work is one LDS read and one 64-bit add.
//  - Threads are laid out (x = vector index inside a row, y = row). Thread
//    x keeps the same position in every row it copies, so which tensor and
//    which head chunk it touches is decided once per thread, not per byte
//    as in the reference's byte-per-thread kernels
//    (crates/sglang-kernel/src/cuda_kv_kernels.rs:11-99).
//  - Each thread issues the loads of SGLKV_ROWS_PER_THREAD rows before any
//    store, so a 64-lane wavefront keeps up to 8 KiB in flight.
//  - Accesses are VB-byte vectors (16 B = global_load/store_dwordx4 on the
//    common shapes); consecutive lanes touch consecutive vectors of one row
//    or one head chunk, so every wavefront access is a run of >= 256
//    contiguous bytes for the shapes of this path.
// A slot outside the pool skips the row and raises SGLKV_FLAG_SLOT in the
// device error word, as the reference's kernels do with error_flag.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kv_params.h"

typedef unsigned int sglkv_v4u __attribute__((ext_vector_type(4)));
typedef unsigned int sglkv_v2u __attribute__((ext_vector_type(2)));

// Global-address-space pointers: built from integer addresses, a plain
// pointer would be flat, and flat accesses share the LDS wait counter, which
// would serialise the loads behind the LDS reads of the row offsets.
typedef __attribute__((address_space(1))) const char sglkv_gsrc;
typedef __attribute__((address_space(1))) char sglkv_gdst;

// Tile constants of this code object, read by the launcher at load time.
extern "C" __device__ uint32_t sglkv_rows_per_thread = SGLKV_ROWS_PER_THREAD;
extern "C" __device__ uint32_t sglkv_max_tile_rows = SGLKV_MAX_TILE_ROWS;
extern "C" __device__ uint32_t sglkv_realign_rows_per_thread = SGLKV_REALIGN_ROWS_PER_THREAD;

// Cache policy of each copy direction, as bits: 1 = non-temporal loads,
// 2 = non-temporal stores (they stream past the caches instead of
// allocating lines nothing will reuse). Defaults chosen by measurement on
// MI355X.
#ifndef SGLKV_PACK_NT
#define SGLKV_PACK_NT 1
#endif
#ifndef SGLKV_UNPACK_NT
#define SGLKV_UNPACK_NT 3
#endif
#ifndef SGLKV_TRANSFER_NT
#define SGLKV_TRANSFER_NT 3
#endif
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs
// on XCD b % 8). A remapped direction instead gives each XCD one contiguous
// eighth of the row tiles. The unpack keeps the round-robin order: the rows
// pack has just written are still partly in the Infinity Cache (the later
// part of each layer's rows), and round-robin tiles give every XCD an equal
// share of cached and uncached rows, where contiguous eighths leave the XCDs
// with the uncached first half the long pole (read latency twice that of
// the other half in rocprofv3's per-XCD counters). Measured on MI355X, one
// process per line with both orders on the same pools: unpack per layer C2
// 208.1 -> 206.0 us (180.0 -> 174.7 in the other placement cluster), C3
// 107.9 -> 90.4, C4 117.5 -> 94.9, the C4 key/value pair 192.6 -> 183.8;
// the 64-byte-chunk HND unpack is unchanged. Pack: contiguous eighths were
// 1 % slower.
#ifndef SGLKV_PACK_REMAP
#define SGLKV_PACK_REMAP 0
#endif
#ifndef SGLKV_UNPACK_REMAP
#define SGLKV_UNPACK_REMAP 0
#endif
#ifndef SGLKV_TRANSFER_REMAP
#define SGLKV_TRANSFER_REMAP 2
#endif
#define SGLKV_XCDS 8u

template <typename V, int NT>
__device__ __forceinline__ V sglkv_load(__attribute__((address_space(1))) const V *p) {
    if (NT & 1) return __builtin_nontemporal_load(p);
    return *p;
}

template <typename V, int NT>
__device__ __forceinline__ void sglkv_store(__attribute__((address_space(1))) V *p, V v) {
    if (NT & 2)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

// Logical tile and layer of this workgroup. REMAP 1 gives each XCD one
// contiguous eighth of each layer's tiles. REMAP 2 gives it one contiguous
// eighth of all (tile, layer) pairs, the layers of a tile one after another:
// in a page-major pool they are adjacent, so the rows that an XCD reads (and
// the page regions it writes) close together in time lie close together in
// memory. Measured on MI355X against REMAP 1, 16 layers pool to pool: 40,000
// tokens of 8 x 64 fp8 into head-major pages 261 -> 255 us, token-major 232 ->
// 224, bf16 head-major 449 -> 432; 649-byte rows 136 -> 131; 4 layers of
// 100,000 x 4 KiB 608 -> 593. Launches of up to SGLKV_JOINT_TILES workgroups,
// about two rounds of the chip, keep the layers apart (768: 12.1 us, 12.6 so);
// so do the pack and the unpack (1 to 2 % either way).
#define SGLKV_JOINT_TILES 4096u
template <int REMAP>
__device__ __forceinline__ void sglkv_place(uint32_t *tile, uint32_t *layer) {
    const uint32_t g = gridDim.x, layers = gridDim.y;
    *tile = blockIdx.x;
    *layer = blockIdx.y;
    if (!REMAP) return;
    const uint64_t all = static_cast<uint64_t>(g) * layers;
    const bool joint = REMAP == 2 && layers > 1 && all > SGLKV_JOINT_TILES && all >> 32 == 0;
    const uint32_t n = joint ? static_cast<uint32_t>(all) : g, b = joint ? blockIdx.y * g + blockIdx.x : blockIdx.x;
    const uint32_t q = n / SGLKV_XCDS, r = n % SGLKV_XCDS, x = b % SGLKV_XCDS;
    const uint32_t at = x * q + (x < r ? x : r) + b / SGLKV_XCDS;
    *tile = joint ? at / layers : at;
    if (joint) *layer = at % layers;
}

template <int VB> struct sglkv_vec;
template <> struct sglkv_vec<16> { typedef sglkv_v4u type; };
template <> struct sglkv_vec<8> { typedef sglkv_v2u type; };
template <> struct sglkv_vec<4> { typedef uint32_t type; };
template <> struct sglkv_vec<2> { typedef uint16_t type; };
template <> struct sglkv_vec<1> { typedef uint8_t type; };

// Byte offsets (relative to plane[0] and plane[1]) of `row`'s tensor rows
// in a POOL side: page * page stride + pos * pos_mult[t], or
// SGLKV_INVALID_OFFSET for both after flagging a slot outside the pool. The
// host guarantees slot_count < 2^32, so the page split runs in 32 bits.
__device__ __forceinline__ void sglkv_pool_row(const sglkv_side &s, uint32_t row, uint32_t *flag,
                                               uint32_t *host_flag, uint64_t *off0, uint64_t *off1) {
    const uint64_t slot = s.slots[row];
    if (slot >= s.slot_count) {
        // (A plain store to the host word: the only bit that a copy raises, and
        // an atomic on host memory would need the host link's support.)
        if (host_flag)
            __hip_atomic_store(host_flag, SGLKV_FLAG_SLOT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        else
            atomicOr(flag, SGLKV_FLAG_SLOT);
        *off0 = *off1 = SGLKV_INVALID_OFFSET;
        return;
    }
    const uint32_t sl = static_cast<uint32_t>(slot);
    const uint32_t page = sl / s.page_size;
    const uint32_t pos = sl - page * s.page_size;
    const uint64_t base = static_cast<uint64_t>(page) * s.stride[0];
    *off0 = base + static_cast<uint64_t>(pos) * s.pos_mult[0];
    *off1 = base + static_cast<uint64_t>(pos) * s.pos_mult[1];
}

// Stages the tile's pool-row offsets in LDS (s_src[t][i], s_dst[t][i]:
// tensor t's row of tile row i) and returns whether the tile is "clean":
// every one of its rows exists and resolved to a valid slot.
template <uint32_t SK, uint32_t DK>
__device__ __forceinline__ bool sglkv_stage_tile(const sglkv_side &src, const sglkv_side &dst, uint32_t *flag,
                                                 uint32_t *host_flag, uint64_t row0, uint32_t tile, uint32_t rows, uint64_t *s_src0,
                                                 uint64_t *s_src1, uint64_t *s_dst0, uint64_t *s_dst1) {
    const uint32_t nthreads = blockDim.x * blockDim.y;
    const uint32_t tid = threadIdx.y * blockDim.x + threadIdx.x;
    // 64-bit: the last tile may reach past 2^32 rows.
    int bad = row0 + tile > rows;
    if (SK == SGLKV_SIDE_POOL || DK == SGLKV_SIDE_POOL) {
        for (uint32_t i = tid; i < tile; i += nthreads) {
            const uint64_t r = row0 + i;
            if (r < rows) {
                if (SK == SGLKV_SIDE_POOL) {
                    sglkv_pool_row(src, static_cast<uint32_t>(r), flag, host_flag, &s_src0[i], &s_src1[i]);
                    bad |= s_src0[i] == SGLKV_INVALID_OFFSET;
                }
                if (DK == SGLKV_SIDE_POOL) {
                    sglkv_pool_row(dst, static_cast<uint32_t>(r), flag, host_flag, &s_dst0[i], &s_dst1[i]);
                    bad |= s_dst0[i] == SGLKV_INVALID_OFFSET;
                }
            }
        }
    }
    return !__syncthreads_or(bad);
}

// Per-layer quantisation scales ride along bit-exactly (workgroup 0 of each layer).
__device__ __forceinline__ void sglkv_copy_scales(const float *src, float *dst, uint32_t count) {
    const uint32_t tid = threadIdx.y * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && tid < count) {
        const uint32_t i = blockIdx.y * count + tid;
        reinterpret_cast<uint32_t *>(dst)[i] = reinterpret_cast<const uint32_t *>(src)[i];
    }
}

template <int VB, uint32_t SK, uint32_t DK, int NT, int REMAP>
__device__ __forceinline__ void sglkv_copy_rows(const sglkv_copy_params &p) {
    typedef typename sglkv_vec<VB>::type V;
    constexpr uint32_t RU = SGLKV_ROWS_PER_THREAD;
    __shared__ uint64_t s_src[2][SGLKV_MAX_TILE_ROWS];
    __shared__ uint64_t s_dst[2][SGLKV_MAX_TILE_ROWS];

    const uint32_t tile = p.tile_rows;
    uint32_t at, layer;
    sglkv_place<REMAP>(&at, &layer);
    const uint64_t row0 = static_cast<uint64_t>(at) * tile;

    // Clean tiles (all but the last tile, unless a slot is bad) copy without
    // per-row predicates, so the compiler can pipeline the stores behind the
    // loads instead of draining the memory counter at every branch.
    const bool clean = sglkv_stage_tile<SK, DK>(p.src, p.dst, p.flag, p.host_flag, row0, tile, p.rows, s_src[0], s_src[1],
                                                s_dst[0], s_dst[1]);
    sglkv_copy_scales(p.scale_src, p.scale_dst, p.scale_count);

    // Thread (tx, ty): vector tx of rows ty + k * blockDim.y. Head-major
    // pages with head chunks of under a cache line (line_rows = 128 / chunk
    // bytes > 1) hold line_rows consecutive positions of a head chunk in one
    // line. There the lanes are regrouped so that each run of line_rows *
    // chunk-vectors lanes moves one chunk of line_rows consecutive rows:
    // the line is then written (or read) whole by one wave, not in pieces
    // by the waves of separate rows.
    uint32_t tx = threadIdx.x, ty = threadIdx.y;
    if (p.line_rows > 1) {
        const uint32_t g = p.line_rows, cv = p.vpc[0], span = g * blockDim.x;
        const uint32_t tid = threadIdx.y * blockDim.x + threadIdx.x, j = tid % span;
        tx = (j / (g * cv)) * cv + j % cv;
        ty = (tid / span) * g + (j / cv) % g;
    }

    for (uint32_t j = tx; j < p.vpr; j += blockDim.x) {
        // Select rather than index the kernel-argument arrays: a dynamic
        // index would copy the struct to scratch.
        const uint32_t t = j >= p.vpt;
        const uint32_t jt = t ? j - p.vpt : j;
        const uint32_t vpc = t ? p.vpc[1] : p.vpc[0];
        const uint32_t h = jt / vpc;
        const uint32_t jc = jt - h * vpc;
        const uint64_t src_plane =
            (t ? p.src.plane[1] : p.src.plane[0]) + static_cast<uint64_t>(layer) * p.src.layer_stride;
        const uint64_t dst_plane =
            (t ? p.dst.plane[1] : p.dst.plane[0]) + static_cast<uint64_t>(layer) * p.dst.layer_stride;
        const uint64_t src_stride = t ? p.src.stride[1] : p.src.stride[0];
        const uint64_t dst_stride = t ? p.dst.stride[1] : p.dst.stride[0];
        const uint64_t *so_t = s_src[t];
        const uint64_t *do_t = s_dst[t];
        sglkv_gsrc *sb = reinterpret_cast<sglkv_gsrc *>(
            src_plane + static_cast<uint64_t>(h) * (t ? p.src.head_stride[1] : p.src.head_stride[0]) +
            static_cast<uint64_t>(jc) * VB);
        sglkv_gdst *db = reinterpret_cast<sglkv_gdst *>(
            dst_plane + static_cast<uint64_t>(h) * (t ? p.dst.head_stride[1] : p.dst.head_stride[0]) +
            static_cast<uint64_t>(jc) * VB);

        typedef __attribute__((address_space(1))) const V gload_t;
        typedef __attribute__((address_space(1))) V gstore_t;
        V buf[RU];
        if (clean) {
#pragma unroll
            for (uint32_t k = 0; k < RU; ++k) {
                const uint32_t i = ty + k * blockDim.y;
                const uint64_t so = SK == SGLKV_SIDE_POOL ? so_t[i] : (row0 + i) * src_stride;
                buf[k] = sglkv_load<V, NT>(reinterpret_cast<gload_t *>(sb + so));
            }
#pragma unroll
            for (uint32_t k = 0; k < RU; ++k) {
                const uint32_t i = ty + k * blockDim.y;
                const uint64_t dof = DK == SGLKV_SIDE_POOL ? do_t[i] : (row0 + i) * dst_stride;
                sglkv_store<V, NT>(reinterpret_cast<gstore_t *>(db + dof), buf[k]);
            }
            continue;
        }
        // Ragged or faulty tile (the last tile, or a bad slot): row by row,
        // kept rolled so that it does not inflate the register allocation of
        // the clean path above.
#pragma unroll 1
        for (uint32_t k = 0; k < RU; ++k) {
            const uint32_t i = ty + k * blockDim.y;
            const uint64_t r = row0 + i;
            if (r >= p.rows) break;
            const uint64_t so = SK == SGLKV_SIDE_POOL ? so_t[i] : r * src_stride;
            const uint64_t dof = DK == SGLKV_SIDE_POOL ? do_t[i] : r * dst_stride;
            if (so == SGLKV_INVALID_OFFSET || dof == SGLKV_INVALID_OFFSET) continue;
            sglkv_store<V, NT>(reinterpret_cast<gstore_t *>(db + dof),
                               sglkv_load<V, NT>(reinterpret_cast<gload_t *>(sb + so)));
        }
    }
}

// Dword `i` (0..3) of a 16-byte vector held in four registers, by selects
// (a dynamically indexed register array would live in scratch).
__device__ __forceinline__ uint32_t sglkv_dword(uint32_t i, uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
    return i == 0 ? w0 : i == 1 ? w1 : i == 2 ? w2 : w3;
}

// Writes bytes [lo, hi) of the 16-byte vector (w0..w3) whose aligned
// destination is `d`, as naturally aligned 8, 4, 2 and 1-byte stores.
template <int NT>
__device__ __forceinline__ void sglkv_store_partial(uint64_t d, uint32_t lo, uint32_t hi, uint32_t w0,
                                                    uint32_t w1, uint32_t w2, uint32_t w3) {
    uint32_t pos = lo;
#pragma unroll 1
    while (pos < hi) {
        const uint32_t rem = hi - pos;
        const uint32_t a = sglkv_dword(pos >> 2, w0, w1, w2, w3);
        const uint32_t sh = 8u * (pos & 3u);
        if ((pos & 7u) == 0 && rem >= 8) {
            const sglkv_v2u v = {a, sglkv_dword((pos >> 2) + 1, w0, w1, w2, w3)};
            sglkv_store<sglkv_v2u, NT>(reinterpret_cast<__attribute__((address_space(1))) sglkv_v2u *>(d + pos), v);
            pos += 8;
        } else if ((pos & 3u) == 0 && rem >= 4) {
            sglkv_store<uint32_t, NT>(reinterpret_cast<__attribute__((address_space(1))) uint32_t *>(d + pos), a);
            pos += 4;
        } else if ((pos & 1u) == 0 && rem >= 2) {
            sglkv_store<uint16_t, NT>(reinterpret_cast<__attribute__((address_space(1))) uint16_t *>(d + pos),
                                      static_cast<uint16_t>(a >> sh));
            pos += 2;
        } else {
            sglkv_store<uint8_t, NT>(reinterpret_cast<__attribute__((address_space(1))) uint8_t *>(d + pos),
                                     static_cast<uint8_t>(a >> sh));
            pos += 1;
        }
    }
}

// The byte-realigning copy (sglkv_realign_params): every global access an
// aligned 16-byte vector, whatever the row width and stride. Thread x owns
// LDS vector x of each row (blockDim.x == vrow), thread y a row of each
// group of blockDim.y rows.
template <uint32_t SK, uint32_t DK, int NT, int REMAP>
__device__ __forceinline__ void sglkv_realign_rows(const sglkv_realign_params &p) {
    constexpr uint32_t RU = SGLKV_REALIGN_ROWS_PER_THREAD;
    extern __shared__ __attribute__((aligned(16))) uint8_t sglkv_realign_lds[];
    const uint32_t tile = p.tile_rows;
    uint64_t *s_src0 = reinterpret_cast<uint64_t *>(sglkv_realign_lds);
    uint64_t *s_src1 = s_src0 + tile;
    uint64_t *s_dst0 = s_src1 + tile;
    uint64_t *s_dst1 = s_dst0 + tile;
    // The tile's rows, after a 16-byte pad (16-byte aligned).
    uint8_t *data = reinterpret_cast<uint8_t *>(s_dst1 + tile) + 16;

    uint32_t at, layer;
    sglkv_place<REMAP>(&at, &layer);
    const uint64_t row0 = static_cast<uint64_t>(at) * tile;
    sglkv_stage_tile<SK, DK>(p.src, p.dst, p.flag, p.host_flag, row0, tile, p.rows, s_src0, s_src1, s_dst0, s_dst1);
    sglkv_copy_scales(p.scale_src, p.scale_dst, p.scale_count);

    const uint32_t j = threadIdx.x;
    const uint32_t t = j >= p.vt0;
    const uint32_t jt = t ? j - p.vt0 : j;
    const uint32_t seg = t ? p.seg[1] : p.seg[0];
    const uint32_t h = jt / seg;
    const uint32_t m = jt - h * seg;
    const uint32_t c = t ? p.chunk[1] : p.chunk[0];
    const uint64_t src_base = (t ? p.src.plane[1] : p.src.plane[0]) +
                              static_cast<uint64_t>(layer) * p.src.layer_stride +
                              static_cast<uint64_t>(h) * (t ? p.src.head_stride[1] : p.src.head_stride[0]);
    const uint64_t dst_base = (t ? p.dst.plane[1] : p.dst.plane[0]) +
                              static_cast<uint64_t>(layer) * p.dst.layer_stride +
                              static_cast<uint64_t>(h) * (t ? p.dst.head_stride[1] : p.dst.head_stride[0]);
    const uint64_t src_stride = t ? p.src.stride[1] : p.src.stride[0];
    const uint64_t dst_stride = t ? p.dst.stride[1] : p.dst.stride[0];
    const uint64_t *so_t = t ? s_src1 : s_src0;
    const uint64_t *do_t = t ? s_dst1 : s_dst0;
    // This thread's LDS vector within a row's area: segment start + m.
    uint8_t *lds_vec = data + 16u * j;
    const uint32_t seg_lds = (j - m) * 16u;
    const uint32_t row_lds = p.vrow * 16u;

    typedef __attribute__((address_space(1))) const sglkv_v4u gload_t;
    typedef __attribute__((address_space(1))) sglkv_v4u gstore_t;

    // Phase 1: the aligned source vectors covering each segment -> LDS.
    // Every lane loads (lanes with nothing to load read the context's zero
    // row), so no branch separates the loads and all RU stay in flight.
    sglkv_v4u buf[RU];
    uint32_t live = 0;
    const uint64_t zero = reinterpret_cast<uint64_t>(p.zero);
#pragma unroll
    for (uint32_t k = 0; k < RU; ++k) {
        const uint32_t i = threadIdx.y + k * blockDim.y;
        const uint64_t r = row0 + i;
        const uint64_t so = SK == SGLKV_SIDE_POOL ? so_t[i] : r * src_stride;
        const uint64_t dof = DK == SGLKV_SIDE_POOL ? do_t[i] : 0;
        const uint64_t s = src_base + so;
        const uint32_t sa = static_cast<uint32_t>(s & 15u);
        const bool ok = r < p.rows && so != SGLKV_INVALID_OFFSET && dof != SGLKV_INVALID_OFFSET &&
                        m < ((sa + c + 15u) >> 4);
        buf[k] = sglkv_load<sglkv_v4u, NT>(reinterpret_cast<gload_t *>(ok ? s - sa + 16u * m : zero));
        live |= static_cast<uint32_t>(ok) << k;
    }
#pragma unroll
    for (uint32_t k = 0; k < RU; ++k) {
        const uint32_t i = threadIdx.y + k * blockDim.y;
        if (live & (1u << k)) *reinterpret_cast<sglkv_v4u *>(lds_vec + i * row_lds) = buf[k];
    }
    __syncthreads();

    // Phase 2: each aligned destination vector of each segment, shifted out
    // of LDS by the source/destination misalignment.
    //
    // Where a segment ends part-way into a 16-byte vector and the next tile
    // row's same segment starts right there in the destination (consecutive
    // positions of a page, contiguous transfer rows), the two share that
    // vector: the next row's first lane writes it whole, with this row's
    // last bytes, and this row's last lane writes nothing. Only segments of
    // at least 16 bytes pair up (their first and last vectors are distinct
    // lanes); both lanes decide from the same three facts (the rows are in
    // this tile, both are valid, the destinations touch).
    const uint32_t tile_rows = p.tile_rows;
#pragma unroll 1
    for (uint32_t k = 0; k < RU; ++k) {
        const uint32_t i = threadIdx.y + k * blockDim.y;
        const uint64_t r = row0 + i;
        if (r >= p.rows) break;
        const uint64_t so = SK == SGLKV_SIDE_POOL ? so_t[i] : r * src_stride;
        const uint64_t dof = DK == SGLKV_SIDE_POOL ? do_t[i] : r * dst_stride;
        if (so == SGLKV_INVALID_OFFSET || dof == SGLKV_INVALID_OFFSET) continue;
        const uint32_t sa = static_cast<uint32_t>((src_base + so) & 15u);
        const uint64_t d = dst_base + dof;
        const uint32_t da = static_cast<uint32_t>(d & 15u);
        const uint32_t kvec = (da + c + 15u) >> 4;
        if (m >= kvec) continue;
        const uint32_t lo = m == 0 ? da : 0u;
        const uint32_t end = da + c - 16u * m;
        const uint32_t hi = end < 16u ? end : 16u;
        // The neighbouring tile row's destination offset, when that row
        // exists, is in this tile and is valid (else INVALID).
        bool merge_prev = false;
        if (c >= 16u && lo != 0 && i > 0) {
            const uint64_t pso = SK == SGLKV_SIDE_POOL ? so_t[i - 1] : (r - 1) * src_stride;
            const uint64_t pdo = DK == SGLKV_SIDE_POOL ? do_t[i - 1] : (r - 1) * dst_stride;
            merge_prev = pso != SGLKV_INVALID_OFFSET && pdo != SGLKV_INVALID_OFFSET && pdo + c == dof;
        }
        if (c >= 16u && hi < 16u && m + 1 == kvec && i + 1 < tile_rows && r + 1 < p.rows) {
            const uint64_t nso = SK == SGLKV_SIDE_POOL ? so_t[i + 1] : (r + 1) * src_stride;
            const uint64_t ndo = DK == SGLKV_SIDE_POOL ? do_t[i + 1] : (r + 1) * dst_stride;
            if (nso != SGLKV_INVALID_OFFSET && ndo != SGLKV_INVALID_OFFSET && dof + c == ndo) continue;
        }
        // Segment byte b sits at LDS offset seg + sa + b; destination vector
        // m starts at segment byte 16 m - da. The offset is at least
        // seg - 15, inside the front pad for the first segment.
        const int32_t o = static_cast<int32_t>(i * row_lds + seg_lds + sa + 16u * m) - static_cast<int32_t>(da);
        const uint32_t *wp = reinterpret_cast<const uint32_t *>(data + (o & ~3));
        const uint32_t sh = static_cast<uint32_t>(o) & 3u;
        const uint32_t x0 = wp[0], x1 = wp[1], x2 = wp[2], x3 = wp[3], x4 = wp[4];
        uint32_t w0 = __builtin_amdgcn_alignbyte(x1, x0, sh);
        uint32_t w1 = __builtin_amdgcn_alignbyte(x2, x1, sh);
        uint32_t w2 = __builtin_amdgcn_alignbyte(x3, x2, sh);
        uint32_t w3 = __builtin_amdgcn_alignbyte(x4, x3, sh);
        const uint64_t dv = d - da + 16u * m;
        if (merge_prev) {
            // Bytes [0, da) of the shared vector are the previous row's last
            // da bytes, in its own LDS area.
            const uint64_t pso = SK == SGLKV_SIDE_POOL ? so_t[i - 1] : (r - 1) * src_stride;
            const uint32_t psa = static_cast<uint32_t>((src_base + pso) & 15u);
            const uint32_t po = (i - 1) * row_lds + seg_lds + psa + c - da;
            const uint32_t *pp = reinterpret_cast<const uint32_t *>(data + (po & ~3u));
            const uint32_t psh = po & 3u;
            const uint32_t y0 = pp[0], y1 = pp[1], y2 = pp[2], y3 = pp[3], y4 = pp[4];
            const uint32_t v[4] = {__builtin_amdgcn_alignbyte(y1, y0, psh), __builtin_amdgcn_alignbyte(y2, y1, psh),
                                   __builtin_amdgcn_alignbyte(y3, y2, psh), __builtin_amdgcn_alignbyte(y4, y3, psh)};
            // byte j < da from the previous row
#define SGLKV_MERGE(J, W)                                                                  \
    {                                                                                      \
        const uint32_t nb = da > 4u * (J) ? (da - 4u * (J) >= 4u ? 4u : da - 4u * (J)) : 0u; \
        const uint32_t mask = nb == 4u ? 0xFFFFFFFFu : (1u << (8u * nb)) - 1u;            \
        W = (v[J] & mask) | (W & ~mask);                                                   \
    }
            SGLKV_MERGE(0, w0)
            SGLKV_MERGE(1, w1)
            SGLKV_MERGE(2, w2)
            SGLKV_MERGE(3, w3)
#undef SGLKV_MERGE
        }
        if ((lo == 0 || merge_prev) && hi == 16u) {
            const sglkv_v4u v = {w0, w1, w2, w3};
            sglkv_store<sglkv_v4u, NT>(reinterpret_cast<gstore_t *>(dv), v);
        } else {
            sglkv_store_partial<NT>(dv, merge_prev ? 0u : lo, hi, w0, w1, w2, w3);
        }
    }
}

// Occupancy hint: the waves per SIMD the register allocation must allow
// (0 = the compiler's choice).
#ifndef SGLKV_WAVES_PER_EU
#define SGLKV_WAVES_PER_EU 0
#endif
#if SGLKV_WAVES_PER_EU
#define SGLKV_OCCUPANCY __attribute__((amdgpu_waves_per_eu(SGLKV_WAVES_PER_EU)))
#else
#define SGLKV_OCCUPANCY
#endif

#define SGLKV_COPY_KERNEL(VB, SK, DK, NT, REMAP, NAME)                                 \
    extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) SGLKV_OCCUPANCY void  \
    NAME(const sglkv_copy_params p) {                                                  \
        sglkv_copy_rows<VB, SK, DK, NT, REMAP>(p);                                     \
    }

#define SGLKV_COPY_KERNELS(VB)                                                                 \
    SGLKV_COPY_KERNEL(VB, SGLKV_SIDE_POOL, SGLKV_SIDE_ROWS, SGLKV_PACK_NT, SGLKV_PACK_REMAP,   \
                      sglkv_copy_pool_rows_v##VB)                                               \
    SGLKV_COPY_KERNEL(VB, SGLKV_SIDE_ROWS, SGLKV_SIDE_POOL, SGLKV_UNPACK_NT,                   \
                      SGLKV_UNPACK_REMAP, sglkv_copy_rows_pool_v##VB)                           \
    SGLKV_COPY_KERNEL(VB, SGLKV_SIDE_POOL, SGLKV_SIDE_POOL, SGLKV_TRANSFER_NT,                 \
                      SGLKV_TRANSFER_REMAP, sglkv_copy_pool_pool_v##VB)

SGLKV_COPY_KERNELS(16)
SGLKV_COPY_KERNELS(8)
SGLKV_COPY_KERNELS(4)
SGLKV_COPY_KERNELS(2)
SGLKV_COPY_KERNELS(1)

#define SGLKV_REALIGN_KERNEL(SK, DK, NT, REMAP, NAME)                                  \
    extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void NAME(            \
        const sglkv_realign_params p) {                                                \
        sglkv_realign_rows<SK, DK, NT, REMAP>(p);                                      \
    }

// Cache policy and tile order of the realigning kernels (bits as above).
#ifndef SGLKV_REALIGN_PACK_NT
#define SGLKV_REALIGN_PACK_NT SGLKV_PACK_NT
#endif
#ifndef SGLKV_REALIGN_UNPACK_NT
#define SGLKV_REALIGN_UNPACK_NT SGLKV_UNPACK_NT
#endif
#ifndef SGLKV_REALIGN_TRANSFER_NT
#define SGLKV_REALIGN_TRANSFER_NT SGLKV_TRANSFER_NT
#endif
// The byte-realigning unpack (649-byte packed-MLA rows) keeps contiguous
// eighths: round-robin tiles measured 1.5 % slower there (67.6 -> 68.6 us).
#ifndef SGLKV_REALIGN_REMAP
#define SGLKV_REALIGN_REMAP 1
#endif

SGLKV_REALIGN_KERNEL(SGLKV_SIDE_POOL, SGLKV_SIDE_ROWS, SGLKV_REALIGN_PACK_NT, SGLKV_PACK_REMAP,
                     sglkv_realign_pool_rows)
SGLKV_REALIGN_KERNEL(SGLKV_SIDE_ROWS, SGLKV_SIDE_POOL, SGLKV_REALIGN_UNPACK_NT, SGLKV_REALIGN_REMAP,
                     sglkv_realign_rows_pool)
SGLKV_REALIGN_KERNEL(SGLKV_SIDE_POOL, SGLKV_SIDE_POOL, SGLKV_REALIGN_TRANSFER_NT, SGLKV_TRANSFER_REMAP,
                     sglkv_realign_pool_pool)

// Spans + page table -> one physical slot per row (the decode side's
// dst_kv_indices, crates/sglang-srt/src/pd_bootstrap.rs:416-494, expanded to
// the per-row slot map the copy kernels take). One thread per row; the
// row's span is the last one whose row_start <= row (binary search over
// spans sorted by row_start). Rows no span covers, and rows whose page
// entry is outside the table or the pool, get SGLKV_INVALID_OFFSET and
// raise SGLKV_FLAG_SPAN / SGLKV_FLAG_PAGE.
extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_resolve_spans(
    const sglkv_resolve_params p) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= p.rows) return;
    uint32_t lo = 0, hi = p.span_count;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (p.spans[mid].row_start <= r)
            lo = mid + 1;
        else
            hi = mid;
    }
    uint64_t out = SGLKV_INVALID_OFFSET;
    if (lo == 0) {
        atomicOr(p.flag, SGLKV_FLAG_SPAN);
    } else {
        const sglkv_span s = p.spans[lo - 1];
        const uint32_t k = r - s.row_start;
        if (k >= s.token_count) {
            atomicOr(p.flag, SGLKV_FLAG_SPAN);
        } else {
            const uint64_t token = static_cast<uint64_t>(s.token_offset) + k;
            const uint64_t index = static_cast<uint64_t>(s.page_table_start) + token / p.page_size;
            const int32_t page = index < p.page_table_len ? p.page_table[index] : -1;
            if (page < 0 || static_cast<uint64_t>(page) >= p.page_count) {
                atomicOr(p.flag, SGLKV_FLAG_PAGE);
            } else {
                out = static_cast<uint64_t>(page) * p.page_size + token % p.page_size;
            }
        }
    }
    p.out_slots[r] = out;
}

// Reads and clears error words in one atomic step each: out[i] <-
// *words[i], *words[i] <- 0. A bit raised by work still running elsewhere
// lands either in this read or in the word afterwards, never in neither.
extern "C" __global__ void sglkv_take_flags(uint32_t *word0, uint32_t *word1, uint32_t *out) {
    if (threadIdx.x == 0) out[0] = atomicExch(word0, 0u);
    if (threadIdx.x == 1) out[1] = atomicExch(word1, 0u);
}

// Synthetic-input generator for benchmarks and tests (no reference
// counterpart). Word i (8 bytes) of the buffer derives from
// z = splitmix64(seed + (i + 1) * 0x9E3779B97F4A7C15):
//   kind 0: the word is z itself (reproducible on the host for checks);
//   kind 1: four bf16 N(0, 1) values, Box-Muller on (z, splitmix64(z));
//   kind 2: four bf16 U(-1, 1) values from the four 16-bit fields of z.
// Grid-stride loop; every thread exits after its last word.
__device__ __forceinline__ uint64_t sglkv_mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ uint32_t sglkv_bf16_bits(float f) {
    const uint32_t bits = __float_as_uint(f);
    return (bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16;
}

extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_fill_synthetic(
    uint64_t *out, uint64_t words, uint64_t seed, uint32_t kind) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words;
         i += stride) {
        const uint64_t z = sglkv_mix64(seed + (i + 1) * 0x9E3779B97F4A7C15ull);
        uint64_t w = z;
        if (kind == 1) {
            const uint64_t z2 = sglkv_mix64(z);
            uint32_t v[4];
            for (int k = 0; k < 2; ++k) {
                const uint64_t src = k ? z2 : z;
                // 24-bit uniforms; u1 in (0, 1] keeps the logarithm finite.
                const float u1 = (static_cast<float>(src & 0xFFFFFFu) + 1.0f) * (1.0f / 16777216.0f);
                const float u2 = static_cast<float>((src >> 32) & 0xFFFFFFu) * (1.0f / 16777216.0f);
                const float r = sqrtf(-2.0f * logf(u1));
                float sn, cs;
                sincosf(6.283185307179586f * u2, &sn, &cs);
                v[2 * k] = sglkv_bf16_bits(r * cs);
                v[2 * k + 1] = sglkv_bf16_bits(r * sn);
            }
            w = v[0] | (static_cast<uint64_t>(v[1]) << 16) | (static_cast<uint64_t>(v[2]) << 32) |
                (static_cast<uint64_t>(v[3]) << 48);
        } else if (kind == 2) {
            w = 0;
            for (int k = 0; k < 4; ++k) {
                const float u = static_cast<float>((z >> (16 * k)) & 0xFFFFu) * (2.0f / 65536.0f) - 1.0f;
                w |= static_cast<uint64_t>(sglkv_bf16_bits(u)) << (16 * k);
            }
        }
        out[i] = w;
    }
}

// Executes PD page requests (the descriptors of
// build_mooncake_{,remote_}kv_transfer_requests,
// crates/sglang-srt/src/transfer.rs:1945-2090) as device copies: the
// page-for-page transfer between co-resident pools of equal page size and
// layout, in one launch instead of one transport write per page. Workgroup b
// copies chunk b % chunks (64 KiB) of request b / chunks. A request whose
// source or target range leaves its region, or that is longer than the
// launch's chunks cover, is skipped and raises SGLKV_FLAG_REQUEST.
__device__ __forceinline__ bool sglkv_inside(uint64_t addr, uint64_t len, uint64_t lo, uint64_t hi) {
    return lo <= hi && addr >= lo && len <= hi - lo && addr - lo <= (hi - lo) - len;
}

extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_copy_requests(
    const sglkv_request_params p) {
    const uint64_t b = blockIdx.x;
    const uint64_t index = b / p.chunks;
    const uint64_t chunk = b - index * p.chunks;
    if (index >= p.count) return;
    const sglkv_request r = p.requests[index];
    const uint64_t begin = chunk * SGLKV_REQUEST_CHUNK;
    const bool target_wraps = r.target_offset > ~0ull - p.target_base;
    const uint64_t target = p.target_base + r.target_offset;
    const bool ok = !target_wraps && r.length <= p.chunks * SGLKV_REQUEST_CHUNK &&
                    sglkv_inside(r.source, r.length, p.source_lo, p.source_hi) &&
                    sglkv_inside(target, r.length, p.target_lo, p.target_hi);
    if (!ok) {
        if (chunk == 0 && threadIdx.x == 0) atomicOr(p.flag, SGLKV_FLAG_REQUEST);
        return;
    }
    if (begin >= r.length) return;
    const uint64_t n = r.length - begin < SGLKV_REQUEST_CHUNK ? r.length - begin : SGLKV_REQUEST_CHUNK;
    sglkv_gsrc *s = reinterpret_cast<sglkv_gsrc *>(r.source + begin);
    sglkv_gdst *d = reinterpret_cast<sglkv_gdst *>(target + begin);
    if (((r.source | target | n) & 15u) == 0) {
        typedef __attribute__((address_space(1))) const sglkv_v4u gload_t;
        typedef __attribute__((address_space(1))) sglkv_v4u gstore_t;
        gload_t *sv = reinterpret_cast<gload_t *>(s);
        gstore_t *dv = reinterpret_cast<gstore_t *>(d);
        const uint32_t vecs = static_cast<uint32_t>(n / 16);
        constexpr uint32_t U = 8;
        for (uint32_t base = threadIdx.x; base < vecs; base += U * SGLKV_BLOCK_THREADS) {
            sglkv_v4u buf[U];
#pragma unroll
            for (uint32_t k = 0; k < U; ++k) {
                const uint32_t v = base + k * SGLKV_BLOCK_THREADS;
                if (v < vecs) buf[k] = __builtin_nontemporal_load(sv + v);
            }
#pragma unroll
            for (uint32_t k = 0; k < U; ++k) {
                const uint32_t v = base + k * SGLKV_BLOCK_THREADS;
                if (v < vecs) __builtin_nontemporal_store(buf[k], dv + v);
            }
        }
    } else {
        for (uint64_t i = threadIdx.x; i < n; i += SGLKV_BLOCK_THREADS) d[i] = s[i];
    }
}

// Forward-pass write of a layer's key and value rows (unequal widths) to
// their slots: one launch for both tensors of a layer, where the reference
// copies one (token, tensor) per cuMemcpyDtoD (cuda_mla.rs:256-271 through
// cuda_kv_cache.rs:258-294). A slot >= slot_count raises SGLKV_FLAG_SLOT
// and its row is skipped.
template <int W>
__device__ __forceinline__ void sglkv_pair_slots_body(const sglkv_pair_slots_params &p) {
    const uint64_t per_row = p.pieces[0] + p.pieces[1];
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * SGLKV_BLOCK_THREADS + threadIdx.x;
    const uint64_t row = t / per_row;
    if (row >= p.count) return;
    const uint64_t piece = t - row * per_row;
    const uint64_t slot = p.slots[row];
    if (slot >= p.slot_count) {
        if (piece == 0) atomicOr(p.flag, SGLKV_FLAG_SLOT);
        return;
    }
    const uint32_t k = piece < p.pieces[0] ? 0 : 1;
    const uint64_t pc = k ? piece - p.pieces[0] : piece;
    const uint64_t page = slot / p.page_size, pos = slot - page * p.page_size;
    uint8_t *dst = p.pool + page * p.page_stride + p.offset[k] + pos * p.row_bytes[k] + pc * W;
    const uint8_t *src = p.rows[k] + row * p.row_stride[k] + pc * W;
    if (W == 16)
        *reinterpret_cast<sglkv_v4u *>(dst) = *reinterpret_cast<const sglkv_v4u *>(src);
    else
        *dst = *src;
}

extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_write_pair_slots_v16(
    const sglkv_pair_slots_params p) {
    sglkv_pair_slots_body<16>(p);
}

extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_write_pair_slots_v1(
    const sglkv_pair_slots_params p) {
    sglkv_pair_slots_body<1>(p);
}

// Streaming ceilings of the device, for the benchmark's roofline context:
// a plain contiguous copy, read and write of 16-byte vectors, grid-stride,
// non-temporal, U vectors in flight per thread (the fastest settings of a
// sweep on MI355X). Not used by the transfer path itself.
template <int MODE, int U>
__device__ __forceinline__ void sglkv_stream_body(const sglkv_v4u *src, sglkv_v4u *dst, uint64_t vecs) {
    typedef __attribute__((address_space(1))) const sglkv_v4u gload_t;
    typedef __attribute__((address_space(1))) sglkv_v4u gstore_t;
    const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    sglkv_v4u acc = {0, 0, 0, 0};
    for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * blockDim.x * U + threadIdx.x; base < vecs;
         base += step * U) {
        sglkv_v4u b[U];
        if (MODE != 2) {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const uint64_t i = base + static_cast<uint64_t>(k) * blockDim.x;
                b[k] = __builtin_nontemporal_load(
                    reinterpret_cast<gload_t *>(reinterpret_cast<uint64_t>(src + (i < vecs ? i : 0))));
            }
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const uint64_t i = base + static_cast<uint64_t>(k) * blockDim.x;
            if (MODE == 1) {
                acc ^= b[k];
            } else if (i < vecs) {
                const sglkv_v4u v = MODE == 0 ? b[k] : sglkv_v4u{static_cast<uint32_t>(i), 1u, 2u, 3u};
                __builtin_nontemporal_store(v, reinterpret_cast<gstore_t *>(reinterpret_cast<uint64_t>(dst + i)));
            }
        }
    }
    // The read keeps its loads alive with a store no input can trigger in
    // practice (an XOR of every word equal to this constant).
    if (MODE == 1 && (acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x5D1E5EEDu) dst[0] = acc;
}

extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_stream_copy(const sglkv_v4u *src,
                                                                                   sglkv_v4u *dst,
                                                                                   uint64_t vecs) {
    sglkv_stream_body<0, 4>(src, dst, vecs);
}
extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_stream_read(const sglkv_v4u *src,
                                                                                   sglkv_v4u *dst,
                                                                                   uint64_t vecs) {
    sglkv_stream_body<1, 8>(src, dst, vecs);
}
extern "C" __global__ __launch_bounds__(SGLKV_BLOCK_THREADS) void sglkv_stream_write(const sglkv_v4u *src,
                                                                                    sglkv_v4u *dst,
                                                                                    uint64_t vecs) {
    sglkv_stream_body<2, 8>(src, dst, vecs);
}

// The paged-attention reader of the same pools shares this code object.
#include "kv_attention.hip"
#include "kv_attention_tile.hip"
