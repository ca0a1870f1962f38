// attention_mfma.h — the gfx950 MFMA kernels of the verify attention: one piece of a
// (sequence, kv head) item, and the LPT kernel that runs a plan's pieces.
//
// One 256-thread workgroup per piece. Its G*R query rows
// (G query heads of the kv head x R verify rows, row r = j*G + g) form NT tiles of
// 16 rows; K/V of each 64-token chunk (four 16-token blocks) are read ONCE with
// 16-byte loads and shared by every row — the GQA x draft reuse that turns
// a bandwidth-bound decode into MFMA-friendly tiles. The four waves stream
// disjoint chunks and merge their (max, sum, P.V) states through LDS at the end.
//
// Per chunk (64 tokens for 1-byte pools, 32 for 2-byte pools) and row tile, lane = 16*g4 + c:
//   S^T = K . Q^T   v_mfma_f32_16x16x32_{bf16,f16}: A = K (16 tokens x 32 dims),
//                   B = Q^T. Token m = 4q+i of tile s is (block q, offset 4s+i), so
//                   the output gives lane (g4, c) row c and block g4's offsets 4s..4s+3.
//   P = softmax     online, per row, base-2 exponent; row max via the row-swap permutes.
//   O += P . V      A = P (row c, k = 8*g4+i -> block g4 offset 8*pv+i),
//                   B = V from the dim-major V block: one 16-byte load gives a lane
//                   all 16 offsets of one dim.
// Head dims are permuted consistently in K and Q (lane group g4 owns dims
// 32*g4..32*g4+31), so every K load is a contiguous 32- or 64-byte run.
//
// A piece that is not the machine's whole life is bound by its chain of round trips: table
// entry, block ids, queries, first chunk, then per chunk, then the merges. So a piece's table
// entry holds everything its workgroup would look up (one load), its first block ids go out
// next, its queries before its K/V (loads retire in order: the Q staging waits for them alone),
// the four waves merge four dims per thread, and a split item's records are read two items and
// four records at a time in 8-byte loads. Against one lookup after the other and element-wise
// merges, per pass on one box: one fp8 sequence of 3000 keys over 16 layers 363.7 -> 311.9 µs,
// 16 f16 sequences at head_dim 64 62.6 -> 56.3, 80 bf16 rows per kv head 92.8 -> 74.9, the
// config-2 / 3 / 4 shapes 132.1 -> 127.2 / 239.4 -> 236.0 / 121.1 -> 113.9.
//
// Pool types: BF16 (bf16 MFMA; P split into bf16 hi+lo for two MFMAs so the
// probabilities keep ~16 bits), F16 (f16 MFMA), FP8-E4M3 and INT8 (decoded in
// registers to exact f16 values: E4M3 by the gfx950 pk_f16_fp8 conversion, int8
// via the 0x6400 magic; the per-head / per-block scales are applied to the fp32
// scores and to P, never to the operands).
#pragma once
#include "gg_common.h"
#include "attention_common.h"
#include "attention_rows.h"

#include <type_traits>

namespace gg {
#ifdef GG_TRACE
// Debug builds (-DGG_TRACE) only: the LPT kernel's per-workgroup timeline in wall-clock
// ticks (100 MHz): [4p] start, [4p+1] end, [4p+2] CU id (__smid) | 1 << 32 | XCC << 40 |
// keys << 44, [4p+3] when wave 0's first chunk had arrived. gg_debug_trace_ptr gives its device address.
static __device__ long long g_trace[65536 * 4];
#endif
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef unsigned __int128 u128;

constexpr int kBS = 16;
constexpr int kWaves = 4;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

template <gg_dtype_t DT>
struct PoolTraits;
template <>
struct PoolTraits<GG_DTYPE_BF16> {
    static constexpr int kEB = 2;
    static constexpr bool kBf16 = true;
};
template <>
struct PoolTraits<GG_DTYPE_F16> {
    static constexpr int kEB = 2;
    static constexpr bool kBf16 = false;
};
template <>
struct PoolTraits<GG_DTYPE_FP8_E4M3> {
    static constexpr int kEB = 1;
    static constexpr bool kBf16 = false;
};
template <>
struct PoolTraits<GG_DTYPE_INT8> {
    static constexpr int kEB = 1;
    static constexpr bool kBf16 = false;
};

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c, bool bf16) {
    if (bf16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Four E4M3 bytes -> four f16 (exact: every E4M3 value, subnormals included, is an
// f16 value), two hardware conversions (v_cvt_scalef32_pk_f16_fp8, scale 1).
__device__ __forceinline__ uint2 e4m3x4_to_f16x4(uint32_t w) {
    const f16x2 lo = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
    const f16x2 hi = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
    return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}
// Four int8 -> four f16 (exact): (0x6400 | (b ^ 0x80)) is 1024 + b + 128. Each half is
// one byte permute of (0x64646464 : w), bytes (b, 0x64, b', 0x64): five instructions per
// four bytes with the sign flip and the two subtractions (shift-and-mask takes ten).
__device__ __forceinline__ uint2 i8x4_to_f16x4(uint32_t w) {
    w ^= 0x80808080u;
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
    const f16x2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    f16x2 a = __builtin_bit_cast(f16x2, lo) - bias;
    f16x2 b = __builtin_bit_cast(f16x2, hi) - bias;
    return make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
}
// Eight 1-byte elements (two dwords) -> one 16-byte MFMA operand of f16.
template <gg_dtype_t DT>
__device__ __forceinline__ uint4 bytes8_to_f16x8(uint32_t w0, uint32_t w1) {
    uint2 a, b;
    if constexpr (DT == GG_DTYPE_FP8_E4M3) {
        a = e4m3x4_to_f16x4(w0);
        b = e4m3x4_to_f16x4(w1);
    } else {
        a = i8x4_to_f16x4(w0);
        b = i8x4_to_f16x4(w1);
    }
    return make_uint4(a.x, a.y, b.x, b.y);
}

// The same to bf16 (exact: E4M3 has 4 significant bits, int8 values 7 and a sign).
__device__ __forceinline__ uint2 e4m3x4_to_bf16x4(uint32_t w) {
    const bf16x2v lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false);
    const bf16x2v hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true);
    return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}
// (b ^ 0x80) is b + 128; the upper halves of the four f32 differences are the bf16 values.
__device__ __forceinline__ uint2 i8x4_to_bf16x4(uint32_t w) {
    w ^= 0x80808080u;
    uint32_t f[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = __float_as_uint((float)((w >> (8 * k)) & 0xffu) - 128.0f);
    return make_uint2(__builtin_amdgcn_perm(f[1], f[0], 0x07060302u), __builtin_amdgcn_perm(f[3], f[2], 0x07060302u));
}
template <gg_dtype_t DT>
__device__ __forceinline__ uint4 bytes8_to_bf16x8(uint32_t w0, uint32_t w1) {
    uint2 a, b;
    if constexpr (DT == GG_DTYPE_FP8_E4M3) {
        a = e4m3x4_to_bf16x4(w0);
        b = e4m3x4_to_bf16x4(w1);
    } else {
        a = i8x4_to_bf16x4(w0);
        b = i8x4_to_bf16x4(w1);
    }
    return make_uint4(a.x, a.y, b.x, b.y);
}

// Hardware round-to-nearest-even pair conversions (v_cvt_pk_f16_f32 / v_cvt_pk_bf16_f32)
// for probabilities, which are finite and non-negative.
__device__ __forceinline__ uint32_t cvt_pk_f16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2v));
}
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    return (uint32_t)f32_to_bf16_bits(a) | ((uint32_t)f32_to_bf16_bits(b) << 16);
}
__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
    return (uint32_t)f32_to_f16_bits(a) | ((uint32_t)f32_to_f16_bits(b) << 16);
}

__device__ __forceinline__ uint4 zero4() { return make_uint4(0, 0, 0, 0); }

// Max over lanes l, l^16, l^32, l^48 (the four 16-lane rows of the wave) with the gfx950
// row-swap permutes, which stay in the VALU instead of going through the LDS crossbar.
__device__ __forceinline__ float max_over_rows(float v) {
    const uint32_t u = __float_as_uint(v);
    const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    v = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
    const uint32_t w = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Zero the 1-byte elements at offsets >= nvalid of a 16-offset run.
__device__ __forceinline__ uint4 mask_bytes16(uint4 v, int nvalid) {
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int lo = 4 * k;
        uint32_t m;
        if (nvalid >= lo + 4) m = 0xFFFFFFFFu;
        else if (nvalid <= lo) m = 0u;
        else m = 0xFFFFFFFFu >> (8 * (lo + 4 - nvalid));
        w[k] &= m;
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}
// Zero the bytes at offsets >= nvalid of an 8-offset run starting at `first`.
__device__ __forceinline__ uint2 mask_bytes8(uint2 v, int nvalid, int first) {
    const int n = nvalid - first;
    const uint32_t m0 = n >= 4 ? 0xFFFFFFFFu : (n <= 0 ? 0u : 0xFFFFFFFFu >> (8 * (4 - n)));
    const uint32_t m1 = n >= 8 ? 0xFFFFFFFFu : (n <= 4 ? 0u : 0xFFFFFFFFu >> (8 * (8 - n)));
    return make_uint2(v.x & m0, v.y & m1);
}
// The same for an 8-offset run of 2-byte elements.
__device__ __forceinline__ uint4 mask_halves8(uint4 v, int nvalid, int first) {
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int o0 = first + 2 * k;
        uint32_t m = (o0 < nvalid ? 0x0000FFFFu : 0u) | (o0 + 1 < nvalid ? 0xFFFF0000u : 0u);
        w[k] &= m;
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// Chunk geometry. A chunk is kTok consecutive tokens (kTok/16 blocks). 1-byte pools use
// 64-token chunks, 2-byte pools 32-token chunks, so that in both cases a lane moves
// 256 bytes per chunk: K rows of kTok/16 tiles (32 dims each) and one 16-byte run
// of V offsets for each of the eight dim tiles.
//
// S tile s, M index m = 4q + i (q = m/4) holds token (block bq(q), offset ob(q) + 4s + i):
//   64-token chunks: bq(q) = q,    ob(q) = 0       (tiles s = 0..3)
//   32-token chunks: bq(q) = q/2,  ob(q) = 8*(q%2) (tiles s = 0..1)
// The MFMA output gives lane (g4, c16) row c16 and tokens (bq(g4), ob(g4) + 4s + i), so the
// lane's P values are the consecutive offsets ob(g4) .. ob(g4) + 4*NS - 1 of one block,
// which is exactly the A operand of P.V (k = 8*g4 + i' -> offset ob(g4) + 8*pv + i') and
// one contiguous run of the dim-major V block.
template <int kEB, int TOK, int HD>
struct Geo {
    static constexpr int kTok = TOK;
    static constexpr int kNS = kTok / 16;                 // S tiles (and blocks) per chunk
    static constexpr int kNPV = kNS / 2;                  // P.V MFMAs per dim tile
    static constexpr int kLaneDims = HD / 4;              // dims of a lane group's K rows
    static constexpr int kKVec = kLaneDims * kEB / 16;    // 16-byte loads per lane per K tile
    static constexpr int kMM = HD / 32;                   // S MFMAs per tile (8 dims of a lane group each)
    static constexpr int kDT = HD / 16;                   // 16-dim tiles of V and O
    static constexpr int kVBytes = 8 * kNPV * kEB;        // V bytes per lane per dim tile (16, or 8)
    using VReg = std::conditional_t<kVBytes == 16, uint4, uint2>;
    __device__ static __forceinline__ int bq(int q) { return kTok == 64 ? q : (q >> 1); }
    __device__ static __forceinline__ int ob(int q) { return kTok == 64 ? 0 : 8 * (q & 1); }
};

template <int kEB, int TOK, int HD>
struct ChunkRegs {
    using G = Geo<kEB, TOK, HD>;
    uint4 k[G::kNS][G::kKVec];
    typename G::VReg v[G::kDT];
    float ksc, vsc;  // INT8 pools: scales of the lane's V block, fetched with its V
};

// Block ids of one chunk as this lane uses them: k = the block of its K rows, v = the
// block of its V columns and P run (-1: no block: past the keys, past the piece, or an
// out-of-range table entry). The chunk's kNS ids are read with wave-uniform (scalar)
// loads, so waiting for them never waits on the vector loads of K/V in flight, and are
// narrowed to the lane's two right there, from registers: a later lane-dependent pick
// from a stored array would be folded into an indexed load and spill.
struct LaneBlocks {
    int k, v;
};

// What a piece needs to start streaming: its first chunk's K/V in flight and the block
// ids of its first two chunks (PieceIO::start).
template <gg_dtype_t DT, int TOK, int HD>
struct PieceIn {
    ChunkRegs<PoolTraits<DT>::kEB, TOK, HD> cur;
    LaneBlocks bl_cur, bl_next;
};

// A piece: tokens [t0, t_end) of sequence b against kv head kvh, written to partition
// slot `part` / record `rec` (both < 0: the output), for the query rows from row0 on; ctx
// and nrows are the sequence's keys and rows. Wave-uniform.
struct PieceDesc {
    int b, kvh, t0, t_end, part, rec, row0, ctx, nrows;
};

template <gg_dtype_t DT, int TOK, int HD>
struct PieceIO {
    static constexpr int kEB = PoolTraits<DT>::kEB;
    using Geom = Geo<kEB, TOK, HD>;
    static constexpr int kNS = Geom::kNS;
    static constexpr int kTok = Geom::kTok;

    // Block ids of chunk `ch` of the piece [t0, t_end), in two steps: fetch_blocks issues
    // the kNS table reads together (wave-uniform scalar loads; indices are clamped to the
    // row, so they wait for neither the piece bounds nor the context length), and
    // lane_blocks, called as late as possible, applies the bounds and narrows the ids
    // to the lane's two.
    struct RawBlocks {
        int q[kNS];
        int t;  // first token of the chunk
    };
    __device__ static __forceinline__ RawBlocks fetch_blocks(const AttnArgs& a, int b, int t0, int ch) {
        const int32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
        RawBlocks r;
        r.t = t0 + ch * kTok;
#pragma unroll
        for (int qb = 0; qb < kNS; ++qb) r.q[qb] = bt[min((r.t >> 4) + qb, a.max_blocks - 1)];
        return r;
    }
    __device__ static __forceinline__ LaneBlocks lane_blocks(const KVView& kv, const RawBlocks& r, int t_end) {
        int q[kNS];
#pragma unroll
        for (int qb = 0; qb < kNS; ++qb) {
            const int blk = r.q[qb];
            q[qb] = (r.t + 16 * qb < t_end && blk < kv.num_blocks) ? blk : -1;
        }
        const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
        const int ik = Geom::bq(c16 >> 2), iv = Geom::bq(g4);
        LaneBlocks l{q[0], q[0]};
#pragma unroll
        for (int qb = 1; qb < kNS; ++qb) {
            l.k = ik == qb ? q[qb] : l.k;
            l.v = iv == qb ? q[qb] : l.v;
        }
        return l;
    }
    // The block ids of the wave's first two chunks.
    struct FirstBlocks {
        RawBlocks r0, r1;
    };
    __device__ static __forceinline__ FirstBlocks first_blocks(const AttnArgs& a, const PieceDesc& d) {
        const int wave_u = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        return FirstBlocks{fetch_blocks(a, d.b, d.t0, wave_u), fetch_blocks(a, d.b, d.t0, wave_u + kWaves)};
    }
    // K rows: lane supplies M index c16 of every tile. Loads are unconditional (missing
    // blocks read block 0); such tokens are always masked in S.
    __device__ static __forceinline__ void load_k(const KVView& kv, const LaneBlocks bl, int kvh,
                                                  ChunkRegs<kEB, TOK, HD>& rg) {
        const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4, kq = c16 >> 2;
        const int blk = bl.k;
        const uint8_t* base =
            kv.kc + (((size_t)(blk < 0 ? 0 : blk) * kv.Hkv + kvh) * (size_t)(2 * kBS * HD) + Geom::kLaneDims * g4) * kEB;
#pragma unroll
        for (int s = 0; s < kNS; ++s) {
            const int off = Geom::ob(kq) + 4 * s + (c16 & 3);
#pragma unroll
            for (int v = 0; v < Geom::kKVec; ++v) rg.k[s][v] = *(const uint4*)(base + (size_t)off * HD * kEB + 16 * v);
        }
    }
    // V: lane owns block bq(g4), dim dt*16 + c16, offsets ob(g4) .. ob(g4)+16/kEB-1 (zeroed
    // later when the block is missing or partly past the keys).
    __device__ static __forceinline__ void load_v(const KVView& kv, const LaneBlocks bl, int kvh,
                                                  ChunkRegs<kEB, TOK, HD>& rg) {
        const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
        const int blk = bl.v;
        if constexpr (DT == GG_DTYPE_INT8) {
            // Scales first: the softmax that needs them then waits for nothing behind them.
            const size_t si = (size_t)(blk < 0 ? 0 : blk) * kv.Hkv + kvh;
            rg.ksc = f16_bits_to_f32(kv.k_blk_scale[si]);
            rg.vsc = f16_bits_to_f32(kv.v_blk_scale[si]);
        }
        const uint8_t* base =
            kv.vc + (((size_t)(blk < 0 ? 0 : blk) * kv.Hkv + kvh) * (size_t)(2 * kBS * HD) + Geom::ob(g4)) * kEB;
#pragma unroll
        for (int dt = 0; dt < Geom::kDT; ++dt) {
            const int d = dt * 16 + c16;
            rg.v[dt] = *(const typename Geom::VReg*)(base + (size_t)d * kBS * kEB);
        }
    }
    // Issue the first chunk of piece d (this wave's first chunk is chunk `wave`): its K rows and
    // V columns, from the block ids read ahead.
    __device__ static __forceinline__ void start(const KVView& kv, const PieceDesc& d, const FirstBlocks& fb,
                                                 PieceIn<DT, TOK, HD>& in) {
        in.bl_cur = lane_blocks(kv, fb.r0, d.t_end);
        in.bl_next = lane_blocks(kv, fb.r1, d.t_end);
        load_k(kv, in.bl_cur, d.kvh, in.cur);
        load_v(kv, in.bl_cur, d.kvh, in.cur);
    }
};

// Draft rows a piece appends itself (gg_verify_append_attention_planned on the MFMA path):
// rows [j0, j1) of its sequence (none when j0 == j1), and this thread's work item of them.
struct DeferredRows {
    AppendItem it;
    int j0, j1;
};
// Most draft rows a piece stages in LDS, at any head_dim: the V staging holds a dim's rows in 16
// bytes, eight of a 2-byte pool, and the patch shifts them as one 128-bit value.
constexpr int kAppRows = 8;
static_assert(kAppRows * 2 <= (int)sizeof(uint4), "a dim's staged rows are one 16-byte word");

// Start piece d (PieceIO::start) and, when the call carries draft rows (a.k_new), take
// care of the rows whose key positions lie in the piece. Every workgroup that reads a key
// position appends its row itself first, so none waits for another's stores: without row groups
// one piece alone holds the position; with them the piece of each group appends the same row, and
// the stores write equal bytes (but for PER_BLOCK INT8 pools, whose blocks would be re-scaled by
// each group: those calls append in a launch of their own). Chunks are multiples of 16 tokens, so
// a block's tokens (its K rows and its V columns) are all read by one chunk, and so by one wave.
//   - Rows inside the first chunks that `start` issues (short pieces), more rows than
//     kAppRows, no `ap` (the stream-K loop over pieces, whose registers are full), or a
//     PER_BLOCK INT8 pool (a block's new rows re-scale the whole block; a block lies in one
//     piece, since pieces are whole chunks): appended here by the whole workgroup, then a
//     barrier orders the stores before the piece's loads (within a workgroup a barrier
//     orders global stores before loads: same CU, write-through L1; for INT8, with
//     workgroup-scope release and acquire fences around it).
//   - Otherwise (the usual case: the rows are the item's last positions) their loads are
//     issued here, after `start`, one work item per thread. attn_piece converts them into
//     LDS before its Q-staging barrier; the wave that reads the chunk holding them patches
//     its registers from LDS (the pool still holds stale bytes there) and writes that
//     block's V tile back whole, and the K rows are stored after the loop. No load waits
//     behind these stores (gfx950 counts stores in vmcnt, so a store issued ahead of a
//     chunk's loads would hold up the wait for that chunk).
template <gg_dtype_t DT, int TOK, int HD>
__device__ __forceinline__ void start_piece(const AttnArgs& a, const KVView& kv, const PieceDesc& d,
                                            PieceIn<DT, TOK, HD>& in, DeferredRows* ap) {
    constexpr int kTok = TOK;
    // The in-register patch of the chunk holding the rows needs 16-byte V runs.
    constexpr bool kDefer = DT != GG_DTYPE_INT8 && Geo<PoolTraits<DT>::kEB, TOK, HD>::kVBytes == 16;
    if (ap) ap->j0 = ap->j1 = 0;
    const auto fb = PieceIO<DT, TOK, HD>::first_blocks(a, d);
    if (a.k_new) {
        const int ctx = d.ctx, nrows = d.nrows;
        const int first = ctx - nrows;
        const int j0 = max(0, d.t0 - first), j1 = min(nrows, d.t_end - first);
        if (nrows > 0 && nrows <= ctx && j0 < j1) {
            const int items = (j1 - j0) * (HD / 8);
            static_assert(kAppRows * (HD / 8) <= 256, "one work item per thread");
            if (kDefer && ap && j1 - j0 <= kAppRows && first + j0 >= d.t0 + kWaves * kTok) {
                PieceIO<DT, TOK, HD>::start(kv, d, fb, in);
                ap->j0 = j0;
                ap->j1 = j1;
                ap->it.live = false;
                if ((int)threadIdx.x < items) ap->it = append_load(a, kv, d.b, d.kvh, ctx, nrows, j0, threadIdx.x);
            } else if (DT == GG_DTYPE_INT8) {
                // Re-quantised rows and the block scales are read back by other waves:
                // workgroup-scope release and acquire around the barrier. (Issuing the
                // piece's first chunks before the block update, when the rows lie past
                // them, was slower: 121.4 -> 130.7 µs per call at config 4. Loads retire
                // in order, so the update's small loads waited behind the chunks.)
                append_item_rows(a, kv, d.b, d.kvh, j0, j1);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                __syncthreads();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                PieceIO<DT, TOK, HD>::start(kv, d, fb, in);
            } else {
                append_item_rows(a, kv, d.b, d.kvh, j0, j1);
                __syncthreads();
                PieceIO<DT, TOK, HD>::start(kv, d, fb, in);
            }
            return;
        }
    }
    PieceIO<DT, TOK, HD>::start(kv, d, fb, in);
}

// One piece of work: tokens [t0, t_end) of sequence b against kv head kvh. The result
// goes to the output (part < 0 && rec < 0), to partition slot `part` of the fixed
// partition grid, or to stream-K record `rec`. Must be reached by the whole workgroup.
//
// `in` holds the piece's first chunk, already issued (PieceIO::start).
// Partial records go through device-scope (agent) relaxed atomic stores and loads: they
// bypass the per-XCD caches' stale copies, so a workgroup on another XCD reads what was
// written. Ordering before the merge counter comes from waiting for the stores to
// complete (every record store of the workgroup) before the counter's atomic add.
__device__ __forceinline__ float2 load_agent2(const float* p) {
    const unsigned long long v =
        __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}
__device__ __forceinline__ void store_agent(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent2(float* p, float a, float b) {
    const unsigned long long v = ((unsigned long long)__float_as_uint(b) << 32) | __float_as_uint(a);
    __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Four consecutive output elements in one store. The struct types promise no more than the
// element's own alignment, whatever the caller's buffer has.
__device__ __forceinline__ void store4_from_f32(void* p, gg_dtype_t dt, size_t i, const float (&v)[4]) {
    struct __attribute__((packed, aligned(4))) F4 { float4 v; };
    struct __attribute__((packed, aligned(2))) H4 { uint2 v; };
    if (dt == GG_DTYPE_F32) {
        ((F4*)((float*)p + i))->v = make_float4(v[0], v[1], v[2], v[3]);
        return;
    }
    uint32_t h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) h[k] = dt == GG_DTYPE_BF16 ? f32_to_bf16_bits(v[k]) : f32_to_f16_bits(v[k]);
    ((H4*)((uint16_t*)p + i))->v = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
}

// The piece's queries of a 16-bit type, as the Q staging below takes them (f32 ones are read
// there). Issued before the piece's K and V: loads retire in order, so the staging then waits
// for these alone.
template <int NT>
struct QRaw {
    uint4 v[NT];
};
template <int NT, int HD>
__device__ __forceinline__ QRaw<NT> load_q16(const AttnArgs& a, const KVView& kv, const PieceDesc& d) {
    struct __attribute__((packed, aligned(2))) U4 { uint4 v; };
    QRaw<NT> q;
    if (a.q_dtype == GG_DTYPE_F32) {
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) q.v[rt] = make_uint4(0, 0, 0, 0);
        return q;
    }
    const int G = a.num_q_heads / kv.Hkv, rows = G * d.nrows - d.row0;
    const int c16 = threadIdx.x & 15, g4 = (threadIdx.x >> 4) & 3, mm = (threadIdx.x >> 6) & (HD / 32 - 1);
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
        const int r = rt * 16 + c16 < rows ? d.row0 + rt * 16 + c16 : 0;
        const size_t i = (((size_t)d.b * a.rows + r / G) * a.num_q_heads + (size_t)d.kvh * G + r % G) * HD +
                         HD / 4 * g4 + 8 * mm;
        q.v[rt] = ((const U4*)((const uint16_t*)a.q + i))->v;
    }
    return q;
}

// The piece by the per-row kernel's steps, a row per wave and round: for pieces whose sums are not
// finite (attn_piece). s_row: HD query elements and 64 probabilities per wave. rec_rows: rows per
// record.
template <gg_dtype_t DT, int HD>
__device__ __forceinline__ void piece_by_rows(const AttnArgs& a, const KVView& kv, const PieceDesc& d, int rows, int rec_rows,
                                              float* s_row) {
    constexpr int kDC = HD / 64;
    const int G = a.num_q_heads / kv.Hkv, lane = threadIdx.x & 63;
    float* s_q = s_row;
    float* s_p = s_row + HD;
    for (int r = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); r < rows; r += kWaves) {
        const int j = (d.row0 + r) / G, g = (d.row0 + r) % G;
        const size_t obase = (((size_t)d.b * a.rows + j) * a.num_q_heads + (size_t)d.kvh * G + g) * HD;
        __builtin_amdgcn_wave_barrier();  // (the previous row's reads)
#pragma unroll
        for (int c = 0; c < kDC; ++c) s_q[lane + 64 * c] = load_as_f32(a.q, a.q_dtype, obase + lane + 64 * c);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float acc[kDC], m, l;
        generic_partition<DT, kDC, true>(a, kv, d.b, d.kvh, d.t0, min(d.t_end, d.ctx - d.nrows + j + 1), s_q, s_p, nullptr,
                                         acc, m, l);
        if (d.rec < 0) {
            const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
            for (int c = 0; c < kDC; ++c) store_from_f32(a.out, a.out_dtype, obase + lane + 64 * c, acc[c] * inv);
        } else {
            const size_t q = (size_t)d.rec * rec_rows + r;
#pragma unroll
            for (int c = 0; c < kDC; ++c) store_agent(a.ws_acc + q * HD + lane + 64 * c, acc[c]);
            if (lane == 0) store_agent2(a.ws_ml + q * 2, m, l);
        }
    }
}

template <gg_dtype_t DT, int NT, int HD, bool FULL>
__device__ __forceinline__ void attn_piece(const AttnArgs& a, const KVView& kv, const PieceDesc pd,
                                           PieceIn<DT, attn_chunk_tokens(PoolTraits<DT>::kEB, NT), HD>& in,
                                           const DeferredRows* ap, const QRaw<NT>& q16) {
    const int b = pd.b, kvh = pd.kvh, t0 = pd.t0, t_end = pd.t_end, part = pd.part, rec = pd.rec;
    using T = PoolTraits<DT>;
    // FULL: FP8 and INT8 values go through bf16 as well, whose range holds any block scale.
    constexpr bool kIsBf16 = FULL ? DT != GG_DTYPE_F16 : T::kBf16;
    constexpr int kNP_parts = FULL ? 3 : kIsBf16 ? 2 : 1;  // operands P is split into
    constexpr int kEB = T::kEB;
    constexpr int TOK = attn_chunk_tokens(kEB, NT);
    using Geom = Geo<kEB, TOK, HD>;
    using Regs = ChunkRegs<kEB, TOK, HD>;
    constexpr int kTok = Geom::kTok;
    constexpr int kNS = Geom::kNS;

    const int ctx = pd.ctx;
    const int R = a.rows;
    const int nrows = pd.nrows;
    if (nrows <= 0 || nrows > ctx) return;
    const int Hq = a.num_q_heads;
    const int G = Hq / kv.Hkv;
    const int row0 = FULL ? pd.row0 : 0;
    const int nvalid_rows = G * nrows - row0;  // (may exceed the piece's 16 * NT rows)
    if (FULL && nvalid_rows <= 0) return;
    const bool final_out = part < 0 && rec < 0;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int c16 = lane & 15;
    const int g4 = lane >> 4;

    const int nchunks = (t_end - t0 + kTok - 1) / kTok;
    const int first_masked = ctx - nrows;  // tokens >= this are causally masked for some row

    // Score multiplier (log2 domain) and P.V multiplier per pool type.
    float sscale = a.scale * kLog2e;
    constexpr float kPUnits = 16384.f;  // FULL with f16 operands: P is multiplied in units of 2^-14
    float vfold = FULL && !kIsBf16 ? 1.f / kPUnits : 1.f;
    if constexpr (DT == GG_DTYPE_FP8_E4M3) {
        sscale *= kv.k_head_scale[kvh];
        vfold = kv.v_head_scale[kvh];
    }

    // Draft rows loaded by start_piece: converted into LDS here (the Q-staging barrier
    // below publishes them). The chunk that holds them reads stale pool bytes at their
    // positions; the wave that owns that chunk patches its registers from LDS (see the
    // loop), and the rows go to the pool after the loop, where nothing waits for the
    // stores (on gfx950 stores count in vmcnt, so a store ahead of a chunk's loads would
    // hold up the wait for that chunk). s_app keeps each work item (row, 8 dims) in the
    // pool's format; s_vt the same V values by dim: element r of s_vt[d] is row r's V[d].
    __shared__ AppendBytes s_app[kAppRows * (HD / 8)];
    __shared__ uint4 s_vt[HD];
    int app_lo = 0, app_hi = 0;  // their key positions [app_lo, app_hi)
    if constexpr (DT != GG_DTYPE_INT8) {
        if (ap) {
            const int j0 = __builtin_amdgcn_readfirstlane(ap->j0), j1 = __builtin_amdgcn_readfirstlane(ap->j1);
            if (j0 < j1) {
                const int i = threadIdx.x;
                if (i < (j1 - j0) * (HD / 8)) {
                    const AppendBytes o = append_encode(a, kv, ap->it);
                    s_app[i] = o;
                    const int r = i / (HD / 8), d0 = (i % (HD / 8)) * 8;
                    if constexpr (kEB == 1) {
                        const uint32_t u[2] = {o.v[0].x, o.v[0].y};
#pragma unroll
                        for (int e = 0; e < 8; ++e) ((uint8_t*)&s_vt[d0 + e])[r] = (uint8_t)(u[e >> 2] >> (8 * (e & 3)));
                    } else {
                        const uint32_t u[4] = {o.v[0].x, o.v[0].y, o.v[0].z, o.v[0].w};
#pragma unroll
                        for (int e = 0; e < 8; ++e) ((uint16_t*)&s_vt[d0 + e])[r] = (uint16_t)(u[e >> 1] >> (16 * (e & 1)));
                    }
                }
                app_lo = first_masked + j0;
                app_hi = first_masked + j1;
            }
        }
    }

    // ---- Q operands: B[k = 8*g4+i][n = c16] <- Q[row rt*16+c16][32*g4 + 8*mm + i] ----
    // Staged once per piece in LDS (wave w converts dim group mm = w for every row tile)
    // and read back per chunk one mm at a time, so only NT operands are live in the loop.
    // Loads are issued unconditionally (invalid rows read row 0 and are zeroed).
    // BF16 pools take Q as bf16 hi + lo (two S MFMAs) unless Q already is bf16, so f32
    // and f16 queries keep ~16 bits instead of bf16's 8.
    // FULL takes Q in as many parts as it needs to be exact: one when the operand type
    // holds the query type, two for f16 queries as bf16, three for f32.
    constexpr int kMM = Geom::kMM;
    constexpr int kQParts = FULL ? 3 : kIsBf16 ? 2 : 1;
    __shared__ uint4 s_q[kQParts][NT][kMM][64];  // [part][rt][mm][lane]
    const int qparts = FULL ? (a.q_dtype == GG_DTYPE_F32 ? 3 : kIsBf16 && a.q_dtype == GG_DTYPE_F16 ? 2 : 1)
                            : (kIsBf16 && a.q_dtype != GG_DTYPE_BF16 ? 2 : 1);
    int row_pos[NT];  // last visible key position of the lane's S row (c16)
    {
        const int mm = kMM == 4 ? wave : (wave & (kMM - 1));  // (head_dim 64: waves 2 and 3 stage again)
        size_t qb[NT];
        bool qvalid[NT];
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            const int r = rt * 16 + c16;
            qvalid[rt] = r < nvalid_rows;
            const int j = qvalid[rt] ? (row0 + r) / G : 0;
            const int g = qvalid[rt] ? (row0 + r) % G : 0;
            row_pos[rt] = qvalid[rt] ? first_masked + j : ctx - 1;
            qb[rt] = (((size_t)b * R + j) * Hq + (size_t)kvh * G + g) * HD + Geom::kLaneDims * g4 + 8 * mm;
        }
        if constexpr (FULL) {
            float f[NT][8];
            if (a.q_dtype == GG_DTYPE_F32) {
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) {
                    const float4 x = ((const float4*)((const float*)a.q + qb[rt]))[0];
                    const float4 y = ((const float4*)((const float*)a.q + qb[rt]))[1];
                    const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[rt][e] = qvalid[rt] ? v[e] : 0.f;
                }
            } else {
                const bool src_bf16 = a.q_dtype == GG_DTYPE_BF16;
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) {
                    const uint32_t w[4] = {q16.v[rt].x, q16.v[rt].y, q16.v[rt].z, q16.v[rt].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint16_t h = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
                        const float v = src_bf16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
                        f[rt][e] = qvalid[rt] ? v : 0.f;
                    }
                }
            }
            // f16 operands: the piece's queries are scaled by the power of two that brings the
            // largest |q| just below 2^15, up as well as down, and the score multiplier back.
            if (!kIsBf16 && a.q_dtype != GG_DTYPE_F16) {
                float lm = 0.f;
#pragma unroll
                for (int rt = 0; rt < NT; ++rt)
#pragma unroll
                    for (int e = 0; e < 8; ++e) lm = fmaxf(lm, fabsf(f[rt][e]));
                for (int o = 32; o > 0; o >>= 1) lm = fmaxf(lm, __shfl_xor(lm, o));
                __shared__ float s_fqmax[kWaves];
                if (lane == 0) s_fqmax[wave] = lm;
                __syncthreads();
                const float mx = fmaxf(fmaxf(s_fqmax[0], s_fqmax[1]), fmaxf(s_fqmax[2], s_fqmax[3]));
                int e2 = 0;
                (void)frexpf(mx, &e2);
                const int k = (mx > 0.f && mx <= 3.402823466e38f) ? (e2 - 15 < -100 ? -100 : e2 - 15) : 0;
                const float qs = ldexpf(1.f, -k);
                sscale = ldexpf(sscale, k);
#pragma unroll
                for (int rt = 0; rt < NT; ++rt)
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[rt][e] *= qs;
            }
            for (int part = 0; part < qparts; ++part) {
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) {
                    uint32_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float &x = f[rt][2 * e], &y = f[rt][2 * e + 1];
                        if constexpr (kIsBf16) {
                            h[e] = pack_bf16x2(x, y);
                            x -= __uint_as_float(h[e] << 16);
                            y -= __uint_as_float(h[e] & 0xffff0000u);
                        } else {
                            h[e] = pack_f16x2(x, y);
                            x -= f16_bits_to_f32((uint16_t)h[e]);
                            y -= f16_bits_to_f32((uint16_t)(h[e] >> 16));
                        }
                    }
                    s_q[part][rt][mm][lane] = make_uint4(h[0], h[1], h[2], h[3]);
                }
            }
            // (Positive, whatever the head's scale and the queries' made of it: attn_mfma_scale.)
            sscale = fmaxf(sscale, 0x1p-126f);
            __syncthreads();
        } else {
        // One uniform dtype branch around all row tiles, so their loads issue together.
        uint4 op[NT];
        // Eight values -> MFMA operand (and, for a split, the operand of the remainder).
        auto pack8 = [&](const float* f, uint4& hi, uint4& lo) {
            if constexpr (kIsBf16) {
                uint32_t h[4], l[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    h[k] = pack_bf16x2(f[2 * k], f[2 * k + 1]);
                    l[k] = pack_bf16x2(f[2 * k] - __uint_as_float(h[k] << 16),
                                       f[2 * k + 1] - __uint_as_float(h[k] & 0xffff0000u));
                }
                hi = make_uint4(h[0], h[1], h[2], h[3]);
                lo = make_uint4(l[0], l[1], l[2], l[3]);
            } else {
                hi = make_uint4(pack_f16x2(f[0], f[1]), pack_f16x2(f[2], f[3]), pack_f16x2(f[4], f[5]),
                                pack_f16x2(f[6], f[7]));
                lo = zero4();
            }
        };
        uint4 opl[NT];
        // f16 operands (FP8 / INT8 / F16 pools) hold |q| < 65504. A bf16 or f32 query beyond
        // 2^15 is scaled by 2^-k for the piece (k from the rows' largest |q|) and the score
        // multiplier by 2^k: power-of-two scalings are exact, so in range nothing changes.
        constexpr bool kF16Op = !kIsBf16;
        __shared__ float s_qmax[4];
        auto piece_q_shift = [&](float local_max) -> int {
            for (int o = 32; o > 0; o >>= 1) local_max = fmaxf(local_max, __shfl_xor(local_max, o));
            if (lane == 0) s_qmax[wave] = local_max;
            __syncthreads();
            const float mx = fmaxf(fmaxf(s_qmax[0], s_qmax[1]), fmaxf(s_qmax[2], s_qmax[3]));
            int e = 0;
            (void)frexpf(mx, &e);  // mx = f * 2^e, f in [0.5, 1)
            return (mx == mx && mx <= 3.402823466e38f && e > 15) ? e - 15 : 0;
        };
        if (a.q_dtype == GG_DTYPE_F32) {
            float4 raw[NT][2];
#pragma unroll
            for (int rt = 0; rt < NT; ++rt)
#pragma unroll
                for (int h = 0; h < 2; ++h) raw[rt][h] = ((const float4*)((const float*)a.q + qb[rt]))[h];
            float qs = 1.f;
            if constexpr (kF16Op) {
                float lm = 0.f;
#pragma unroll
                for (int rt = 0; rt < NT; ++rt)
                    if (qvalid[rt])
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            lm = fmaxf(lm, fmaxf(fmaxf(fabsf(raw[rt][h].x), fabsf(raw[rt][h].y)),
                                                 fmaxf(fabsf(raw[rt][h].z), fabsf(raw[rt][h].w))));
                const int k = piece_q_shift(lm);
                qs = ldexpf(1.f, -k);
                sscale = ldexpf(sscale, k);
            }
#pragma unroll
            for (int rt = 0; rt < NT; ++rt) {
                const float f[8] = {raw[rt][0].x * qs, raw[rt][0].y * qs, raw[rt][0].z * qs, raw[rt][0].w * qs,
                                    raw[rt][1].x * qs, raw[rt][1].y * qs, raw[rt][1].z * qs, raw[rt][1].w * qs};
                pack8(f, op[rt], opl[rt]);
            }
        } else {
            const bool src_bf16 = a.q_dtype == GG_DTYPE_BF16;
#pragma unroll
            for (int rt = 0; rt < NT; ++rt) {
                op[rt] = q16.v[rt];
                opl[rt] = zero4();
            }
            // Convert when the Q type differs from the MFMA operand type.
            if (src_bf16 != kIsBf16) {
                float f[NT][8];
                float lm = 0.f;
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) {
                    const uint32_t w[4] = {op[rt].x, op[rt].y, op[rt].z, op[rt].w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint16_t lo = (uint16_t)w[k], hi = (uint16_t)(w[k] >> 16);
                        f[rt][2 * k] = src_bf16 ? bf16_bits_to_f32(lo) : f16_bits_to_f32(lo);
                        f[rt][2 * k + 1] = src_bf16 ? bf16_bits_to_f32(hi) : f16_bits_to_f32(hi);
                    }
                    if (qvalid[rt])
#pragma unroll
                        for (int k = 0; k < 8; ++k) lm = fmaxf(lm, fabsf(f[rt][k]));
                }
                if constexpr (kF16Op) {
                    const int k = piece_q_shift(lm);
                    if (k > 0) {
                        const float qs = ldexpf(1.f, -k);
#pragma unroll
                        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
                            for (int e = 0; e < 8; ++e) f[rt][e] *= qs;
                        sscale = ldexpf(sscale, k);
                    }
                }
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) pack8(f[rt], op[rt], opl[rt]);
            }
        }
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            s_q[0][rt][mm][lane] = qvalid[rt] ? op[rt] : zero4();
            if constexpr (kIsBf16) s_q[kQParts - 1][rt][mm][lane] = qvalid[rt] ? opl[rt] : zero4();
        }
        __syncthreads();
        }
    }

    f32x4 o[NT][Geom::kDT];
    float m_run[NT], l_run[NT];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
        m_run[rt] = -1e30f;
        l_run[rt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < Geom::kDT; ++dt) o[rt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    using IO = PieceIO<DT, TOK, HD>;

    Regs& cur = in.cur;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    // Block ids run two chunks ahead and are requested after the softmax: the LDS
    // reads of Q at the top of the next chunk wait on every outstanding scalar load,
    // and by then these have had the whole P.V stage to arrive.
    LaneBlocks& bl_cur = in.bl_cur;
    LaneBlocks& bl_next = in.bl_next;

    for (int ch = wave_u; ch < nchunks; ch += kWaves) {
        const int blk_v = bl_cur.v;
        const int tc = t0 + ch * kTok;
        const int tlane = tc + 16 * Geom::bq(g4) + Geom::ob(g4);  // first token of the lane's P run
        // Valid offsets of the lane's V block (offsets counted from the block start).
        const int nvalid_v = blk_v < 0 ? 0 : ctx - (tc + 16 * Geom::bq(g4));

        // (A missing block reads block 0's scales; its tokens are masked either way.) A K
        // scale of 0 (a block never written, or one whose rows are all zero, so every K
        // byte is 0) is taken as 1: the scores it scales are 0 either way, and masked
        // scores must stay -inf rather than become -inf * 0 = NaN.
        const float kblk_scale = DT == GG_DTYPE_INT8 ? (cur.ksc > 0.f ? cur.ksc : 1.f) : 1.f;
        const float vblk_scale = DT == GG_DTYPE_INT8 ? cur.vsc : 1.f;

        // Draft rows in this chunk: their K rows replace the stale pool bytes just read.
        const bool app_here = DT != GG_DTYPE_INT8 && app_lo < app_hi && tc < app_hi && tc + kTok > app_lo;
        if constexpr (DT != GG_DTYPE_INT8) {
            if (app_here) {
                const int kq = c16 >> 2;
#pragma unroll
                for (int s = 0; s < kNS; ++s) {
                    const int r = tc + 16 * Geom::bq(kq) + Geom::ob(kq) + 4 * s + (c16 & 3) - app_lo;
                    if (r >= 0 && r < app_hi - app_lo) {
#pragma unroll
                        for (int v = 0; v < Geom::kKVec; ++v) {
                            if constexpr (kEB == 1) {
                                const int g = Geom::kLaneDims / 8 * g4 + 2 * v;
                                const uint4 A = s_app[r * (HD / 8) + g].k[0], B = s_app[r * (HD / 8) + g + 1].k[0];
                                cur.k[s][v] = make_uint4(A.x, A.y, B.x, B.y);
                            } else {
                                cur.k[s][v] = s_app[r * (HD / 8) + Geom::kLaneDims / 8 * g4 + v].k[0];
                            }
                        }
                    }
                }
            }
        }

        // ---- S^T = K . Q^T for kTok tokens x all row tiles; each K tile decoded once ----
        // The Q index is opaque to the optimiser so that the LDS reads stay in the loop
        // instead of being hoisted into registers for the whole piece.
        // (Non-volatile and without a memory clobber, the asm leaves the block-table
        // loads free to stay scalar; the chunk index input keeps it inside the loop.)
        int qlane;
        asm("" : "=v"(qlane) : "0"(lane), "s"(ch));
        f32x4 sacc[NT][kNS];
#pragma unroll
        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
            for (int s = 0; s < kNS; ++s) sacc[rt][s] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto k_operand = [&](int s, int mm) -> uint4 {
            if constexpr (kEB == 2) {
                return cur.k[s][mm];
            } else {
                const uint4 r = cur.k[s][mm >> 1];
                if constexpr (kIsBf16) return (mm & 1) ? bytes8_to_bf16x8<DT>(r.z, r.w) : bytes8_to_bf16x8<DT>(r.x, r.y);
                else return (mm & 1) ? bytes8_to_f16x8<DT>(r.z, r.w) : bytes8_to_f16x8<DT>(r.x, r.y);
            }
        };
        auto s_part = [&](int part) {
#pragma unroll
            for (int mm = 0; mm < kMM; ++mm) {
                uint4 qop[NT];
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) qop[rt] = s_q[part][rt][mm][qlane];
#pragma unroll
                for (int s = 0; s < kNS; ++s) {
                    const uint4 kop = k_operand(s, mm);
#pragma unroll
                    for (int rt = 0; rt < NT; ++rt) sacc[rt][s] = mfma(kop, qop[rt], sacc[rt][s], kIsBf16);
                }
            }
        };
        s_part(0);
        if constexpr (kQParts > 1) {
            if (qparts > 1) s_part(1);
        }
        if constexpr (kQParts > 2) {
            if (qparts > 2) s_part(2);
        }
        // Next chunk's K rows stream in while this chunk finishes.
        IO::load_k(kv, bl_next, kvh, cur);
#ifdef GG_TRACE
        if (ch == wave_u && threadIdx.x == 0) g_trace[4 * blockIdx.x + 3] = wall_clock64();
#endif

        // ---- online softmax; P packed as MFMA A operands ----
        // Masked scores: causal (keys past the row's position, which covers keys past the
        // context) and every key of a missing block (its K was read from block 0). A
        // lane's scores all come from its V block, so a missing block masks whole lanes.
        const bool blk_missing = blk_v < 0;
        const bool need_mask = tc + kTok - 1 >= first_masked || __any(blk_missing);
        const float mult = DT == GG_DTYPE_INT8 ? sscale * kblk_scale : sscale;
        constexpr int kNP = 4 * kNS;  // P values per lane per row tile
        uint4 pop[NT][Geom::kNPV][kNP_parts];
        // One wave-uniform branch around all the masking, so that chunks with nothing to
        // mask (most of them) skip it instead of running it as selects.
        if (__builtin_expect(need_mask, 0)) {
#pragma unroll
            for (int rt = 0; rt < NT; ++rt)
#pragma unroll
                for (int s = 0; s < kNS; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        sacc[rt][s][i] = (!blk_missing && (tlane + 4 * s + i) <= row_pos[rt]) ? sacc[rt][s][i] : -INFINITY;
        }
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            // The multiplier is positive, so the scaled maximum is the maximum of the raw
            // scores times the lane's multiplier (rounding is monotonic); the scale then
            // folds into the exponent's FMA.
            float sc[kNP];
            float cmax = -INFINITY;
#pragma unroll
            for (int s = 0; s < kNS; ++s) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = sacc[rt][s][i];
                    sc[4 * s + i] = v;
                    cmax = fmaxf(cmax, v);
                }
            }
            cmax = max_over_rows(cmax * mult);
            const float m_new = fmaxf(m_run[rt], cmax);
            const float alpha = __builtin_amdgcn_exp2f(m_run[rt] - m_new);
            m_run[rt] = m_new;
            float psum = 0.f;
#pragma unroll
            for (int k = 0; k < kNP; ++k) {
                sc[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[k], mult, -m_new));
                psum += sc[k];
            }
            l_run[rt] = l_run[rt] * alpha + psum;
            // Rescale O rows (4*g4 + i) by their rows' alpha; skipped by the whole wave
            // when no row max moved (the common case once the running max has settled).
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float al = __shfl(alpha, 4 * g4 + i);
#pragma unroll
                    for (int dt = 0; dt < Geom::kDT; ++dt) o[rt][dt][i] *= al;
                }
            }
            if constexpr (DT == GG_DTYPE_INT8) {
#pragma unroll
                for (int k = 0; k < kNP; ++k) sc[k] *= vblk_scale;
            }
#pragma unroll
            for (int pv = 0; pv < Geom::kNPV; ++pv) {
                const float* pp = sc + 8 * pv;
                if constexpr (FULL) {
                    // P as hi + mid + lo: three bf16 parts hold all 24 bits, three f16 ones those
                    // above 2^-39 (in units of 2^-14 the smallest f16 is 2^-38).
                    float x[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) x[k] = kIsBf16 ? pp[k] : pp[k] * kPUnits;
#pragma unroll
                    for (int part = 0; part < kNP_parts; ++part) {
                        uint32_t h[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            if constexpr (kIsBf16) {
                                h[k] = cvt_pk_bf16(x[2 * k], x[2 * k + 1]);
                                x[2 * k] -= __uint_as_float(h[k] << 16);
                                x[2 * k + 1] -= __uint_as_float(h[k] & 0xffff0000u);
                            } else {
                                h[k] = cvt_pk_f16(x[2 * k], x[2 * k + 1]);
                                x[2 * k] -= f16_bits_to_f32((uint16_t)h[k]);
                                x[2 * k + 1] -= f16_bits_to_f32((uint16_t)(h[k] >> 16));
                            }
                        }
                        pop[rt][pv][part] = make_uint4(h[0], h[1], h[2], h[3]);
                    }
                } else if constexpr (kIsBf16) {
                    // P = hi + lo, both bf16, so the probabilities keep ~16 bits.
                    uint32_t hw[4], lw[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        hw[k] = cvt_pk_bf16(pp[2 * k], pp[2 * k + 1]);
                        const float h0 = __uint_as_float(hw[k] << 16), h1 = __uint_as_float(hw[k] & 0xffff0000u);
                        lw[k] = cvt_pk_bf16(pp[2 * k] - h0, pp[2 * k + 1] - h1);
                    }
                    pop[rt][pv][0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
                    pop[rt][pv][kIsBf16 ? 1 : 0] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
                } else {
                    pop[rt][pv][0] = make_uint4(cvt_pk_f16(pp[0], pp[1]), cvt_pk_f16(pp[2], pp[3]),
                                                cvt_pk_f16(pp[4], pp[5]), cvt_pk_f16(pp[6], pp[7]));
                }
            }
        }

        const typename IO::RawBlocks raw_after = IO::fetch_blocks(a, b, t0, ch + 2 * kWaves);

        // ---- O += P . V; each V dim tile decoded once for all row tiles ----
        // Draft rows in this chunk: their V columns replace the stale pool bytes. The lane's
        // run is offsets ob(g4) .. of its block, rows base + offset of the staged rows.
        // Lanes whose block holds draft rows then write their runs back to the pool: the
        // runs of a block cover its whole dim-major V tile, so these are full-line stores
        // (the draft rows alone would be 1- or 2-byte pieces of every line, each a partial
        // write to memory); the other offsets are written back with the bytes just read.
        if constexpr (DT != GG_DTYPE_INT8 && Geom::kVBytes == 16) {
            if (app_here) {
                const int blk0 = tc + 16 * Geom::bq(g4) - app_lo;  // staged row of the block's offset 0
                const int base = blk0 + Geom::ob(g4);
                const int nr = app_hi - app_lo;
                constexpr int kE = 8 * kEB;  // bits per element
                constexpr int kRun = 16 / kEB;  // elements per 16-byte run
                if (base < nr && base + kRun > 0) {
                    // Element o of the run takes staged row base + o.
                    const int lo_bits = (nr - (base > 0 ? base : 0)) * kE;
                    u128 mask = lo_bits >= 128 ? ~(u128)0 : (((u128)1 << lo_bits) - 1);
                    if (base < 0) mask <<= (-base) * kE;
#pragma unroll
                    for (int dt = 0; dt < Geom::kDT; ++dt) {
                        const uint4 sv = s_vt[dt * 16 + c16];
                        u128 nv = ((u128)sv.w << 96) | ((u128)sv.z << 64) | ((u128)sv.y << 32) | sv.x;
                        if (kEB == 1) nv &= ((u128)1 << (8 * kAppRows)) - 1;  // (staged rows of one byte)
                        nv = base < 0 ? nv << ((-base) * kE) : nv >> (base * kE);
                        const uint4 c = cur.v[dt];
                        u128 cv = ((u128)c.w << 96) | ((u128)c.z << 64) | ((u128)c.y << 32) | c.x;
                        cv = (cv & ~mask) | (nv & mask);
                        cur.v[dt] = make_uint4((uint32_t)cv, (uint32_t)(cv >> 32), (uint32_t)(cv >> 64),
                                               (uint32_t)(cv >> 96));
                    }
                }
                if (blk_v >= 0 && blk0 < nr && blk0 + kBS > 0) {
                    uint8_t* vbase = const_cast<uint8_t*>(kv.vc) +
                                     (((size_t)blk_v * kv.Hkv + kvh) * (size_t)(2 * kBS * HD) + Geom::ob(g4)) * kEB;
#pragma unroll
                    for (int dt = 0; dt < Geom::kDT; ++dt) *(uint4*)(vbase + (size_t)(dt * 16 + c16) * kBS * kEB) = cur.v[dt];
                }
            }
        }
        if (nvalid_v < kBS) {
#pragma unroll
            for (int dt = 0; dt < Geom::kDT; ++dt) {
                if constexpr (kEB == 2) cur.v[dt] = mask_halves8(cur.v[dt], nvalid_v, Geom::ob(g4));
                else if constexpr (Geom::kVBytes == 16) cur.v[dt] = mask_bytes16(cur.v[dt], nvalid_v);
                else cur.v[dt] = mask_bytes8(cur.v[dt], nvalid_v, Geom::ob(g4));
            }
        }
#pragma unroll
        for (int dt = 0; dt < Geom::kDT; ++dt) {
#pragma unroll
            for (int pv = 0; pv < Geom::kNPV; ++pv) {
                uint4 vop;
                if constexpr (kEB == 2) {
                    vop = cur.v[dt];
                } else if constexpr (Geom::kVBytes == 16) {
                    const uint4 r = cur.v[dt];
                    if constexpr (kIsBf16) vop = pv ? bytes8_to_bf16x8<DT>(r.z, r.w) : bytes8_to_bf16x8<DT>(r.x, r.y);
                    else vop = pv ? bytes8_to_f16x8<DT>(r.z, r.w) : bytes8_to_f16x8<DT>(r.x, r.y);
                } else if constexpr (kIsBf16) {
                    vop = bytes8_to_bf16x8<DT>(cur.v[dt].x, cur.v[dt].y);
                } else {
                    vop = bytes8_to_f16x8<DT>(cur.v[dt].x, cur.v[dt].y);
                }
#pragma unroll
                for (int rt = 0; rt < NT; ++rt) {
#pragma unroll
                    for (int part = 0; part < kNP_parts; ++part)
                        o[rt][dt] = mfma(pop[rt][pv][part], vop, o[rt][dt], kIsBf16);
                }
            }
        }
        // Next chunk's V columns.
        IO::load_v(kv, bl_next, kvh, cur);
        bl_cur = bl_next;
        bl_next = IO::lane_blocks(kv, raw_after, t_end);
    }

    // The draft rows' K to the pool (their V went back with the patched runs), now that no
    // load of this piece waits behind the stores.
    if constexpr (DT != GG_DTYPE_INT8) {
        if (app_lo < app_hi)
            for (int i = threadIdx.x; i < (app_hi - app_lo) * (HD / 8); i += blockDim.x) append_write_k(kv, s_app[i]);
    }

    // ---- merge the four waves' states through LDS ----
    __shared__ float s_m[kWaves][64];
    __shared__ float s_l[kWaves][64];
    __shared__ __align__(16) float s_o[kWaves][16][HD + 4];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
        float lt = l_run[rt];
        lt += __shfl_xor(lt, 16);
        lt += __shfl_xor(lt, 32);
        if (g4 == 0) {
            s_m[wave][rt * 16 + c16] = m_run[rt];
            s_l[wave][rt * 16 + c16] = lt;
        }
    }
    __shared__ int s_bad[FULL ? kWaves : 1];
    if constexpr (FULL) {
        // A NaN or infinity among the queries, keys or values reaches rows that it should not
        // touch: a hidden key's P is 0, and 0 times it is NaN; the parts of P give infinities of
        // both signs; an infinite query sets the scale of the piece's other queries. Each leaves a
        // sum that is not finite, and the piece is then computed row by row.
        float z = 0.f;
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            z = __builtin_fmaf(l_run[rt], 0.f, z);
#pragma unroll
            for (int dt = 0; dt < Geom::kDT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) z = __builtin_fmaf(o[rt][dt][i], 0.f, z);
        }
        const bool any = __any(z != 0.f);
        if (lane == 0) s_bad[wave] = any;
    }
    __syncthreads();
    if constexpr (FULL) {
        if (__builtin_expect(s_bad[0] | s_bad[1] | s_bad[2] | s_bad[3], 0)) {
            piece_by_rows<DT, HD>(a, kv, pd, min(nvalid_rows, 16 * NT), 16 * NT, &s_o[wave][0][0]);
            return;
        }
    }

    const size_t zbase = (size_t)b * R;
    for (int rt = 0; rt < NT; ++rt) {
        // Each wave writes its O rows scaled to the common row max.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = 4 * g4 + i;
            const int r = rt * 16 + rr;
            float mx = s_m[0][r];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, s_m[w][r]);
            const float f = __builtin_amdgcn_exp2f(s_m[wave][r] - mx);
#pragma unroll
            for (int dt = 0; dt < Geom::kDT; ++dt) s_o[wave][rr][dt * 16 + c16] = o[rt][dt][i] * f;
        }
        __syncthreads();
        // 256 threads sum the four waves' copies, four dims of a row at a time.
#pragma unroll
        for (int e = threadIdx.x; e < 16 * (HD / 4); e += 256) {
            const int rr = e / (HD / 4), d = 4 * (e % (HD / 4));
            const int r = rt * 16 + rr;
            if (r >= nvalid_rows) continue;
            float mx = s_m[0][r];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, s_m[w][r]);
            float L = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                L += s_l[w][r] * __builtin_amdgcn_exp2f(s_m[w][r] - mx);
                const float4 v = *(const float4*)&s_o[w][rr][d];
                acc[0] += v.x;
                acc[1] += v.y;
                acc[2] += v.z;
                acc[3] += v.w;
            }
            const int j = (row0 + r) / G, g = (row0 + r) % G;
            const size_t z = zbase + j;
            const int h = kvh * G + g;
            if (final_out) {
                float val[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) val[k] = L > 0.f ? acc[k] * vfold / L : 0.f;
                store4_from_f32(a.out, a.out_dtype, (z * Hq + h) * HD + d, val);
            } else {
                const size_t pidx = rec >= 0 ? (size_t)rec * (size_t)(FULL ? 16 * NT : G * R) + (size_t)r
                                             : (z * Hq + h) * a.max_parts + part;
                // Device-scope stores: they reach the point every XCD reads from, so the
                // last piece of an LPT item can merge the records in the same launch.
                store_agent2(a.ws_acc + pidx * HD + d, acc[0] * vfold, acc[1] * vfold);
                store_agent2(a.ws_acc + pidx * HD + d + 2, acc[2] * vfold, acc[3] * vfold);
                if (d == 0) store_agent2(a.ws_ml + pidx * 2, mx > -1e29f ? mx * kLn2 : -1e30f, L);
            }
        }
        __syncthreads();
    }
}

// Chunks of work of sequence b (0 when it has nothing to compute).
__device__ __forceinline__ int seq_chunks(const AttnArgs& a, int b, int tok) {
    const int ctx = seq_keys(a, b, kBS);
    const int nrows = seq_rows(a, b);
    if (nrows <= 0 || nrows > ctx) return 0;
    return (ctx + tok - 1) / tok;
}

// ---- LPT schedule: pieces of a few mean slot loads at most, longest first ----
//
// Items longer than T chunks (attention_common.h) are cut: while the items fill the slots,
// into pieces of T chunks and a shorter last piece; with fewer items, into equal pieces of at
// most T chunks. attn_lpt_plan_kernel orders the pieces by size,
// descending (ties: sequence, then piece, then kv head), and the main launch runs them in
// that order (with
// few items the first round pairs long and shorter pieces per CU, lpt_slot): dispatched in
// order, the longest pieces start first and the shortest fill the tail.
// The last piece of a split item to finish merges the item's partial records
// (lpt_merge_if_last), so the schedule is one launch. Its records are written and read
// with device-scope stores and loads; a device-scope fence instead would write back or
// invalidate a whole L2 here, which costs more than a separate merge launch.
//
// Plan layout (ints, in the workspace after the records), P = piece bound (lpt_pieces), B =
// sequences, H = heads (kv heads, times the row groups of a shape whose rows are cut):
//   [0 .. 15]                 unused
//   [16 + 8p ..]              piece p: sequence (-1 past the last piece), head | pieces of
//                             the item << 16, first token, end token, keys and rows of the
//                             sequence, the item's first record, piece j of the item: all a
//                             workgroup needs to start, in one load
//   [16 + 8P + b*H + h]       merge counter of (sequence b, head h)
// The records of split item (b, h) are first, first + H, ... in piece order, numbered by
// sequence; items of one piece have none.
__device__ __forceinline__ int* lpt_table(int* plan) { return plan + 16; }
// Workgroup of the piece of rank r. While the
// (sequence, kv head) items do not outnumber the S slots: over the first W = min(S,
// pieces) ranks, the groups of eight ranks in [H, W), H = W/2, are taken in reverse order,
// so workgroup w + H gets a rank near W - 1 - w. Dispatched round-robin, workgroups w and
// w + H land on one CU as its first two slots, which then hold a long and a shorter piece
// instead of two long ones. Measured, same box (with the ranks of [H, W) reversed one by
// one): config 2 (items = S/2) 73.3 -> 71.1 µs; over eight seeded config-3 layouts (items =
// S) the mean 127.2 -> 126.1 µs and the worst layout 136.8 -> 129.4 µs; config 5 (items =
// 2S) 128.3 -> 129.2 µs, so more items than slots keep the plain order.
// Reversing whole groups of eight keeps every workgroup's index congruent to its rank
// modulo 8, and workgroup w runs on XCD w mod 8. A sequence's kv-head items have
// consecutive ranks from a multiple of Hkv, so with Hkv = 8 item (b, h) runs on XCD
// (first rank of b + h) mod 8 = h mod 8 whether b's items are long or short, and two
// sequences that share prefix blocks read each shared block of a head on one XCD, the
// second read mostly from that XCD's L2. (Reversed one by one, a short sequence's head h
// ran on XCD 7 - h, and a shared block's second read went to another XCD's L2.) Config 3
// (20 % of the blocks shared by pairs of sequences), same box: attention reads 291,491 ->
// 282,994 KiB per call (FETCH_SIZE; 597.0 -> 579.6 MB, the unique pool bytes are 579.2 MB),
// 117.5 -> 116.9 µs per call; configs 2 and 5 unchanged.
__device__ __forceinline__ int lpt_slot(int r, int S, int total, bool pair) {
    const int W = min(S, total);
    const int H = W / 2;
    if (pair && r >= H && r < W) {
        const int q = r - H, G = (W - H) / 8;
        return q < 8 * G ? H + 8 * (G - 1 - q / 8) + (q & 7) : r;
    }
    return r;
}
// Merge counters, one per (sequence, kv head): pieces of a split item that have written
// their records. The plan clears them; the piece that merges an item clears its counter.
__device__ __forceinline__ int* lpt_count(int* plan, int pieces) { return plan + 16 + 8 * pieces; }

// The piece of a split item that finishes last merges the item's records: the online
// log-sum-exp over its pieces in piece order, as a merge launch of its own would. Each
// piece waits until its record stores have completed, then counts itself in the item's
// counter (a device-scope atomic, no fence: the records were written with device-scope
// stores, and the merging workgroup reads them with device-scope loads). No workgroup
// waits for another, so there is no spinning; the merge costs the last piece a read of
// the item's records.
// Ordering, on gfx950 (gg_kv_create refuses other devices): a device-scope relaxed store
// is issued with the system-coherent bit, so it is written through the XCD's L2 to the
// coherence point, and it counts in vmcnt until that write is acknowledged;
// `s_waitcnt vmcnt(0)` therefore returns only once every record store of the thread is
// visible at the coherence point. The barrier orders all threads' waits before thread 0's
// counter add, which is performed at the coherence point. The merging piece sees the final
// count in the add's return value and only then issues its record loads, which are
// device-scope (system-coherent bit: served from the coherence point, never from a stale
// line of its own XCD's L2). So every record load follows, in time, the completion of the
// record's store. The language-level way (a release add and an acquire read) writes back
// and invalidates the whole XCD L2 on this device and costs config 3 about 4 % (measured).
// h: the item's head (with row groups, group * kv heads + kv head); RW: rows per record;
// first: the item's first record, the others `heads` apart.
template <int HD>
__device__ __forceinline__ void lpt_merge_if_last(const AttnArgs& a, int Hkv, int heads, const PieceDesc& d, int h, int np,
                                                  int first, int RW) {
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's record stores are done
    __syncthreads();
    int* cnt = lpt_count(a.plan, lpt_pieces(a.sk_grid, a.num_seqs, heads)) + d.b * heads + h;
    if (threadIdx.x == 0)
        s_last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == np - 1;
    __syncthreads();
    if (!s_last) return;
    const int G = a.num_q_heads / Hkv;
    const int items = min(G * d.nrows - d.row0, RW) * (HD / 4);  // (row, 4 dims)
    // Two items per thread and up to four records per step, their loads issued together: the
    // merge is a chain of round trips to the coherence point.
    for (int e0 = threadIdx.x; e0 < items; e0 += 2 * blockDim.x) {
        const int e[2] = {e0, min(e0 + (int)blockDim.x, items - 1)};
        float M[2] = {-1e30f, -1e30f}, L[2] = {0.f, 0.f}, acc[2][4] = {};
        int jp = 0;
        auto merge = [&](auto n) {
            constexpr int N = decltype(n)::value;
            float2 ml[2][N], v[2][N][2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const size_t q = (size_t)(first + (jp + u) * heads) * RW + e[i] / (HD / 4);
                    const float* x = a.ws_acc + q * HD + 4 * (e[i] % (HD / 4));
                    ml[i][u] = load_agent2(a.ws_ml + q * 2);
                    v[i][u][0] = load_agent2(x);
                    v[i][u][1] = load_agent2(x + 2);
                }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const float mn = fmaxf(M[i], ml[i][u].x);
                    const float fo = __expf(M[i] - mn), fn = __expf(ml[i][u].x - mn);
                    M[i] = mn;
                    L[i] = L[i] * fo + ml[i][u].y * fn;
                    acc[i][0] = acc[i][0] * fo + v[i][u][0].x * fn;
                    acc[i][1] = acc[i][1] * fo + v[i][u][0].y * fn;
                    acc[i][2] = acc[i][2] * fo + v[i][u][1].x * fn;
                    acc[i][3] = acc[i][3] * fo + v[i][u][1].y * fn;
                }
            jp += N;
        };
        while (jp + 4 <= np) merge(std::integral_constant<int, 4>{});
        if (jp + 2 <= np) merge(std::integral_constant<int, 2>{});
        if (jp < np) merge(std::integral_constant<int, 1>{});
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (i == 1 && e0 + (int)blockDim.x >= items) break;
            const int r = d.row0 + e[i] / (HD / 4), d4 = 4 * (e[i] % (HD / 4));
            const float inv = L[i] > 0.f ? 1.f / L[i] : 0.f;
            const float o[4] = {acc[i][0] * inv, acc[i][1] * inv, acc[i][2] * inv, acc[i][3] * inv};
            store4_from_f32(a.out, a.out_dtype,
                            (((size_t)d.b * a.rows + r / G) * a.num_q_heads + (size_t)d.kvh * G + r % G) * HD + d4, o);
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next layer
}

// Workgroup p computes the piece at table entry p (exits past the last piece); the last
// piece of a split item to finish merges it.
template <gg_dtype_t DT, int NT, int HD, bool FULL>
__global__ void __launch_bounds__(256, attn_occupancy(PoolTraits<DT>::kEB, NT, HD)) attn_mfma_lpt_kernel(AttnArgs a, KVView kv) {
    const int p = blockIdx.x;
#ifdef GG_TRACE
    const long long tr_t0 = wall_clock64();
#endif
    // One load tells the workgroup everything about its piece.
    const int4 e = ((const int4*)lpt_table(a.plan))[2 * p], f = ((const int4*)lpt_table(a.plan))[2 * p + 1];
    if (e.x < 0) return;  // past the last piece
    const int h = e.y & 0xffff, np = e.y >> 16;
    const int heads = FULL ? kv.Hkv * a.row_groups : kv.Hkv;
    const int kvh = FULL ? h % kv.Hkv : h;
    const int row0 = FULL ? h / kv.Hkv * (16 * NT) : 0;
    const PieceDesc d{e.x, kvh, e.z, e.w, -1, np > 1 ? f.z + f.w * heads : -1, row0, f.x, f.y};
    PieceIn<DT, attn_chunk_tokens(PoolTraits<DT>::kEB, NT), HD> in;
    DeferredRows ap;
    const QRaw<NT> q16 = load_q16<NT, HD>(a, kv, d);
    start_piece(a, kv, d, in, &ap);
    attn_piece<DT, NT, HD, FULL>(a, kv, d, in, &ap, q16);
    if (np > 1 && (!FULL || a.num_q_heads / kv.Hkv * d.nrows > row0))
        lpt_merge_if_last<HD>(a, kv.Hkv, heads, d, h, np, f.z, FULL ? 16 * NT : a.num_q_heads / kv.Hkv * a.rows);
#ifdef GG_TRACE
    if (threadIdx.x == 0) {
        g_trace[4 * p + 0] = tr_t0;
        g_trace[4 * p + 1] = wall_clock64();
        // CU id, a valid bit, the XCC (hardware register XCC_ID) and the piece's key count
        const long long xcc = (long long)(__builtin_amdgcn_s_getreg(20 | (15 << 11)) & 0xf);
        g_trace[4 * p + 2] = (long long)__smid() | (1LL << 32) | (xcc << 40) | ((long long)(e.w - e.z) << 44);
    }
#endif
}

}  // namespace
}  // namespace gg
