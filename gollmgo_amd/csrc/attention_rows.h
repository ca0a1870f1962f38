// attention_rows.h — one partition of one (row, head) of the verify attention by one wave, keys
// and dims in fp32: the phase-1 step of the per-row kernel, and of pieces of the MFMA kernels
// that are computed row by row (piece_by_rows).
#pragma once
#include "gg_common.h"
#include "attention_common.h"

namespace gg {
namespace {

// One pool element as f32 (raw, before its block / head scale), pool type fixed.
template <gg_dtype_t DT>
__device__ __forceinline__ float pool_elem(const uint8_t* base, size_t i) {
    if constexpr (DT == GG_DTYPE_F32) return ((const float*)base)[i];
    else if constexpr (DT == GG_DTYPE_F16) return f16_bits_to_f32(((const uint16_t*)base)[i]);
    else if constexpr (DT == GG_DTYPE_BF16) return bf16_bits_to_f32(((const uint16_t*)base)[i]);
    else if constexpr (DT == GG_DTYPE_FP8_E4M3) return fp8e4m3_to_f32(base[i]);
    else return (float)((const int8_t*)base)[i];
}

// The pool elements in 16 bytes, as f32.
template <gg_dtype_t DT>
struct Pool16 {
    static constexpr int kN = DT == GG_DTYPE_F32 ? 4 : (DT == GG_DTYPE_F16 || DT == GG_DTYPE_BF16) ? 8 : 16;
    __device__ static __forceinline__ void decode(const uint4 r, float (&f)[kN]) {
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int k = 0; k < kN; ++k) {
            if constexpr (DT == GG_DTYPE_F32) f[k] = __uint_as_float(w[k]);
            else if constexpr (DT == GG_DTYPE_F16) f[k] = f16_bits_to_f32((uint16_t)(w[k >> 1] >> (16 * (k & 1))));
            else if constexpr (DT == GG_DTYPE_BF16) f[k] = bf16_bits_to_f32((uint16_t)(w[k >> 1] >> (16 * (k & 1))));
            else if constexpr (DT == GG_DTYPE_FP8_E4M3)
                f[k] = (k & 3) == 0   ? fp8e4m3_to_f32<0>(w[k >> 2])
                       : (k & 3) == 1 ? fp8e4m3_to_f32<1>(w[k >> 2])
                       : (k & 3) == 2 ? fp8e4m3_to_f32<2>(w[k >> 2])
                                      : fp8e4m3_to_f32<3>(w[k >> 2]);
            else f[k] = (float)(int8_t)(uint8_t)(w[k >> 2] >> (8 * (k & 3)));
        }
    }
};

// One partition of one (row, head), by one wave: keys in tiles of 64, lane i scoring key i of
// the tile against the whole query (in LDS), one wave max and sum per tile, then P.V with each
// lane owning dims lane + 64c. A tile's K rows and V runs are all requested before its scores
// are needed, so a tile waits for one round trip to its block ids and one to its K and V. V
// comes in 16-byte runs of offsets where blocks are whole runs and tiles whole blocks
// (kVRun), by element elsewhere; the products are added in key order either way.
// Bound by those round trips: with four K vectors and sixteen V elements in flight (V at a
// line per lane and key) and the merge in a launch, 4 x 5 rows of 8 heads over 64-256 fp32 keys
// took 14.0 + 4.2 µs, now 8.8; per call on one box, four fp32 sequences of 100-700 keys at
// head_dim 128 64 -> 25 µs, eight bf16 ones at head_dim 96 132 -> 24.
template <gg_dtype_t DT, int DC, bool kVRun>
__device__ __forceinline__ void generic_partition(const AttnArgs& a, const KVView& kv, int b, int kvh, int t0, int t1,
                                                  const float* s_q, float* s_p, size_t* s_vrow, float (&acc)[DC], float& m,
                                                  float& l) {
    const int lane = threadIdx.x & 63;
    const int D = kv.D;
    const int32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
    const uint8_t* vc = kv.vc;
    constexpr int kN = Pool16<DT>::kN;
    constexpr int kRuns = 64 / kN;  // 16-byte V runs of a tile per dim
    m = -1e30f;
    l = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c) acc[c] = 0.f;
    for (int tb = t0; tb < t1; tb += 64) {
        const int t = tb + lane;
        const int ntile = min(64, t1 - tb);
        int blk = -1, off = 0;
        if (t < t1) {
            blk = bt[t / kv.bs];
            off = t % kv.bs;
            if (blk < 0 || blk >= kv.num_blocks) blk = -1;  // invalid table entry: key skipped
        }
        // (Skipped keys read block 0.)
        const size_t vrow = kv.tile0(max(blk, 0), kvh) + off;
        [[maybe_unused]] uint4 vr[kVRun ? DC : 1][kVRun ? kRuns : 1];
        if constexpr (kVRun) {
#pragma unroll
            for (int r = 0; r < kRuns; ++r) {
                const size_t base = ((size_t)__shfl((unsigned)(vrow >> 32), r * kN) << 32) | (unsigned)__shfl((unsigned)vrow, r * kN);
#pragma unroll
                for (int c = 0; c < DC; ++c) {
                    const int d = min(lane + 64 * c, D - 1);
                    // (A run past the tile reads its key 0's block: not used.)
                    vr[c][r] = *(const uint4*)(vc + (base + (size_t)d * kv.bs) * dtype_bytes(DT));
                }
            }
        }
        float sc = -INFINITY;
        if (blk >= 0) {
            // The lane's key row is contiguous: 16-byte loads when rows are whole
            // multiples of 16 bytes (pools are 256-byte aligned), else element loads.
            const uint8_t* krow = kv.kc + (kv.tile0(blk, kvh) + (size_t)off * D) * dtype_bytes(DT);
            float dot = 0.f;
            if (D % kN == 0) {
#pragma unroll(DT == GG_DTYPE_F32 ? 16 : 4)
                for (int v = 0; v < D / kN; ++v) {
                    float f[kN];
                    Pool16<DT>::decode(((const uint4*)krow)[v], f);
#pragma unroll
                    for (int e = 0; e < kN; ++e) dot += s_q[v * kN + e] * f[e];
                }
            } else {
#pragma unroll 16
                for (int d = 0; d < D; ++d) dot += s_q[d] * pool_elem<DT>(krow, d);
            }
            sc = dot * a.scale * kv.k_scale(blk, kvh);
        }
        float mt = sc;
        for (int o = 32; o > 0; o >>= 1) mt = fmaxf(mt, __shfl_xor(mt, o));
        const float m_new = fmaxf(m, mt);
        const float alpha = __expf(m - m_new);
        const float p = blk >= 0 ? __expf(sc - m_new) : 0.f;
        float ps = p;
        for (int o = 32; o > 0; o >>= 1) ps += __shfl_xor(ps, o);
        l = l * alpha + ps;
        m = m_new;
#pragma unroll
        for (int c = 0; c < DC; ++c) acc[c] *= alpha;
        // The tile's probabilities (and by element, V offsets) go through LDS, so the key loop
        // below has no cross-lane operations. (Masked and skipped keys have p = 0.)
        // One wave's own slots: its LDS operations complete in order.
        __builtin_amdgcn_wave_barrier();
        s_p[lane] = blk >= 0 ? p * kv.v_scale(blk, kvh) : 0.f;
        if constexpr (!kVRun) s_vrow[lane] = vrow;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (kVRun) {
#pragma unroll
            for (int r = 0; r < kRuns; ++r) {
                if (r * kN >= ntile) break;
                float pi[kN];
#pragma unroll
                for (int e = 0; e < kN; ++e) pi[e] = s_p[r * kN + e];
#pragma unroll
                for (int c = 0; c < DC; ++c) {
                    float f[kN];
                    Pool16<DT>::decode(vr[c][r], f);
#pragma unroll
                    for (int e = 0; e < kN; ++e) acc[c] += pi[e] * (r * kN + e < ntile ? f[e] : 0.f);
                }
            }
        } else {
#pragma unroll 16
            for (int i = 0; i < ntile; ++i) {
                const float pi = s_p[i];
                const size_t vr0 = s_vrow[i];
#pragma unroll
                for (int c = 0; c < DC; ++c) {
                    const int d = lane + 64 * c;
                    if (d < D) acc[c] += pi * pool_elem<DT>(vc, vr0 + (size_t)d * kv.bs);
                }
            }
        }
    }
}

}  // namespace
}  // namespace gg
