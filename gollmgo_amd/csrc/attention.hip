// attention.hip — multi-query split-K paged attention for the verify rows.
//
// Semantics: textbook softmax attention per (sequence, draft row, query head),
// as the reference's v1 kernel defines it for one query
// (kernels/gollmgo_paged_attn.cu:38-119: GQA kv_head = h / (Hq/Hkv), scores
// q.k*scale, max-subtracted softmax, P.V) extended to R causal rows per sequence
// with the mask of naive_attention (kernels/gollmgo_ops.cu:178: key j is visible
// to row i iff position_j <= position_i). Long contexts are split into
// partitions whose (max, sum, unnormalised P.V) partials are merged with the
// log-sum-exp identity — the job of paged_attention_v2_{phase1,reduce}
// (kernels/gollmgo_paged_attn.cu:234-384), whose reduce is not followed because it
// normalises only in thread 0 and mixes partial strides.
//
// Phase-1 kernels:
//   - attention_mfma.hip: gfx950 MFMA path for head_dim 128, block_size 16,
//     BF16/F16/FP8/INT8 pools, G*R <= 64 rows per kv head;
//   - attention_full.hip: the same pieces for head_dim 64 and for more rows per kv head, at
//     the precision of the per-row kernel (automatic schedule, up to kLptMaxSeqs sequences, where
//     attn_rows_faster does not prefer the per-row kernel);
//   - attn_generic_kernel (here): any head_dim <= 1024 / block size / pool dtype,
//     one wave per (row, head, partition), scalar online softmax. Used for the
//     shapes the MFMA tiling does not cover (fp32 pools, other head_dims and block sizes), for
//     narrow tables and explicit partitions of attention_full.hip's shapes, and for scales that
//     the MFMA softmax does not take (attn_mfma_scale). Its partitions and the MFMA partition grid
//     share one partial format and one combine kernel.
#include <type_traits>

#include "gg_common.h"
#include "attention_common.h"
#include "attention_rows.h"

namespace gg {
namespace {

constexpr int kMaxDC = 16;  // head_dim <= 1024 -> up to 16 dims per lane

// Most partitions of a (row, head) that one workgroup takes, a wave each, merging them in LDS.
constexpr int kFuseParts = 8;

// kFused: workgroup (h, z) takes every partition of a (row, head), wave w partition w, and
// merges them through LDS in partition order (the combine kernel's sums); else workgroup
// (part, h, z) takes one and the combine kernel merges.
template <gg_dtype_t DT, int DC, bool kVRun, bool kFused>
__global__ void __launch_bounds__(kFused ? 64 * kFuseParts : 64) attn_generic_kernel(AttnArgs a, KVView kv) {
    const int wave = kFused ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    const int part = kFused ? wave : (int)blockIdx.x;
    const int h = blockIdx.y;
    const int z = blockIdx.z;  // b*R + j
    const int b = z / a.rows, j = z % a.rows;
    const int nrows = seq_rows(a, b);
    if (j >= nrows) return;
    const int ctx = seq_keys(a, b, kv.bs);
    if (ctx <= 0 || nrows > ctx) return;
    const int P = a.partition;
    const int nparts = (ctx + P - 1) / P;
    if (!kFused && part >= nparts) return;
    const int pos = ctx - nrows + j;
    const int t0 = part * P;
    const int t1 = min(t0 + P, pos + 1);
    const int kvh = h / (a.num_q_heads / kv.Hkv);
    const int lane = threadIdx.x & 63;
    const int D = kv.D;
    constexpr int kW = kFused ? kFuseParts : 1;
    __shared__ float s_q[64 * DC];
    __shared__ __align__(16) float s_p[kW][64];
    __shared__ size_t s_vrow[kVRun ? 1 : kW][kVRun ? 1 : 64];
    const size_t qbase = ((size_t)z * a.num_q_heads + h) * D;
    for (int d = threadIdx.x; d < D; d += blockDim.x) s_q[d] = load_as_f32(a.q, a.q_dtype, qbase + d);
    __syncthreads();
    float acc[DC], m, l;
    generic_partition<DT, DC, kVRun>(a, kv, b, kvh, t0, part < nparts ? t1 : t0, s_q, s_p[wave], s_vrow[kVRun ? 0 : wave],
                                     acc, m, l);
    if constexpr (kFused) {
        __shared__ float s_acc[kFuseParts][64 * DC];
        __shared__ float s_ml[kFuseParts][2];
        if (nparts > 1) {
#pragma unroll
            for (int c = 0; c < DC; ++c) s_acc[wave][lane + 64 * c] = acc[c];
            if (lane == 0) {
                s_ml[wave][0] = m;
                s_ml[wave][1] = l;
            }
            __syncthreads();
            float M = -1e30f, total = 0.f;
            for (int p = 0; p < nparts; ++p) M = fmaxf(M, s_ml[p][0]);
            for (int p = 0; p < nparts; ++p) total += __expf(s_ml[p][0] - M) * s_ml[p][1];
            const float inv = total > 0.f ? 1.0f / total : 0.f;
            for (int d = threadIdx.x; d < D; d += blockDim.x) {
                float o = 0.f;
                for (int p = 0; p < nparts; ++p) o += __expf(s_ml[p][0] - M) * s_acc[p][d];
                store_from_f32(a.out, a.out_dtype, qbase + d, o * inv);
            }
            return;
        }
        if (wave) return;
    }
    if (nparts == 1) {
        const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) store_from_f32(a.out, a.out_dtype, qbase + d, acc[c] * inv);
        }
        return;
    }
    if constexpr (!kFused) {
        const size_t pidx = ((size_t)z * a.num_q_heads + h) * a.max_parts + part;
        if (lane == 0) {
            a.ws_ml[pidx * 2 + 0] = m;
            a.ws_ml[pidx * 2 + 1] = l;
        }
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) a.ws_acc[pidx * D + d] = acc[c];
        }
    }
}

// Merge the partitions of one (row, head): out = sum_p e^{m_p-M} acc_p / sum_p e^{m_p-M} l_p.
__global__ void __launch_bounds__(128) attn_combine_kernel(AttnArgs a, int D) {
    const int h = blockIdx.x;
    const int z = blockIdx.y;
    const int b = z / a.rows, j = z % a.rows;
    const int nrows = seq_rows(a, b);
    if (j >= nrows) return;
    const int ctx = seq_keys(a, b, a.kv_bs);
    const int nparts = (ctx + a.partition - 1) / a.partition;
    if (nparts <= 1 || nrows > ctx) return;
    const size_t base = ((size_t)z * a.num_q_heads + h) * a.max_parts;
    __shared__ float wgt[512];
    __shared__ float inv_total;
    float M = -1e30f;
    for (int p = 0; p < nparts; ++p) M = fmaxf(M, a.ws_ml[(base + p) * 2]);
    // nparts <= max_parts; weights are staged in chunks of 512 partitions.
    float acc_local[8];
    const int DPT = (D + blockDim.x - 1) / blockDim.x;  // <= 8 for D <= 1024
    for (int c = 0; c < 8; ++c) acc_local[c] = 0.f;
    float total = 0.f;
    for (int p0 = 0; p0 < nparts; p0 += 512) {
        const int pn = min(512, nparts - p0);
        __syncthreads();
        for (int p = threadIdx.x; p < pn; p += blockDim.x)
            wgt[p] = __expf(a.ws_ml[(base + p0 + p) * 2] - M);
        __syncthreads();
        for (int p = 0; p < pn; ++p) total += wgt[p] * a.ws_ml[(base + p0 + p) * 2 + 1];
        for (int c = 0; c < DPT; ++c) {
            const int d = threadIdx.x + c * blockDim.x;
            if (d >= D) break;
            float s = 0.f;
            for (int p = 0; p < pn; ++p) s += wgt[p] * a.ws_acc[(base + p0 + p) * D + d];
            acc_local[c] += s;
        }
    }
    if (threadIdx.x == 0) inv_total = total > 0.f ? 1.0f / total : 0.f;
    __syncthreads();
    const size_t obase = ((size_t)z * a.num_q_heads + h) * D;
    for (int c = 0; c < DPT; ++c) {
        const int d = threadIdx.x + c * blockDim.x;
        if (d >= D) break;
        store_from_f32(a.out, a.out_dtype, obase + d, acc_local[c] * inv_total);
    }
}

// Standalone draft-KV append from the block tables: workgroup (item) = (b, kvh).
__global__ void __launch_bounds__(256) append_from_tables_kernel(AttnArgs a, KVView kv) {
    append_item_rows(a, kv, blockIdx.x / kv.Hkv, blockIdx.x % kv.Hkv);
}

}  // namespace

gg_status_t launch_append_from_tables(const AttnArgs& a, const KVView& kv, hipStream_t s) {
    append_from_tables_kernel<<<a.num_seqs * kv.Hkv, 256, 0, s>>>(a, kv);
    return check_hip(hipGetLastError(), "append launch");
}

int attn_generic_partition(const KV* kv, int num_seqs, int rows, int num_q_heads, int max_blocks) {
    // One wave per (row, head, partition): partitions of 64..512 keys, as many as
    // it takes to reach about 2048 waves (the kernel's time is the longest wave's
    // chain of 64-key tiles; the merge costs one small launch).
    const long long waves = (long long)num_seqs * rows * num_q_heads;
    const long long want = waves > 0 ? (2048 + waves - 1) / waves : 1;
    const long long keys = (long long)max_blocks * kv->block_size;
    long long part = (keys + want - 1) / want;
    part = (part + 63) / 64 * 64;
    part = part < 64 ? 64 : (part > 512 ? 512 : part);
    return (int)part;
}

AttnPlan attn_plan(const KV* kv, int num_seqs, int rows, int num_q_heads, int max_blocks,
                   int partition_tokens) {
    if (partition_tokens > 0) return {ATTN_SCHED_GRID, partition_tokens};
    const AttnShape sh = attn_shape(kv, rows, num_q_heads);
    // (2^18 heads over all sequences: a plan of a few MB.)
    if (sh.full && num_seqs <= kLptMaxSeqs && (long long)num_seqs * kv->num_kv_heads * sh.groups <= (1 << 18))
        return {ATTN_SCHED_LPT, 0};
    if (!attn_mfma_supported(kv, rows, num_q_heads)) {
        return {ATTN_SCHED_GRID, attn_generic_partition(kv, num_seqs, rows, num_q_heads, max_blocks)};
    }
    // Longest-first pieces (LPT: long items cut, dispatched longest first, split items merged
    // inside the launch) at every batch the plan kernel can rank. Few items too: against the
    // even stream-K split that served items below a quarter of the slots, per call with the
    // plan of its step: one fp8 sequence of 3000 keys 38 -> 22.5 µs, eight of 300-1500 keys 49 ->
    // 21.7 µs, two int8 sequences of 300 keys 60.5 -> 25.7 µs, eight int8 sequences of
    // 16k-32k keys 121.1 -> 121.1 (112 without the plan launch); planned and run in one call,
    // 34.3 -> 26.1 µs (one sequence), 45.6 -> 24.7 (eight), 137.0 -> 131.1 (eight long).
    // Past kLptMaxSeqs sequences: one workgroup per item, or stream-K where contexts are long.
    const long long max_keys = (long long)max_blocks * kv->block_size;
    const long long items = (long long)num_seqs * kv->num_kv_heads;
    const long long slots = (long long)device_cu_count() * attn_occupancy((int)dtype_bytes(kv->dtype), sh.nt, kv->head_dim);
    if (num_seqs <= kLptMaxSeqs) return {ATTN_SCHED_LPT, 0};
    if (items >= slots && max_keys <= kMfmaMaxPartition)
        return {ATTN_SCHED_GRID, (int)((max_keys + 63) / 64 * 64)};
    return {ATTN_SCHED_STREAMK, 0};
}

// Narrow tables at head_dim 64 or in row groups: the per-row kernel reads K/V once per query row,
// the MFMA kernels once per item but at the price of a piece's start, and a call that plans for
// itself runs the plan kernel first. Both are estimated in µs, at contexts of three quarters of
// the table's width, from 1128 shapes measured on one box (head_dim 64 and 128, 1 to 512 sequences,
// 1 to 512 query rows per kv head, F16, FP8 and INT8 pools; BF16 costs what F16 does). A call that
// plans for itself takes its faster kernel but for 14 shapes, where it loses 10 to 41 %. 256
// sequences of up to 32 keys, 32 heads of one row, INT8: 125.7 -> 10.8 µs, planned 92 -> 10.8; 64,
// 8 heads, BF16: 14.8 -> 5.3. Past 512 keys the per-row kernel needs more partitions than one
// workgroup merges, and loses except for one row per head.
bool attn_rows_faster(const KV* kv, int num_seqs, int rows, int num_q_heads, int max_blocks, bool plans) {
    const AttnShape sh = attn_shape(kv, rows, num_q_heads);
    const long long keys = (long long)max_blocks * kv->block_size;
    if (!sh.full || keys > 64 * kFuseParts) return false;
    const bool wide = kv->head_dim == 128, byte = dtype_bytes(kv->dtype) == 1;
    const double k = (double)keys, heads = (double)num_seqs * rows * num_q_heads;
    const double items = (double)num_seqs * kv->num_kv_heads * sh.groups;
    // The latency of one workgroup, and the throughput per query row and head.
    const double by_rows = (wide ? 5.3 + 0.01 * k : 4.5 + 0.005 * k) +
                           heads * 1e-3 * (wide ? 0.8 + (byte ? 0.024 : 0.035) * k : 0.5 + (byte ? 0.018 : 0.02) * k);
    // The latency of a piece, and the items past the resident ones.
    double by_pieces = (wide ? (byte ? 12.3 : 10.7) : (byte ? 6.8 : 6.3) + 2 * (sh.nt - 1)) + 0.005 * k +
                       (items > 512 ? (items - 512) * (wide ? (byte ? 0.022 : 0.019) : (byte ? 0.0108 : 0.0072)) : 0);
    // A planned call's pieces append the draft rows too; the per-row kernel has a launch for them.
    by_pieces += plans ? 4 + 0.07 * num_seqs + 0.0007 * items : -1;
    return by_rows < by_pieces;
}

size_t attn_workspace_bytes(const KV* kv, int num_seqs, int rows, int num_q_heads, int max_blocks,
                            int partition) {
    const int max_parts = (max_blocks * kv->block_size + partition - 1) / partition;
    if (max_parts <= 1) return 0;
    size_t n_ml = (size_t)num_seqs * rows * num_q_heads * max_parts * 2;
    n_ml = ((n_ml + 63) / 64) * 64;
    size_t n_acc = (size_t)num_seqs * rows * num_q_heads * max_parts * kv->head_dim;
    return (n_ml + n_acc) * sizeof(float);
}

gg_status_t launch_verify_attention(const AttnArgs& a, hipStream_t s) {
    const KV* kv = a.kv;
    KVView view = make_kv_view(kv, a.layer);
    const bool mfma = attn_mfma_scale(a.scale) &&
                      (a.sched != ATTN_SCHED_GRID
                           ? !attn_rows_faster(kv, a.num_seqs, a.rows, a.num_q_heads, a.max_blocks, !a.plan_ready)
                           : attn_mfma_supported(kv, a.rows, a.num_q_heads) && a.partition % 64 == 0 &&
                                 a.partition <= kMfmaMaxPartition);
    bool combine = true;  // (the partition grid's merge launch)
    AttnArgs m = a;
    if (!mfma && a.sched != ATTN_SCHED_GRID) {
        // A planned shape at another scale, or a narrow one: partitions that one workgroup merges,
        // which need none of the workspace. (The schedules' shapes have head_dim 64 or 128.)
        const long long keys = (long long)a.max_blocks * kv->block_size;
        m.sched = ATTN_SCHED_GRID;
        m.partition = (int)(((keys + kFuseParts - 1) / kFuseParts + 63) / 64 * 64);
        m.max_parts = (int)((keys + m.partition - 1) / m.partition);
    }
    // Draft rows of the call: the MFMA kernels append them piece by piece (start_piece); the
    // generic path takes a launch of its own first, and so do the row groups of an INT8 item: each
    // would re-quantise the block it appends to.
    if (a.k_new && (!mfma || (a.row_groups > 1 && kv->dtype == GG_DTYPE_INT8))) {
        const gg_status_t st = launch_append_from_tables(a, view, s);
        if (st != GG_OK) return st;
        m.k_new = nullptr;
    }
    if (mfma) {
        // Stream-K and LPT launch their own merge over their record layout.
        gg_status_t st = launch_attn_mfma(m, view, s);
        if (st != GG_OK) return st;
        if (a.sched != ATTN_SCHED_GRID) return check_hip(hipGetLastError(), "verify_attention launch");
    } else {
        // Dims per lane rounded up to 1, 2, 4, 8 or 16 (the excess lanes idle).
        const int dc = (kv->head_dim + 63) / 64;
        const int DC = dc <= 1 ? 1 : dc <= 2 ? 2 : dc <= 4 ? 4 : dc <= 8 ? 8 : 16;
        if (dc > kMaxDC) return fail(GG_ERR_INVALID, "attention: head_dim too large");
        // V by 16-byte runs: a block is whole runs, a tile of 64 keys whole blocks, and a lane's
        // runs of a tile fit its registers. Every partition of a row in one workgroup: few
        // partitions, few enough dims for the LDS they meet in.
        const bool vrun = kv->block_size * dtype_bytes(kv->dtype) % 16 == 0 && 64 % kv->block_size == 0 && DC <= 2;
        const bool fused = m.max_parts <= kFuseParts && DC <= 2;
        const dim3 grid(fused ? 1 : m.max_parts, m.num_q_heads, m.num_seqs * m.rows);
        const int threads = fused ? 64 * m.max_parts : 64;
        auto launch = [&](auto dt_tag) {
            constexpr gg_dtype_t DT = decltype(dt_tag)::value;
            auto small = [&](auto dc_tag) {
                constexpr int N = decltype(dc_tag)::value;
                if (vrun && fused) attn_generic_kernel<DT, N, true, true><<<grid, threads, 0, s>>>(m, view);
                else if (vrun) attn_generic_kernel<DT, N, true, false><<<grid, threads, 0, s>>>(m, view);
                else if (fused) attn_generic_kernel<DT, N, false, true><<<grid, threads, 0, s>>>(m, view);
                else attn_generic_kernel<DT, N, false, false><<<grid, threads, 0, s>>>(m, view);
            };
            switch (DC) {
                case 1: small(std::integral_constant<int, 1>{}); break;
                case 2: small(std::integral_constant<int, 2>{}); break;
                case 4: attn_generic_kernel<DT, 4, false, false><<<grid, threads, 0, s>>>(m, view); break;
                case 8: attn_generic_kernel<DT, 8, false, false><<<grid, threads, 0, s>>>(m, view); break;
                default: attn_generic_kernel<DT, 16, false, false><<<grid, threads, 0, s>>>(m, view); break;
            }
        };
        combine = !fused;
        switch (kv->dtype) {
            case GG_DTYPE_F32: launch(std::integral_constant<gg_dtype_t, GG_DTYPE_F32>{}); break;
            case GG_DTYPE_F16: launch(std::integral_constant<gg_dtype_t, GG_DTYPE_F16>{}); break;
            case GG_DTYPE_BF16: launch(std::integral_constant<gg_dtype_t, GG_DTYPE_BF16>{}); break;
            case GG_DTYPE_FP8_E4M3: launch(std::integral_constant<gg_dtype_t, GG_DTYPE_FP8_E4M3>{}); break;
            case GG_DTYPE_INT8: launch(std::integral_constant<gg_dtype_t, GG_DTYPE_INT8>{}); break;
            default: return fail(GG_ERR_INVALID, "attention: pool dtype");
        }
    }
    if (combine && m.max_parts > 1) {
        attn_combine_kernel<<<dim3(m.num_q_heads, m.num_seqs * m.rows), 128, 0, s>>>(m, kv->head_dim);
    }
    static_assert(kMaxDC == 16, "generic kernel instantiations cover head_dim <= 1024");
    return check_hip(hipGetLastError(), "verify_attention launch");
}

}  // namespace gg
