// attention_full.hip — the LPT attention kernels for head_dim 64, and for more than 64 query
// rows per kv head.
//
// The same pieces as attention_mfma.hip's (attention_mfma.h), at the precision of the per-row
// kernel that used to serve these shapes: queries in as many operand parts as they need to be
// exact, probabilities as three parts: bf16 ones (24 bits; FP8 and INT8 values are exact in bf16)
// or, for F16 pools, f16 ones in units of 2^-14. More than 16 * nt rows are cut into
// groups of row tiles, each an item of its own that reads the same K/V (from HBM once: the
// groups of a kv head run side by side).
//
// The per-row kernel read every K/V row once per query row and head: 4 FLOPs per element
// through L2, 1057 µs a call for 16 f16 sequences of 512-4096 keys at head_dim 64 (32 query
// heads on 8, five rows; 79 MB of K/V) and 2504 µs for 80 rows per kv head at head_dim 128
// (bf16, 41 MB). Here 22 and 30 µs: bound by the pieces' start, merge and dependency chain
// (19 chunks of work per slot at most), no longer by re-reading. Error against fp64, 2-norm
// over nine shapes, as a share of the per-row kernel's, for bf16 / f16 / f32 queries: BF16
// pools 0.77 / 0.89 / 0.83, F16 0.75 / 0.67 / 0.68, FP8 0.80 / 0.89 / 0.84, INT8 0.81 / 0.86 /
// 0.82. (F16 with two parts of P, and the 2^14 inside the exponent, where it takes four of the
// argument's bits: 1.38 / 1.20 / 0.99, for 0.1 µs a call less at head_dim 64.)
#include "attention_mfma.h"

namespace gg {
namespace {

template <gg_dtype_t DT>
gg_status_t launch_full_dt(const AttnArgs& a, const KVView& kv, const AttnShape& sh, hipStream_t s) {
    const int pieces = lpt_pieces(a.sk_grid, a.num_seqs, kv.Hkv * sh.groups);
    if (kv.D == 128) {
        // (More than four row tiles in groups of at most two.)
        attn_mfma_lpt_kernel<DT, 2, 128, true><<<pieces, 256, 0, s>>>(a, kv);
        return check_hip(hipGetLastError(), "verify_attention launch");
    }
    switch (sh.nt) {
        case 1: attn_mfma_lpt_kernel<DT, 1, 64, true><<<pieces, 256, 0, s>>>(a, kv); break;
        case 2: attn_mfma_lpt_kernel<DT, 2, 64, true><<<pieces, 256, 0, s>>>(a, kv); break;
        case 3: attn_mfma_lpt_kernel<DT, 3, 64, true><<<pieces, 256, 0, s>>>(a, kv); break;
        default: attn_mfma_lpt_kernel<DT, 4, 64, true><<<pieces, 256, 0, s>>>(a, kv); break;
    }
    return check_hip(hipGetLastError(), "verify_attention launch");
}

}  // namespace

gg_status_t launch_attn_full(const AttnArgs& a, const KVView& kv, const AttnShape& sh, hipStream_t s) {
    if (a.sched != ATTN_SCHED_LPT) return fail(GG_ERR_INTERNAL, "attention: full-precision rows run the LPT schedule only");
    switch (kv.dt) {
        case GG_DTYPE_BF16: return launch_full_dt<GG_DTYPE_BF16>(a, kv, sh, s);
        case GG_DTYPE_F16: return launch_full_dt<GG_DTYPE_F16>(a, kv, sh, s);
        case GG_DTYPE_FP8_E4M3: return launch_full_dt<GG_DTYPE_FP8_E4M3>(a, kv, sh, s);
        case GG_DTYPE_INT8: return launch_full_dt<GG_DTYPE_INT8>(a, kv, sh, s);
        default: return fail(GG_ERR_INVALID, "attention: pool dtype not on the MFMA path");
    }
}

}  // namespace gg
