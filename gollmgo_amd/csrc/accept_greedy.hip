// accept_greedy.hip — greedy verify on the device.
//
// Replaces the host-side Verify/argmax loop (internal/engine/speculative.go:68-84,
// internal/engine/sampling.go:75-85) driven by emitSpeculative
// (internal/engine/serving.go:514-566). Two launches:
//   1) segment argmax: each wave scans 4096 logits of one row with 16-byte loads and
//      writes (value, index) of their first maximum;
//   2) decide: one block per sequence merges the segments of rows 0..n, every row at
//      once (a lane group per row), then walks the drafts in order: the first row whose
//      argmax differs from its draft ends the accepted prefix and supplies the corrected
//      token; if none differs, row n supplies the bonus token.
// Tie rule: first index of the maximum. NaN never wins; a NaN at element 0 makes
// the row's argmax 0 (the reference scans with `>` from element 0).
#include <type_traits>

#include "gg_common.h"
#include "gg_draw.h"

namespace gg {
namespace {

constexpr int kSeg = 4096;
constexpr int kThreads = 256;
constexpr int kNone = 0x7fffffff;

struct ArgBest {
    float v;
    int i;
};

__device__ __forceinline__ ArgBest wave_best(ArgBest b) {
    for (int o = 32; o > 0; o >>= 1) {
        float ov = __shfl_xor(b.v, o);
        int oi = __shfl_xor(b.i, o);
        if (oi != kNone && (b.i == kNone || ov > b.v || (ov == b.v && oi < b.i))) {
            b.v = ov;
            b.i = oi;
        }
    }
    return b;
}

// First maximum of elements [base, end) of a row, at most LEN, by one wave: 16-byte vectors
// aligned in memory, lane l taking vectors l, l + 64, ..., all of their loads in flight at once.
// A lane's indices ascend, so a strict `>` keeps its first maximum and never takes NaN. The
// vectors that the segment cuts (a row need not start on 16 bytes) are read by element.
template <gg_dtype_t DT, int LEN>
__device__ __forceinline__ ArgBest scan_segment(const void* row, int base, int end) {
    constexpr int kEB = DT == GG_DTYPE_F32 ? 4 : 2;
    constexpr int kPer = 16 / kEB;
    constexpr int kIters = LEN / (64 * kPer);
    const int lane = threadIdx.x & 63;
    const uint8_t* p = (const uint8_t*)row + (size_t)base * kEB;
    const int shift = (int)((uintptr_t)p & 15) / kEB;  // elements between the aligned start and base
    const uint8_t* al = p - shift * kEB;
    const int first = base - shift;
    uint4 raw[kIters];
    bool whole[kIters];
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const int j = it * 64 + lane, e0 = first + j * kPer;
        whole[it] = e0 >= base && e0 + kPer <= end;
        raw[it] = whole[it] ? *(const uint4*)(al + (size_t)j * 16) : make_uint4(0, 0, 0, 0);
    }
    ArgBest b{-INFINITY, kNone};
    auto by_element = [&](int e0) {
        for (int e = max(e0, base); e < min(e0 + kPer, end); ++e) {
            const float v = load_as_f32(row, DT, e);
            if (v > b.v) b = ArgBest{v, e};
        }
    };
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const int e0 = first + (it * 64 + lane) * kPer;
        if (whole[it]) {
            const uint32_t w[4] = {raw[it].x, raw[it].y, raw[it].z, raw[it].w};
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                float v;
                if constexpr (DT == GG_DTYPE_F32) {
                    v = __uint_as_float(w[k]);
                } else {
                    const uint16_t h = (uint16_t)(w[k >> 1] >> ((k & 1) * 16));
                    v = DT == GG_DTYPE_BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
                }
                if (v > b.v) b = ArgBest{v, e0 + k};
            }
        } else if (e0 < end) {
            by_element(e0);
        }
    }
    if (first + kIters * 64 * kPer < end && lane == 0) by_element(first + kIters * 64 * kPer);
    return b;
}

// One wave per 4096-element segment (SPLIT 1). A 256-thread block per segment had two loads in
// flight per thread and spent most of its life in the reduction: 32 x 5 rows of 128256 bf16 logits
// (41 MB) 15.4 -> 10.5 us, 128 x 6 rows (197 MB) 57 -> 34 us (5.8 TB/s).
// SPLIT 4, a wave per quarter: where the waves of whole segments are fewer than the SIMDs, a
// wave's own chain of loads and compares is the time (launch_accept_greedy).
template <gg_dtype_t DT, int SPLIT>
__global__ void __launch_bounds__(kThreads) greedy_segment_kernel(const void* __restrict__ logits, int rows, int R, int V,
                                                                  int nseg, const int32_t* __restrict__ n_drafts,
                                                                  float2* __restrict__ ws) {
    constexpr int kWaves = kThreads / 64, kLen = kSeg / SPLIT;
    static_assert(SPLIT == 1 || SPLIT == kWaves, "a block is one segment or a segment per wave");
    const int wave = threadIdx.x >> 6;
    const int w = SPLIT == 1 ? blockIdx.x * kWaves + wave : blockIdx.x;  // row * nseg + segment
    const int row = __builtin_amdgcn_readfirstlane(w / nseg), seg = __builtin_amdgcn_readfirstlane(w % nseg);
    if (row >= rows) return;
    const int b = row / R, j = row % R;
    const int nb = n_drafts[b];
    if (j > (nb < 0 ? 0 : nb)) return;  // rows 0..n, n clamped as the decide kernel clamps it
    const void* rowp = (const uint8_t*)logits + (size_t)row * V * dtype_bytes(DT);
    const int base = __builtin_amdgcn_readfirstlane(seg * kSeg + (SPLIT == 1 ? 0 : wave * kLen));
    ArgBest best = wave_best(scan_segment<DT, kLen>(rowp, base, min(base + kLen, V)));  // (none past the row)
    if constexpr (SPLIT > 1) {
        __shared__ ArgBest s_best[kWaves];
        if ((threadIdx.x & 63) == 0) s_best[wave] = best;
        __syncthreads();
        if (threadIdx.x) return;
        best = s_best[0];
        for (int i = 1; i < kWaves; ++i)
            if (s_best[i].v > best.v) best = s_best[i];  // (-inf where none; the first maximum wins)
    }
    if ((threadIdx.x & 63) == 0) ws[(size_t)row * nseg + seg] = make_float2(best.v, __int_as_float(best.i));
}

// Lane group of g = 2^ceil(log2 nseg) lanes per row (lane s of a group reads segment s,
// and s + g, ... past 64), kDecideThreads / g rows per pass; each row's argmax lands in LDS
// and thread 0 walks the rows. (Walking row by row, each row's loads waiting for the
// previous row's decision, took 13 us for nine rows.)
constexpr int kDecideThreads = 512;
constexpr int kMaxRows = 65;  // rows per sequence: max_drafts + 1, max_drafts <= 64 (checked by the ABI)
// DRAW: the sequence's draw is set up here too (its bonus row when every draft was accepted,
// none otherwise): the row's maximum is at hand, and the draw needs no launch for it.
template <bool DRAW>
__global__ void __launch_bounds__(kDecideThreads) greedy_decide_kernel(
    const void* __restrict__ logits, gg_dtype_t dt, int K, int V, int nseg,
    const int32_t* __restrict__ drafts, const int32_t* __restrict__ n_drafts,
    const float2* __restrict__ ws, int32_t* __restrict__ out_acc, int32_t* __restrict__ out_tok,
    fd::DrawParams P, int force_exact) {
    const int b = blockIdx.x;
    const int R = K + 1;
    int n = n_drafts[b];
    n = n < 0 ? 0 : (n > K ? K : n);
    __shared__ int s_am[kMaxRows];
    __shared__ ArgBest s_last;  // row n's first maximum
    __shared__ int s_draw;
    int g = 1;
    while (g < nseg && g < 64) g <<= 1;
    const int per_pass = kDecideThreads / g;
    const int jl = threadIdx.x / g, sl = threadIdx.x % g;
    for (int j0 = 0; j0 <= n; j0 += per_pass) {
        const int j = j0 + jl;
        const bool live = j <= n;
        const int row = b * R + (live ? j : 0);
        const float first = load_as_f32(logits, dt, (size_t)row * V);
        ArgBest best{-INFINITY, kNone};
        for (int s = sl; s < nseg; s += g) {
            const float2 p = ws[(size_t)row * nseg + s];
            const int pi = __float_as_int(p.y);
            if (pi != kNone && (best.i == kNone || p.x > best.v || (p.x == best.v && pi < best.i))) {
                best.v = p.x;
                best.i = pi;
            }
        }
        for (int o = g >> 1; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best.v, o);
            const int oi = __shfl_xor(best.i, o);
            if (oi != kNone && (best.i == kNone || ov > best.v || (ov == best.v && oi < best.i))) {
                best.v = ov;
                best.i = oi;
            }
        }
        if (live && sl == 0) s_am[j] = (first != first || best.i == kNone) ? 0 : best.i;
        if (DRAW && j == n && sl == 0) s_last = best;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int accepted = n, token = s_am[n];
        for (int j = 0; j < n; ++j) {
            if (s_am[j] != drafts[(size_t)b * K + j]) {
                accepted = j;
                token = s_am[j];
                break;
            }
        }
        out_acc[b] = accepted;
        out_tok[b] = token;
        if constexpr (DRAW) {
            s_draw = accepted == n;
            fd::prep_row(P, b, accepted == n ? n : -1, -1, s_last.v, s_last.i != kNone, 0ull, 0.0, force_exact);
        }
    }
    if constexpr (DRAW) {
        __syncthreads();
        if (!s_draw || !P.filtered) return;
        for (int i = threadIdx.x; i < fd::kBins; i += kDecideThreads) {
            P.hcnt[(size_t)b * fd::kBins + i] = 0;
            if (!P.top_list) P.hmass[(size_t)b * fd::kBins + i] = 0.0;
        }
    }
}

}  // namespace

size_t greedy_workspace_bytes(int num_seqs, int max_drafts, int vocab) {
    int nseg = (vocab + kSeg - 1) / kSeg;
    return (size_t)num_seqs * (max_drafts + 1) * nseg * sizeof(float2);
}

gg_status_t launch_accept_greedy(const void* logits, gg_dtype_t dt, int num_seqs, int max_drafts,
                                 int vocab, const int32_t* drafts, const int32_t* n_drafts,
                                 int32_t* out_acc, int32_t* out_tok, void* ws, hipStream_t s,
                                 const fd::DrawParams* draw, bool force_exact) {
    const int R = max_drafts + 1;
    if (R > kMaxRows) return fail(GG_ERR_INVALID, "accept_greedy: more than 64 drafts per sequence");
    const int nseg = (vocab + kSeg - 1) / kSeg;
    const int rows = num_seqs * R;
    // Quarters up to one segment per SIMD. Calls with whole / quarter segments, f32: 1 x 1 row of 1000
    // (1 segment) 5.8 / 5.5 us, 1 x 9 of 1000 6.8 / 6.1, 8 x 1 of 128256 (256) 8.0 / 6.9, 32 x 1
    // (1024) 8.3 / 7.7; bf16: 1 x 5 of 128256 (160) 7.8 / 6.7, 16 x 5 of 50257 (1040) 8.9 / 8.9, 16 x 3 of
    // 128256 (1536) 8.2 / 8.5, 16 x 9 of 50257 (1872) 9.5 / 10.8.
    const long long segs = (long long)rows * nseg;
    const bool split = segs <= 4 * device_cu_count();
    const unsigned grid = (unsigned)(split ? segs : (segs + kThreads / 64 - 1) / (kThreads / 64));
    float2* seg = (float2*)ws;
    auto scan = [&](auto dt_tag) {
        constexpr gg_dtype_t DT = decltype(dt_tag)::value;
        if (split) greedy_segment_kernel<DT, 4><<<grid, kThreads, 0, s>>>(logits, rows, R, vocab, nseg, n_drafts, seg);
        else greedy_segment_kernel<DT, 1><<<grid, kThreads, 0, s>>>(logits, rows, R, vocab, nseg, n_drafts, seg);
    };
    switch (dt) {
        case GG_DTYPE_F32: scan(std::integral_constant<gg_dtype_t, GG_DTYPE_F32>{}); break;
        case GG_DTYPE_BF16: scan(std::integral_constant<gg_dtype_t, GG_DTYPE_BF16>{}); break;
        default: scan(std::integral_constant<gg_dtype_t, GG_DTYPE_F16>{}); break;
    }
    if (draw)
        greedy_decide_kernel<true><<<num_seqs, kDecideThreads, 0, s>>>(logits, dt, max_drafts, vocab, nseg, drafts, n_drafts,
                                                                      seg, out_acc, out_tok, *draw, force_exact);
    else
        greedy_decide_kernel<false><<<num_seqs, kDecideThreads, 0, s>>>(logits, dt, max_drafts, vocab, nseg, drafts, n_drafts,
                                                                       seg, out_acc, out_tok, fd::DrawParams{}, 0);
    return check_hip(hipGetLastError(), "accept_greedy launch");
}

}  // namespace gg
