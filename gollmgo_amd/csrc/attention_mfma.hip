// attention_mfma.hip — the MFMA attention launches: the partition grid, stream-K, and the LPT
// schedule with its plan (kernels of a piece: attention_mfma.h).
#include "attention_mfma.h"

#include <algorithm>

namespace gg {
namespace {

constexpr int kHD = 128;  // head_dim of the kernels here

// Fixed partition grid: workgroup (part, kvh, b) takes tokens [part*P, (part+1)*P).
template <gg_dtype_t DT, int NT>
__global__ void __launch_bounds__(256, attn_occupancy(PoolTraits<DT>::kEB, NT, kHD)) attn_mfma_kernel(AttnArgs a, KVView kv) {
    const int part = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const int ctx = seq_keys(a, b, kBS);
    const int P = a.partition;
    const int nparts = (ctx + P - 1) / P;
    if (part >= nparts) return;
    const PieceDesc d{b, kvh, part * P, min(part * P + P, ctx), nparts == 1 ? -1 : part, -1, 0, ctx, seq_rows(a, b)};
    PieceIn<DT, attn_chunk_tokens(PoolTraits<DT>::kEB, NT), kHD> in;
    DeferredRows ap;
    const QRaw<NT> q16 = load_q16<NT, kHD>(a, kv, d);
    start_piece(a, kv, d, in, &ap);
    attn_piece<DT, NT, kHD, false>(a, kv, d, in, &ap, q16);
}

// Stream-K: the (sequence, kv head) items are laid end to end in chunk units; the grid
// of gridDim.x workgroups splits that total evenly (at least sk_min_chunks each). A
// workgroup's range is cut at item boundaries into pieces; a piece that is a whole item
// writes the output, any other piece writes record (workgroup + item), and
// attn_streamk_combine_kernel merges the records of split items.
template <gg_dtype_t DT, int NT>
__global__ void __launch_bounds__(256, attn_occupancy(PoolTraits<DT>::kEB, NT, kHD)) attn_mfma_streamk_kernel(AttnArgs a, KVView kv) {
    constexpr int kTok = attn_chunk_tokens(PoolTraits<DT>::kEB, NT);
    const int w = blockIdx.x;
    const int Hkv = kv.Hkv;
    __shared__ long long s_scan[256];
    __shared__ long long s_total;
    __shared__ int s_b0;
    __shared__ long long s_base0;
    // Per-thread slice of sequences, its work, and an exclusive scan over threads.
    const int B = a.num_seqs;
    const int per_t = (B + 255) / 256;
    const int b_lo = min(B, (int)threadIdx.x * per_t), b_hi = min(B, b_lo + per_t);
    long long mine = 0;
    for (int bb = b_lo; bb < b_hi; ++bb) mine += (long long)Hkv * seq_chunks(a, bb, kTok);
    s_scan[threadIdx.x] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long c = 0;
        for (int t = 0; t < 256; ++t) {
            const long long v = s_scan[t];
            s_scan[t] = c;
            c += v;
        }
        s_total = c;
        s_b0 = B;
        s_base0 = c;
    }
    __syncthreads();
    const long long C = s_total;
    const long long per = max((C + gridDim.x - 1) / gridDim.x, (long long)a.sk_min_chunks);
    const long long g0 = (long long)w * per;
    if (g0 >= C) return;
    const long long g1 = min(g0 + per, C);
    // The thread whose slice holds chunk g0 finds the sequence.
    {
        long long gb = s_scan[threadIdx.x];
        if (gb <= g0 && g0 < gb + mine) {
            for (int bb = b_lo; bb < b_hi; ++bb) {
                const long long wk = (long long)Hkv * seq_chunks(a, bb, kTok);
                if (g0 < gb + wk) {
                    s_b0 = bb;
                    s_base0 = gb;
                    break;
                }
                gb += wk;
            }
        }
    }
    __syncthreads();
    // Loop state is wave-uniform 32-bit (chunk totals stay far below 2^31) and kept in
    // scalar registers.
    int b = __builtin_amdgcn_readfirstlane(s_b0);
    int gb = __builtin_amdgcn_readfirstlane((int)s_base0);  // chunk index where sequence b starts
    int g = __builtin_amdgcn_readfirstlane((int)g0);
    const int ge = __builtin_amdgcn_readfirstlane((int)g1);
    // The next piece of [g, ge): advances (g, b, gb); false when the range is done.
    auto next_piece = [&](PieceDesc& d) -> bool {
        while (g < ge && b < B) {
            const int nch = __builtin_amdgcn_readfirstlane(seq_chunks(a, b, kTok));
            const int wk = Hkv * nch;
            if (nch == 0 || g >= gb + wk) {
                gb += wk;
                ++b;
                continue;
            }
            const int off = g - gb;
            const int kvh = off / nch;
            const int c0 = off % nch;
            const int c1 = min(nch, c0 + (ge - g));
            const int item = b * Hkv + kvh;
            const bool whole = c0 == 0 && c1 == nch;
            const int ctx = __builtin_amdgcn_readfirstlane(seq_keys(a, b, kBS));
            d = PieceDesc{b, kvh, c0 * kTok, min(c1 * kTok, ctx), -1, whole ? -1 : w + item, 0, ctx,
                          __builtin_amdgcn_readfirstlane(seq_rows(a, b))};
            g = __builtin_amdgcn_readfirstlane(g + (c1 - c0));
            return true;
        }
        return false;
    };
    PieceDesc d;
    while (next_piece(d)) {
        PieceIn<DT, attn_chunk_tokens(PoolTraits<DT>::kEB, NT), kHD> in;
        const QRaw<NT> q16 = load_q16<NT, kHD>(a, kv, d);
        start_piece(a, kv, d, in, nullptr);
        attn_piece<DT, NT, kHD, false>(a, kv, d, in, nullptr, q16);
    }
}

// Sum over an N-thread workgroup (wave sums, then the wave totals).
template <int N>
__device__ __forceinline__ unsigned long long block_sum(unsigned long long v, unsigned long long* s_w) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long t = 0;
#pragma unroll
    for (int w = 0; w < N / 64; ++w) t += s_w[w];
    return t;
}

// Exclusive prefix sums over an N-thread workgroup of two non-negative ints (sums below 2^31)
// in one pass, packed (lo, hi), and their totals.
template <int N>
__device__ __forceinline__ unsigned long long block_excl_scan2(int lo, int hi, unsigned long long* s_w,
                                                               unsigned long long* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long v = ((unsigned long long)hi << 32) | (unsigned)lo;
    unsigned long long inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long t = __shfl_up(inc, o);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_w[w] = inc;
    __syncthreads();
    unsigned long long before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < N / 64; ++i) {
        before += i < w ? s_w[i] : 0;
        all += s_w[i];
    }
    *total = all;
    return before + inc - v;
}

// Place of row group rg of unit u (a piece of one kv head) in a block of `units` equal pieces
// of each of `groups` groups: the groups of a unit eight places apart, in blocks of eight
// units. Workgroup w runs on XCD w mod 8, so the groups of a unit, which read the same K/V at
// the same time, share one XCD's L2. (One group: u itself.) Three groups of 80 bf16 rows per kv
// head, two kv heads, 16 sequences: 34.1 -> 30.3 µs a call.
__device__ __forceinline__ int lpt_place(int u, int rg, int units, int groups) {
    const int first = u & ~7;
    return first * groups + rg * min(8, units - first) + (u & 7);
}

// One workgroup of N threads (one sequence per thread): sizes, ranks and lays out the pieces.
// A chain of barriers and short loops of one workgroup, paid once per step: N is 256 for up
// to 256 sequences (four waves meet at its barriers), the table is written by all threads, and
// no 64-bit division is left (the fp64 quotients are exact where rounding matters: both
// operands are integers below 2^53 and no non-integer quotient comes within 2^-28 of one).
// Per call, 64 sequences 9.4 -> 7.6 µs, one 6.7 -> 5.2.
template <int N>
__global__ void __launch_bounds__(N) attn_lpt_plan_kernel(AttnArgs a, int Hkv, int tok_log2, int slots, int pieces) {
    __shared__ __align__(16) int s_key[N];  // piece size in chunks (0: no work)
    __shared__ __align__(16) int s_cnt[N];  // pieces of the sequence over all kv heads
    __shared__ int s_nch[N], s_ctx[N], s_rows[N], s_first[N], s_pos[N], s_np[N];
    __shared__ unsigned long long s_sum[N / 64], s_scan[N / 64];
    __shared__ int s_t;
    const int B = a.num_seqs, tok = 1 << tok_log2;
    const int b = threadIdx.x;
    const int ctx = b < B ? seq_keys(a, b, kBS) : 0;
    const int nrows = b < B ? seq_rows(a, b) : 0;
    const int nch = nrows > 0 && nrows <= ctx ? (ctx + tok - 1) >> tok_log2 : 0;  // (seq_chunks)
    s_nch[b] = nch;
    s_ctx[b] = ctx;
    s_rows[b] = nrows;
    const double C = (double)(block_sum<N>((unsigned long long)nch, s_sum) * (unsigned long long)Hkv);
    const bool few = lpt_few_items(slots, B, Hkv);
    const int tmin = lpt_min_chunks(tok);
    int T;
    if (few) {
        // Fewer items than slots: every long item has to be cut to fill the slots, into equal
        // pieces. T is the shortest piece length whose pieces still fit one round of slots:
        // 64 candidate lengths from the mean slot load up, each counted by one thread per wave
        // over a slice of the sequences.
        const int t_lo = max((int)ceil(C / slots), tmin);
        const int t_step = (t_lo + kLptTSpan - 1) / kLptTSpan;
        const int cand = t_lo + (threadIdx.x & 63) * t_step;
        int count = 0;
        for (int q = threadIdx.x >> 6; q < B; q += N / 64) count += (s_nch[q] + cand - 1) / cand;
        s_cnt[threadIdx.x] = count;
        __syncthreads();
        if (threadIdx.x < 64) {
            int sum = 0;
#pragma unroll
            for (int w = 0; w < N / 64; ++w) sum += s_cnt[64 * w + threadIdx.x];
            const unsigned long long fits = __ballot(sum * Hkv <= slots);
            // (None fits, for instance when the items nearly fill the slots: the longest one.)
            if (threadIdx.x == 0) s_t = t_lo + (fits ? __builtin_ctzll(fits) : 63) * t_step;
        }
        __syncthreads();
        T = s_t;
    } else {
        T = max((int)ceil(C * kLptPieceNum / ((double)slots * kLptPieceDen)), tmin);
    }
    // The ranks: with few items all pieces by size; else the full pieces (by sequence), then the
    // last pieces by size, descending (ties: sequence). Records of split sequences by (sequence,
    // piece, kv head).
    const int np = nch ? (nch + T - 1) / T : 0;
    const int key = few ? (np ? (nch + np - 1) / np : 0) : (np ? nch - (np - 1) * T : 0);
    const int cnt = few ? np * Hkv : (np ? Hkv : 0);  // pieces ranked by key
    const int nfull = !few && np > 1 ? (np - 1) * Hkv : 0;
    // (Entries past B, up to a multiple of 8, read as empty.)
    s_key[b] = key;
    s_cnt[b] = cnt;
    unsigned long long sums;
    const unsigned long long before = block_excl_scan2<N>(nfull, np > 1 ? np * Hkv : 0, s_scan, &sums);
    const int full_pos = (int)(unsigned)before, F = (int)(unsigned)sums;  // (its barrier publishes s_key / s_cnt)
    s_first[b] = (int)(before >> 32);
    // Pieces ahead of this sequence's: larger ones, then equal ones of lower sequences. Eight
    // sequences per step from 16-byte LDS reads (independent adds, no serial chain).
    int pos = F, all = F;
    if (b < B || b == 0) {
        for (int t0 = 0; t0 < B; t0 += 8) {
            const int4 k0 = *(const int4*)&s_key[t0], k1 = *(const int4*)&s_key[t0 + 4];
            const int4 n0 = *(const int4*)&s_cnt[t0], n1 = *(const int4*)&s_cnt[t0 + 4];
            const int kk[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
            const int nn[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int t = t0 + e;
                pos += (kk[e] > key || (kk[e] == key && t < b)) ? nn[e] : 0;
                all += nn[e];
            }
        }
        if (b == 0) s_t = all;
    }
    s_pos[b] = pos;
    s_np[b] = np | (full_pos << 10);
    __syncthreads();
    const int total = s_t;
    // The table, by all threads: several per (sequence, kv head) when those are few.
    int* plan = a.plan;
    int4* table = (int4*)lpt_table(plan);
    const int heads = B * Hkv;
    const int kvh_n = Hkv / a.row_groups;
    int sub = 1;
    while (sub * 2 * heads <= N) sub *= 2;
    for (int i = threadIdx.x; i < heads * sub; i += N) {
        const int item = i / sub, q = item / Hkv, h = item % Hkv;
        const int n = s_nch[q], qc = s_ctx[q], qr = s_rows[q], first = s_first[q] + h, qp = s_pos[q];
        const int qn = s_np[q] & 1023, qf = s_np[q] >> 10;
        if (i % sub == 0) lpt_count(plan, pieces)[item] = 0;
        const int size = few && qn ? n / qn : T, extra = few ? n - size * qn : 0;
        for (int j = i % sub; j < qn; j += sub) {
            const int c0 = j * size + min(j, extra);
            const int c1 = few ? c0 + size + (j < extra ? 1 : 0) : min(c0 + size, n);
            // Equal pieces of a sequence have a block of ranks: few, all of them; else its full
            // pieces, and its last ones.
            const bool full = !few && j < qn - 1;
            const int units = (few ? qn : full ? qn - 1 : 1) * kvh_n;
            const int u = (few || full ? j * kvh_n : 0) + h % kvh_n;
            const int r = (full ? qf : qp) + lpt_place(u, h / kvh_n, units, a.row_groups);
            int4* t = table + 2 * lpt_slot(r, slots, total, heads <= slots);
            t[0] = make_int4(q, h | (qn << 16), c0 << tok_log2, min(c1 << tok_log2, qc));
            t[1] = make_int4(qc, qr, first, j);
        }
    }
    // Entries past the last piece tell their workgroups to exit.
    for (int q = total + threadIdx.x; q < pieces; q += N) table[2 * q] = make_int4(-1, 0, 0, 0);
}

template <gg_dtype_t DT>
gg_status_t launch_dt(const AttnArgs& a, const KVView& kv, int nt, hipStream_t s) {
    if (a.sched == ATTN_SCHED_LPT) {
        const int pieces = lpt_pieces(a.sk_grid, a.num_seqs, kv.Hkv);
        switch (nt) {
            case 1: attn_mfma_lpt_kernel<DT, 1, kHD, false><<<pieces, 256, 0, s>>>(a, kv); break;
            case 2: attn_mfma_lpt_kernel<DT, 2, kHD, false><<<pieces, 256, 0, s>>>(a, kv); break;
            case 3: attn_mfma_lpt_kernel<DT, 3, kHD, false><<<pieces, 256, 0, s>>>(a, kv); break;
            case 4: attn_mfma_lpt_kernel<DT, 4, kHD, false><<<pieces, 256, 0, s>>>(a, kv); break;
            default: return fail(GG_ERR_INVALID, "attention: too many rows per kv head for the MFMA path");
        }
        return GG_OK;
    }
    if (a.sched == ATTN_SCHED_STREAMK) {
        const int grid = a.sk_grid;
        switch (nt) {
            case 1: attn_mfma_streamk_kernel<DT, 1><<<grid, 256, 0, s>>>(a, kv); break;
            case 2: attn_mfma_streamk_kernel<DT, 2><<<grid, 256, 0, s>>>(a, kv); break;
            case 3: attn_mfma_streamk_kernel<DT, 3><<<grid, 256, 0, s>>>(a, kv); break;
            case 4: attn_mfma_streamk_kernel<DT, 4><<<grid, 256, 0, s>>>(a, kv); break;
            default: return fail(GG_ERR_INVALID, "attention: too many rows per kv head for the MFMA path");
        }
        return GG_OK;
    }
    dim3 grid(a.max_parts, kv.Hkv, a.num_seqs);
    switch (nt) {
        case 1: attn_mfma_kernel<DT, 1><<<grid, 256, 0, s>>>(a, kv); break;
        case 2: attn_mfma_kernel<DT, 2><<<grid, 256, 0, s>>>(a, kv); break;
        case 3: attn_mfma_kernel<DT, 3><<<grid, 256, 0, s>>>(a, kv); break;
        case 4: attn_mfma_kernel<DT, 4><<<grid, 256, 0, s>>>(a, kv); break;
        default: return fail(GG_ERR_INVALID, "attention: too many rows per kv head for the MFMA path");
    }
    return GG_OK;
}

// Merge the stream-K records of one (sequence, kv head) item that was split over
// several workgroups. Workgroup (item, y) takes rows 4y .. 4y+3 of the item; each thread
// one row and four dims, merged in one online pass whose record loads are independent.
__global__ void __launch_bounds__(128) attn_streamk_combine_kernel(AttnArgs a, int Hkv, int tok, int grid) {
    const int item = blockIdx.x;
    const int b = item / Hkv, kvh = item % Hkv;
    const int G = a.num_q_heads / Hkv;
    const int nrows = seq_rows(a, b);
    const int r = blockIdx.y * 4 + (threadIdx.x >> 5);
    const int d4 = threadIdx.x & 31;
    const int nch = seq_chunks(a, b, tok);
    if (nch == 0 || (int)blockIdx.y * 4 >= G * nrows) return;
    // Chunks before sequence b and in total (same arithmetic as the producer).
    __shared__ long long s_before[128], s_total[128];
    long long before = 0, total = 0;
    for (int bb = threadIdx.x; bb < a.num_seqs; bb += 128) {
        const long long wk = (long long)Hkv * seq_chunks(a, bb, tok);
        total += wk;
        if (bb < b) before += wk;
    }
    s_before[threadIdx.x] = before;
    s_total[threadIdx.x] = total;
    __syncthreads();
    for (int o = 64; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            s_before[threadIdx.x] += s_before[threadIdx.x + o];
            s_total[threadIdx.x] += s_total[threadIdx.x + o];
        }
        __syncthreads();
    }
    before = s_before[0];
    total = s_total[0];
    const long long per = max((total + grid - 1) / grid, (long long)a.sk_min_chunks);
    const long long gi0 = before + (long long)kvh * nch, gi1 = gi0 + nch;
    const int w0 = (int)(gi0 / per), w1 = (int)((gi1 - 1) / per);
    if (w0 == w1 || r >= G * nrows) return;  // one piece: the producer wrote the output
    const int RW = G * a.rows;
    float M = -1e30f, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int w = w0; w <= w1; ++w) {
        const size_t p = (size_t)(w + item) * RW + r;
        const float2 ml = *(const float2*)(a.ws_ml + p * 2);
        const float4 v = ((const float4*)(a.ws_acc + p * kHD))[d4];
        const float mn = fmaxf(M, ml.x);
        const float fo = __expf(M - mn), fn = __expf(ml.x - mn);
        M = mn;
        L = L * fo + ml.y * fn;
        acc.x = acc.x * fo + v.x * fn;
        acc.y = acc.y * fo + v.y * fn;
        acc.z = acc.z * fo + v.z * fn;
        acc.w = acc.w * fo + v.w * fn;
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const int j = r / G, g = r % G;
    const size_t obase = (((size_t)b * a.rows + j) * a.num_q_heads + (size_t)kvh * G + g) * kHD + 4 * d4;
    store_from_f32(a.out, a.out_dtype, obase + 0, acc.x * inv);
    store_from_f32(a.out, a.out_dtype, obase + 1, acc.y * inv);
    store_from_f32(a.out, a.out_dtype, obase + 2, acc.z * inv);
    store_from_f32(a.out, a.out_dtype, obase + 3, acc.w * inv);
}

}  // namespace

gg_status_t launch_attn_mfma(const AttnArgs& a, const KVView& kv, hipStream_t s) {
    const AttnShape sh = attn_shape(a.kv, a.rows, a.num_q_heads);
    const int G = a.num_q_heads / kv.Hkv;
    const int nt = sh.nt;
    const int tok = attn_chunk_tokens(dtype_bytes(kv.dt), nt);
    if (a.sched == ATTN_SCHED_LPT && !a.plan_ready) {
        const gg_status_t st = launch_attn_plan(a, s);
        if (st != GG_OK) return st;
    }
    if (sh.full) return launch_attn_full(a, kv, sh, s);
    gg_status_t st;
    switch (kv.dt) {
        case GG_DTYPE_BF16: st = launch_dt<GG_DTYPE_BF16>(a, kv, nt, s); break;
        case GG_DTYPE_F16: st = launch_dt<GG_DTYPE_F16>(a, kv, nt, s); break;
        case GG_DTYPE_FP8_E4M3: st = launch_dt<GG_DTYPE_FP8_E4M3>(a, kv, nt, s); break;
        case GG_DTYPE_INT8: st = launch_dt<GG_DTYPE_INT8>(a, kv, nt, s); break;
        default: return fail(GG_ERR_INVALID, "attention: pool dtype not on the MFMA path");
    }
    if (st != GG_OK) return st;
    const dim3 cgrid(a.num_seqs * kv.Hkv, (G * a.rows + 3) / 4);
    if (a.sched == ATTN_SCHED_STREAMK) attn_streamk_combine_kernel<<<cgrid, 128, 0, s>>>(a, kv.Hkv, tok, a.sk_grid);
    // (LPT: the split items are merged inside the main launch, lpt_merge_if_last.)
    return GG_OK;
}

gg_status_t launch_attn_plan(const AttnArgs& a, hipStream_t s) {
    if (a.sched != ATTN_SCHED_LPT) return GG_OK;
    if (a.num_seqs > kLptMaxSeqs) return fail(GG_ERR_INTERNAL, "attention: LPT plan over too many sequences");
    const KV* kv = a.kv;
    const int Hkv = kv->num_kv_heads;
    const AttnShape sh = attn_shape(kv, a.rows, a.num_q_heads);
    const int heads = Hkv * sh.groups;
    const int tok = attn_chunk_tokens(dtype_bytes(kv->dtype), sh.nt);
    const int pieces = lpt_pieces(a.sk_grid, a.num_seqs, heads);
    const int tok_log2 = tok == 64 ? 6 : 5;
    if (a.num_seqs <= 256) attn_lpt_plan_kernel<256><<<1, 256, 0, s>>>(a, heads, tok_log2, a.sk_grid, pieces);
    else attn_lpt_plan_kernel<kLptMaxSeqs><<<1, kLptMaxSeqs, 0, s>>>(a, heads, tok_log2, a.sk_grid, pieces);
    return check_hip(hipGetLastError(), "verify_attention plan launch");
}

int attn_slots(const KV* kv, int rows, int num_q_heads) {
    // One resident wave of workgroups: each CU holds attn_occupancy of them.
    return device_cu_count() * attn_occupancy((int)dtype_bytes(kv->dtype), attn_shape(kv, rows, num_q_heads).nt, kv->head_dim);
}

size_t attn_record_workspace_bytes(const KV* kv, int sched, int num_seqs, int rows, int num_q_heads, int max_blocks,
                                   size_t* ml_elems, size_t* acc_elems) {
    const AttnShape sh = attn_shape(kv, rows, num_q_heads);
    const int slots = attn_slots(kv, rows, num_q_heads);
    const int heads = kv->num_kv_heads * sh.groups;
    const size_t items = (size_t)num_seqs * heads;
    const size_t gr = (size_t)(num_q_heads / kv->num_kv_heads) * rows;
    const bool lpt = sched == ATTN_SCHED_LPT;
    auto bytes = [&](size_t records, size_t rw, size_t plan_ints) {
        return ((records * rw * 2 + 63) / 64 * 64 + records * rw * kv->head_dim) * sizeof(float) + plan_ints * sizeof(int);
    };
    // LPT: records of split items only. Stream-K: one per workgroup and item.
    const size_t records = lpt ? (size_t)lpt_records(slots) : (size_t)slots + items;
    const size_t rw = sh.full ? (size_t)16 * sh.nt : gr;
    if (ml_elems) *ml_elems = records * rw * 2;
    if (acc_elems) *acc_elems = records * rw * kv->head_dim;
    const size_t need = bytes(records, rw, lpt ? 16 + 8 * (size_t)lpt_pieces(slots, num_seqs, heads) + items : 0);
    // The size asked for is never below a record per slot and item and its plan, or, for the
    // shapes the per-row kernel also serves, that kernel's: callers size buffers by it, and
    // gg_verify_attention_noalloc takes the calls that fit its fixed array by this measure.
    const size_t asked = sh.full ? attn_workspace_bytes(kv, num_seqs, rows, num_q_heads, max_blocks,
                                                        attn_generic_partition(kv, num_seqs, rows, num_q_heads, max_blocks))
                                 : bytes((size_t)slots + items, gr, 16 + 4 * ((size_t)slots + items) + 2 * (size_t)num_seqs + items);
    return std::max(need, asked);
}

#ifdef GG_TRACE
extern "C" __attribute__((visibility("default"))) void* gg_debug_trace_ptr() {
    void* p = nullptr;
    (void)hipGetSymbolAddress(&p, HIP_SYMBOL(g_trace));
    return p;
}
#endif

}  // namespace gg
