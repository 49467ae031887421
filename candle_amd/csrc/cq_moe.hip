// Expert-grouped quantized matmul for gfx950: QTensor::indexed_moe_forward and
// candle_nn::moe::moe_gemm_gguf behind one kernel pair.
//
// Both entry points are lists of "pairs" (expert, activation row, output row, scale):
//   indexed_moe_forward (candle-core/src/quantized/cuda.rs:505-584, candle-kernels/src/quantized.cu:4670-4760)
//       pair p = b * topk + t : expert ids[p], activation row (input_dim1 == 1 ? b : p), output row p, scale 1
//   moe_gemm_gguf (candle-nn/src/moe.rs:169-337, candle-kernels/src/moe/moe_gguf.cu:55-132)
//       pair m : expert expert_ids[m], tok = sorted_token_ids[m],
//                activation row (topk_weights ? tok : tok / topk), output row tok, scale topk_weights[tok] or 1
//
// Step 1 quantizes the activation rows exactly as the CPU path does.  Step 2 (one workgroup)
// buckets the pairs by expert with a counting sort, so the input order does not matter (the
// reference sorts with an unstable sort, candle-core/src/sort.rs:282-297).  Step 3 streams every
// hit expert's rows once: workgroup (row tile, expert) keeps the decoded weight registers and loops
// over that expert's pairs — unlike the reference kernels, which re-read the expert's weights for
// every pair routed to it.  (Few pairs skip steps 1 and 2: a fused matvec per pair.  Hundreds of pairs take step 3 on the matrix
// cores: Q4_K and Q5_K experts with up to two dozen pairs each (few of long rows: 64) as batched matvecs over their pairs, cq_matvec_batch.hip, the rest as tiles of
// expert-sorted rows through the prefill kernel of the format.)
#include <algorithm>
#include "cq_device.h"
#include "cq_fmt.h"
#include "cq_launch.h"

namespace {

struct MoeWorkspace {
    int64_t act_off, offsets_off, cursor_off, pin_off, pout_off, pscale_off, chunk_off, max_chunks, rows_alloc, extra_off, total;
};

inline MoeWorkspace moe_workspace(int w_dtype, int64_t num_experts, int64_t n_pairs, int64_t x_rows, int64_t k) {
    MoeWorkspace w;
    w.act_off = 0;
    // the chunked path quantizes the activation rows in expert-sorted pair order (plus one chunk of padding rows);
    // the older per-expert kernel quantizes the x rows as they are: room for the larger of the two
    w.rows_alloc = n_pairs + CQ_MOE_CHUNK;
    w.max_chunks = n_pairs / CQ_MOE_CHUNK + (num_experts < n_pairs ? num_experts : n_pairs) + 1;
    w.offsets_off = cq_act_layout(w_dtype, k, w.rows_alloc > x_rows ? w.rows_alloc : x_rows).total;
    // (experts run as batched matvecs keep their pairs' rows as operand tiles instead)
    if ((w_dtype == CQ_Q4K || w_dtype == CQ_Q5K) && k % 256 == 0) w.offsets_off = std::max<int64_t>(w.offsets_off, cq_align256(cq_moe_stream_operand_bytes(num_experts, n_pairs, k)));
    w.cursor_off = w.offsets_off + cq_align256((num_experts + 1) * 4);
    w.pin_off = w.cursor_off + cq_align256(num_experts * 4);
    w.pout_off = w.pin_off + cq_align256(n_pairs * 4);
    w.pscale_off = w.pout_off + cq_align256(n_pairs * 4);
    w.chunk_off = w.pscale_off + cq_align256(n_pairs * 4);
    w.extra_off = w.chunk_off + cq_align256((3 * w.max_chunks + 1) * 4);  // n_chunks | expert[] | first[] | count[]
    // further passes of the experts with more than 32 pairs, for the batched-matvec form: n | two counters | (expert, pass)[]
    w.total = w.extra_off + cq_align256((CQ_MOE_EXTRA_HEADER + 2 * (n_pairs / 32 + 1)) * 4);
    return w;
}

// offsets[e] .. offsets[e+1] is expert e's segment of pair_in / pair_out / pair_scale.
// LC: the per-expert counters live in LDS (up to GROUP_LDS_EXPERTS experts) instead of the global `cursor` array: the
// two passes of atomics are then LDS atomics, not trips of one workgroup to the L2.
// (Lists of expert, token pairs: moe_group_wide_kernel, up to its number of experts.)
// The first KEEP pairs of every thread stay in registers between the two passes.  Decoding a pair is two dependent loads.  MANY: all first ones are asked for before any is
// used, then all second ones, whether a thread has that many pairs or not, which pays from 6144 pairs on (12000 pairs on 1500 experts: a call of 121 us takes 117).
constexpr int GROUP_LDS_EXPERTS = 4096, GROUP_MANY_PAIRS = 6144;
template <bool LC, bool MANY>
__global__ __launch_bounds__(1024) void moe_group_kernel(PairSource ps, int *__restrict__ offsets, int *__restrict__ cursor,
                                                         int *__restrict__ pair_in, int *__restrict__ pair_out,
                                                         float *__restrict__ pair_scale, float *__restrict__ out, int n, int *__restrict__ chunks,
                                                         int max_chunks, int chunk, int *__restrict__ extra) {
    __shared__ int carry, n_chunks, n_extra;
    __shared__ int buf[1024];
    __shared__ int lcur[LC ? GROUP_LDS_EXPERTS : 1];
    int *cur = LC ? lcur : cursor;
    const int tid = threadIdx.x;
    const int E = ps.num_experts;
    for (int e = tid; e < E; e += 1024) cur[e] = 0;
    __syncthreads();
    constexpr int KEEP = MANY ? 12 : 4;
    int ke[KEEP], kin[KEEP], kout[KEEP];
    float ksc[KEEP];
    bool kok[KEEP];
    const int last = ps.n_pairs - 1;
    if (!MANY) {
#pragma unroll
        for (int i = 0; i < KEEP; i++) kok[i] = tid + i * 1024 <= last && pair_decode(ps, tid + i * 1024, ke[i], kin[i], kout[i], ksc[i]);
    } else if (ps.mode == MOE_INDEXED) {
#pragma unroll
        for (int i = 0; i < KEEP; i++) ke[i] = (int)ps.ids_u32[min(tid + i * 1024, last)];
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            kout[i] = min(tid + i * 1024, last);
            kin[i] = ps.input_dim1 == 1 ? kout[i] / ps.topk : kout[i];
            ksc[i] = 1.0f;
            kok[i] = tid + i * 1024 <= last && (uint32_t)ke[i] < (uint32_t)E;
        }
    } else {
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            ke[i] = ps.expert_ids[min(tid + i * 1024, last)];
            kout[i] = ps.sorted_token_ids[min(tid + i * 1024, last)];
        }
#pragma unroll
        for (int i = 0; i < KEEP; i++) ksc[i] = ps.topk_weights ? ps.topk_weights[min(max(kout[i], 0), last)] : 1.0f;
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            kin[i] = ps.topk_weights ? kout[i] : kout[i] / ps.topk;
            kok[i] = tid + i * 1024 <= last && ke[i] >= 0 && ke[i] < E && kout[i] >= 0 && kout[i] <= last && kin[i] < ps.x_rows;
        }
    }
#pragma unroll
    for (int i = 0; i < KEEP; i++)
        if (kok[i]) atomicAdd(&cur[ke[i]], 1);
    for (int p = tid + KEEP * 1024; p < ps.n_pairs; p += 1024) {
        int e, in_row, out_row;
        float scale;
        if (pair_decode(ps, p, e, in_row, out_row, scale)) atomicAdd(&cur[e], 1);
    }
    if (tid == 0) { carry = 0; n_chunks = 0; n_extra = 0; }
    __syncthreads();
    // exclusive scan of the counts, 1024 experts per sweep (only as many doubling steps as the sweep is wide)
    for (int base = 0; base < E; base += 1024) {
        int e = base + tid;
        int c = e < E ? cur[e] : 0;
        const int width = min(1024, E - base);
        buf[tid] = c;
        __syncthreads();
        for (int o = 1; o < width; o <<= 1) {
            int v = tid >= o ? buf[tid - o] : 0;
            __syncthreads();
            buf[tid] += v;
            __syncthreads();
        }
        int start = carry + buf[tid] - c;
        if (e < E) {
            offsets[e] = start;
            cur[e] = start;
            // chunk table: expert e's segment in pieces of `chunk` pairs (any order: chunks are independent)
            // (the batched-matvec form takes 32 pairs of an expert per pass over its weights: every further pass is an item of a
            // list that the workgroups of that launch share out among themselves once their own pass is done)
            if (extra && c > 32) {
                const int np = (c + 31) / 32 - 1;
                const int eb = atomicAdd(&n_extra, np);
                for (int i = 0; i < np; i++) {
                    extra[CQ_MOE_EXTRA_HEADER + 2 * (eb + i)] = e;
                    extra[CQ_MOE_EXTRA_HEADER + 2 * (eb + i) + 1] = i + 1;
                }
            }
            const int cc = (c + chunk - 1) / chunk;
            if (cc > 0) {
                const int cb = atomicAdd(&n_chunks, cc);
                for (int i = 0; i < cc; i++) {
                    chunks[1 + cb + i] = e;
                    chunks[1 + max_chunks + cb + i] = start + i * chunk;
                    chunks[1 + 2 * max_chunks + cb + i] = min(chunk, c - i * chunk);
                }
            }
        }
        __syncthreads();
        if (tid == width - 1) carry += buf[tid];              // the inclusive sum of the sweep
        __syncthreads();
    }
    if (tid == 0) {
        offsets[E] = carry;
        chunks[0] = n_chunks;
        if (extra) { extra[0] = n_extra; extra[1] = 0; extra[2] = 0; }         // the list's length, and the two launches' counters
    }
    // positions behind the last valid pair are never part of a chunk, but the gathering quantizer walks all n_pairs
    // rows: give them a valid source row
    for (int p = carry + tid; p < ps.n_pairs; p += 1024) pair_in[p] = 0;
    auto place = [&](int p, bool ok, int e, int in_row, int out_row, float scale) {
        if (ok) {
            int pos = atomicAdd(&cur[e], 1);
            pair_in[pos] = in_row;
            pair_out[pos] = out_row;
            pair_scale[pos] = scale;
        } else if (ps.mode == MOE_INDEXED) {
            for (int c = 0; c < n; c++) out[(int64_t)p * n + c] = 0.0f;   // id out of range: defined output
        }
    };
#pragma unroll
    for (int i = 0; i < KEEP; i++)
        if (tid + i * 1024 < ps.n_pairs) place(tid + i * 1024, kok[i], ke[i], kin[i], kout[i], ksc[i]);
    for (int p = tid + KEEP * 1024; p < ps.n_pairs; p += 1024) {
        int e, in_row, out_row;
        float scale;
        const bool ok = pair_decode(ps, p, e, in_row, out_row, scale);
        place(p, ok, e, in_row, out_row, scale);
    }
}

// The same with a workgroup per expert, for lists of (expert, token) pairs of up to GROUP_WIDE_EXPERTS experts: every workgroup counts the whole list in LDS, which
// comes out of the L2, and then places the pairs of its own expert.  One workgroup for all of them takes 1.7 us per 1000 pairs: its loads, atomics and
// stores wait for each other on one unit (12000 pairs of 128 experts 25.8 -> 9.6 us; a layer of 256 tokens 142 -> 138).  That every workgroup reads the whole list shows
// where there are many: beyond 512 experts, one round of workgroups, up to 4096 pairs are grouped by one (a call of 1024 experts in us, by one / by all: 600 pairs 40.0 /
// 44.3, 2400: 57.6 / 58.7, 5000: 69.4 / 66.1, 12000: 96.9 / 87.8; in a list sorted by expert 5000: 64.1 / 66.8, 12000: 85.8 / 89.3, 48000: 266 / 239).
// inverse: pair_in[p] is the place of pair p (-1: none) instead of the row at a place.
constexpr int GROUP_WIDE_EXPERTS = 1024, GROUP_WIDE_ROUND = 512, GROUP_WIDE_PAIRS = 4096;
// From here on the pairs of a token are quantized once: fewer take no longer by a wave for each row of a pair (a call of 600 Q8_0 pairs on 512 experts in us, once / pair by
// pair: 40.6 / 39.8, on 128: 64.0 / 63.5, 1200: 65.7 / 67.4; sorted by expert 600 on 512: 42.8 / 39.8, 1200 on 128: 69.3 / 68.4, 2400: 76.5 / 74.3; 2400 in token order 72.2 /
// 74.7, 12000: 161 / 174).
constexpr int SPREAD_PAIRS = 2048;
__global__ __launch_bounds__(1024) void moe_group_wide_kernel(PairSource ps, int *__restrict__ offsets, int *__restrict__ pair_in, int *__restrict__ pair_out,
                                                              float *__restrict__ pair_scale, int *__restrict__ chunks, int max_chunks, int chunk,
                                                              int *__restrict__ extra, int inverse) {
    __shared__ int cnt[GROUP_WIDE_EXPERTS], before[4], own;
    const int tid = threadIdx.x, e = blockIdx.x, E = ps.num_experts, n = ps.n_pairs;
    // tokens below this have a row and, where rows are weighed, a weight
    const int limit = (int)min((int64_t)n, ps.topk_weights ? (int64_t)ps.x_rows : (int64_t)ps.x_rows * ps.topk);
    for (int i = tid; i < E; i += 1024) cnt[i] = 0;
    if (tid == 0) own = 0;
    __syncthreads();
    constexpr int U = 6;                       // pairs of a thread asked for at a time
    auto each = [&](auto &&f) {
        for (int p0 = tid; p0 < n; p0 += U * 1024) {
            int ke[U], to[U];
#pragma unroll
            for (int i = 0; i < U; i++) {
                ke[i] = ps.expert_ids[min(p0 + 1024 * i, n - 1)];
                to[i] = ps.sorted_token_ids[min(p0 + 1024 * i, n - 1)];
            }
#pragma unroll
            for (int i = 0; i < U; i++)
                if (p0 + 1024 * i < n) f(p0 + 1024 * i, (uint32_t)ke[i] < (uint32_t)E && to[i] >= 0 && to[i] < limit, ke[i], to[i]);
        }
    };
    // pairs of one expert in a row, as in a list sorted by expert, are counted by the first of them: one by one their lanes would wait for each other (48000 sorted pairs
    // of 512 experts: a call of 207 us takes 161)
    each([&](int, bool ok, int expert, int) {
        const int lane = tid & 63, x = ok ? expert : -1;
        const bool head = __builtin_amdgcn_update_dpp(-2, x, 0x138, 0xf, 0xf, false) != x;      // (the lane before; -2 in front of the first)
        const uint64_t heads = __ballot(head), here = __ballot(1);
        int count = 1;
        if (heads != here) {
            const uint64_t after = heads >> lane >> 1;
            count = after ? __builtin_ctzll(after) + 1 : __popcll(here) - lane;
        }
        if (head && ok) atomicAdd(&cnt[x], count);
    });
    __syncthreads();
    auto passes = [](int c) { return c > 32 ? (c + 31) / 32 - 1 : 0; };       // (of an expert's pairs beyond the first 32, for the batched matvecs)
    if (tid < 64) {
        int sum[4] = {0, 0, 0, 0};
        for (int i = tid; i < E; i += 64) {
            const int c = cnt[i];
            sum[3] += c;
            if (i < e) {
                sum[0] += c;
                sum[1] += (c + chunk - 1) / chunk;
                sum[2] += passes(c);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            for (int o = 32; o; o >>= 1) sum[i] += __shfl_xor(sum[i], o, 64);
            if (tid == 0) before[i] = sum[i];
        }
    }
    __syncthreads();
    const int c = cnt[e], start = before[0], n_chunks = (c + chunk - 1) / chunk, cb = before[1], n_extra = extra ? passes(c) : 0, eb = before[2], all = before[3];
    if (tid == 0) {
        offsets[e] = start;
        if (e == E - 1) {
            offsets[E] = all;
            chunks[0] = cb + n_chunks;
            if (extra) { extra[0] = eb + n_extra; extra[1] = 0; extra[2] = 0; }
        }
    }
    for (int i = tid; i < n_chunks; i += 1024) {
        chunks[1 + cb + i] = e;
        chunks[1 + max_chunks + cb + i] = start + i * chunk;
        chunks[1 + 2 * max_chunks + cb + i] = min(chunk, c - i * chunk);
    }
    for (int i = tid; i < n_extra; i += 1024) {
        extra[CQ_MOE_EXTRA_HEADER + 2 * (eb + i)] = e;
        extra[CQ_MOE_EXTRA_HEADER + 2 * (eb + i) + 1] = i + 1;
    }
    each([&](int p, bool ok, int x, int tok) {
        if (ok && x == e) {
            const int pos = start + atomicAdd(&own, 1);
            if (inverse) pair_in[p] = pos;
            else pair_in[pos] = ps.topk_weights ? tok : tok / ps.topk;
            pair_out[pos] = tok;
            pair_scale[pos] = ps.topk_weights ? ps.topk_weights[tok] : 1.0f;
        }
        if (!ok && inverse && e == 0) pair_in[p] = -1;
    });
    // places behind the last valid pair are in no chunk, but a gathering quantizer walks all of them
    if (!inverse && e == 0)
        for (int p = all + tid; p < n; p += 1024) pair_in[p] = 0;
}

// Workgroup (blockIdx.x = row tile, blockIdx.y = expert); 4 waves x R rows.  Pairs of the expert are
// taken PB at a time with the decoded weight registers held across them.
template <int DT, int R, int PB>
__global__ __launch_bounds__(256) void moe_matvec_kernel(const uint8_t *__restrict__ w, ActView av, float *__restrict__ out,
                                                         const int *__restrict__ offsets, const int *__restrict__ pair_in,
                                                         const int *__restrict__ pair_out, const float *__restrict__ pair_scale,
                                                         int k, int n) {
    typedef Fmt<DT> F;
    const int e = blockIdx.y;
    const int seg0 = offsets[e], seg1 = offsets[e + 1];
    if (seg0 == seg1) return;
    const int lane = threadIdx.x & 63;
    const int64_t row0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
    if (row0 >= n) return;
    const int nblk = k / BlockInfo<DT>::elems;
    const int units = nblk * F::UPB;
    const int64_t row_bytes = (int64_t)nblk * BlockInfo<DT>::bytes;
    const uint8_t *we = w + (int64_t)e * n * row_bytes;

    for (int s0 = seg0; s0 < seg1; s0 += PB) {
        int arow[PB];
#pragma unroll
        for (int b = 0; b < PB; b++) arow[b] = pair_in[s0 + b < seg1 ? s0 + b : seg1 - 1];
        float acc[R][PB];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int b = 0; b < PB; b++) acc[r][b] = 0.0f;

        ActRow arow_p[PB];
#pragma unroll
        for (int b = 0; b < PB; b++) arow_p[b] = act_row(av.qs, av.d, av.bsums, DT, arow[b], k);
        for (int u = lane; u < units; u += CQ_WAVE) {
            typename F::W wr[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                int64_t row = row0 + r < n ? row0 + r : n - 1;
                F::load_w(wr[r], we + row * row_bytes, u);
            }
            typename F::A ar[PB];
#pragma unroll
            for (int b = 0; b < PB; b++) F::load_a(ar[b], arow_p[b], u);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int b = 0; b < PB; b++) acc[r][b] += F::dot(wr[r], ar[b], u);
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int b = 0; b < PB; b++) {
                float v = wave_sum(acc[r][b]);
                if (lane == 0 && row0 + r < n && s0 + b < seg1)
                    out[(int64_t)pair_out[s0 + b] * n + row0 + r] = v * pair_scale[s0 + b];
            }
    }
}

template <int DT>
int launch_moe_matvec(const MoeArgs &a, const ActView &av, const int *offsets, const int *pin, const int *pout, const float *pscale,
                      hipStream_t s) {
    constexpr int R = 2, PB = 4;
    int64_t tiles = (a.n + 4 * R - 1) / (4 * R);
    if (tiles > 0x7fffffffLL || a.num_experts > 65535) return CQ_ERR_RANGE;
    hipLaunchKernelGGL((moe_matvec_kernel<DT, R, PB>), dim3((unsigned)tiles, (unsigned)a.num_experts), dim3(256), 0, s,
                       (const uint8_t *)a.w, av, a.out, offsets, pin, pout, pscale, (int)a.k, (int)a.n);
    return (int)hipGetLastError();
}

}  // namespace

int64_t cq_moe_workspace_bytes_impl(int w_dtype, int64_t num_experts, int64_t n_pairs, int64_t x_rows, int64_t k) {
    return moe_workspace(w_dtype, num_experts, n_pairs, x_rows, k).total;
}

// Does a call with this many pairs group them by expert and run the matrix-core kernel of the format over expert tiles?
static bool moe_takes_mfma(int w_dtype, const void *w, const void *w_b, int64_t n_pairs, int64_t k) {
    // (the matrix-core kernel of the 32-element formats copies weight rows in 8-byte pieces: experts at another alignment take
    // the matvec passes)
    const bool q0_ok = (w_dtype == CQ_Q4_0 || w_dtype == CQ_Q8_0) && ((uintptr_t)w & 7) == 0 && (!w_b || ((uintptr_t)w_b & 7) == 0);
    return k % 256 == 0 && (cq_is_kquant(w_dtype) || q0_ok) && cq_has_mfma(w_dtype) && n_pairs >= CQ_MOE_MFMA_MIN_PAIRS;
}
// Rows of a tile of one expert's pairs, 32, or 128 of which parts of 32 rows that are not there are left out.  A tile of 128 reads and converts an expert's weights once where those of 32 do it
// for every 32 pairs, but takes 5 - 20 % longer for the same rows: which is better depends on whether the second tiles of experts with more than 32 pairs fit into the rounds of workgroups that
// the first ones leave part-filled.  With p pairs an expert on average about (p - 18) / 22 of them have a second tile (between even and as uneven as those of a model), so:
// time in tiles of 128 over that in tiles of 32, p = 20, 24, 28, 33, 38 with even loads and, behind the bar, uneven ones:
//   Q8_0 16 experts of 2048 x 1024 (64 workgroups)  1.08 1.17 1.17 1.16 1.17 | 1.08 1.17 1.19 1.18 1.19      40 of 2048 x 1024 (160)  1.07 1.09 1.14 1.11 0.73 | 1.14 1.14 1.14 1.28 1.28
//   Q8_0 64 experts of 2048 x 1024 (256)  1.05 0.73 0.74 0.76 0.76 | 0.75 0.76 0.77 0.84 0.84      128 of 2048 x 768 (384)  1.08 1.09 1.11 0.88 0.89 | 1.13 1.20 0.94 0.94 0.93
//   Q6_K as Q8_0 (the first 1.09 1.09 1.16 1.16 1.15, the last 1.04 1.05 1.06 0.84 0.85), Q4_0 of more than 1024 columns too (24 of 4096 x 1280, 120: 1.06 1.06 1.19 1.19 1.18; 32 of 4096 x 2048,
//   256: 1.08 1.07 0.78 0.79 0.80).  Q4_K and Q5_K (what is not batched matvecs): a second tile pays up to 64 pairs
//   (32 rows by the batched matvecs 0.8 where 128 take 0.9 - 1.15 of their time, 64 and 96 workgroups).
// General kernels, whose tiles of 32 rows are 128 columns wide and those of 128 rows 64, over 780 shapes of 8 to 160 experts, time against the better of the two with the limit below (and without
// a split by workgroups): Q2_K 1.008 (at 27 1.026, at 60 1.017); Q3_K 1.026 (at 18 1.033, at 39 1.055), where 39 is the better one for few workgroups; Q6_K of rows below 1536 1.024 (1.027, 1.085);
// Q4_0 of up to 1024 columns 1.044 (at 18 1.034, but up to 1.11 of what tiles of 32 rows took where this is at most 1.08; at 39 1.106).
// n, k: columns and rows' length of the weights (of a gate / up call, whose grouping the down projection takes over: of that call).
static int moe_tile_rows(int w_dtype, int64_t n_pairs, int64_t num_experts, int64_t n, int64_t k) {
    const int64_t wide = num_experts * ((n + 255) / 256), narrow = num_experts * ((n + 127) / 128), room = (wide + 255) / 256 * 256;
    int64_t small = 18 + 22 * (room - wide) / wide;        // pairs an expert up to which tiles of 32 rows are taken
    small = std::min<int64_t>(std::max<int64_t>(small, 18), w_dtype == CQ_Q4K || w_dtype == CQ_Q5K ? 64 : 39);
    if (w_dtype == CQ_Q4_0 && n <= 1024) small = narrow <= 64 ? 30 : 24;
    if (w_dtype == CQ_Q2K) small = 39;
    if (w_dtype == CQ_Q3K) small = narrow <= 64 ? 39 : 27;
    if (w_dtype == CQ_Q6K && k < 1536) small = narrow <= 224 ? 30 : 21;
    return n_pairs < (small + 1) * num_experts ? CQ_MOE_TILE_SMALL : CQ_MOE_TILE_LARGE;
}

// Gate and up in one launch, which has tiles of 128 rows whatever their number (twice as many workgroups as a launch for one of them): from 19 pairs an expert on where a
// product is not batched matvecs, and from 28 where it is: a layer gains more by the one launch.  us of a layer, each product batched / gate and up in one launch: 12 experts of 2560 x 1024, 28 each,
// Q4_K 85 65, Q5_K 90 77, 16 and 50 each 106 71, 111 84, 6 and 50 76 64, 79 76; 8 of 2048 x 512, 50 each, 56 53, 58 63 (few and short ones of Q5_K are what loses: 150 layers of 6 - 32 experts
// 0.90 on average, 11 of them above 1.04, 1.21 at most; Q4_K 0.81 and 1.04).
static bool moe_swiglu_pairs(int w_dtype, int64_t num_experts, int64_t n_pairs, int64_t k, int64_t n) {
    return n_pairs >= 19 * num_experts && (n_pairs > 27 * num_experts || !cq_moe_stream_shape(w_dtype, num_experts, n_pairs, k, n));
}

int cq_moe_down_after_pair_launch(int w_dtype, const void *w_down, const float *gate, const float *up, const float *topk_weights, float *out,
                                  int64_t num_experts, int64_t topk, int64_t n_pairs, int64_t n, int64_t k, int64_t k_pair, void *workspace,
                                  hipStream_t s) {
    if (n_pairs > 0x7fffffffLL || topk <= 0 || n_pairs % topk) return CQ_ERR_RANGE;
    // what the gate / up call did with these pairs, and what this one needs
    // (K-quants only: whether Q4_0 / Q8_0 experts were grouped for the matrix cores also depended on that call's weight addresses)
    if (!cq_is_kquant(w_dtype)) return CQ_ERR_RANGE;
    if (cq_moe_direct(w_dtype, num_experts, n_pairs, k_pair) || !moe_takes_mfma(w_dtype, nullptr, nullptr, n_pairs, k_pair)) return CQ_ERR_RANGE;
    if (!moe_takes_mfma(w_dtype, w_down, nullptr, n_pairs, k)) return CQ_ERR_RANGE;
    const MoeWorkspace ws = moe_workspace(w_dtype, num_experts, n_pairs, n_pairs / topk, k_pair);
    // the pair call ran its experts as batched matvecs (chunks of 16 pairs): this one must be able to as well
    // (n of the pair call = this call's k; its expert tensors were 16-byte aligned or it returned CQ_ERR_ALIGN)
    if (!up && !moe_swiglu_pairs(w_dtype, num_experts, n_pairs, k_pair, k)) return CQ_ERR_RANGE;
    if (up && cq_moe_stream_shape(w_dtype, num_experts, n_pairs, k_pair, k)) {
        if (!cq_moe_stream_takes(w_dtype, w_down, nullptr, num_experts, n_pairs, k, n)) return CQ_ERR_RANGE;
        if (cq_align256(cq_moe_stream_operand_bytes(num_experts, n_pairs, k)) > ws.offsets_off) return CQ_ERR_RANGE;
        uint8_t *b = (uint8_t *)workspace;
        const int *offsets = (const int *)(b + ws.offsets_off);
        const int *pout = (const int *)(b + ws.pout_off);
        float *pscale = (float *)(b + ws.pscale_off);
        const int *chunks = (const int *)(b + ws.chunk_off);
        int rc = cq_moe_stream_quantize_launch(gate, up, pout, topk_weights, pscale, chunks, ws.max_chunks, num_experts, n_pairs, offsets, b + ws.act_off, k, s);
        if (rc) return rc;
        return cq_moe_stream_launch(w_dtype, w_down, nullptr, out, nullptr, b + ws.act_off, offsets, pout, pscale, (int *)(b + ws.extra_off), 1,
                                    num_experts, k, n, s);
    }
    // the rows of this call are quantized into the front of the workspace: they must end before that call's tables begin
    if (cq_act_layout(w_dtype, k, ws.rows_alloc).total > ws.offsets_off) return CQ_ERR_RANGE;
    uint8_t *b = (uint8_t *)workspace;
    const int *pout = (const int *)(b + ws.pout_off);
    float *pscale = (float *)(b + ws.pscale_off);
    const int *chunks = (const int *)(b + ws.chunk_off);
    // pair i of the expert-sorted list reads row pair_out[i] (one row per pair here) and is scaled by that pair's routing weight
    const int *n_valid = (const int *)(b + ws.offsets_off) + num_experts;          // the end of the last expert's segment
    int rc = cq_quantize_act_swiglu_gather_launch(w_dtype, gate, up, pout, n_valid, topk_weights, pscale, b + ws.act_off, k, n_pairs, ws.rows_alloc, s);
    if (rc) return rc;
    MoeChunks mc{chunks, chunks + 1, chunks + 1 + ws.max_chunks, chunks + 1 + 2 * ws.max_chunks, pout, pscale, (int)ws.max_chunks};
    const int tile_rows = up ? moe_tile_rows(w_dtype, n_pairs, num_experts, k, k_pair) : CQ_MOE_TILE_LARGE;
    return cq_matmul_moe_launch(w_dtype, w_down, b + ws.act_off, ws.rows_alloc, out, mc, num_experts, k, n, tile_rows, s);
}

int cq_moe_launch(const MoeArgs &a, void *workspace, hipStream_t s) {
    if (a.n_pairs > 0x7fffffffLL || a.x_rows > 0x7fffffffLL) return CQ_ERR_RANGE;
    const bool mfma = moe_takes_mfma(a.w_dtype, a.w, a.w_b, a.n_pairs, a.k);
    const bool stream_shape = mfma && !a.swiglu && !cq_moe_direct(a.w_dtype, a.num_experts, a.n_pairs, a.k) && cq_moe_stream_shape(a.w_dtype, a.num_experts, a.n_pairs, a.k, a.n);
    const bool stream = stream_shape && cq_moe_stream_takes(a.w_dtype, a.w, a.w_b, a.num_experts, a.n_pairs, a.k, a.n);
    // (a later cq_moe_down_after_pair_launch tells from the shape alone how this call chunked its pairs)
    if (a.w_b && stream_shape && !stream) return CQ_ERR_ALIGN;
    if (a.swiglu && (!mfma || cq_moe_direct(a.w_dtype, a.num_experts, a.n_pairs, a.k) || !moe_swiglu_pairs(a.w_dtype, a.num_experts, a.n_pairs, a.k, a.n) ||
                     a.x_rows * a.k > 0x7fffffffLL ||                          // (tokens' rows are named by 32-bit offsets)
                     !cq_qtile_moe_takes_swiglu(a.w_dtype, a.w, a.w_b, a.num_experts, a.k, a.n)))
        return CQ_ERR_RANGE;
    if (a.w_b && !mfma) {
        // only the MFMA path shares its grouping pass and quantized activations between two weight tensors
        MoeArgs one = a;
        one.w_b = nullptr; one.out_b = nullptr;
        int rc = cq_moe_launch(one, workspace, s);
        if (rc) return rc;
        one.w = a.w_b; one.out = a.out_b;
        return cq_moe_launch(one, workspace, s);
    }
    PairSource ps;
    ps.mode = a.mode; ps.ids_u32 = a.ids_u32; ps.sorted_token_ids = a.sorted_token_ids; ps.expert_ids = a.expert_ids;
    ps.topk_weights = a.topk_weights; ps.topk = (int)a.topk; ps.input_dim1 = (int)a.input_dim1;
    ps.n_pairs = (int)a.n_pairs; ps.num_experts = (int)a.num_experts; ps.x_rows = (int)a.x_rows;
    // Few pairs (decode): every pair is its own fused matvec (activation quantization in the kernel, no scratch,
    // no grouping pass); an expert hit by two pairs is simply read twice, the second time from cache.
    if (cq_moe_direct(a.w_dtype, a.num_experts, a.n_pairs, a.k)) {
        int rc = cq_moe_pairs_launch(a.w_dtype, a.w, a.x, a.out, ps, a.k, a.n, s);
        if (rc != CQ_ERR_RANGE) return rc;
    }
    MoeWorkspace ws = moe_workspace(a.w_dtype, a.num_experts, a.n_pairs, a.x_rows, a.k);
    uint8_t *b = (uint8_t *)workspace;
    int rc;
    int *offsets = (int *)(b + ws.offsets_off), *cursor = (int *)(b + ws.cursor_off);
    int *pin = (int *)(b + ws.pin_off), *pout = (int *)(b + ws.pout_off);
    float *pscale = (float *)(b + ws.pscale_off);
    int *chunks = (int *)(b + ws.chunk_off);
    int *extra = (int *)(b + ws.extra_off);
    // Hundreds of pairs per call: the expert-sorted rows go through the MFMA prefill kernel of the format in tiles of up to
    // 128 rows of one expert (integer-exact like the dense paths).  Otherwise 8 pairs per matvec pass.
    const int tile_rows = a.swiglu ? CQ_MOE_TILE_LARGE : moe_tile_rows(a.w_dtype, a.n_pairs, a.num_experts, a.n, a.k);
    const bool many = a.n_pairs > GROUP_MANY_PAIRS;
    auto *const group = a.num_experts <= GROUP_LDS_EXPERTS ? (many ? moe_group_kernel<true, true> : moe_group_kernel<true, false>)
                                                           : (many ? moe_group_kernel<false, true> : moe_group_kernel<false, false>);
    const int chunk = stream ? CQ_MOE_STREAM_CHUNK : mfma ? tile_rows : CQ_MOE_CHUNK;
    const bool wide = a.mode != MOE_INDEXED && (a.num_experts <= GROUP_WIDE_ROUND || (a.num_experts <= GROUP_WIDE_EXPERTS && a.n_pairs > GROUP_WIDE_PAIRS));
    // pairs of the gate / up products: the same row goes to all experts of a token
    const bool spread = wide && mfma && !stream && !a.swiglu && !a.topk_weights && a.topk > 1 && a.n_pairs > SPREAD_PAIRS;
    if (wide)
        hipLaunchKernelGGL(moe_group_wide_kernel, dim3((unsigned)a.num_experts), dim3(1024), 0, s, ps, offsets, pin, pout, pscale, chunks, (int)ws.max_chunks, chunk,
                           stream ? extra : nullptr, (int)spread);
    else
        hipLaunchKernelGGL(group, dim3(1), dim3(1024), 0, s, ps, offsets, cursor, pin, pout, pscale, a.out, (int)a.n, chunks, (int)ws.max_chunks, chunk,
                           stream ? extra : nullptr);
    if ((rc = (int)hipGetLastError())) return rc;
    if (stream) {
        // every expert a batched matvec over its own pairs: the weights of an expert are streamed once per 32 pairs
        if (cq_align256(cq_moe_stream_operand_bytes(a.num_experts, a.n_pairs, a.k)) > ws.offsets_off) return CQ_ERR_RANGE;      // (the workspace layout above reserves it)
        if ((rc = cq_moe_stream_quantize_launch(a.x, nullptr, pin, nullptr, nullptr, chunks, ws.max_chunks, a.num_experts, a.n_pairs, offsets, b + ws.act_off, a.k, s))) return rc;
        return cq_moe_stream_launch(a.w_dtype, a.w, a.w_b, a.out, a.out_b, b + ws.act_off, offsets, pout, pscale, extra, 0, a.num_experts, a.k, a.n, s);
    }
    if (mfma) {
        // gate and up in one launch: each token's row once, and the product asks for the rows that its pairs name (1500 rows of 2048, 8 pairs each: 12.9 us for a copy to every pair -> 5.9;
        // the product waits a memory trip longer for its first rows, 130.2 us for 128.1)
        rc = a.swiglu ? cq_quantize_act_launch(a.w_dtype, a.x, CQ_F32, b + ws.act_off, a.k, a.x_rows, s)
             : spread ? cq_quantize_act_spread_launch(a.w_dtype, a.x, a.sorted_token_ids, pin, a.topk, b + ws.act_off, a.k, a.n_pairs, ws.rows_alloc, s)
                      : cq_quantize_act_gather_launch(a.w_dtype, a.x, pin, b + ws.act_off, a.k, a.n_pairs, ws.rows_alloc, s);
        if (rc) return rc;
        MoeChunks mc{chunks, chunks + 1, chunks + 1 + ws.max_chunks, chunks + 1 + 2 * ws.max_chunks, pout, pscale, (int)ws.max_chunks};
        if (a.swiglu) {
            mc.src = pin;
            return cq_qtile_moe_swiglu_launch(a.w_dtype, a.w, a.w_b, cq_act_view(b + ws.act_off, a.w_dtype, a.k, a.x_rows), a.out, mc, a.num_experts, a.n_pairs, a.k, a.n, s);
        }
        rc = cq_matmul_moe_launch(a.w_dtype, a.w, b + ws.act_off, ws.rows_alloc, a.out, mc, a.num_experts, a.k, a.n, tile_rows, s);
        if (!rc && a.w_b) rc = cq_matmul_moe_launch(a.w_dtype, a.w_b, b + ws.act_off, ws.rows_alloc, a.out_b, mc, a.num_experts, a.k, a.n, tile_rows, s);
        return rc;
    }
    if (a.k % 256 == 0) {
        // Many pairs: activation rows quantized in expert-sorted order, then CQ_MOE_CHUNK pairs of an expert per pass
        // over its rows (the matvec body with 8 activation rows in LDS).
        if ((rc = cq_quantize_act_gather_launch(a.w_dtype, a.x, pin, b + ws.act_off, a.k, a.n_pairs, ws.rows_alloc, s))) return rc;
        MoeChunks mc{chunks, chunks + 1, chunks + 1 + ws.max_chunks, chunks + 1 + 2 * ws.max_chunks, pout, pscale, (int)ws.max_chunks};
        rc = cq_moe_chunks_launch(a.w_dtype, a.w, b + ws.act_off, ws.rows_alloc, a.out, mc, a.k, a.n, s);
        if (rc != CQ_ERR_RANGE) return rc;
    }
    if ((rc = cq_quantize_act_launch(a.w_dtype, a.x, CQ_F32, b + ws.act_off, a.k, a.x_rows, s))) return rc;
    ActView av = cq_act_view(b + ws.act_off, a.w_dtype, a.k, a.x_rows);
    switch (a.w_dtype) {
        case CQ_Q4_0: return launch_moe_matvec<CQ_Q4_0>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q8_0: return launch_moe_matvec<CQ_Q8_0>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q4K: return launch_moe_matvec<CQ_Q4K>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q5K: return launch_moe_matvec<CQ_Q5K>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q6K: return launch_moe_matvec<CQ_Q6K>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q2K: return launch_moe_matvec<CQ_Q2K>(a, av, offsets, pin, pout, pscale, s);
        case CQ_Q3K: return launch_moe_matvec<CQ_Q3K>(a, av, offsets, pin, pout, pscale, s);
    }
    return CQ_ERR_DTYPE;
}
