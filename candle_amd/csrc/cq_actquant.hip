// Stand-alone activation quantization kernels: one wave64 per 256-element span, writing the
// device-private scratch layout of cq_device.h.  The arithmetic lives in cq_actquant.h.
#include "cq_actquant.h"
#include "cq_launch.h"

namespace {

template <int XDT>
__global__ __launch_bounds__(256) void quantize_q8k_kernel(const void *__restrict__ x, int8_t *__restrict__ qs,
                                                           float *__restrict__ dout, int16_t *__restrict__ bsums, int64_t n_blocks) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= n_blocks) return;
    cq_quantize_q8k_span<XDT>(x, blk, threadIdx.x & 63, qs, dout, bsums);
}

template <int XDT>
__global__ __launch_bounds__(256) void quantize_q80_kernel(const void *__restrict__ x, int8_t *__restrict__ qs,
                                                           float *__restrict__ ds, int64_t total) {
    const int64_t span = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    cq_quantize_q80_span<XDT>(x, span, threadIdx.x & 63, total, qs, ds);
}

// Gathering variants (f32 rows): destination row i of the scratch is row row_map[i] of x.  k is a multiple of 256.
__global__ __launch_bounds__(256) void quantize_q8k_gather_kernel(const float *__restrict__ x, const int *__restrict__ row_map, int kb,
                                                                  int8_t *__restrict__ qs, float *__restrict__ dout, int16_t *__restrict__ bsums,
                                                                  int64_t n_blocks) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= n_blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = blk / kb, b = blk - row * kb;
    float v[4];
    cq_load4<CQ_F32>(x, ((int64_t)row_map[row] * kb + b) * 256 + lane * 4, v);
    cq_quantize_q8k_vals(v, blk, lane, qs, dout, bsums);
}
__global__ __launch_bounds__(256) void quantize_q80_gather_kernel(const float *__restrict__ x, const int *__restrict__ row_map, int kb,
                                                                  int8_t *__restrict__ qs, float *__restrict__ ds, int64_t n_spans) {
    const int64_t span = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (span >= n_spans) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = span / kb, b = span - row * kb;
    float v[4];
    cq_load4<CQ_F32>(x, ((int64_t)row_map[row] * kb + b) * 256 + lane * 4, v);
    cq_quantize_q80_vals(v, true, span * 256 + lane * 4, lane, qs, ds);
}

// Spreading variant: every pair of a list of (row of x, place in the scratch) gets its row.  A wave takes `group` pairs that follow each other.  In a list in token order
// they share a row, which is quantized once: 12000 pairs of 1500 rows of 2048, 30.4 -> 12.9 us, of which the 28 MB written take 6.  In a list sorted by expert they are as many
// rows: those of eight pairs are asked for before the first is quantized, and no wave has more than sixteen (a call of 12000 pairs, 64 of them a token: 104 -> 67 us sorted, 66 ->
// 58 in token order).
constexpr int SPREAD_GROUP = 16;
template <bool Q8K>
__global__ __launch_bounds__(256) void quantize_spread_kernel(const float *__restrict__ x, const int *__restrict__ tokens, const int *__restrict__ place, int topk, int group,
                                                              int n_pairs, int kb, int8_t *__restrict__ qs, float *__restrict__ dout, int16_t *__restrict__ bsums,
                                                              int64_t n_units) {
    constexpr int U = 8;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (unit >= n_units) return;
    const int lane = threadIdx.x & 63;
    const int64_t g = unit / kb, b = unit - g * kb, p = g * group + lane;
    const bool live = lane < group && p < n_pairs;
    const int to = live ? place[p] : -1, from = live ? tokens[p] / topk : 0;       // (negative: a pair that names no expert or row)
    int row = -1;                              // the row in q8k / q80
    Q8kBlock q8k;
    Q80Block q80;
    for (int j0 = 0; j0 < group; j0 += U) {
        float v[U][4];
        bool other[U];                         // than the row before
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int t = __builtin_amdgcn_readlane(to, j0 + j), f = __builtin_amdgcn_readlane(from, j0 + j);
            other[j] = t >= 0 && f != row;
            if (!other[j]) continue;
            cq_load4<CQ_F32>(x, ((int64_t)f * kb + b) * 256 + lane * 4, v[j]);
            row = f;
        }
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int t = __builtin_amdgcn_readlane(to, j0 + j);
            if (t < 0) continue;
            if (other[j]) {
                if (Q8K) q8k = cq_quantize_q8k_regs(v[j], lane);
                else q80 = cq_quantize_q80_regs(v[j]);
            }
            const int64_t blk = (int64_t)t * kb + b;
            if (Q8K) q8k.store(blk, lane, qs, dout, bsums);
            else q80.store(blk * 256 + lane * 4, lane, qs, dout);
        }
    }
}

__global__ __launch_bounds__(256) void quantize_q8k_swiglu_kernel(const float *__restrict__ gate, const float *__restrict__ up, int64_t gate_stride,
                                                                  int64_t up_stride, int kb, int8_t *__restrict__ qs, float *__restrict__ dout,
                                                                  int16_t *__restrict__ bsums, int64_t n_blocks) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= n_blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = blk / kb, off = (blk - row * kb) * 256 + lane * 4;
    float v[4];
    cq_load_swiglu4(gate, up, row * gate_stride + off, row * up_stride + off, v);
    cq_quantize_q8k_vals(v, blk, lane, qs, dout, bsums);
}
__global__ __launch_bounds__(256) void quantize_q80_swiglu_kernel(const float *__restrict__ gate, const float *__restrict__ up, int64_t gate_stride,
                                                                  int64_t up_stride, int kb, int8_t *__restrict__ qs, float *__restrict__ ds,
                                                                  int64_t n_spans) {
    const int64_t span = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (span >= n_spans) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = span / kb, off = (span - row * kb) * 256 + lane * 4;
    float v[4];
    cq_load_swiglu4(gate, up, row * gate_stride + off, row * up_stride + off, v);
    cq_quantize_q80_vals(v, true, span * 256 + lane * 4, lane, qs, ds);
}

// rms_norm_kernel of cq_nn.hip (the same sums in the same order) for rows of which only the quantized form is wanted: a workgroup's wave has 256 elements that follow each other, a
// block, in registers.  Bound by memory (1000 rows of 4096: 52 MB, 11 us at the rate of a copy): 16 us in a llama's prompt, where norm and quantizers, one for each format, took 12 + 2 x 6.8 in front
// of attention and 12 + 6.8 in front of the feed-forward (1000 tokens, four layers: 2956 -> 2901 us).
template <int KEEP>
__global__ __launch_bounds__(256) void quantize_q8k_norm_kernel(const float *x, const float *__restrict__ delta, const float *__restrict__ w, float *sum_out, int dim, float eps,
                                                                int8_t *__restrict__ qs, float *__restrict__ dout, int16_t *__restrict__ bsums) {
    __shared__ float red[4];
    const int64_t base = (int64_t)blockIdx.x * dim;
    const int n4 = dim >> 2, lane = threadIdx.x & 63;
    const f32x4 *const x4 = reinterpret_cast<const f32x4 *>(x + base), *const d4 = reinterpret_cast<const f32x4 *>(delta + base), *const w4 = reinterpret_cast<const f32x4 *>(w);
    f32x4 keep[KEEP], a[KEEP];
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < KEEP; c++) {
        const int i = threadIdx.x + 256 * c;
        if (i >= n4) continue;                             // (whole waves: rows are whole blocks)
        keep[c] = x4[i];
        if (delta) keep[c] += d4[i];
        a[c] = w4[i];
    }
#pragma unroll
    for (int c = 0; c < KEEP; c++) {
        const int i = threadIdx.x + 256 * c;
        if (i >= n4) continue;
        if (sum_out) reinterpret_cast<f32x4 *>(sum_out + base)[i] = keep[c];
#pragma unroll
        for (int e = 0; e < 4; e++) acc += keep[c][e] * keep[c][e];
    }
    acc = wave_sum(acc);
    if (lane == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float m = sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)dim + eps);
#pragma unroll
    for (int c = 0; c < KEEP; c++) {
        const int i = threadIdx.x + 256 * c;
        if (i >= n4) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = keep[c][e] / m * a[c][e];
        cq_quantize_q8k_vals(v, (int64_t)blockIdx.x * (dim >> 8) + (i >> 6), lane, qs, dout, bsums);
    }
}

template <int XDT>
int launch_quantize_act(int w_dtype, const void *x, void *scratch, int64_t k, int64_t rows, hipStream_t s) {
    ActLayout L = cq_act_layout(w_dtype, k, rows);
    uint8_t *b = (uint8_t *)scratch;
    int64_t total = rows * k;
    int64_t spans = (total + 255) / 256;
    if (spans == 0) return CQ_OK;
    int64_t grid = (spans + 3) / 4;
    if (grid > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (cq_is_kquant(w_dtype))
        hipLaunchKernelGGL((quantize_q8k_kernel<XDT>), dim3((unsigned)grid), dim3(256), 0, s, x, (int8_t *)(b + L.qs_off),
                           (float *)(b + L.d_off), (int16_t *)(b + L.bs_off), total / 256);
    else
        hipLaunchKernelGGL((quantize_q80_kernel<XDT>), dim3((unsigned)grid), dim3(256), 0, s, x, (int8_t *)(b + L.qs_off),
                           (float *)(b + L.d_off), total);
    return (int)hipGetLastError();
}

// Scratch row i = quantized silu(gate[row_map[i]]) * up[row_map[i]] (rows of k contiguous floats), and scale_out[i] =
// scale_in[row_map[i]], for i < *n_valid: the down projection of an expert MLP over pairs that an earlier call has bucketed by expert.  PLAIN: of gate alone.
template <bool PLAIN>
__global__ __launch_bounds__(256) void quantize_q8k_swiglu_gather_kernel(const float *__restrict__ gate, const float *__restrict__ up,
                                                                         const int *__restrict__ row_map, const int *__restrict__ n_valid,
                                                                         const float *__restrict__ scale_in, float *__restrict__ scale_out, int kb,
                                                                         int8_t *__restrict__ qs, float *__restrict__ dout,
                                                                         int16_t *__restrict__ bsums, int64_t n_blocks) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= n_blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = blk / kb, b = blk - row * kb;
    const int src = row < *n_valid ? row_map[row] : 0;          // (rows behind the last valid pair are in no tile: any valid source)
    const int64_t off = ((int64_t)src * kb + b) * 256 + lane * 4;
    float v[4];
    if constexpr (PLAIN) cq_load4<CQ_F32>(gate, off, v);
    else cq_load_swiglu4(gate, up, off, off, v);
    cq_quantize_q8k_vals(v, blk, lane, qs, dout, bsums);
    if (b == 0 && lane == 0) scale_out[row] = scale_in[src];
}
__global__ __launch_bounds__(256) void quantize_q80_swiglu_gather_kernel(const float *__restrict__ gate, const float *__restrict__ up,
                                                                         const int *__restrict__ row_map, const int *__restrict__ n_valid,
                                                                         const float *__restrict__ scale_in, float *__restrict__ scale_out, int kb,
                                                                         int8_t *__restrict__ qs, float *__restrict__ ds, int64_t n_spans) {
    const int64_t span = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (span >= n_spans) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = span / kb, b = span - row * kb;
    const int src = row < *n_valid ? row_map[row] : 0;          // (rows behind the last valid pair are in no tile: any valid source)
    const int64_t off = ((int64_t)src * kb + b) * 256 + lane * 4;
    float v[4];
    cq_load_swiglu4(gate, up, off, off, v);
    cq_quantize_q80_vals(v, true, span * 256 + lane * 4, lane, qs, ds);
    if (b == 0 && lane == 0) scale_out[row] = scale_in[src];
}

}  // namespace

// k is a multiple of the weight type's block size (256 for K-quants, 32 for Q4_0 / Q8_0); the API
// layer checks it.
int cq_quantize_act_launch(int w_dtype, const void *x, int x_dtype, void *scratch, int64_t k, int64_t rows, hipStream_t s) {
    switch (x_dtype) {
        case CQ_F32: return launch_quantize_act<CQ_F32>(w_dtype, x, scratch, k, rows, s);
        case CQ_F16: return launch_quantize_act<CQ_F16>(w_dtype, x, scratch, k, rows, s);
        case CQ_BF16: return launch_quantize_act<CQ_BF16>(w_dtype, x, scratch, k, rows, s);
    }
    return CQ_ERR_DTYPE;
}

// Scratch rows [0, rows) = quantized x[row_map[i]]; the layout is that of `rows_alloc` rows (rows_alloc >= rows).
int cq_quantize_act_gather_launch(int w_dtype, const float *x, const int *row_map, void *scratch, int64_t k, int64_t rows, int64_t rows_alloc,
                                  hipStream_t s) {
    if (k % 256) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    ActLayout L = cq_act_layout(w_dtype, k, rows_alloc);
    uint8_t *b = (uint8_t *)scratch;
    const int64_t spans = rows * (k / 256);
    const int64_t grid = (spans + 3) / 4;
    if (grid > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (cq_is_kquant(w_dtype))
        hipLaunchKernelGGL(quantize_q8k_gather_kernel, dim3((unsigned)grid), dim3(256), 0, s, x, row_map, (int)(k / 256), (int8_t *)(b + L.qs_off),
                           (float *)(b + L.d_off), (int16_t *)(b + L.bs_off), spans);
    else
        hipLaunchKernelGGL(quantize_q80_gather_kernel, dim3((unsigned)grid), dim3(256), 0, s, x, row_map, (int)(k / 256), (int8_t *)(b + L.qs_off),
                           (float *)(b + L.d_off), spans);
    return (int)hipGetLastError();
}

// Scratch row place[p] = quantized x[tokens[p] / topk] for the pairs p whose place is not negative; the layout is that of `rows_alloc` rows.
int cq_quantize_act_spread_launch(int w_dtype, const float *x, const int *tokens, const int *place, int64_t topk, void *scratch, int64_t k, int64_t n_pairs,
                                  int64_t rows_alloc, hipStream_t s) {
    if (k % 256) return CQ_ERR_SHAPE;
    if (n_pairs == 0) return CQ_OK;
    ActLayout L = cq_act_layout(w_dtype, k, rows_alloc);
    uint8_t *b = (uint8_t *)scratch;
    const int64_t group = topk < SPREAD_GROUP ? topk : SPREAD_GROUP, units = (n_pairs + group - 1) / group * (k / 256), grid = (units + 3) / 4;
    if (grid > 0x7fffffffLL) return CQ_ERR_RANGE;
    auto *const fn = cq_is_kquant(w_dtype) ? quantize_spread_kernel<true> : quantize_spread_kernel<false>;
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, s, x, tokens, place, (int)topk, (int)group, (int)n_pairs, (int)(k / 256), (int8_t *)(b + L.qs_off),
                       (float *)(b + L.d_off), (int16_t *)(b + L.bs_off), units);
    return (int)hipGetLastError();
}

// Scratch rows [0, rows) = quantized silu(gate[row_map[i]]) * up[row_map[i]] (without up, of K formats: gate[row_map[i]]), scale_out[i] = scale_in[row_map[i]].
int cq_quantize_act_swiglu_gather_launch(int w_dtype, const float *gate, const float *up, const int *row_map, const int *n_valid, const float *scale_in,
                                         float *scale_out, void *scratch, int64_t k, int64_t rows, int64_t rows_alloc, hipStream_t s) {
    if (k % 256) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    ActLayout L = cq_act_layout(w_dtype, k, rows_alloc);
    uint8_t *b = (uint8_t *)scratch;
    const int64_t spans = rows * (k / 256);
    const int64_t grid = (spans + 3) / 4;
    if (grid > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (!up && !cq_is_kquant(w_dtype)) return CQ_ERR_DTYPE;
    if (cq_is_kquant(w_dtype))
        hipLaunchKernelGGL(up ? quantize_q8k_swiglu_gather_kernel<false> : quantize_q8k_swiglu_gather_kernel<true>, dim3((unsigned)grid), dim3(256), 0, s, gate, up, row_map, n_valid, scale_in, scale_out, (int)(k / 256),
                           (int8_t *)(b + L.qs_off), (float *)(b + L.d_off), (int16_t *)(b + L.bs_off), spans);
    else
        hipLaunchKernelGGL(quantize_q80_swiglu_gather_kernel, dim3((unsigned)grid), dim3(256), 0, s, gate, up, row_map, n_valid, scale_in, scale_out, (int)(k / 256),
                           (int8_t *)(b + L.qs_off), (float *)(b + L.d_off), spans);
    return (int)hipGetLastError();
}

// Scratch rows [0, rows) = quantized silu(gate[r]) * up[r].  k is a multiple of 256; strides in floats, multiples of 4.
int cq_quantize_act_swiglu_launch(int w_dtype, const float *gate, const float *up, int64_t gate_stride, int64_t up_stride, void *scratch, int64_t k,
                                  int64_t rows, hipStream_t s) {
    if (k % 256) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    ActLayout L = cq_act_layout(w_dtype, k, rows);
    uint8_t *b = (uint8_t *)scratch;
    const int64_t spans = rows * (k / 256);
    const int64_t grid = (spans + 3) / 4;
    if (grid > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (cq_is_kquant(w_dtype))
        hipLaunchKernelGGL(quantize_q8k_swiglu_kernel, dim3((unsigned)grid), dim3(256), 0, s, gate, up, gate_stride, up_stride, (int)(k / 256),
                           (int8_t *)(b + L.qs_off), (float *)(b + L.d_off), (int16_t *)(b + L.bs_off), spans);
    else
        hipLaunchKernelGGL(quantize_q80_swiglu_kernel, dim3((unsigned)grid), dim3(256), 0, s, gate, up, gate_stride, up_stride, (int)(k / 256),
                           (int8_t *)(b + L.qs_off), (float *)(b + L.d_off), spans);
    return (int)hipGetLastError();
}

// Scratch rows = quantized rms_norm(x + delta) * w, sum_out (may be x) = x + delta.  dim: whole blocks of 256, at most 8192.
int cq_quantize_norm_launch(const float *x, const float *delta, const float *w, float *sum_out, void *scratch, int64_t dim, int64_t rows, float eps, hipStream_t s) {
    if (dim % 256 || dim > 8192 || rows > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (rows == 0) return CQ_OK;
    const ActLayout L = cq_act_layout(CQ_Q4K, dim, rows);
    uint8_t *const b = (uint8_t *)scratch;
    auto *const fn = dim <= 4096 ? quantize_q8k_norm_kernel<4> : quantize_q8k_norm_kernel<8>;
    hipLaunchKernelGGL(fn, dim3((unsigned)rows), dim3(256), 0, s, x, delta, w, sum_out, (int)dim, eps, (int8_t *)(b + L.qs_off), (float *)(b + L.d_off), (int16_t *)(b + L.bs_off));
    return (int)hipGetLastError();
}
