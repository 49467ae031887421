// Sequence mixers with a recurrent matrix state per head: linear attention with a fixed decay (retention) and the generalized
// delta rule.  States are f32 and stored by columns, [head][value column][state_pad]: a wave holds four columns with 16 lanes
// on the rows of each, so a step over one token needs 16-lane sums only.
#include "cq_mix.h"

namespace {

// ---- retention, several tokens ----------------------------------------------------------------------------------------------
// Chunks of 64 tokens on v_mfma_f32_16x16x4; workgroup: 4 waves on one head and 64 value columns.  With gamma the head's decay, i and j
// places in the chunk and S the state before it:
//   o_i = gamma^(i+1) S^T q_i + sum_{j<=i} gamma^(i-j) (q_i . k_j) v_j,     S' = gamma^n S + sum_j gamma^(n-1-j) k_j v_j^T
// A long call is cut into segments of whole chunks that run side by side: retention_segment_kernel leaves what each segment adds to the
// state (Z), retention_prefix_kernel turns Z into the state before each segment and forms the final one.
constexpr int RC = 64, RLD = 68;                     // chunk length; LDS row of 64 columns (16 rows x 4 fall on 64 banks)

struct Retention {
    const float *q, *k, *v, *log2_decay;
    float *state, *out, *z;
    int64_t v_stride, out_stride;
    int rows, heads, dp, vdim, sp, nvb, nseg, seg_len;      // sp: state_pad
};

__device__ __forceinline__ float *segment_z(const Retention &a, int h, int vb, int seg) {
    return a.z + (((int64_t)h * a.nvb + vb) * a.nseg + seg) * a.dp * 64;
}

// V of a chunk as operand: vf[s][n] = v[t0 + 4 s + lk][64 vb + 16 n + lr] (rows beyond the chunk repeat its last one: their weights are zero)
__device__ __forceinline__ void load_v(const Retention &a, int h, int vb, int t0, int n_tok, int lr, int lk, float (&vf)[16][4]) {
#pragma unroll
    for (int s = 0; s < 16; s++) {
        const float *vr = a.v + (int64_t)(t0 + min(4 * s + lk, n_tok - 1)) * a.v_stride + (int64_t)h * a.vdim;
#pragma unroll
        for (int n = 0; n < 4; n++) vf[s][n] = vr[min(64 * vb + 16 * n + lr, a.vdim - 1)];
    }
}

// acc[n] += sum_j gamma^(n_tok-1-j) k_j[16 dt + lr ...] v_j[...] over the chunk
__device__ __forceinline__ void add_kv(const Retention &a, int h, int dt, int t0, int n_tok, float l2, int lr, int lk, const float (&vf)[16][4],
                                       f32x4 (&acc)[4]) {
    float kf[16];
#pragma unroll
    for (int s = 0; s < 16; s++) kf[s] = a.k[((int64_t)(t0 + min(4 * s + lk, n_tok - 1)) * a.heads + h) * a.dp + 16 * dt + lr];
#pragma unroll
    for (int s = 0; s < 16; s++) {
        const int j = 4 * s + lk;
        const float kw = j < n_tok ? kf[s] * exp2f(l2 * (float)(n_tok - 1 - j)) : 0.0f;
#pragma unroll
        for (int n = 0; n < 4; n++) acc[n] = mfma4(kw, vf[s][n], acc[n]);
    }
}

__global__ __launch_bounds__(256) void retention_segment_kernel(Retention a) {
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const int h = blockIdx.x / a.nvb, vb = blockIdx.x % a.nvb, seg = blockIdx.y;
    const float l2 = a.log2_decay[h];
    const int t_end = min(a.rows, (seg + 1) * a.seg_len);
    float *z = segment_z(a, h, vb, seg);
    for (int dt = wv; dt < a.dp / 16; dt += 4) {
        f32x4 acc[4];
#pragma unroll
        for (int n = 0; n < 4; n++) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int t0 = seg * a.seg_len; t0 < t_end; t0 += RC) {
            const int n_tok = min(RC, t_end - t0);
            float vf[16][4];
            load_v(a, h, vb, t0, n_tok, lr, lk, vf);
            const float g = exp2f(l2 * (float)n_tok);
#pragma unroll
            for (int n = 0; n < 4; n++) acc[n] *= g;
            add_kv(a, h, dt, t0, n_tok, l2, lr, lk, vf, acc);
        }
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int e = 0; e < 4; e++) z[(16 * dt + 4 * lk + e) * 64 + 16 * n + lr] = acc[n][e];
    }
}

__global__ __launch_bounds__(256, 2) void retention_kernel(Retention a) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float *S = smem, *A = S + a.dp * RLD;                 // state [dp][64], decayed q k^T [64][64]
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const int h = blockIdx.x / a.nvb, vb = blockIdx.x % a.nvb, seg = blockIdx.y;
    const float l2 = a.log2_decay[h];
    const int seg0 = seg * a.seg_len, t_end = min(a.rows, seg0 + a.seg_len);
    float *state = a.state + (int64_t)h * a.vdim * a.sp;

    if (a.nseg > 1) {
        const float *z = segment_z(a, h, vb, seg);
        for (int i = tid; i < a.dp * 64; i += 256) S[(i >> 6) * RLD + (i & 63)] = z[i];
    } else {
        for (int i = tid; i < a.dp * 64; i += 256) {
            const int col = i / a.dp, d = i - col * a.dp;      // rows of a column follow each other in memory
            S[d * RLD + col] = 64 * vb + col < a.vdim ? state[(int64_t)(64 * vb + col) * a.sp + d] : 0.0f;
        }
    }
    __syncthreads();

    const int n_d = a.dp / 16;
    for (int t0 = seg0; t0 < t_end; t0 += RC) {
        const int n_tok = min(RC, t_end - t0);
        float vf[16][4];
        load_v(a, h, vb, t0, n_tok, lr, lk, vf);
        // rows 16 wv .. of the chunk: A and S^T q
        f32x4 sc[4], o[4];
#pragma unroll
        for (int n = 0; n < 4; n++) sc[n] = o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        const float *qr = a.q + ((int64_t)(t0 + min(16 * wv + lr, n_tok - 1)) * a.heads + h) * a.dp + 4 * lk;
        const float *kr[4];
#pragma unroll
        for (int n = 0; n < 4; n++) kr[n] = a.k + ((int64_t)(t0 + min(16 * n + lr, n_tok - 1)) * a.heads + h) * a.dp + 4 * lk;
        for (int c = 0; c < n_d; c++) {
            const f32x4 qf = *reinterpret_cast<const f32x4 *>(qr + 16 * c);
            f32x4 kf[4];
#pragma unroll
            for (int n = 0; n < 4; n++) kf[n] = *reinterpret_cast<const f32x4 *>(kr[n] + 16 * c);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    if (n <= wv) sc[n] = mfma4(qf[e], kf[n][e], sc[n]);
                    o[n] = mfma4(qf[e], S[(16 * c + 4 * lk + e) * RLD + 16 * n + lr], o[n]);
                }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int i = 16 * wv + 4 * lk + e;
            const float g = exp2f(l2 * (float)(i + 1));
#pragma unroll
            for (int n = 0; n < 4; n++) {
                o[n][e] *= g;
                const int j = 16 * n + lr;
                A[i * RLD + j] = j <= i && j < n_tok ? sc[n][e] * exp2f(l2 * (float)(i - j)) : 0.0f;
            }
        }
        __syncthreads();                                    // A is written, and every wave has read S
#pragma unroll
        for (int s = 0; s < 16; s++)
            if (s < 4 * (wv + 1)) {
                const float w = A[(16 * wv + lr) * RLD + 4 * s + lk];
#pragma unroll
                for (int n = 0; n < 4; n++) o[n] = mfma4(w, vf[s][n], o[n]);
            }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int i = 16 * wv + 4 * lk + e;
            if (i >= n_tok) continue;
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const int col = 64 * vb + 16 * n + lr;
                if (col < a.vdim) a.out[(int64_t)(t0 + i) * a.out_stride + (int64_t)h * a.vdim + col] = o[n][e];
            }
        }
        if (t0 + RC < t_end || a.nseg == 1) {
            const float g = exp2f(l2 * (float)n_tok);
            for (int dt = wv; dt < n_d; dt += 4) {
                f32x4 acc[4];
#pragma unroll
                for (int n = 0; n < 4; n++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[n][e] = g * S[(16 * dt + 4 * lk + e) * RLD + 16 * n + lr];
                add_kv(a, h, dt, t0, n_tok, l2, lr, lk, vf, acc);
#pragma unroll
                for (int n = 0; n < 4; n++)
#pragma unroll
                    for (int e = 0; e < 4; e++) S[(16 * dt + 4 * lk + e) * RLD + 16 * n + lr] = acc[n][e];
            }
        }
        __syncthreads();
    }
    if (a.nseg == 1)
        for (int i = tid; i < a.dp * 64; i += 256) {
            const int col = i / a.dp, d = i - col * a.dp;
            if (64 * vb + col < a.vdim) state[(int64_t)(64 * vb + col) * a.sp + d] = S[d * RLD + col];
        }
}

__global__ __launch_bounds__(256) void retention_prefix_kernel(Retention a) {
    const int h = blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;             // element of the [nvb][dp][64] Z of a segment
    if (i >= a.nvb * a.dp * 64) return;
    const int vb = i / (a.dp * 64), in = i - vb * a.dp * 64, d = in >> 6, col = 64 * vb + (in & 63);
    const float l2 = a.log2_decay[h], g = exp2f(l2 * (float)a.seg_len), g_last = exp2f(l2 * (float)(a.rows - (a.nseg - 1) * a.seg_len));
    float *st = a.state + ((int64_t)h * a.vdim + min(col, a.vdim - 1)) * a.sp + d;
    float *z = segment_z(a, h, vb, 0) + in;
    const int64_t step = (int64_t)a.dp * 64;
    float s = col < a.vdim ? st[0] : 0.0f;
    constexpr int B = 8;                                      // the loads of eight segments before their chain
    for (int x0 = 0; x0 < a.nseg; x0 += B) {
        float v[B];
#pragma unroll
        for (int x = 0; x < B; x++) v[x] = z[min(x0 + x, a.nseg - 1) * step];
#pragma unroll
        for (int x = 0; x < B; x++)
            if (x0 + x < a.nseg) {
                z[(x0 + x) * step] = s;
                s = fmaf(x0 + x == a.nseg - 1 ? g_last : g, s, v[x]);
            }
    }
    if (col < a.vdim) st[0] = s;
}

// Segments of at least two chunks, or of one (`fine`, where the workspace holds their states: 8 heads of 128 in us, of two chunks -> of one: 2048 rows 55.2 -> 48.9, 1000: 52.7 ->
// 38.0, 300: 64.7 -> 32.6, 100: 36.1 -> 30.9).  Two or three chunks stay one segment where the heads alone are many workgroups, whose states are then neither written nor
// read (whole / cut to chunks: 64 heads of 64, 100 rows 23.1 / 24.3, 180: 32.0 / 26.0; 128 heads 23.5 / 29.2, 180: 32.1 / 35.8, 200: 40.3 / 35.8; 256 heads, 65: 23.8 / 41.4).
void retention_plan(int64_t rows, int64_t heads, int64_t vdim, bool fine, int *nseg, int *seg_len) {
    const int64_t wg = heads * ((vdim + 63) / 64), chunks = (rows + RC - 1) / RC, least = fine && chunks >= (wg <= 48 ? 2 : wg <= 64 ? 3 : 4) ? 1 : 2;
    int64_t n = 512 / wg;
    n = n < chunks / least ? n : chunks / least;
    n = n < 1 ? 1 : n;
    const int64_t per = (chunks + n - 1) / n;
    *seg_len = (int)(per * RC);
    *nseg = (int)((rows + *seg_len - 1) / *seg_len);
}
int64_t retention_bytes(int64_t heads, int64_t dim, int64_t vdim, int nseg) { return nseg > 1 ? heads * ((vdim + 63) / 64) * nseg * ((dim + 15) / 16 * 16) * 64 * 4 : 0; }

// ---- one token: merge of the attention records, and the retention step --------------------------------------------------------
struct StepArgs {
    const float *rec;
    int n_head, att_vdim, window, keep_first, ctx, splits, split_keys;
    float att_scale, ret_scale, eps;
    float *att_out, *state, *ret_out;
    const float *row, *decay;
    cq_mix_heads gq, gk;
    int64_t v_off, g_off;
    int heads, vdim;
};

// The state columns of a wave are requested before q and k are worked out.
template <int NR>
__device__ __forceinline__ void retention_step(const StepArgs &a, int h, int p, float *sm) {
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), sub = lane & 15, cg = lane >> 4;
    constexpr int SP = 64 * NR;
    float *qs = sm, *ks = qs + SP, *os = ks + SP;
    __shared__ float s_inv;
    f32x4 s[NR];
    float vj;
    auto load = [&](int c0) {
        const int col = min(c0 + cg, a.vdim - 1);
        const float *st = a.state + ((int64_t)h * a.vdim + col) * SP + 4 * sub;
#pragma unroll
        for (int c = 0; c < NR; c++) s[c] = *reinterpret_cast<const f32x4 *>(st + 64 * c);
        vj = a.row[a.v_off + (int64_t)h * a.vdim + col];
    };
    load(4 * wv);
    if (wv < 2) {
        const cq_mix_heads &g = wv == 0 ? a.gq : a.gk;
        HeadShared<NR> sh;
        HeadRegs<NR> x;
        sh.load(g, p, lane);
        x.load(g, a.row + g.src_off + (int64_t)h * g.dim, lane);
        sh.ready(g, lane);
        x.finish(g, sh, a.eps, lane);
#pragma unroll
        for (int e = 0; e < NR; e++) sm[wv * SP + lane + 64 * e] = x.v[e];
    }
    const float dec = a.decay[h];
    __syncthreads();
    f32x4 qv[NR], kv[NR];
#pragma unroll
    for (int c = 0; c < NR; c++) {
        qv[c] = *reinterpret_cast<const f32x4 *>(qs + 64 * c + 4 * sub);
        kv[c] = *reinterpret_cast<const f32x4 *>(ks + 64 * c + 4 * sub);
    }
    for (int c0 = 4 * wv; c0 < a.vdim; c0 += 64) {
        if (c0 >= 64) load(c0);
        float o = 0.0f;
#pragma unroll
        for (int c = 0; c < NR; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                s[c][e] = fmaf(dec, s[c][e], kv[c][e] * vj);
                o = fmaf(s[c][e], qv[c][e], o);
            }
        o = row16_sum(o);
        if (c0 + cg < a.vdim) {
            float *st = a.state + ((int64_t)h * a.vdim + c0 + cg) * SP + 4 * sub;
#pragma unroll
            for (int c = 0; c < NR; c++) *reinterpret_cast<f32x4 *>(st + 64 * c) = s[c];
            if (sub == 0) os[c0 + cg] = o;
        }
    }
    __syncthreads();
    if (wv == 0) {
        const float inv = head_inv_rms(os, a.vdim, a.eps, lane);
        if (lane == 0) s_inv = inv;
    }
    __syncthreads();
    for (int e = tid; e < a.vdim; e += 1024) {
        const float g = a.row[a.g_off + (int64_t)h * a.vdim + e];
        a.ret_out[(int64_t)h * a.vdim + e] = a.ret_scale * os[e] * s_inv * (g * mix_sigmoid(g));
    }
}

// Blocks [0, n_head): out of one attention head from its records; blocks behind them: one retention head each.
template <int NR>
__global__ __launch_bounds__(1024) void talk_merge_retention_kernel(StepArgs a, const int32_t *__restrict__ pos_dev, int pos0) {
    extern __shared__ __attribute__((aligned(16))) float sm[];          // max(splits + 1024, 2 * 64 NR + vdim)
    __shared__ float red[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = pos0 + (pos_dev ? pos_dev[0] : 0);
    if (p >= a.ctx) return;
    if ((int)blockIdx.x >= a.n_head) {
        retention_step<NR>(a, blockIdx.x - a.n_head, p, sm);
        return;
    }
    const int h = blockIdx.x, stride = talk_record(a.att_vdim);
    const int n = (visible_keys(p, a.window, a.keep_first).n + a.split_keys - 1) / a.split_keys;      // splits that hold keys
    const float *rec = a.rec + (int64_t)h * a.splits * stride;
    float *wt = sm, *part = sm + (n + 3) / 4 * 4;
    float m = -INFINITY;
    for (int s = tid; s < n; s += 1024) m = fmaxf(m, wt[s] = rec[(int64_t)s * stride + stride - 4]);
    m = wave_max(m);
    if (lane == 0) red[wv] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < 16; w++) m = fmaxf(m, red[w]);
    float l = 0.0f;
    for (int s = tid; s < n; s += 1024) {                    // the thread's own wt entries
        const float w = __expf(wt[s] - m);
        wt[s] = w;
        l = fmaf(w, rec[(int64_t)s * stride + stride - 3], l);
    }
    l = wave_sum(l);
    __syncthreads();
    if (lane == 0) red[wv] = l;
    __syncthreads();
    l = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; w++) l += red[w];
    // 64 columns at a time, the waves share out the splits
    for (int e0 = 0; e0 < a.att_vdim; e0 += 64) {
        const int e = min(e0 + lane, a.att_vdim - 1);
        float acc = 0.0f;
#pragma unroll 4
        for (int s = wv; s < n; s += 16) acc = fmaf(wt[s], rec[(int64_t)s * stride + e], acc);
        __syncthreads();
        part[wv * 64 + lane] = acc;
        __syncthreads();
        if (wv == 0 && e0 + lane < a.att_vdim) {
            float t = 0.0f;
#pragma unroll
            for (int w = 0; w < 16; w++) t += part[w * 64 + lane];
            a.att_out[(int64_t)h * a.att_vdim + e0 + lane] = a.att_scale * t / l;
        }
    }
}

// ---- generalized delta rule ---------------------------------------------------------------------------------------------------
constexpr float DELTA_UNIT_EPS = 1e-6f;              // inside the root of the unit key
constexpr float DELTA_DECAY = 0.60653065971263342f;  // exp(-1/2)

__device__ __forceinline__ float delta_decay(float wl, float w0) { return expf(-DELTA_DECAY * mix_sigmoid(wl + w0)); }

// One head of a token as four vectors of `sp` floats, w | a u | u | r, zero beyond dim, and |k| (k = |k| u).  One wave.
template <typename WL>
__device__ __forceinline__ void delta_pack(const float *r, const float *k, const float *al, WL wl, const float *w0, const float *ab, float *dst, float *k_norm, int dim,
                                           int sp, int lane) {
    float s = 0.0f;
    for (int d = lane; d < dim; d += 64) s = fmaf(k[d], k[d], s);
    const float norm = sqrtf(wave_sum(s) + DELTA_UNIT_EPS), inv = 1.0f / norm;
    if (lane == 0) k_norm[0] = norm;
    for (int d = lane; d < sp; d += 64) {
        const bool ok = d < dim;
        const float u = ok ? k[d] * inv : 0.0f;
        dst[d] = ok ? delta_decay(wl(d), w0[d]) : 0.0f;
        dst[sp + d] = ok ? mix_sigmoid(al[d] + ab[d]) * u : 0.0f;
        dst[2 * sp + d] = u;
        dst[3 * sp + d] = ok ? r[d] : 0.0f;
    }
}

__global__ __launch_bounds__(256) void delta_prep_kernel(const float *__restrict__ row, int64_t row_stride, int64_t r_off, int64_t k_off, int64_t a_off,
                                                         const float *__restrict__ wl, int64_t wl_stride, const float *__restrict__ w0,
                                                         const float *__restrict__ ab, float *__restrict__ packed, int64_t rows, int heads, int dim, int sp) {
    const int lane = threadIdx.x & 63, h = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (h >= heads) return;
    const int64_t t = blockIdx.x, id = t * heads + h, hd = (int64_t)h * dim;
    const float *s = row + t * row_stride + hd, *w = wl + t * wl_stride + hd;
    delta_pack(s + r_off, s + k_off, s + a_off, [&](int d) { return w[d]; }, w0 + hd, ab + hd, packed + id * 4 * sp, packed + rows * heads * 4 * sp + id, dim, sp, lane);
}

// The rows of a column that a lane holds, and one token's vectors on them.
template <int NR>
struct DeltaRows {
    f32x4 w[NR], b[NR], u[NR], r[NR];
    __device__ __forceinline__ void load(const float *vec, int sub) {
#pragma unroll
        for (int c = 0; c < NR; c++) {
            const float *x = vec + 64 * c + 4 * sub;
            w[c] = *reinterpret_cast<const f32x4 *>(x);
            b[c] = *reinterpret_cast<const f32x4 *>(x + 64 * NR);
            u[c] = *reinterpret_cast<const f32x4 *>(x + 2 * 64 * NR);
            r[c] = *reinterpret_cast<const f32x4 *>(x + 3 * 64 * NR);
        }
    }
};

// One column step: s <- w s - b (u . s) + u v (v: the value times |k|); returns this lane's part of r . s.
template <int NR>
__device__ __forceinline__ float delta_column(f32x4 (&s)[NR], const DeltaRows<NR> &x, float v) {
    float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        x0 = fmaf(x.u[c].x, s[c].x, x0);
        x1 = fmaf(x.u[c].y, s[c].y, x1);
        x0 = fmaf(x.u[c].z, s[c].z, x0);
        x1 = fmaf(x.u[c].w, s[c].w, x1);
    }
    const float us = row16_sum(x0 + x1);
    float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int c = 0; c < NR; c++) {
#pragma unroll
        for (int e = 0; e < 4; e++) s[c][e] = fmaf(-x.b[c][e], us, fmaf(x.w[c][e], s[c][e], x.u[c][e] * v));
        o0 = fmaf(x.r[c].x, s[c].x, o0);
        o1 = fmaf(x.r[c].y, s[c].y, o1);
        o0 = fmaf(x.r[c].z, s[c].z, o0);
        o1 = fmaf(x.r[c].w, s[c].w, o1);
    }
    return o0 + o1;
}

// Token after token.  Workgroup: 16 value columns of one head, 4 waves x 4 columns; the packed vectors of TB tokens at a time go
// through LDS (double-buffered: the next block's loads are in flight while this one runs) and from there, one token ahead, into
// registers.  The lanes' parts of r . s are collected for the block and summed 16 tokens at a time, off the chain of state updates.
template <int NR, int TB>
__global__ __launch_bounds__(256) void delta_scan_kernel(const float *__restrict__ packed, const float *__restrict__ v, int64_t v_stride,
                                                         float *__restrict__ state, float *__restrict__ out, int64_t out_stride, int rows, int heads, int dim,
                                                         int ncb) {
    constexpr int SP = 64 * NR, VEC = 4 * SP, LOADS = TB * VEC / 4 / 256;
    static_assert(TB * VEC % 1024 == 0 && TB <= 16, "whole float4 per thread");
    extern __shared__ __attribute__((aligned(16))) float smem[];         // 2 x { packed [TB][VEC], v [TB][16] }
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), sub = lane & 15, cg = lane >> 4;
    // workgroups of one head on one XCD (dealt round-robin): they read the same packed vectors
    const int hb = blockIdx.x / (8 * ncb), in = blockIdx.x % (8 * ncb);
    const int h = hb * 8 + in % 8, cb = in / 8;
    if (h >= heads) return;
    const int col = 16 * cb + 4 * wv + cg, colc = min(col, dim - 1);
    float *st = state + ((int64_t)h * dim + colc) * SP + 4 * sub;
    f32x4 s[NR];
#pragma unroll
    for (int c = 0; c < NR; c++) s[c] = *reinterpret_cast<const f32x4 *>(st + 64 * c);
    const int64_t tok = (int64_t)heads * VEC;
    const float *src = packed + (int64_t)h * VEC;
    const float *knorm = packed + (int64_t)rows * tok + h;
    const float *vsrc = v + (int64_t)h * dim + min(16 * cb + (tid & 15), dim - 1);
    float *dst = out + (int64_t)h * dim + col;

    f32x4 ld[LOADS];
    float ldv = 0.0f, ldk = 0.0f;
    auto fetch = [&](int t0) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const int x = tid + 256 * i, t = min(t0 + x / (VEC / 4), rows - 1);
            ld[i] = *reinterpret_cast<const f32x4 *>(src + t * tok + 4 * (x % (VEC / 4)));
        }
        if (tid < TB * 16) {
            const int64_t t = min(t0 + (tid >> 4), rows - 1);
            ldv = vsrc[t * v_stride];
            ldk = knorm[t * heads];
        }
    };
    auto stage = [&](float *to) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) *reinterpret_cast<f32x4 *>(to + 4 * (tid + 256 * i)) = ld[i];
        if (tid < TB * 16) to[TB * VEC + tid] = ldv * ldk;
    };
    constexpr int BUF = TB * VEC + TB * 16;
    fetch(0);
    stage(smem);
    __syncthreads();
    int cur = 0;
    for (int t0 = 0; t0 < rows; t0 += TB) {
        const bool more = t0 + TB < rows;
        if (more) fetch(t0 + TB);
        const float *b = smem + cur * BUF, *bv = b + TB * VEC + 4 * wv + cg;
        const int n = min(TB, rows - t0);
        if (n == TB) {
            DeltaRows<NR> x[2];
            float vx[2], o[TB];
            x[0].load(b, sub);
            vx[0] = bv[0];
#pragma unroll
            for (int t = 0; t < TB; t++) {
                if (t + 1 < TB) {
                    x[(t + 1) & 1].load(b + (t + 1) * VEC, sub);
                    vx[(t + 1) & 1] = bv[16 * (t + 1)];
                }
                o[t] = delta_column<NR>(s, x[t & 1], vx[t & 1]);
            }
            // lane `sub` ends with the sum of token t0 + sub
            float mine = 0.0f;
#pragma unroll
            for (int t = 0; t < TB; t++) {
                const float sum = row16_sum(o[t]);
                mine = sub == t ? sum : mine;
            }
            if (sub < TB && col < dim) dst[(int64_t)(t0 + sub) * out_stride] = mine;
        } else {
            for (int t = 0; t < n; t++) {
                DeltaRows<NR> x;
                x.load(b + t * VEC, sub);
                const float o = row16_sum(delta_column<NR>(s, x, bv[16 * t]));
                if (sub == 0 && col < dim) dst[(int64_t)(t0 + t) * out_stride] = o;
            }
        }
        if (more) {
            stage(smem + (cur ^ 1) * BUF);
            __syncthreads();
            cur ^= 1;
        }
    }
    if (col < dim) {
#pragma unroll
        for (int c = 0; c < NR; c++) *reinterpret_cast<f32x4 *>(st + 64 * c) = s[c];
    }
}

// ---- generalized delta rule, many tokens of heads of up to 64 dimensions: chunks of 16 tokens on the matrix cores ------------------------
// Token after token the rule is one serial chain of 16-lane sums, 109 ns a token whatever the chip.  Inside a chunk let W_t be the product of its first t decays
// (element by element), v' = |k| v and S the state before the chunk.  With
//   ut_t = u_t W_(t-1),   rt_t = r_t W_t,   uh_s = u_s / W_s,   bh_s = a u_s / W_s
// the state after token t is S_t = W_t (S + sum_{s<=t} uh_s v'_s - bh_s x_s), where the removed rows x_t = u_t . S_(t-1) solve the unit lower triangular system
//   x_t + sum_{s<t} (ut_t . bh_s) x_s = ut_t S + sum_{s<t} (ut_t . uh_s) v'_s           =>   X = P S + Q V'
// the outputs are o_t = rt_t S + sum_{s<=t} (rt_t . uh_s) v'_s - (rt_t . bh_s) x_s      =>   O = Ro S + Qo V'
// and the state after the chunk is                                                        S' = W_16 S - B (P S) + U V',   B = W_16 bh^T, U = W_16 uh^T - B Q.
// delta_chunk_kernel finds P, Ro, Qo, B, U and V' of all chunks side by side, delta_chain_kernel then takes two products that wait for each other per 16 tokens.
// A decay is at least exp(-exp(-1/2)) = 0.545, so W stays above 6e-5; it and the four products of rows are formed in 64 bits and rounded once, which leaves the
// error of the whole against 64 bits where that of the scan is (2-norm, 32 heads of 64, 64 - 2048 tokens: outputs 1.20 - 1.33e-7 against 1.20 - 1.41e-7, states 1.00 -
// 1.18e-7 against 1.03 - 1.30e-7).
// 32 heads of 64 in us, packing and scan -> chunks and chain: 2048 tokens 25 + 223 -> 40 + 70, 256: 37.1 -> 23.4, 100: 18.0 -> 14.3; 16 heads, 1500 tokens 177 -> 71.
// The chunks are bound by the bytes of rows and records (64 + 89 MB of 2048 tokens) and the latencies between four barriers, with five workgroups on a CU; the chain
// by the latencies of a chunk: eight products in a row (8 x 32 cycles) and a way through LDS.
constexpr int KC = 16, KLD = 68;                     // chunk length; LDS row of 64 dimensions
// A record per (chunk, head), as the chain's lanes (lr = lane % 16, lk = lane / 16) take it, float4 [4 waves][64 lanes] each: P and Ro [t = lr][d = 16 wave + 4 lk ..],
// U and B [d = 16 wave + lr][s = 4 lk ..], V' [s = 4 lk ..][column 16 wave + lr]; then W_16 [64], and Qo [4 waves][64 lanes] of [t = lr][s = 4 lk + wave].
constexpr int KREC_W = 5 * 1024, KREC_Q = KREC_W + 64, KREC = KREC_Q + 256;
typedef double f64x4 __attribute__((ext_vector_type(4)));

struct DeltaRowsIn {
    const float *row, *wl, *w0, *ab;
    int64_t row_stride, r_off, k_off, v_off, a_off, wl_stride;
    int rows, heads, dim;
};

// A workgroup per chunk and head; lane: dimension, wave g: tokens 4 g ... .  The four products of rows are one wave each.
__global__ __launch_bounds__(256) void delta_chunk_kernel(DeltaRowsIn a, float *__restrict__ rec) {
    constexpr int LD = 20, MAT = KC * LD;                  // [t][s] of ut.uh, ut.bh, rt.uh, rt.bh
    __shared__ __attribute__((aligned(16))) float arr[5][KC * KLD], mat[4 * MAT];
    __shared__ double prod[4][64];
    float *const s_ut = arr[0], *const s_rt = arr[1], *const s_uh = arr[2], *const s_bh = arr[3], *const s_bt = arr[4];
    const int tid = threadIdx.x, lane = tid & 63, g = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const int h = blockIdx.y, t0 = blockIdx.x * KC, n = min(KC, a.rows - t0);
    const bool ok = lane < a.dim;
    const int64_t hd = (int64_t)h * a.dim + min(lane, a.dim - 1);
    float *const r = rec + ((int64_t)blockIdx.x * a.heads + h) * KREC;
    f32x4 *const r4 = reinterpret_cast<f32x4 *>(r);
    const int own = lk * 64 + 16 * g + lr;                 // the place of four tokens 4 g .. of dimension `lane` in an operand

    float k[4], al[4], wl[4], rr[4];
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t x = t0 + min(4 * g + i, n - 1);
        const float *s = a.row + x * a.row_stride + hd;
        k[i] = s[a.k_off];
        al[i] = s[a.a_off];
        wl[i] = a.wl[x * a.wl_stride + hd];
        rr[i] = s[a.r_off];
        v[i] = s[a.v_off];
    }
    const float w0 = a.w0[hd], ab = a.ab[hd];
    float sq = 0.0f;                                       // lane i: |k|^2 of token i
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (!ok || 4 * g + i >= n) k[i] = al[i] = rr[i] = v[i] = 0.0f;
        const float q = wave_sum(k[i] * k[i]);
        sq = lane == i ? q : sq;
    }
    const float norm = sqrtf(sq + DELTA_UNIT_EPS), inv_norm = 1.0f / norm;
    float u[4], b[4];
    double W[4], P = 1.0;                                  // products of this wave's decays
#pragma unroll
    for (int i = 0; i < 4; i++) {
        u[i] = k[i] * __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, inv_norm), i));
        v[i] *= __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, norm), i));
        b[i] = mix_sigmoid(al[i] + ab) * u[i];
        P *= ok && 4 * g + i < n ? (double)delta_decay(wl[i], w0) : 1.0;
        W[i] = P;
    }
    prod[g][lane] = P;
    __syncthreads();
    double before = 1.0, all = 1.0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const double q = prod[i][lane];
        before = i < g ? before * q : before;
        all *= q;
    }
    f32x4 bt;
    float un[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const double Wt = before * W[i], Wp = i ? before * W[i - 1] : before, x = (double)__builtin_amdgcn_rcpf((float)Wt), inv = fma(fma(-Wt, x, 1.0), x, x), f = all * inv;
        const int at = (4 * g + i) * KLD + lane;
        s_ut[at] = (float)((double)u[i] * Wp);
        s_rt[at] = rr[i] = (float)((double)rr[i] * Wt);
        s_uh[at] = (float)((double)u[i] * inv);
        s_bh[at] = (float)((double)b[i] * inv);
        un[i] = (float)((double)u[i] * f);
        s_bt[at] = bt[i] = (float)((double)b[i] * f);
    }
    r4[768 + own] = bt;
    r4[1024 + own] = v;
    if (g == 0) r[KREC_W + lane] = (float)all;
    __syncthreads();
    {
        const float *x = (g < 2 ? s_ut : s_rt) + lr * KLD + 4 * lk, *y = (g & 1 ? s_bh : s_uh) + lr * KLD + 4 * lk;
        f64x4 m = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const f32x4 fx = *reinterpret_cast<const f32x4 *>(x + 16 * c), fy = *reinterpret_cast<const f32x4 *>(y + 16 * c);
#pragma unroll
            for (int e = 0; e < 4; e++) m = __builtin_amdgcn_mfma_f64_16x16x4f64((double)fx[e], (double)fy[e], m, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {                      // (64-bit results: row lk + 4 e, column lr)
            const int t = lk + 4 * e;
            mat[g * MAT + t * LD + lr] = lr < t || (g >= 2 && lr == t) ? (float)m[e] : 0.0f;
        }
    }
    __syncthreads();
    // the triangular system, row by row: wave 0 has the columns of P (dimensions), wave 1 those of Q (tokens; in place)
    if (g < 2) {
        float *const x = g == 0 ? s_ut + lane : mat + lr;
        const int ld = g == 0 ? KLD : LD;
        float p[KC];
#pragma unroll
        for (int t = 0; t < KC; t++) p[t] = x[t * ld];
#pragma unroll
        for (int t = 1; t < KC; t++) {
            float sum = 0.0f;
#pragma unroll
            for (int s4 = 0; 4 * s4 < t; s4++) {
                const f32x4 l = *reinterpret_cast<const f32x4 *>(mat + MAT + t * LD + 4 * s4);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (4 * s4 + e < t) sum = fmaf(l[e], p[4 * s4 + e], sum);
            }
            p[t] -= sum;
        }
        if (g == 0 || lk == 0)
#pragma unroll
            for (int t = 0; t < KC; t++) x[t * ld] = p[t];
    }
    __syncthreads();
    r4[tid] = *reinterpret_cast<const f32x4 *>(s_ut + lr * KLD + 16 * g + 4 * lk);
    {
        const int j = 4 * lk + g;                          // Qo: [t = lr][s = 4 lk + g]
        float sum = 0.0f;
#pragma unroll
        for (int s = 0; s < KC; s++) {
            const float more = fmaf(mat[3 * MAT + lr * LD + s], mat[s * LD + j], sum);
            sum = s <= lr ? more : sum;
        }
        r[KREC_Q + tid] = mat[2 * MAT + lr * LD + j] - sum;
    }
    // Ro and U of the wave's own tokens (beyond the triangles the matrices are zero, but P and Q of a token that is no number are none either, and may not reach the
    // tokens before it)
    float ro[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4 lost = {0.f, 0.f, 0.f, 0.f};
    auto removed = [&](int s4, auto whole) {
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; e++) p[e] = s_ut[(4 * s4 + e) * KLD + lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const f32x4 l = *reinterpret_cast<const f32x4 *>(mat + 3 * MAT + (4 * g + i) * LD + 4 * s4);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (whole || e <= i) ro[i] = fmaf(l[e], p[e], ro[i]);
        }
    };
    for (int s4 = 0; s4 < g; s4++) removed(s4, std::integral_constant<bool, true>{});
    removed(g, std::integral_constant<bool, false>{});
    for (int t = 4 * g + 1; t < KC; t++) {
        const f32x4 q = *reinterpret_cast<const f32x4 *>(mat + t * LD + 4 * g);
        const float x = s_bt[t * KLD + lane];
#pragma unroll
        for (int i = 0; i < 4; i++) lost[i] = fmaf(q[i], x, lost[i]);
    }
    r4[512 + own] = f32x4{un[0], un[1], un[2], un[3]} - lost;
#pragma unroll
    for (int i = 0; i < 4; i++) s_rt[(4 * g + i) * KLD + lane] = rr[i] - ro[i];
    __syncthreads();
    r4[256 + tid] = *reinterpret_cast<const f32x4 *>(s_rt + lr * KLD + 16 * g + 4 * lk);
}

// Chunk after chunk.  Workgroup: 16 value columns of one head.  Of its eight waves the first four carry the state: wave wv keeps rows 16 wv .. as a result tile, which
// is at the same time the operand of its quarter of P S; the quarters meet in LDS (one barrier a chunk), and their sum is again a result tile and the operand of the
// update.  The other four form the outputs from the states that the first ones leave in LDS, each a quarter, and write the sums of the quarters one chunk later.  All
// that waves hand to each other lies in LDS twice, for even and odd chunks: what is written between barriers c - 1 and c is read between c and c + 1, and its place written
// again behind c + 1.
struct DeltaPart {
    f32x4 a, u, b, v, w;                                   // a: P (state waves) or Ro (output waves)
    float qo;
};
__global__ __launch_bounds__(512, 2) void delta_chain_kernel(const float *__restrict__ rec, float *__restrict__ state, float *__restrict__ out, int64_t out_stride, int rows,
                                                             int heads, int dim, int ncb) {
    __shared__ f32x4 px[2][4][64], ps[2][4][64], po[2][4][64];      // [chunk % 2][wave][lane]: quarters of P S, states, quarters of the outputs
    const int tid = threadIdx.x & 255, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const bool outputs = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) != 0;
    // workgroups of one head on one XCD (dealt round-robin): they read the same records
    const int hb = blockIdx.x / (8 * ncb), in = blockIdx.x % (8 * ncb);
    const int h = hb * 8 + in % 8, cb = in / 8;
    if (h >= heads) return;
    const int chunks = (rows + KC - 1) / KC;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const float *const r0 = rec + (int64_t)h * KREC;
    const int64_t r_step = (int64_t)heads * KREC;
    // barrier c: the quarters of P S and the state of chunk c are there, and those of the outputs of chunk c - 1 (__syncthreads would wait for the records on their way)
    auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    if (outputs) {
        const int oc = 16 * cb + lr, ot = tid >> 4;        // thread: token tid / 16, column tid % 16
        float *const dst = out + (int64_t)h * dim + oc;
        const float *const src = reinterpret_cast<const float *>(&po[0][0][0]) + (wv * 16 + lr) * 4 + lk;
        auto load = [&](DeltaPart &x, int c) {             // (past the end: the last chunk again, for nobody)
            const float *r = r0 + min(c, chunks - 1) * r_step;
            x.a = reinterpret_cast<const f32x4 *>(r)[256 + tid];
            x.v = reinterpret_cast<const f32x4 *>(r)[1024 + 64 * cb + lane];
            x.qo = r[KREC_Q + tid];
        };
        auto value = [&](const DeltaPart &x) { return wv & 2 ? (wv & 1 ? x.v[3] : x.v[2]) : (wv & 1 ? x.v[1] : x.v[0]); };      // of token 4 lk + wv
        auto marked = [&](const DeltaPart &x) { return __any(!(fabsf(value(x)) < INFINITY)) != 0; };
        bool mark;                                         // one of the chunk's values is no number (found out a step ahead: in front of the products it costs 2 %)
        auto step = [&](const DeltaPart &x, const DeltaPart &next, int c) {
            const float vs = value(x);
            f32x4 o0 = zero, o1 = zero;
            if (!mark) o1 = mfma4(x.qo, vs, zero);
            else {                                         // such a value counts from its own token on: zero times it is no number either
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    const float va = __shfl(vs, 16 * a + lr, 64);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float q = __shfl(x.qo, 16 * a + 4 * lk + e, 64), more = fmaf(q, va, o1[e]);
                        o1[e] = 4 * a + wv <= 4 * lk + e ? more : o1[e];
                    }
                }
            }
            meet();
            const f32x4 s = ps[c & 1][wv][lane];
            if (c > 0 && oc < dim) {                       // (whole chunks)
                const float *p = src + (~c & 1) * 1024;
                dst[(int64_t)(KC * (c - 1) + ot) * out_stride] = (p[0] + p[256]) + (p[512] + p[768]);
            }
#pragma unroll
            for (int e = 0; e < 2; e++) {
                o0 = mfma4(x.a[e], s[e], o0);
                o1 = mfma4(x.a[2 + e], s[2 + e], o1);
            }
            po[c & 1][wv][lane] = o0 + o1;
            mark = marked(next);
        };
        DeltaPart x[4];
        load(x[0], 0);
        load(x[1], 1);
        load(x[2], 2);
        mark = marked(x[0]);
        for (int c = 0; c < chunks; c += 4) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (c + j >= chunks) break;
                load(x[(j + 3) & 3], c + j + 3);
                step(x[j], x[(j + 1) & 3], c + j);
            }
        }
        meet();
        const int c = chunks - 1;
        const float *p = src + (c & 1) * 1024;
        if (KC * c + ot < rows && oc < dim) dst[(int64_t)(KC * c + ot) * out_stride] = (p[0] + p[256]) + (p[512] + p[768]);
        return;
    }

    float *const st = state + ((int64_t)h * dim + min(16 * cb + lr, dim - 1)) * 64 + 16 * wv + 4 * lk;
    f32x4 s = *reinterpret_cast<const f32x4 *>(st);
    auto load = [&](DeltaPart &x, int c) {
        const float *r = r0 + min(c, chunks - 1) * r_step;
        const f32x4 *r4 = reinterpret_cast<const f32x4 *>(r);
        x.a = r4[tid];
        x.u = r4[512 + tid];
        x.b = r4[768 + tid];
        x.v = r4[1024 + 64 * cb + lane];
        x.w = *reinterpret_cast<const f32x4 *>(r + KREC_W + 16 * wv + 4 * lk);
    };
    auto step = [&](const DeltaPart &x, int c) {
        f32x4 xp = zero, nv = zero, rm = zero;
#pragma unroll
        for (int e = 0; e < 4; e++) xp = mfma4(x.a[e], s[e], xp);
        __builtin_amdgcn_sched_barrier(0);
        ps[c & 1][wv][lane] = s;
        nv = mfma4(x.u[0], x.v[0], nv);
        px[c & 1][wv][lane] = xp;
        __builtin_amdgcn_sched_barrier(0);
        meet();
        const f32x4 x0 = px[c & 1][0][lane], x1 = px[c & 1][1][lane], x2 = px[c & 1][2][lane], x3 = px[c & 1][3][lane];
#pragma unroll
        for (int e = 1; e < 4; e++) nv = mfma4(x.u[e], x.v[e], nv);
        __builtin_amdgcn_sched_barrier(0);
        const f32x4 xs = (x0 + x1) + (x2 + x3);
#pragma unroll
        for (int e = 0; e < 4; e++) rm = mfma4(x.b[e], -xs[e], rm);
#pragma unroll
        for (int e = 0; e < 4; e++) s[e] = fmaf(x.w[e], s[e], rm[e] + nv[e]);
    };
    DeltaPart x[4];
    load(x[0], 0);
    load(x[1], 1);
    load(x[2], 2);
    for (int c = 0; c < chunks; c += 4) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (c + j >= chunks) break;
            load(x[(j + 3) & 3], c + j + 3);
            step(x[j], c + j);
        }
    }
    meet();
    if (16 * cb + lr < dim) *reinterpret_cast<f32x4 *>(st) = s;
}

// Chunks for heads of at most 64 dimensions (their operators have 64 rows) and from so many tokens on that they take no longer than packing and scan, whose time grows by the
// token: with more heads a chunk's work fills the chip and shows (us, packing and scan / chunks: 32 heads of 64, 32 tokens 8.2 / 10.0, 48: 10.5 / 11.1, 56: 12.2 / 11.9,
// 64 heads, 56: 13.6 / 13.2; 128 heads, 64: 18.9 / 19.0, 96: 25.8 / 23.0; 200 heads of 16, 64: 19.5 / 22.1, 96: 25.5 / 24.8; 400 heads of 16, 128: 41.3 / 43.7, 256: 73.3 / 73.0).
bool delta_chunked(int64_t rows, int64_t heads, int64_t dim) { return dim <= 64 && heads <= 65535 && rows >= (heads <= 64 ? 56 : heads <= 200 ? 96 : 256); }

struct DeltaStep {
    const float *row, *w0, *ab, *weight;
    const uint16_t *w2;
    float *state, *out;
    int64_t r_off, k_off, v_off, g_off, a_off, low_off, ldw2;
    int rank, heads, dim;
    float eps;
};

// One token, one head per workgroup of 16 waves.  The first 64 state columns are requested before anything else.
template <int NR>
__global__ __launch_bounds__(1024) void delta_step_kernel(DeltaStep a) {
    constexpr int SP = 64 * NR;
    extern __shared__ __attribute__((aligned(16))) float low[];           // tanh of the rank values, zero up to ldw2
    __shared__ __attribute__((aligned(16))) float vec[4 * SP], wl[SP], os[SP];
    __shared__ float s_inv, k_norm;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), sub = lane & 15, cg = lane >> 4;
    const int h = blockIdx.x;
    const int64_t hd = (int64_t)h * a.dim;
    f32x4 s[NR];
    float vj;
    auto load = [&](int c0) {
        const int col = min(c0 + cg, a.dim - 1);
        const float *st = a.state + (hd + col) * SP + 4 * sub;
#pragma unroll
        for (int c = 0; c < NR; c++) s[c] = *reinterpret_cast<const f32x4 *>(st + 64 * c);
        vj = a.row[a.v_off + hd + col];
    };
    load(4 * wv);
    for (int i = tid; i < a.ldw2; i += 1024) low[i] = i < a.rank ? tanhf(a.row[a.low_off + i]) : 0.0f;
    __syncthreads();
    for (int i0 = wv * 4; i0 < a.dim; i0 += 64) {
        const uint16_t *w = a.w2 + (hd + min(i0 + cg, a.dim - 1)) * a.ldw2;
        float acc = 0.0f;
        for (int j = 4 * sub; j < a.ldw2; j += 64) {
            const u32x2 x = *reinterpret_cast<const u32x2 *>(w + j);
            const f32x4 y = *reinterpret_cast<const f32x4 *>(low + j);
            acc = fmaf(__builtin_bit_cast(float, x.x << 16), y.x, acc);
            acc = fmaf(__builtin_bit_cast(float, x.x & 0xffff0000u), y.y, acc);
            acc = fmaf(__builtin_bit_cast(float, x.y << 16), y.z, acc);
            acc = fmaf(__builtin_bit_cast(float, x.y & 0xffff0000u), y.w, acc);
        }
        acc = row16_sum(acc);
        if (sub == 0 && i0 + cg < a.dim) wl[i0 + cg] = acc;
    }
    __syncthreads();
    if (wv == 0) {
        const float *x = a.row + hd;
        delta_pack(x + a.r_off, x + a.k_off, x + a.a_off, [&](int d) { return wl[d]; }, a.w0 + hd, a.ab + hd, vec, &k_norm, a.dim, SP, lane);
    }
    __syncthreads();
    DeltaRows<NR> x;
    x.load(vec, sub);
    for (int c0 = 4 * wv; c0 < a.dim; c0 += 64) {
        if (c0 >= 64) load(c0);
        const float o = row16_sum(delta_column<NR>(s, x, vj * k_norm));
        if (c0 + cg < a.dim) {
            float *st = a.state + (hd + c0 + cg) * SP + 4 * sub;
#pragma unroll
            for (int c = 0; c < NR; c++) *reinterpret_cast<f32x4 *>(st + 64 * c) = s[c];
            if (sub == 0) os[c0 + cg] = o;
        }
    }
    __syncthreads();
    if (wv == 0) {
        const float inv = head_inv_rms(os, a.dim, a.eps, lane);
        if (lane == 0) s_inv = inv;
    }
    __syncthreads();
    for (int e = tid; e < a.dim; e += 1024) a.out[hd + e] = os[e] * s_inv * a.weight[hd + e] * mix_sigmoid(a.row[a.g_off + hd + e]);
}

}  // namespace

extern "C" {

int64_t cq_mix_state_pad(int64_t dim) { return dim > 0 && dim <= CQ_MIX_MAX_DIM ? (dim <= 64 ? 64 : (dim <= 128 ? 128 : 256)) : -1; }

int64_t cq_mix_retention_workspace_bytes(int64_t rows, int64_t heads, int64_t dim, int64_t vdim) {
    if (rows <= 0 || heads <= 0 || dim <= 0 || vdim <= 0) return 0;
    int nseg, seg_len;
    retention_plan(rows, heads, vdim, true, &nseg, &seg_len);
    return retention_bytes(heads, dim, vdim, nseg);
}

int cq_mix_retention(const float *q_dev, const float *k_dev, const float *v_dev, int64_t v_stride, const float *log2_decay_dev, float *state_dev,
                     float *out_dev, int64_t out_stride, int64_t rows, int64_t heads, int64_t dim, int64_t dim_pad, int64_t vdim, void *workspace_dev,
                     int64_t workspace_bytes, void *stream) {
    if (rows < 0 || heads <= 0 || dim <= 0 || vdim <= 0 || dim_pad != (dim + 15) / 16 * 16 || v_stride < heads * vdim || out_stride < heads * vdim)
        return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    if (!q_dev || !k_dev || !v_dev || !log2_decay_dev || !state_dev || !out_dev) return CQ_ERR_NULL;
    if (mix_misaligned(q_dev, 16) || mix_misaligned(k_dev, 16)) return CQ_ERR_ALIGN;
    if (dim > CQ_MIX_MAX_DIM || rows > (1 << 24) || heads * ((vdim + 63) / 64) > (1 << 20) || heads > 65535) return CQ_ERR_RANGE;
    Retention a;
    a.q = q_dev; a.k = k_dev; a.v = v_dev; a.log2_decay = log2_decay_dev;
    a.state = state_dev; a.out = out_dev; a.z = (float *)workspace_dev;
    a.v_stride = v_stride; a.out_stride = out_stride;
    a.rows = (int)rows; a.heads = (int)heads; a.dp = (int)dim_pad; a.vdim = (int)vdim; a.sp = (int)cq_mix_state_pad(dim);
    a.nvb = (a.vdim + 63) / 64;
    retention_plan(rows, heads, vdim, true, &a.nseg, &a.seg_len);
    if (!workspace_dev || workspace_bytes < retention_bytes(heads, dim, vdim, a.nseg)) {
        retention_plan(rows, heads, vdim, false, &a.nseg, &a.seg_len);
        if (a.nseg > 1 && (!workspace_dev || workspace_bytes < retention_bytes(heads, dim, vdim, a.nseg))) return CQ_ERR_WORKSPACE;
    }
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)(a.heads * a.nvb), (unsigned)a.nseg);
    const size_t lds = (size_t)(a.dp + RC) * RLD * sizeof(float);
    if (lds > 64 * 1024) {
        const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(retention_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e) return e;
    }
    if (a.nseg > 1) {
        hipLaunchKernelGGL(retention_segment_kernel, grid, dim3(256), 0, s, a);
        hipLaunchKernelGGL(retention_prefix_kernel, dim3((unsigned)((a.nvb * a.dp * 64 + 255) / 256), (unsigned)heads), dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL(retention_kernel, grid, dim3(256), lds, s, a);
    return (int)hipGetLastError();
}

int cq_mix_talk_merge_retention_step(const void *workspace_dev, int64_t n_head, int64_t att_vdim, int64_t window, int64_t keep_first, int64_t ctx,
                                     float att_scale, float *att_out_dev, const float *row_dev, const cq_mix_heads *qk, int64_t v_off, int64_t g_off,
                                     const float *decay_dev, float *state_dev, int64_t heads, int64_t vdim, float eps, float ret_scale,
                                     float *ret_out_dev, const int32_t *pos_dev, int64_t pos, void *stream) {
    if (n_head <= 0 || att_vdim <= 0 || window < 1 || keep_first < 0 || ctx <= 0 || heads <= 0 || vdim <= 0 || v_off < 0 || g_off < 0 || pos < 0)
        return CQ_ERR_SHAPE;
    if (!workspace_dev || !att_out_dev || !row_dev || !qk || !decay_dev || !state_dev || !ret_out_dev) return CQ_ERR_NULL;
    for (int i = 0; i < 2; i++) {
        const int e = mix_check_group(qk[i], true);
        if (e) return e;
    }
    if (qk[0].heads != heads || qk[1].heads != heads || qk[0].dim != qk[1].dim) return CQ_ERR_SHAPE;
    if (mix_misaligned(state_dev, 16)) return CQ_ERR_ALIGN;
    if (qk[0].dim > CQ_MIX_MAX_DIM || vdim > 8192 || ctx > (1 << 28) || (!pos_dev && pos >= ctx)) return CQ_ERR_RANGE;
    StepArgs a;
    a.rec = (const float *)workspace_dev;
    a.n_head = (int)n_head; a.att_vdim = (int)att_vdim; a.ctx = (int)ctx;
    a.window = (int)(window < ctx ? window : ctx); a.keep_first = (int)(keep_first < ctx ? keep_first : ctx);
    const int64_t n_max = talk_max_keys(window, keep_first, ctx);
    a.splits = talk_splits(n_max); a.split_keys = talk_split_keys(n_max);
    a.att_scale = att_scale; a.ret_scale = ret_scale; a.eps = eps;
    a.att_out = att_out_dev; a.state = state_dev; a.ret_out = ret_out_dev; a.row = row_dev; a.decay = decay_dev;
    a.gq = qk[0]; a.gk = qk[1]; a.v_off = v_off; a.g_off = g_off; a.heads = (int)heads; a.vdim = (int)vdim;
    const int sp = (int)cq_mix_state_pad(qk[0].dim);
    const int f0 = (a.splits + 3) / 4 * 4 + 1024, f1 = 2 * sp + a.vdim;
    const size_t lds = (size_t)(f0 > f1 ? f0 : f1) * sizeof(float);
    if (lds > 64 * 1024) return CQ_ERR_RANGE;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)(n_head + heads));
    if (sp == 64) hipLaunchKernelGGL(talk_merge_retention_kernel<1>, grid, dim3(1024), lds, s, a, pos_dev, (int)pos);
    else if (sp == 128) hipLaunchKernelGGL(talk_merge_retention_kernel<2>, grid, dim3(1024), lds, s, a, pos_dev, (int)pos);
    else hipLaunchKernelGGL(talk_merge_retention_kernel<4>, grid, dim3(1024), lds, s, a, pos_dev, (int)pos);
    return (int)hipGetLastError();
}

int cq_mix_delta_prep(const float *row_dev, int64_t row_stride, int64_t r_off, int64_t k_off, int64_t a_off, const float *wl_dev, int64_t wl_stride,
                      const float *w0_dev, const float *a_bias_dev, float *packed_dev, int64_t rows, int64_t heads, int64_t dim, void *stream) {
    if (rows < 0 || heads <= 0 || dim <= 0 || r_off < 0 || k_off < 0 || a_off < 0 || wl_stride < heads * dim) return CQ_ERR_SHAPE;
    const int64_t top = (r_off > k_off ? r_off : k_off) > a_off ? (r_off > k_off ? r_off : k_off) : a_off;
    if (row_stride < top + heads * dim) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    if (!row_dev || !wl_dev || !w0_dev || !a_bias_dev || !packed_dev) return CQ_ERR_NULL;
    if (dim > CQ_MIX_MAX_DIM || heads > 4 * 65535 || rows > 0x7fffffffLL) return CQ_ERR_RANGE;
    hipLaunchKernelGGL(delta_prep_kernel, dim3((unsigned)rows, (unsigned)((heads + 3) / 4)), dim3(256), 0, (hipStream_t)stream, row_dev, row_stride, r_off, k_off, a_off,
                       wl_dev, wl_stride, w0_dev, a_bias_dev, packed_dev, rows, (int)heads, (int)dim, (int)cq_mix_state_pad(dim));
    return (int)hipGetLastError();
}

int cq_mix_delta_scan(const float *packed_dev, const float *v_dev, int64_t v_stride, float *state_dev, float *out_dev, int64_t out_stride, int64_t rows,
                      int64_t heads, int64_t dim, void *stream) {
    if (rows < 0 || heads <= 0 || dim <= 0 || v_stride < heads * dim || out_stride < heads * dim) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    if (!packed_dev || !v_dev || !state_dev || !out_dev) return CQ_ERR_NULL;
    if (mix_misaligned(packed_dev, 16) || mix_misaligned(state_dev, 16)) return CQ_ERR_ALIGN;
    if (dim > CQ_MIX_MAX_DIM || heads > (1 << 20) || rows > (1 << 24)) return CQ_ERR_RANGE;
    const int ncb = (int)((dim + 15) / 16), sp = (int)cq_mix_state_pad(dim);
    const dim3 grid((unsigned)((heads + 7) / 8 * 8 * ncb));
    hipStream_t s = (hipStream_t)stream;
#define CQ_DS(NR_, TB_)                                                                                                                                   \
    do {                                                                                                                                                   \
        const size_t lds = (size_t)2 * (TB_ * 4 * 64 * NR_ + TB_ * 16) * sizeof(float);                                                                    \
        if (lds > 64 * 1024) {                                                                                                                             \
            const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(delta_scan_kernel<NR_, TB_>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
            if (e) return e;                                                                                                                               \
        }                                                                                                                                                  \
        hipLaunchKernelGGL((delta_scan_kernel<NR_, TB_>), grid, dim3(256), lds, s, packed_dev, v_dev, v_stride, state_dev, out_dev, out_stride, (int)rows,  \
                           (int)heads, (int)dim, ncb);                                                                                                     \
    } while (0)
    if (sp == 64) CQ_DS(1, 16);
    else if (sp == 128) CQ_DS(2, 8);
    else CQ_DS(4, 8);
#undef CQ_DS
    return (int)hipGetLastError();
}

int64_t cq_mix_delta_rows_workspace_bytes(int64_t rows, int64_t heads, int64_t dim) {
    if (rows <= 0 || heads <= 0 || dim <= 0 || dim > CQ_MIX_MAX_DIM) return 0;
    if (delta_chunked(rows, heads, dim)) return (rows + KC - 1) / KC * heads * KREC * 4;
    return rows * heads * (4 * cq_mix_state_pad(dim) + 1) * 4;
}

int cq_mix_delta_rows(const float *row_dev, int64_t row_stride, int64_t r_off, int64_t k_off, int64_t v_off, int64_t a_off, const float *wl_dev, int64_t wl_stride,
                      const float *w0_dev, const float *a_bias_dev, float *state_dev, float *out_dev, int64_t out_stride, int64_t rows, int64_t heads, int64_t dim,
                      void *workspace_dev, int64_t workspace_bytes, void *stream) {
    if (rows < 0 || heads <= 0 || dim <= 0 || r_off < 0 || k_off < 0 || v_off < 0 || a_off < 0 || wl_stride < heads * dim || out_stride < heads * dim) return CQ_ERR_SHAPE;
    int64_t top = r_off > k_off ? r_off : k_off;
    top = top > v_off ? top : v_off;
    top = top > a_off ? top : a_off;
    if (row_stride < top + heads * dim) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    if (!row_dev || !wl_dev || !w0_dev || !a_bias_dev || !state_dev || !out_dev) return CQ_ERR_NULL;
    if (mix_misaligned(state_dev, 16) || mix_misaligned(workspace_dev, 16)) return CQ_ERR_ALIGN;
    if (dim > CQ_MIX_MAX_DIM || heads > 4 * 65535 || rows > (1 << 24)) return CQ_ERR_RANGE;
    if (!workspace_dev || workspace_bytes < cq_mix_delta_rows_workspace_bytes(rows, heads, dim)) return CQ_ERR_WORKSPACE;
    float *const ws = (float *)workspace_dev;
    if (!delta_chunked(rows, heads, dim)) {
        const int e = cq_mix_delta_prep(row_dev, row_stride, r_off, k_off, a_off, wl_dev, wl_stride, w0_dev, a_bias_dev, ws, rows, heads, dim, stream);
        return e ? e : cq_mix_delta_scan(ws, row_dev + v_off, row_stride, state_dev, out_dev, out_stride, rows, heads, dim, stream);
    }
    DeltaRowsIn a;
    a.row = row_dev; a.wl = wl_dev; a.w0 = w0_dev; a.ab = a_bias_dev;
    a.row_stride = row_stride; a.r_off = r_off; a.k_off = k_off; a.v_off = v_off; a.a_off = a_off; a.wl_stride = wl_stride;
    a.rows = (int)rows; a.heads = (int)heads; a.dim = (int)dim;
    const int ncb = (int)((dim + 15) / 16);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(delta_chunk_kernel, dim3((unsigned)((rows + KC - 1) / KC), (unsigned)heads), dim3(256), 0, s, a, ws);
    hipLaunchKernelGGL(delta_chain_kernel, dim3((unsigned)((heads + 7) / 8 * 8 * ncb)), dim3(512), 0, s, ws, state_dev, out_dev, out_stride, (int)rows, (int)heads, (int)dim, ncb);
    return (int)hipGetLastError();
}

int cq_mix_delta_step(const float *row_dev, int64_t r_off, int64_t k_off, int64_t v_off, int64_t g_off, int64_t a_off, int64_t low_off, const void *w2_dev,
                      int64_t ldw2, int64_t rank, const float *w0_dev, const float *a_bias_dev, const float *weight_dev, float *state_dev, float *out_dev,
                      int64_t heads, int64_t dim, float eps, void *stream) {
    if (heads <= 0 || dim <= 0 || rank <= 0 || ldw2 < rank || ldw2 % 64 || r_off < 0 || k_off < 0 || v_off < 0 || g_off < 0 || a_off < 0 || low_off < 0)
        return CQ_ERR_SHAPE;
    if (!row_dev || !w2_dev || !w0_dev || !a_bias_dev || !weight_dev || !state_dev || !out_dev) return CQ_ERR_NULL;
    if (mix_misaligned(w2_dev, 16) || mix_misaligned(state_dev, 16)) return CQ_ERR_ALIGN;
    if (dim > CQ_MIX_MAX_DIM || heads > (1 << 20) || ldw2 > 8192) return CQ_ERR_RANGE;
    DeltaStep a;
    a.row = row_dev; a.w0 = w0_dev; a.ab = a_bias_dev; a.weight = weight_dev; a.w2 = (const uint16_t *)w2_dev; a.state = state_dev; a.out = out_dev;
    a.r_off = r_off; a.k_off = k_off; a.v_off = v_off; a.g_off = g_off; a.a_off = a_off; a.low_off = low_off; a.ldw2 = ldw2;
    a.rank = (int)rank; a.heads = (int)heads; a.dim = (int)dim; a.eps = eps;
    const size_t lds = (size_t)ldw2 * sizeof(float);
    hipStream_t s = (hipStream_t)stream;
    const int sp = (int)cq_mix_state_pad(dim);
    if (sp == 64) hipLaunchKernelGGL(delta_step_kernel<1>, dim3((unsigned)heads), dim3(1024), lds, s, a);
    else if (sp == 128) hipLaunchKernelGGL(delta_step_kernel<2>, dim3((unsigned)heads), dim3(1024), lds, s, a);
    else hipLaunchKernelGGL(delta_step_kernel<4>, dim3((unsigned)heads), dim3(1024), lds, s, a);
    return (int)hipGetLastError();
}

}  // extern "C"
