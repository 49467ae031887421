// Softmax attention whose scores are mixed across heads before the softmax, over a sliding window plus the first tokens of
// the sequence.  Mixing couples the heads, so one workgroup holds the scores of all heads for its queries and keys.
// f32 throughout (v_mfma_f32_16x16x4): scores, weights, caches.
#include <algorithm>
#include "cq_mix.h"

namespace {

// A load from a wave-uniform base with a 32-bit byte offset: the address costs one register per lane.
template <typename T> __device__ __forceinline__ T ld_at(const float *base, uint32_t bytes) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
}

// ---- several queries ------------------------------------------------------------------------------------------------------
// Workgroup: 16 query rows x all heads, NW waves, keys in tiles of KT, one pass with a running maximum.  Per tile:
//   scores   wave w takes heads [w NHW, (w + 1) NHW): q k^T into LDS, [head][query][key]
//   mixing   wave w takes 16 / NW queries of every head: talk x scores on the matrix cores (heads are the contracted
//            dimension), mask, running softmax in registers, weights back into the same LDS words, rescale factors to `alpha`
//   values   wave w takes U units (head, 64 output columns): weights x V added to the outputs it holds in registers, V read once per VS units
// blockIdx.y: units beyond NW U (the scores are computed again there).  blockIdx.z: split of the key tiles, for calls with too few
// query rows to fill the chip; a split leaves unnormalized outputs with their maximum and sum, talk_combine_kernel merges them.
// LDS strides: query rows of KT + 4 floats (16 rows x 4 keys of an operand read fall on 64 banks), head blocks of 16 rows + 16
// (4 heads x 16 keys likewise).
template <int NW, int NHW, bool SHARED_K, int U, int VS, int KT, typename OT>
__global__ __launch_bounds__(64 * NW) void talk_attention_kernel(const float *__restrict__ q, const float *__restrict__ k_cache, const float *__restrict__ v_cache,
                                                             const float *__restrict__ talk, float scale, int window, int keep_first, float out_scale,
                                                             OT *__restrict__ out, int64_t out_stride, float *__restrict__ part, int pos, int rows, int H, int G,
                                                             int dp, int vdim, int vp, int ctx) {
    constexpr int NHT = (NW * NHW + 15) / 16, HP = 16 * NHT, NT = 64 * NW, RW = 16 / NW;       // heads padded to tiles of 16; queries per wave
    constexpr int RS = KT + 4, HS = 16 * RS + 16, TS = HP + 4, KTL = KT / 16;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float *S = smem, *T = S + HP * HS, *alpha = T + HP * TS, *m_run = alpha + HP * 16, *l_run = m_run + HP * 16;      // the last three: [head][query]
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const int r0 = blockIdx.x * 16, nr = min(16, rows - r0);
    const int p0 = pos + r0, last = p0 + nr - 1;                         // positions of the first and last query
    const int R = H / G, nvc = (vp + 63) / 64;

    for (int i = tid; i < HP * HP; i += NT) {
        const int h = i / HP, g = i - h * HP;
        T[h * TS + g] = h < H && g < H ? talk[h * H + g] * scale : 0.0f;
    }
    for (int i = tid; i < (HP - H) * HS; i += NT) S[H * HS + i] = 0.0f;

    for (int i = tid; i < HP * 16; i += NT) {
        m_run[i] = -INFINITY;
        l_run[i] = 0.0f;
    }
    __syncthreads();
    f32x4 o[U][4];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int n = 0; n < 4; n++) o[u][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int h0 = wv * NHW;
    const float *qb = q + (int64_t)r0 * H * dp;
    const uint32_t q_at = (min(lr, nr - 1) * H * dp + 4 * lk) * 4;
    const int u0 = ((int)blockIdx.y * NW + wv) * U, n_units = H * nvc;

    // tiles of the kept first tokens, then of the window
    const int t_lo = max(0, p0 - window + 1) / KT, t_hi = last / KT;
    const int n_keep = min((keep_first + KT - 1) / KT, t_lo);
    const int n_tiles = n_keep + t_hi - t_lo + 1, nz = gridDim.z, z = blockIdx.z;
    for (int it = n_tiles * z / nz; it < n_tiles * (z + 1) / nz; it++) {
        const int j0 = (it < n_keep ? it : t_lo + it - n_keep) * KT;
        // ---- scores ----
        if (h0 < H) {
            f32x4 acc[NHW][KTL];
#pragma unroll
            for (int i = 0; i < NHW; i++)
#pragma unroll
                for (int t = 0; t < KTL; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            uint32_t k_at[KTL];
#pragma unroll
            for (int t = 0; t < KTL; t++) k_at[t] = (min(j0 + 16 * t + lr, last) * dp + 4 * lk) * 4u;
            const int64_t kv_stride = (int64_t)ctx * dp;
            for (int c = 0; c < dp; c += 16) {
                f32x4 kf[KTL], qf[NHW];
                if (SHARED_K) {
#pragma unroll
                    for (int t = 0; t < KTL; t++) kf[t] = ld_at<f32x4>(k_cache + (h0 / R) * kv_stride + c, k_at[t]);
                }
#pragma unroll
                for (int i = 0; i < NHW; i++) qf[i] = ld_at<f32x4>(qb + min(h0 + i, H - 1) * dp + c, q_at);
#pragma unroll
                for (int i = 0; i < NHW; i++) {
                    if (!SHARED_K) {
#pragma unroll
                        for (int t = 0; t < KTL; t++) kf[t] = ld_at<f32x4>(k_cache + (min(h0 + i, H - 1) / R) * kv_stride + c, k_at[t]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int t = 0; t < KTL; t++) acc[i][t] = mfma4(qf[i][e], kf[t][e], acc[i][t]);
                }
            }
#pragma unroll
            for (int i = 0; i < NHW; i++)
                if (h0 + i < H) {
#pragma unroll
                    for (int t = 0; t < KTL; t++)
#pragma unroll
                        for (int e = 0; e < 4; e++) S[(h0 + i) * HS + (4 * lk + e) * RS + 16 * t + lr] = acc[i][t][e];
                }
        }
        __syncthreads();

        // ---- mixing and softmax: queries RW wv .., one after the other ----
#pragma unroll
        for (int a = 0; a < RW; a++) {
            f32x4 acc[KTL][NHT];
#pragma unroll
            for (int t = 0; t < KTL; t++)
#pragma unroll
                for (int b = 0; b < NHT; b++) acc[t][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
            for (int s = 0; s < HP / 4; s++) {
                float tf[NHT], sf[KTL];
#pragma unroll
                for (int b = 0; b < NHT; b++) tf[b] = T[(16 * b + lr) * TS + 4 * s + lk];
#pragma unroll
                for (int t = 0; t < KTL; t++) sf[t] = S[(4 * s + lk) * HS + (RW * wv + a) * RS + 16 * t + lr];
#pragma unroll
                for (int t = 0; t < KTL; t++)
#pragma unroll
                    for (int b = 0; b < NHT; b++) acc[t][b] = mfma4(tf[b], sf[t], acc[t][b]);
            }
            const int p = p0 + RW * wv + a;
            bool vis[KTL];
#pragma unroll
            for (int t = 0; t < KTL; t++) {
                const int j = j0 + 16 * t + lr;
                vis[t] = j <= p && (p - j < window || j < keep_first);
            }
#pragma unroll
            for (int b = 0; b < NHT; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float s[KTL], mx = -INFINITY, sum = 0.0f;
#pragma unroll
                    for (int t = 0; t < KTL; t++) {
                        s[t] = vis[t] ? acc[t][b][e] : -INFINITY;
                        mx = fmaxf(mx, s[t]);
                    }
                    const int h = 16 * b + 4 * lk + e, hr = h * 16 + RW * wv + a;
                    const float m_old = m_run[hr], m = fmaxf(m_old, row16_max(mx));
                    const float al = m_old > -INFINITY ? __expf(m_old - m) : 0.0f;
#pragma unroll
                    for (int t = 0; t < KTL; t++) {
                        const float w = vis[t] ? __expf(s[t] - m) : 0.0f;
                        sum += w;
                        S[h * HS + (RW * wv + a) * RS + 16 * t + lr] = w;
                    }
                    sum = row16_sum(sum);
                    m_run[hr] = m;                       // the same value from 16 lanes
                    l_run[hr] = l_run[hr] * al + sum;
                    alpha[hr] = al;
                }
        }
        __syncthreads();

        // ---- values (units beyond the last repeat it and are not stored) ----
        if (u0 < n_units) {
#pragma unroll
            for (int ub = 0; ub < U; ub += VS) {
                const int uc = min(u0 + ub, n_units - VS);
                const int g = uc / (R * nvc), c = (uc / R) % nvc, h0v = g * R + uc % R;
                const float *vb = v_cache + (int64_t)g * ctx * vp + 64 * c;
#pragma unroll
                for (int half = 0; half < KTL; half++) {
                    float vf[4][4];
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        const uint32_t at = min(j0 + 16 * half + 4 * s + lk, last) * vp;
#pragma unroll
                        for (int n = 0; n < 4; n++) vf[s][n] = ld_at<float>(vb, (at + min(16 * n + lr, vp - 64 * c - 1)) * 4u);
                    }
#pragma unroll
                    for (int v = 0; v < VS; v++) {
                        const int u = ub + v, h = h0v + v;
                        if (half == 0) {
                            const f32x4 al = *reinterpret_cast<const f32x4 *>(&alpha[h * 16 + 4 * lk]);
#pragma unroll
                            for (int n = 0; n < 4; n++) o[u][n] *= al;
                        }
#pragma unroll
                        for (int s = 0; s < 4; s++) {
                            const float w = S[h * HS + lr * RS + 16 * half + 4 * s + lk];
#pragma unroll
                            for (int n = 0; n < 4; n++) o[u][n] = mfma4(w, vf[s][n], o[u][n]);
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (u0 + u >= n_units) continue;
        const int g = (u0 + u) / (R * nvc), c = ((u0 + u) / R) % nvc, h = g * R + (u0 + u) % R;
#pragma unroll
        for (int n = 0; n < 4; n++) {
            const int col = 64 * c + 16 * n + lr;
            if (col >= vdim) continue;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = 4 * lk + e;
                if (row >= nr) continue;
                if (nz == 1) out[(int64_t)(r0 + row) * out_stride + (int64_t)h * vdim + col] = (OT)(out_scale * o[u][n][e] / l_run[h * 16 + row]);
                else part[((int64_t)(z * rows + r0 + row) * H + h) * vdim + col] = o[u][n][e];
            }
        }
    }
    if (nz > 1 && blockIdx.y == 0) {
        float *ml = part + (int64_t)nz * rows * H * vdim;                 // [split][row][head] of (m, l)
        for (int i = tid; i < nr * H; i += NT) {
            const int row = i / H, h = i - row * H;
            float *x = ml + 2 * ((int64_t)(z * rows + r0 + row) * H + h);
            x[0] = m_run[h * 16 + row];
            x[1] = l_run[h * 16 + row];
        }
    }
}

// ---- several queries, heads of 128 dimensions in groups of R = 2, 4 or 8 on one kv head, H = 8 or 16 of them -----------------------------------
// Workgroup: 16 query rows x all heads, one wave a head, keys in tiles of 16.  Above, every wave reads its queries, keys and values from the caches for every tile, 40 KB a
// wave and 32 keys through a unit's 64 bytes a cycle, and three barriers separate that from the mixing.  Here the queries stay in registers, and copies that no
// register sees bring keys and values to LDS two tiles ahead, once for the R heads that share them.  Per tile:
//   mixing   wave w takes 16 / H queries of all heads, as above; running maxima and sums in its registers
//   values   wave w: the weights of head w x V onto its outputs, then the scores of the next tile, which replace those weights when they are formed
// so that only the mixing stands between two barriers.
// LDS rows of 512 bytes in 32 16-byte chunks: keys' chunk c of row r at c ^ r, values as they are; both without bank conflicts.
// 16 heads in us, above -> this: 2048 rows (window 1024) 327 -> 185, 500: 111 -> 43, 100: 65 -> 30; the error against 64 bits falls (2048 rows 4.9e-7 -> 4.0e-7: scores in two
// sums).  Bound by the f32 matrix instructions, 68 of 32 cycles a wave and tile, four waves to a matrix core: 62 % of a unit's busy cycles, the rest barriers and
// the mixing.
typedef __attribute__((address_space(3))) void talk_lds;
// The tiles of all blocks of 16 rows form one sequence, of which every workgroup takes `chunk`: the first rows see fewer keys than the last, and equal parts of each block left
// a quarter of the units' time idle (2048 rows 210 -> 185 us, 6000 rows 730 -> 530, 8 heads and 2048 rows 132 -> 106).  A part costs 12 us beside its tiles of 5.5: the
// queries and the first keys arrive, every tile at first brings new maxima, and its results go to the workspace.  So a block counts for `lead` tiles more than it has (with none
// the workgroup that gets the six first blocks ended last, 256 us; with 1: 218, 2: 185, 3: 185, and 4096 rows 422, 371, 358), and where the chunks are of
// few tiles (lead 0) none crosses into another block.
constexpr int TT_RS = 20, TT_HS = 16 * TT_RS + 16, TT_ROW = 512, TT_TILE = 16 * TT_ROW;      // floats of a query's weights, of a head's; bytes of a key, of a tile
__host__ __device__ constexpr int talk_tile_lds(int H, int R) { return 4 * (H / R) * TT_TILE + (H * TT_HS + 3 * 256) * 4; }

// The tiles of keys that the 16 rows from r0 on see: those of the kept first tokens, then the window's from t_lo on.
struct TalkTiles {
    int t_lo, n_keep, n, last;
};
__host__ __device__ __forceinline__ TalkTiles talk_tiles_of(int r0, int rows, int pos, int window, int keep_first) {
    TalkTiles t;
    const int p0 = pos + r0, lo = p0 - window + 1, kt = (keep_first + 15) / 16;
    t.last = pos + (r0 + 16 < rows ? r0 + 16 : rows) - 1;
    t.t_lo = (lo > 0 ? lo : 0) / 16;
    t.n_keep = kt < t.t_lo ? kt : t.t_lo;
    t.n = t.n_keep + t.last / 16 - t.t_lo + 1;
    return t;
}
// What a block of n tiles counts in the common sequence: `lead` more than it has, or for lead 0 whole chunks.
__host__ __device__ __forceinline__ int talk_length(int n, int chunk, int lead) { return lead ? n + lead : (n + chunk - 1) / chunk * chunk; }
__host__ __device__ constexpr int64_t talk_slot(int H) { return 16 * H * 130; }      // floats of a partial result: outputs [row][head][128], (m, l) [row][head]

template <int H, int R, typename OT>
__global__ __launch_bounds__(64 * H) void talk_tile_kernel(const float *__restrict__ q, const float *__restrict__ k_cache, const float *__restrict__ v_cache,
                                                           const float *__restrict__ talk, float scale, int window, int keep_first, float out_scale, OT *__restrict__ out,
                                                           int64_t out_stride, float *__restrict__ part, int2 *__restrict__ span, int chunk, int lead, int pos, int rows, int vdim,
                                                           int ctx) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler does not know the buffer accesses)
    constexpr int G = H / R, RW = 16 / H, NI = 8 / R, HALF = G * TT_TILE;       // queries of a wave in the mixing; copies of a wave for a tile of keys
    extern __shared__ __attribute__((aligned(16))) uint8_t tt_smem[];
    uint8_t *const kbuf = tt_smem, *const vbuf = tt_smem + 2 * HALF;
    float *const S = reinterpret_cast<float *>(tt_smem + 4 * HALF), *const alpha = S + H * TT_HS, *const m_run = alpha + 256, *const l_run = m_run + 256;
    const int lane = threadIdx.x & 63, h = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lk = lane >> 4;
    const int w = blockIdx.x, blocks = (rows + 15) / 16;
    int b = blocks - 1 - w, first = 0, todo = 0;           // block of rows (whole ones: the long ones first), the tile of it to start with, tiles left
    if (chunk) {
        int before = 0;                                    // tiles of the blocks before b
        for (int b0 = 0; b0 < blocks; b0 += 64) {
            int sum = b0 + lane < blocks ? talk_length(talk_tiles_of(16 * (b0 + lane), rows, pos, window, keep_first).n, chunk, lead) : 0;
#pragma unroll
            for (int d = 1; d < 64; d *= 2) {
                const int x = __shfl_up(sum, d);
                if (lane >= d) sum += x;
            }
            const int skip = __popcll(__ballot(before + sum <= w * chunk));
            b = b0 + skip;
            if (skip < 64) {
                if (skip) before += __shfl(sum, skip - 1);
                break;
            }
            before += __shfl(sum, 63);
        }
        b = __builtin_amdgcn_readfirstlane(b);
        first = __builtin_amdgcn_readfirstlane(w * chunk - before);
        todo = chunk;
    }
    for (bool head = true; b < blocks; b++, first = 0, head = false) {
    const int r0 = 16 * b, nr = min(16, rows - r0), p0 = pos + r0;
    const TalkTiles tiles = talk_tiles_of(r0, rows, pos, window, keep_first);
    const int t_lo = tiles.t_lo, n_keep = tiles.n_keep, last = tiles.last, it0 = max(first - lead, 0), it1 = chunk ? min(tiles.n, first - lead + todo) : tiles.n;
    const bool whole = it0 == 0 && it1 == tiles.n;
    todo -= it1 - (first - lead);
    if (it1 <= 0) break;                                   // (nothing but the lead)
    auto first_key = [&](int it) { return 16 * (it < n_keep ? it : t_lo + it - n_keep); };

    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)k_cache, 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)v_cache, 0, -1, 0x00020000);
    // two rows an instruction, rows beyond the last visible key repeat it (past the last tile: that one again, for nobody)
    auto copy = [&](auto values, int it) {
        uint8_t *const to = (values ? vbuf : kbuf) + ((it - it0) & 1) * HALF;
        const int j0 = first_key(min(it, it1 - 1));
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const int u = h + H * j, g = u >> 3, row = 2 * (u & 7) + (lane >> 5), c = values ? lane & 31 : (lane & 31) ^ row;
            const uint32_t at = (uint32_t)(g * ctx + min(j0 + row, last)) * TT_ROW + 16 * c;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(values ? vrs : krs, (talk_lds *)(to + 1024 * u), 16, at, 0, 0, 0);
        }
        asm volatile("" ::: "memory");
    };
    constexpr std::integral_constant<bool, false> keys{};
    constexpr std::integral_constant<bool, true> values{};
    f32x4 qd[8];                                           // dims 16 c + 4 lk .. of query lr
    float tf[H / 4], m[RW][4], l[RW][4];                   // mixing weights [head lr][4 s + lk]; of head 4 lk + e and the wave's queries (l: of this lane's keys)
    {
        int dim0 = 4 * lk;
        asm("" : "+v"(dim0));
        const float *qr = q + ((int64_t)(r0 + min(lr, nr - 1)) * H + h) * 128 + dim0;
#pragma unroll
        for (int c = 0; c < 8; c++) qd[c] = *reinterpret_cast<const f32x4 *>(qr + 16 * c);
    }
#pragma unroll
    for (int s = 0; s < H / 4; s++) tf[s] = lr < H ? talk[min(lr, H - 1) * H + 4 * s + lk] * scale : 0.0f;
#pragma unroll
    for (int a = 0; a < RW; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            m[a][e] = -INFINITY;
            l[a][e] = 0.0f;
        }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 o[2][4];                                         // queries 4 lk .. of column 64 x + 4 lr + n
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int n = 0; n < 4; n++) o[x][n] = zero;
    bool stale[RW];
#pragma unroll
    for (int a = 0; a < RW; a++) stale[a] = true;                // (the first tile rescales, also for a query that sees nothing of it)
    float *const Sh = S + h * TT_HS;
    auto scores = [&](int it) {                            // of the wave's head, into S
        const uint8_t *const kt = kbuf + ((it - it0) & 1) * HALF + (h / R) * TT_TILE + lr * TT_ROW;
        f32x4 sc[2] = {zero, zero};
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const f32x4 kf = *reinterpret_cast<const f32x4 *>(kt + 16 * ((4 * c + lk) ^ lr));
#pragma unroll
            for (int e = 0; e < 4; e++) sc[c & 1] = mfma4(qd[c][e], kf[e], sc[c & 1]);
        }
        const f32x4 s = sc[0] + sc[1];
#pragma unroll
        for (int e = 0; e < 4; e++) Sh[(4 * lk + e) * TT_RS + lr] = s[e];
    };
    if (it0 < it1) {
        copy(keys, it0);
        copy(values, it0);
        copy(keys, it0 + 1);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NI) : "memory");
        scores(it0);
    }
    for (int it = it0; it < it1; it++) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the scores of all heads are there
        const int j = first_key(it) + lr;
#pragma unroll
        for (int a = 0; a < RW; a++) {
            const int qi = RW * h + a, p = p0 + qi;
            f32x4 acc = zero;
#pragma unroll
            for (int s = 0; s < H / 4; s++) acc = mfma4(tf[s], S[(4 * s + lk) * TT_HS + qi * TT_RS + lr], acc);
            const bool vis = j <= p && (p - j < window || j < keep_first);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = vis ? acc[e] : -INFINITY;
            const bool up = acc[0] > m[a][0] || acc[1] > m[a][1] || acc[2] > m[a][2] || acc[3] > m[a][3];
            if (__any(up) || stale[a]) {                   // a new maximum, or one in the tile before
                stale[a] = __any(up);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float top = fmaxf(m[a][e], row16_max(acc[e])), al = m[a][e] > -INFINITY ? __expf(m[a][e] - top) : 0.0f;
                    m[a][e] = top;
                    l[a][e] *= al;
                    if (H == 16 || lk < 2) alpha[(4 * lk + e) * 16 + qi] = al;      // (the same value from 16 lanes)
                }
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float w = vis ? __expf(acc[e] - m[a][e]) : 0.0f;
                l[a][e] += w;
                if (H == 16 || lk < 2) S[(4 * lk + e) * TT_HS + qi * TT_RS + lr] = w;
            }
        }
        // the weights of all queries are there, and so are the values of this tile and the keys of the next
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        copy(values, it + 1);
        copy(keys, it + 2);
        const f32x4 al = *reinterpret_cast<const f32x4 *>(&alpha[h * 16 + 4 * lk]);
        if (__any(al.x != 1.0f || al.y != 1.0f || al.z != 1.0f || al.w != 1.0f)) {
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int n = 0; n < 4; n++) o[x][n] *= al;
        }
        const uint8_t *const vt = vbuf + ((it - it0) & 1) * HALF + (h / R) * TT_TILE + lk * TT_ROW + 16 * lr;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const float w = Sh[lr * TT_RS + 4 * s + lk];
#pragma unroll
            for (int x = 0; x < 2; x++) {
                const f32x4 vf = *reinterpret_cast<const f32x4 *>(vt + 4 * s * TT_ROW + 256 * x);
#pragma unroll
                for (int n = 0; n < 4; n++) o[x][n] = mfma4(w, vf[n], o[x][n]);
            }
        }
        if (it + 1 < it1) scores(it + 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (copies may not outlive the workgroup)
#pragma unroll
    for (int a = 0; a < RW; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            l_run[(4 * lk + e) * 16 + RW * h + a] = row16_sum(l[a][e]);
            m_run[(4 * lk + e) * 16 + RW * h + a] = m[a][e];
        }
    __syncthreads();
    float *const slot = part + (2 * (int64_t)w + !head) * talk_slot(H);
    int row0 = 4 * lk, col0 = 4 * lr;
    asm("" : "+v"(row0), "+v"(col0));                    // (addresses made from these stay out of the loop's registers)
    if (whole) {
        const f32x4 lh = *reinterpret_cast<const f32x4 *>(&l_run[h * 16 + row0]);
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = row0 + e, col = 64 * x + col0;
                if (row >= nr) continue;
#pragma unroll
                for (int n = 0; n < 4; n++)
                    if (col + n < vdim) out[(int64_t)(r0 + row) * out_stride + (int64_t)h * vdim + col + n] = (OT)(out_scale * o[x][n][e] / lh[e]);
            }
    } else {
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                *reinterpret_cast<f32x4 *>(&slot[((row0 + e) * H + h) * 128 + 64 * x + col0]) = f32x4{o[x][0][e], o[x][1][e], o[x][2][e], o[x][3][e]};
        for (int i = threadIdx.x; i < 16 * H; i += 64 * H) {
            const int row = i / H, hh = i - row * H;
            slot[16 * H * 128 + 2 * i] = m_run[hh * 16 + row];
            slot[16 * H * 128 + 2 * i + 1] = l_run[hh * 16 + row];
        }
    }
    // the partial results of a block: the slot of its first part, the workgroup of its last; whole ones are done
    if (chunk && threadIdx.x == 0) {
        if (it0 == 0) span[b].x = whole ? -1 : 2 * w + !head;
        if (it1 == tiles.n) span[b].y = w;
    }
    if (todo <= 0 || !lead) break;
    }
#endif
}

// The partial results of talk_tile_kernel; half a wave per (row, head).  2048 rows of 16 heads: 12.6 us, of which most is their memory.
template <typename OT>
__global__ __launch_bounds__(256) void talk_tile_combine_kernel(const float *__restrict__ part, const int2 *__restrict__ span, int H, int vdim, float out_scale,
                                                                OT *__restrict__ out, int64_t out_stride) {
    const int lane = threadIdx.x & 31, h = blockIdx.y * 8 + (threadIdx.x >> 5), r = blockIdx.x, i = (r & 15) * H + h;
    const int2 sp = span[r >> 4];
    if (sp.x < 0) return;
    const int64_t step = talk_slot(H);
    auto slot = [&](int z) { return part + (z ? 2 * ((sp.x >> 1) + z) : sp.x) * step; };      // the others are the first of their workgroups
    auto stat = [&](int z) { return *reinterpret_cast<const float2 *>(slot(z) + 16 * H * 128 + 2 * i); };
    const int nz = sp.y - (sp.x >> 1) + 1;
    float m = -INFINITY, l = 0.0f;
    for (int z = 0; z < nz; z++) m = fmaxf(m, stat(z).x);
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < nz; z++) {
        const float2 ml = stat(z);
        const f32x4 v = *reinterpret_cast<const f32x4 *>(slot(z) + (int64_t)i * 128 + 4 * lane);
        const float w = ml.x > -INFINITY ? __expf(ml.x - m) : 0.0f;
        l = fmaf(w, ml.y, l);
#pragma unroll
        for (int e = 0; e < 4; e++) a[e] = fmaf(w, v[e], a[e]);
    }
    OT *o = out + (int64_t)r * out_stride + (int64_t)h * vdim + 4 * lane;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (4 * lane + e < vdim) o[e] = (OT)(out_scale * a[e] / l);
}

// one wave per (row, head)
template <typename OT>
__global__ __launch_bounds__(256) void talk_combine_kernel(const float *__restrict__ part, int nz, int64_t rows, int H, int vdim, float out_scale,
                                                           OT *__restrict__ out, int64_t out_stride) {
    const int lane = threadIdx.x & 63, h = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (h >= H) return;
    const int64_t r = blockIdx.x, id = r * H + h, n = rows * H;
    const float *ml = part + nz * n * vdim + 2 * id;
    float m = -INFINITY, l = 0.0f;
    for (int z = 0; z < nz; z++) m = fmaxf(m, ml[2 * n * z]);
    for (int z = 0; z < nz; z++) l = fmaf(ml[2 * n * z] > -INFINITY ? __expf(ml[2 * n * z] - m) : 0.0f, ml[2 * n * z + 1], l);
    OT *o = out + r * out_stride + (int64_t)h * vdim;
    for (int e = lane; e < vdim; e += 64) {
        float a = 0.0f;
        for (int z = 0; z < nz; z++) {
            const float w = ml[2 * n * z] > -INFINITY ? __expf(ml[2 * n * z] - m) : 0.0f;
            a = fmaf(w, part[(n * z + id) * vdim + e], a);
        }
        o[e] = (OT)(out_scale * a / l);
    }
}

// Splits of the key tiles: as many as bring the launch to one workgroup per CU, each with at least four tiles of keys.
int talk_key_splits(int64_t rows, int64_t unit_blocks, int64_t max_keys) {
    const int64_t wg = (rows + 15) / 16 * unit_blocks, tiles = max_keys / 32;
    int64_t n = 256 / wg;
    n = n < tiles / 4 ? n : tiles / 4;
    return (int)(n < 1 ? 1 : (n > 16 ? 16 : n));
}
constexpr int TALK_MAX_BLOCKS = 1024, TALK_LEAD = 3;
// Tiles of keys of a workgroup of talk_tile_kernel when the workspace holds `slots` partial results; 0: one workgroup per 16 rows.  The balanced sequence pays from 8 tiles
// a unit on (us balanced / whole chunks: 2048 rows 190 / 213, 1200: 90 / 96, 1000: 78 / 75, 700: 54 / 53); at most 17 parts a block, of two tiles and more; beyond TALK_MAX_BLOCKS
// the order of the blocks balances as well (12000 rows 1054 us, one workgroup per block 1094).
struct TalkPlan {
    int chunk = 0, lead = 0, workgroups = 0;
};
TalkPlan talk_tile_plan(int64_t rows, int64_t window, int64_t keep_first, int64_t pos, int64_t slots) {
    const int blocks = (int)((rows + 15) / 16);
    TalkPlan plan{0, 0, blocks};
    if (blocks > TALK_MAX_BLOCKS || slots < 2) return plan;
    auto total = [&](int chunk, int lead) {
        int64_t n = 0;
        for (int b = 0; b < blocks; b++) n += talk_length(talk_tiles_of(16 * b, (int)rows, (int)pos, (int)window, (int)keep_first).n, chunk, lead);
        return n;
    };
    int most = 0;
    for (int b = 0; b < blocks; b++) most = std::max(most, talk_tiles_of(16 * b, (int)rows, (int)pos, (int)window, (int)keep_first).n);
    const int64_t units = std::min<int64_t>(256, slots / 2), tiles = total(1, 0);
    const int lead = tiles >= 8 * 256 ? TALK_LEAD : 0;
    if (!lead && blocks > units) return plan;
    int64_t chunk = std::max<int64_t>({(tiles + (int64_t)lead * blocks + units - 1) / units, 2, (most + 15) / 16});
    while (!lead && total((int)chunk, 0) > units * chunk) chunk++;
    if (chunk + lead < (int64_t)((blocks + 255) / 256) * (most + lead)) plan = {(int)chunk, lead, (int)((total((int)chunk, lead) + chunk - 1) / chunk)};
    return plan;
}
// Which calls talk_tile_kernel takes: what it has instances for, LDS for up to four kv heads, offsets of 32 bits into the caches.  It is the faster one at all sizes
// (16 heads: 20 rows 22.8 -> 20.7 us, 100: 65 -> 30, 500: 111 -> 43, 2048: 327 -> 185; 8 heads, 2048 rows 196 -> 106).
bool talk_by_tiles(int64_t H, int64_t G, int64_t dim_pad, int64_t vdim_pad, int64_t ctx) {
    const int64_t R = H / G;
    return dim_pad == 128 && vdim_pad == 128 && (H == 8 || H == 16) && (R == 4 || R == 8 || (R == 2 && H == 8)) && G * ctx < (1LL << 23);
}
int talk_unit_blocks(int64_t H, int64_t vp) {               // units a launch takes: NW * U of the instance for H heads
    const int64_t per = H <= 8 ? 16 : (H <= 16 ? 32 : 64);
    return (int)((H * ((vp + 63) / 64) + per - 1) / per);
}

template <int NW, int NHW, bool SHARED_K, int U, int VS, int KT, typename OT>
int talk_launch(const float *q, const float *kc, const float *vc, const float *talk, float scale, int window, int keep, float out_scale, OT *out,
                int64_t out_stride, float *part, int nz, int pos, int rows, int H, int G, int dp, int vdim, int vp, int ctx, hipStream_t s) {
    constexpr int HP = (NW * NHW + 15) / 16 * 16;
    constexpr size_t lds = (size_t)(HP * (16 * (KT + 4) + 16) + HP * (HP + 4) + 3 * HP * 16) * sizeof(float);
    if (lds > 64 * 1024) {
        const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(talk_attention_kernel<NW, NHW, SHARED_K, U, VS, KT, OT>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e) return e;
    }
    const int units = H * ((vp + 63) / 64);
    hipLaunchKernelGGL((talk_attention_kernel<NW, NHW, SHARED_K, U, VS, KT, OT>), dim3((rows + 15) / 16, (units + NW * U - 1) / (NW * U), nz), dim3(64 * NW), lds,
                       s, q, kc, vc, talk, scale, window, keep, out_scale, out, out_stride, part, pos, rows, H, G, dp, vdim, vp, ctx);
    if (nz > 1)
        hipLaunchKernelGGL(talk_combine_kernel<OT>, dim3((unsigned)rows, (unsigned)((H + 3) / 4)), dim3(256), 0, s, (const float *)part, nz, (int64_t)rows, H, vdim, out_scale,
                           out, out_stride);
    return (int)hipGetLastError();
}

template <int H, int R, typename OT>
int talk_tile_launch(const float *q, const float *kc, const float *vc, const float *talk, float scale, int window, int keep, float out_scale, OT *out, int64_t out_stride,
                     float *part, const TalkPlan &plan, int pos, int rows, int vdim, int ctx, hipStream_t s) {
    constexpr int lds = talk_tile_lds(H, R);
    int2 *const span = reinterpret_cast<int2 *>(part + 2 * plan.workgroups * talk_slot(H));
    const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(talk_tile_kernel<H, R, OT>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e) return e;
    hipLaunchKernelGGL((talk_tile_kernel<H, R, OT>), dim3(plan.workgroups), dim3(64 * H), lds, s, q, kc, vc, talk, scale, window, keep, out_scale, out, out_stride, part, span,
                       plan.chunk, plan.lead, pos, rows, vdim, ctx);
    if (plan.chunk)
        hipLaunchKernelGGL(talk_tile_combine_kernel<OT>, dim3((unsigned)rows, H / 8), dim3(256), 0, s, (const float *)part, (const int2 *)span, H, vdim, out_scale, out, out_stride);
    return (int)hipGetLastError();
}

// ---- one query --------------------------------------------------------------------------------------------------------------
// Workgroup: KD of the visible keys x all heads, 16 waves.  The first K and V rows and the head mixing matrix are requested before
// anything else; meanwhile the workgroup normalizes and rotates q itself.  The one that holds the last visible key (the new token) does
// the same for k and v, appends them to the caches and uses its own copies.
//   scores  16 lanes per (kv head, key), each key row read once for the heads that share it
//   mixing  one thread per (head, key)
//   values  four lanes per (kv head, four columns), each on a quarter of the keys, four heads at a time
template <int NC, int KD>
__global__ __launch_bounds__(1024) void talk_decode_kernel(const float *__restrict__ row, cq_mix_heads gq, cq_mix_heads gk, cq_mix_heads gv, float eps,
                                                           const float *__restrict__ talk, float scale, int window, int keep_first,
                                                           const int32_t *__restrict__ pos_dev, int pos0, float *__restrict__ rec, int splits) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int H = gq.heads, G = gk.heads, R = H / G, dp = gk.dim_pad, vdim = gv.dim, vp = gv.dim_pad, ctx = gk.ctx;
    constexpr int SS = KD + 4, PB = 2;                               // rows of scores start on 16 bytes
    float *qs = smem, *kn = qs + H * dp, *vn = kn + G * dp, *sc = vn + G * vp, *mx = sc + H * SS, *T = mx + H * SS;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), sp = blockIdx.x;
    const int p = pos0 + (pos_dev ? pos_dev[0] : 0);
    const Visible vis = visible_keys(p, window, keep_first);
    const int s0 = sp * KD, cnt = min(KD, vis.n - s0);
    if (p >= ctx || cnt <= 0) return;                                // uniform: no key of this split is visible yet
    const bool owner = s0 + cnt == vis.n;                            // key cnt - 1 is the new token
    auto key_of = [&](int j) {                                       // j-th key of the split, clamped to one that exists
        const int s = s0 + min(j, cnt - 1);
        return s < vis.keep ? s : vis.lo + s - vis.keep;
    };
    const int sub = lane & 15, grp = wv * 4 + (lane >> 4), pairs = G * KD, items = G * vp / 4;
    const int quarter = tid & 3;                                     // of every 16 keys
    f32x4 kd[PB][NC], vv[4];
    auto load_k = [&](int b) {
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int pr = min(b + 64 * i, pairs - 1), g = pr / KD;
            const float *kr = gk.dst_dev + g * gk.dst_head_stride + (int64_t)key_of(pr - g * KD) * gk.dst_row_stride;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int d = 64 * c + 4 * sub;
                kd[i][c] = d < dp ? *reinterpret_cast<const f32x4 *>(kr + d) : f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    auto load_v = [&](int i, int jb) {                               // i: four columns of a kv head
        const int g = i / (vp / 4);
        const float *vb = gv.dst_dev + g * gv.dst_head_stride + 4 * (i - g * (vp / 4));
#pragma unroll
        for (int j = 0; j < 4; j++) vv[j] = *reinterpret_cast<const f32x4 *>(vb + (int64_t)key_of(jb + 4 * quarter + j) * gv.dst_row_stride);
    };
    // Loads complete in the order they are asked for: first what the preparation needs (two query heads per wave, and for the new token
    // one head of k or v), then the mixing matrix, K and V.
    const int h2 = min(wv + 16, H - 1), xn = min(wv, 2 * G - 1);
    const cq_mix_heads &gn = xn < G ? gk : gv;
    HeadShared<NC> qsh, nsh;
    HeadRegs<NC> qa, qb, nw;
    qsh.load(gq, p, lane);
    qa.load(gq, row + gq.src_off + (int64_t)min(wv, H - 1) * gq.dim, lane);
    if (H > 16) qb.load(gq, row + gq.src_off + (int64_t)h2 * gq.dim, lane);
    if (owner) {
        nsh.load(gn, p, lane);
        nw.load(gn, row + gn.src_off + (int64_t)(xn < G ? xn : xn - G) * gn.dim, lane);
    }
    const float tv = talk[min(tid, H * H - 1)];
    load_k(grp);
    load_v(min(tid >> 2, items - 1), 0);
    qsh.ready(gq, lane);
    auto keep_q = [&](HeadRegs<NC> &x, int h) {
        x.finish(gq, qsh, eps, lane);
#pragma unroll
        for (int e = 0; e < NC; e++)
            if (h < H && lane + 64 * e < dp) qs[h * dp + lane + 64 * e] = x.v[e];
    };
    auto keep_new = [&](HeadRegs<NC> &x, int i) {
        const cq_mix_heads &gr = i < G ? gk : gv;
        const int hh = i < G ? i : i - G;
        float *dst = gr.dst_dev + hh * gr.dst_head_stride + (int64_t)p * gr.dst_row_stride, *own = (i < G ? kn : vn) + hh * gr.dim_pad;
        nsh.ready(gr, lane);
        x.finish(gr, nsh, eps, lane);
#pragma unroll
        for (int e = 0; e < NC; e++)
            if (i < 2 * G && lane + 64 * e < gr.dim_pad) dst[lane + 64 * e] = own[lane + 64 * e] = x.v[e];
    };
    keep_q(qa, wv);
    if (H > 16) keep_q(qb, wv + 16);
    if (owner && wv < 2 * G) keep_new(nw, wv);
    for (int h = wv + 32; h < H; h += 16) {
        qa.load(gq, row + gq.src_off + (int64_t)h * gq.dim, lane);
        keep_q(qa, h);
    }
    if (owner)
        for (int x = wv + 16; x < 2 * G; x += 16) {
            const cq_mix_heads &gr = x < G ? gk : gv;
            nsh.load(gr, p, lane);
            nw.load(gr, row + gr.src_off + (int64_t)(x < G ? x : x - G) * gr.dim, lane);
            keep_new(nw, x);
        }
    if (tid < H * H) T[tid] = tv * scale;
    for (int i = tid + 1024; i < H * H; i += 1024) T[i] = talk[i] * scale;
    __syncthreads();

    // ---- scores ----
    for (int b = grp; b < pairs; b += 64 * PB) {
        if (b != grp) load_k(b);
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int pr = min(b + 64 * i, pairs - 1), g = pr / KD, j = pr - g * KD;
            if (owner && j >= cnt - 1) {
#pragma unroll
                for (int c = 0; c < NC; c++)
                    if (64 * c + 4 * sub < dp) kd[i][c] = *reinterpret_cast<const f32x4 *>(kn + g * dp + 64 * c + 4 * sub);
            }
            for (int r = 0; r < R; r += 4) {                         // four heads side by side (the last one repeated)
                float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    const int d = min(64 * c + 4 * sub, dp - 4);     // where dp ends, kd is zero
#pragma unroll
                    for (int x = 0; x < 4; x++) {
                        const f32x4 qv = *reinterpret_cast<const f32x4 *>(qs + (g * R + min(r + x, R - 1)) * dp + d);
                        a[x] = fmaf(qv.x, kd[i][c].x, a[x]);
                        a[x] = fmaf(qv.y, kd[i][c].y, a[x]);
                        a[x] = fmaf(qv.z, kd[i][c].z, a[x]);
                        a[x] = fmaf(qv.w, kd[i][c].w, a[x]);
                    }
                }
#pragma unroll
                for (int x = 0; x < 4; x++) a[x] = row16_sum(a[x]);
                if (sub < 4 && r + sub < R) sc[(g * R + r + sub) * SS + j] = sub == 0 ? a[0] : (sub == 1 ? a[1] : (sub == 2 ? a[2] : a[3]));
            }
        }
    }
    __syncthreads();
    // ---- mixing ----
    for (int i = tid; i < H * KD; i += 1024) {
        const int h = i / KD, j = i - h * KD;
        const float *t = T + h * H;
        float a0 = 0.0f, a1 = 0.0f;
        int g = 0;
#pragma unroll 2
        for (; g + 8 <= H; g += 8) {
            float tv8[8], sv[8];
#pragma unroll
            for (int x = 0; x < 8; x++) {
                tv8[x] = t[g + x];
                sv[x] = sc[(g + x) * SS + j];
            }
#pragma unroll
            for (int x = 0; x < 8; x += 2) {
                a0 = fmaf(tv8[x], sv[x], a0);
                a1 = fmaf(tv8[x + 1], sv[x + 1], a1);
            }
        }
        for (; g < H; g++) a0 = fmaf(t[g], sc[g * SS + j], a0);
        mx[h * SS + j] = j < cnt ? a0 + a1 : -INFINITY;
    }
    __syncthreads();
    // ---- softmax of the split: 16 lanes per head ----
    const int stride = talk_record(vdim);
    for (int h = grp; h < H; h += 64) {
        float s[KD / 16], m = -INFINITY, l = 0.0f;
#pragma unroll
        for (int i = 0; i < KD / 16; i++) {
            s[i] = mx[h * SS + 16 * i + sub];
            m = fmaxf(m, s[i]);
        }
        m = row16_max(m);
#pragma unroll
        for (int i = 0; i < KD / 16; i++) {
            s[i] = s[i] > -INFINITY ? __expf(s[i] - m) : 0.0f;
            l += s[i];
            sc[h * SS + 16 * i + sub] = s[i];
        }
        l = row16_sum(l);
        if (sub == 0) {
            float *r = rec + ((int64_t)h * splits + sp) * stride + stride - 4;
            r[0] = m;
            r[1] = l;
        }
    }
    __syncthreads();
    // ---- values ----
    const int v4 = (vdim + 3) / 4;
    for (int i = tid >> 2; i < items; i += 256) {
        const int g = i / (vp / 4), e4 = i - g * (vp / 4);
        for (int r = 0; r < R; r += 4) {
            f32x4 a[4];
#pragma unroll
            for (int x = 0; x < 4; x++) a[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int jb = 0; jb < KD; jb += 16) {
                if (i != (tid >> 2) || jb > 0 || (KD > 16 && r > 0)) load_v(i, jb);
                if (owner) {
                    const f32x4 x = *reinterpret_cast<const f32x4 *>(vn + g * vp + 4 * e4);
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (jb + 4 * quarter + j >= cnt - 1) vv[j] = x;
                }
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const f32x4 w = *reinterpret_cast<const f32x4 *>(sc + (g * R + min(r + x, R - 1)) * SS + jb + 4 * quarter);
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) a[x][e] = fmaf(w[j], vv[j][e], a[x][e]);
                }
            }
            // the sum of the four quarters in every lane; lane `quarter` stores head r + quarter
            f32x4 mine = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float s = quad_sum_f(a[x][e]);
                    mine[e] = quarter == x ? s : mine[e];
                }
            if (e4 < v4 && r + quarter < R) *reinterpret_cast<f32x4 *>(rec + ((int64_t)(g * R + r + quarter) * splits + sp) * stride + 4 * e4) = mine;
        }
    }
}

template <int NC, int KD>
int talk_decode_launch(const float *row, const cq_mix_heads *g, float eps, const float *talk, float scale, int window, int keep, const int32_t *pos_dev, int pos,
                       float *rec, int splits, hipStream_t s) {
    const int H = g[0].heads, G = g[1].heads;
    const size_t lds = (size_t)(H * (g[1].dim_pad + 2 * (KD + 4) + H) + G * (g[1].dim_pad + g[2].dim_pad)) * sizeof(float);
    if (lds > 160 * 1024) return CQ_ERR_RANGE;
    if (lds > 64 * 1024) {
        const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(talk_decode_kernel<NC, KD>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                               160 * 1024);
        if (e) return e;
    }
    hipLaunchKernelGGL((talk_decode_kernel<NC, KD>), dim3(splits), dim3(1024), lds, s, row, g[0], g[1], g[2], eps, talk, scale, window, keep, pos_dev, pos, rec,
                       splits);
    return (int)hipGetLastError();
}

int64_t talk_split_bytes(int64_t rows, int64_t H, int64_t vdim) { return rows * H * (vdim + 2) * 4; }
int64_t talk_plan_bytes(const TalkPlan &plan, int64_t rows, int H) { return 2 * plan.workgroups * talk_slot(H) * 4 + (rows + 15) / 16 * 8; }
int64_t talk_workspace_bytes(int64_t rows, int64_t n_head, int64_t vdim, int64_t window, int64_t keep_first, int64_t pos) {
    if (rows <= 0 || n_head <= 0 || vdim <= 0 || window < 1 || keep_first < 0 || pos < 0) return 0;
    const int64_t max_keys = talk_max_keys(window, keep_first, pos + rows), vp = (vdim + 15) / 16 * 16;
    const int nz = talk_key_splits(rows, talk_unit_blocks(n_head, vp), max_keys);
    int64_t bytes = nz > 1 ? talk_split_bytes(rows, n_head, vdim) * nz : 0;
    if (vp == 128 && (n_head == 8 || n_head == 16) && pos + rows <= 0x7fffffff) {
        const TalkPlan plan = talk_tile_plan(rows, std::min<int64_t>(window, 0x7fffffff), std::min<int64_t>(keep_first, 0x7ffffff0), pos, 512);
        if (plan.chunk) bytes = std::max(bytes, talk_plan_bytes(plan, rows, (int)n_head));
    }
    return bytes;
}

template <typename OT>
int talk_attention(const float *q_dev, const float *k_cache_dev, const float *v_cache_dev, const float *talk_dev, float scale, int64_t window,
                   int64_t keep_first, float out_scale, OT *out_dev, int64_t out_stride, int64_t pos, int64_t rows, int64_t n_head,
                   int64_t n_kv_head, int64_t dim_pad, int64_t vdim, int64_t vdim_pad, int64_t ctx, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    if (rows < 0 || pos < 0 || n_head <= 0 || n_kv_head <= 0 || n_head % n_kv_head || dim_pad <= 0 || dim_pad % 16 || vdim <= 0 || 
        vdim_pad != (vdim + 15) / 16 * 16 || ctx <= 0 || window < 1 || keep_first < 0 || out_stride < n_head * vdim)
        return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    if (!q_dev || !k_cache_dev || !v_cache_dev || !talk_dev || !out_dev) return CQ_ERR_NULL;
    if (mix_misaligned(q_dev, 16) || mix_misaligned(k_cache_dev, 16) || mix_misaligned(v_cache_dev, 16)) return CQ_ERR_ALIGN;
    if (pos + rows > ctx || ctx > (1 << 28) || n_head > CQ_MIX_MAX_HEADS || dim_pad > CQ_MIX_MAX_DIM || vdim_pad > CQ_MIX_MAX_DIM) return CQ_ERR_RANGE;
    if (ctx * (dim_pad > vdim_pad ? dim_pad : vdim_pad) * 4 > 0x7fffffffLL) return CQ_ERR_RANGE;      // byte offsets inside a kv head are 32-bit
    const int w = (int)(window < ctx ? window : ctx), keep = (int)(keep_first < ctx ? keep_first : ctx);
    const int H = (int)n_head, G = (int)n_kv_head, R = H / G;
    const bool by_tiles = talk_by_tiles(n_head, n_kv_head, dim_pad, vdim_pad, ctx);
    const int64_t max_keys = talk_max_keys(window, keep_first, pos + rows);
    const int64_t split_bytes = talk_split_bytes(rows, n_head, vdim);
    const int nz = talk_key_splits(rows, talk_unit_blocks(n_head, vdim_pad), max_keys);
    if (nz > 1 && (!workspace_dev || workspace_bytes < nz * split_bytes)) return CQ_ERR_WORKSPACE;
    TalkPlan plan;
    if (by_tiles)                                          // (as many partial results as the workspace holds)
        plan = talk_tile_plan(rows, w, keep, pos, workspace_dev && !mix_misaligned(workspace_dev, 16) ? std::max<int64_t>(0, workspace_bytes - (rows + 15) / 16 * 8) / (talk_slot(H) * 4) : 0);
    hipStream_t s = (hipStream_t)stream;
#define CQ_TA(NW_, NHW_, SH_, U_, VS_, KT_)                                                                                                            \
    talk_launch<NW_, NHW_, SH_, U_, VS_, KT_>(q_dev, k_cache_dev, v_cache_dev, talk_dev, scale, w, keep, out_scale, out_dev, out_stride,      \
                                              (float *)workspace_dev, nz, (int)pos, (int)rows, H, G, (int)dim_pad, (int)vdim, (int)vdim_pad, (int)ctx, s)
    if (by_tiles) {
#define CQ_TT(H_, R_)                                                                                                                                  \
    talk_tile_launch<H_, R_>(q_dev, k_cache_dev, v_cache_dev, talk_dev, scale, w, keep, out_scale, out_dev, out_stride, (float *)workspace_dev, plan, (int)pos, (int)rows, \
                             (int)vdim, (int)ctx, s)
        if (H == 16 && R == 4) return CQ_TT(16, 4);
        if (H == 16 && R == 8) return CQ_TT(16, 8);
        if (H == 8 && R == 2) return CQ_TT(8, 2);
        if (H == 8 && R == 4) return CQ_TT(8, 4);
        if (H == 8 && R == 8) return CQ_TT(8, 8);
#undef CQ_TT
    }
    if (H <= 8) return R % 2 ? CQ_TA(8, 1, true, 2, 1, 32) : CQ_TA(8, 1, true, 2, 2, 32);
    if (H <= 16) return R % 2 ? CQ_TA(16, 1, true, 2, 1, 32) : CQ_TA(16, 1, true, 2, 2, 32);
    if (H <= 32) return R % 2 ? CQ_TA(16, 2, false, 4, 1, 32) : (R % 4 ? CQ_TA(16, 2, true, 4, 2, 32) : CQ_TA(16, 2, true, 4, 4, 32));
    return R % 4 ? CQ_TA(16, 4, false, 4, 1, 16) : CQ_TA(16, 4, true, 4, 4, 16);
#undef CQ_TA
}

}  // namespace

extern "C" {

int64_t cq_mix_talk_attention_workspace_bytes(int64_t rows, int64_t n_head, int64_t vdim, int64_t window, int64_t keep_first, int64_t pos) {
    return talk_workspace_bytes(rows, n_head, vdim, window, keep_first, pos);
}

int cq_mix_talk_attention(const float *q_dev, const float *k_cache_dev, const float *v_cache_dev, const float *talk_dev, float scale, int64_t window,
                          int64_t keep_first, float out_scale, float *out_dev, int64_t out_stride, int64_t pos, int64_t rows, int64_t n_head,
                          int64_t n_kv_head, int64_t dim_pad, int64_t vdim, int64_t vdim_pad, int64_t ctx, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    return talk_attention(q_dev, k_cache_dev, v_cache_dev, talk_dev, scale, window, keep_first, out_scale, out_dev, out_stride, pos, rows, n_head, n_kv_head, dim_pad, vdim,
                          vdim_pad, ctx, workspace_dev, workspace_bytes, stream);
}

int cq_mix_talk_attention_bf16(const float *q_dev, const float *k_cache_dev, const float *v_cache_dev, const float *talk_dev, float scale, int64_t window,
                               int64_t keep_first, float out_scale, void *out_bf16_dev, int64_t out_stride, int64_t pos, int64_t rows, int64_t n_head,
                               int64_t n_kv_head, int64_t dim_pad, int64_t vdim, int64_t vdim_pad, int64_t ctx, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    return talk_attention(q_dev, k_cache_dev, v_cache_dev, talk_dev, scale, window, keep_first, out_scale, (__bf16 *)out_bf16_dev, out_stride, pos, rows, n_head, n_kv_head,
                          dim_pad, vdim, vdim_pad, ctx, workspace_dev, workspace_bytes, stream);
}

int64_t cq_mix_talk_decode_workspace_bytes(int64_t n_head, int64_t vdim, int64_t window, int64_t keep_first, int64_t ctx) {
    if (n_head <= 0 || vdim <= 0 || window < 1 || keep_first < 0 || ctx <= 0) return -1;
    return n_head * talk_splits(talk_max_keys(window, keep_first, ctx)) * talk_record((int)vdim) * 4;
}

int cq_mix_talk_decode(const float *row_dev, const cq_mix_heads *qkv, float eps, const float *talk_dev, float scale, int64_t window, int64_t keep_first,
                       const int32_t *pos_dev, int64_t pos, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    if (!row_dev || !qkv || !talk_dev || !workspace_dev) return CQ_ERR_NULL;
    const cq_mix_heads &q = qkv[0], &k = qkv[1], &v = qkv[2];
    for (int i = 0; i < 3; i++) {
        const int e = mix_check_group(qkv[i], i == 0);
        if (e) return e;
    }
    if (q.heads % k.heads || v.heads != k.heads || q.dim != k.dim || !k.by_position || !v.by_position || k.ctx != v.ctx || k.dim_pad % 16 || v.dim_pad % 16 ||
        window < 1 || keep_first < 0 || pos < 0 || k.dst_row_stride % 4 || k.dst_head_stride % 4 ||
        v.dst_row_stride % 4 || v.dst_head_stride % 4)
        return CQ_ERR_SHAPE;
    if (mix_misaligned(k.dst_dev, 16) || mix_misaligned(v.dst_dev, 16) || mix_misaligned(workspace_dev, 16)) return CQ_ERR_ALIGN;
    if (q.heads > CQ_MIX_MAX_HEADS || k.dim_pad > CQ_MIX_MAX_DIM || v.dim_pad > CQ_MIX_MAX_DIM || k.ctx > (1 << 28) || (!pos_dev && pos >= k.ctx)) return CQ_ERR_RANGE;
    const int64_t n_max = talk_max_keys(window, keep_first, k.ctx);
    if (workspace_bytes < cq_mix_talk_decode_workspace_bytes(q.heads, v.dim, window, keep_first, k.ctx)) return CQ_ERR_WORKSPACE;
    const int w = (int)(window < k.ctx ? window : k.ctx), keep = (int)(keep_first < k.ctx ? keep_first : k.ctx), splits = talk_splits(n_max);
    hipStream_t s = (hipStream_t)stream;
#define CQ_TD(NC_, KD_) talk_decode_launch<NC_, KD_>(row_dev, qkv, eps, talk_dev, scale, w, keep, pos_dev, (int)pos, (float *)workspace_dev, splits, s)
    const bool fine = talk_split_keys(n_max) == 16;
    const int widest = k.dim_pad > v.dim_pad ? k.dim_pad : v.dim_pad;
    if (widest <= 64) return fine ? CQ_TD(1, 16) : CQ_TD(1, 64);
    if (widest <= 128) return fine ? CQ_TD(2, 16) : CQ_TD(2, 64);
    return fine ? CQ_TD(4, 16) : CQ_TD(4, 64);
#undef CQ_TD
}

}  // extern "C"
