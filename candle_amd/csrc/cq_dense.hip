// Matrix products with unquantized bfloat16 weights: MFMA tiles for several activation rows (bf16 or f32 products, f32
// accumulation), plain, batched or grouped by expert; a weight-streaming matvec for one row with the norm / activation of the
// input as prologue and the residual add as epilogue.  Activations and results are f32 in memory, like everywhere in this library
// (the bf16 product rounds them on the way into LDS), or bfloat16 where a caller feeds another bf16 product.
#include "cq_dense.h"

namespace {

__device__ __forceinline__ bf16x8 round_bf16(const f32x4 &a, const f32x4 &b) {
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r[i] = (__bf16)a[i];
        r[4 + i] = (__bf16)b[i];
    }
    return r;
}

// where a tile's results go: the plane of a k split, or dst with the epilogue
struct Out {
    void *dst;
    const float *add;
    int64_t ldd, ld_add;
    float *planes;          // != nullptr: [splits][m][n4]
    int64_t n4;             // n rounded up to 4
    int accumulate, act, bf16;
    const float *row_scale;
    const int32_t *rows;    // row m goes to row rows[m] of dst
    int64_t batch;          // elements of dst per batch
};

// what a tile reads: weights and activations (f32 or bf16), which row of x row m is, and the group of a tile of rows
struct Src {
    const uint16_t *w;
    const void *x;
    int64_t ldw, ldx, w_batch, x_batch;
    const int32_t *rows;
    const cq_dense_tile *tiles;
    const int32_t *n_tiles;
};

__device__ __forceinline__ void put(const Out &o, int64_t at, float v) {
    if (o.bf16) reinterpret_cast<__bf16 *>(o.dst)[at] = (__bf16)v;
    else reinterpret_cast<float *>(o.dst)[at] = v;
}

// Where row m of a product goes and its factor.
struct Row {
    int64_t at;
    float scale;
    bool there;
};
__device__ __forceinline__ Row row_of(const Out &o, int64_t m, int64_t M) {
    const int64_t mm = min(m, M - 1);
    return Row{o.rows ? o.rows[mm] : mm, o.row_scale ? o.row_scale[mm] : 1.0f, m < M};
}

// Four consecutive columns from column n on of f32 values at p, those of them that there are.
__device__ __forceinline__ f32x4 some4(const float *p, int n, int N) {
    if (n + 4 <= N && (reinterpret_cast<uintptr_t>(p) & 15) == 0) return *reinterpret_cast<const f32x4 *>(p);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (n + i < N) v[i] = p[i];
    return v;
}
__device__ __forceinline__ void store4(float *p, const f32x4 &v, int n, int N) {
    if (n + 4 <= N && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
        *reinterpret_cast<f32x4 *>(p) = v;
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (n + i < N) p[i] = v[i];
}

// four consecutive columns n .. n+3 of a row (n % 4 == 0)
__device__ __forceinline__ void emit4(const Out &o, f32x4 v, const Row &row, int n, int N) {
    if (o.act == CQ_DENSE_ACT_SWIGLU) {                    // columns are gate, up, gate, up
        const float a = row.scale * dense_silu(v.x) * v.y, b = row.scale * dense_silu(v.z) * v.w;
        const int64_t at = row.at * o.ldd + (n >> 1);
        put(o, at, a);
        if (n + 3 < N) put(o, at + 1, b);
        return;
    }
    if (o.act == CQ_DENSE_ACT_RELU2) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = fmaxf(v[i], 0.0f) * fmaxf(v[i], 0.0f);
    }
    if (o.row_scale) v *= row.scale;
    if (o.bf16) {
        __bf16 *d = reinterpret_cast<__bf16 *>(o.dst) + row.at * o.ldd + n;
        if (n + 4 <= N && (reinterpret_cast<uintptr_t>(d) & 7) == 0) {
            bf16x4 b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = (__bf16)v[i];
            *reinterpret_cast<bf16x4 *>(d) = b;
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (n + i < N) d[i] = (__bf16)v[i];
        return;
    }
    float *d = reinterpret_cast<float *>(o.dst) + row.at * o.ldd + n;
    if (o.accumulate) v += some4(d, n, N);
    if (o.add) v += some4(o.add + row.at * o.ld_add + n, n, N);
    store4(d, v, n, N);
}

__device__ __forceinline__ uint32_t pair_bf16(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
}
// a, b: of the four groups of sixteen lanes, a0 a1 a2 a3 and b0 b1 b2 b3 -> a0 a1 b0 b1 and a2 a3 b2 b3 (halves), a0 b0 a2 b2 and a1 b1 a3 b3 (rows)
__device__ __forceinline__ void swap_halves(uint32_t &a, uint32_t &b) {
#ifdef __HIP_DEVICE_COMPILE__
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
#endif
}
__device__ __forceinline__ void swap_rows(uint32_t &a, uint32_t &b) {
#ifdef __HIP_DEVICE_COMPILE__
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
#endif
}

// Whether results of columns n .. n + wide - 1 lie on 16 bytes, in f32 without an activation: whole rows of them in one go.
__device__ __forceinline__ bool plain_f32(const Out &o, int n, int wide, int N) {
    return !o.bf16 && o.act == CQ_DENSE_ACT_NONE && n + wide <= N && ((o.ldd | (o.add ? o.ld_add : 0)) & 3) == 0 &&
           ((reinterpret_cast<uintptr_t>(o.dst) | reinterpret_cast<uintptr_t>(o.add)) & 15) == 0;
}
// One row of them: NF times four columns, number f from column(f) on, added to what is there and to the addend.
template <int NF, class At>
__device__ __forceinline__ void sum_f32(const Out &o, const Row &row, f32x4 (&old)[NF], f32x4 (&more)[NF], At column) {
#pragma unroll
    for (int f = 0; f < NF; f++) {
        if (o.accumulate) old[f] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(o.dst) + row.at * o.ldd + column(f));
        if (o.add) more[f] = *reinterpret_cast<const f32x4 *>(o.add + row.at * o.ld_add + column(f));
    }
}
template <int NF, class At, class Of>
__device__ __forceinline__ void store_f32(const Out &o, const Row &row, Of sums, const f32x4 (&old)[NF], const f32x4 (&more)[NF], At column) {
#pragma unroll
    for (int f = 0; f < NF; f++) {
        f32x4 v = sums(f);
        if (o.row_scale) v *= row.scale;
        if (o.accumulate) v += old[f];
        if (o.add) v += more[f];
        *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(o.dst) + row.at * o.ldd + column(f)) = v;
    }
}

// The sums of a wave: of row m(i) of lane % 16 columns nw + 16 j + 4 (lane / 16) .. + 3.  Whatever memory holds beside them (where a row goes, its factor, what the sums are added to) is
// asked for in front of the stores: a load behind a store waits for it, since both are counted in one order, and per four columns that was sixteen round trips a workgroup.
// bfloat16 results change lanes first, so that four lanes write 64 bytes in a row; as two and eight bytes a lane they were as many instructions again.
// Products of 1500 rows on 64 experts of 2048 x 1408, six a row (unevenly loaded), 240 -> 211 us (gate and up) and 138 -> 125 (down); 1500 x 5632 x 2048 with silu 65 -> 58; a prompt
// of 1500 of such a model 1965 -> 1826.
template <int TM, int TN, class At>
__device__ __forceinline__ void put_sums(const Out &o, const f32x4 (&acc)[TM][TN], At m, int nw, int lk, int64_t M, int N, int split) {
    if (o.planes) {                                        // a part of k: nothing to look up (70 to 350 rows of small products lost 1 - 2 % on the way past the questions below)
#pragma unroll
        for (int i = 0; i < TM; i++) {
            float *const at = o.planes + ((int64_t)split * M + m(i)) * o.n4 + nw + 4 * lk;
            if (m(i) < M)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    if (nw + 16 * j + 4 * lk < N) *reinterpret_cast<f32x4 *>(at + 16 * j) = acc[i][j];
        }
        return;
    }
    Row row[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) row[i] = row_of(o, m(i), M);
    auto column = [&](int j) { return nw + 16 * j + 4 * lk; };
    if (plain_f32(o, nw, 16 * TN, N)) {
        f32x4 old[2][TN], more[2][TN];                     // the next row's in front of this one's stores
        if (row[0].there) sum_f32(o, row[0], old[0], more[0], column);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (i + 1 < TM && row[i + 1].there) sum_f32(o, row[i + 1], old[(i + 1) & 1], more[(i + 1) & 1], column);
            if (row[i].there) store_f32(o, row[i], [&](int j) { return acc[i][j]; }, old[i & 1], more[i & 1], column);
        }
        return;
    }
    if constexpr (TN % 2 == 0) {
        if (o.bf16 && nw + 16 * TN <= N && (TN == 4 || o.act != CQ_DENSE_ACT_SWIGLU) && o.ldd % 8 == 0 && (reinterpret_cast<uintptr_t>(o.dst) & 15) == 0) {
            uint16_t *const dst = reinterpret_cast<uint16_t *>(o.dst);
            if constexpr (TN == 4) if (o.act == CQ_DENSE_ACT_SWIGLU) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    uint32_t p[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const f32x4 v = acc[i][j];
                        p[j] = pair_bf16(row[i].scale * dense_silu(v.x) * v.y, row[i].scale * dense_silu(v.z) * v.w);
                    }
                    swap_halves(p[0], p[2]);
                    swap_halves(p[1], p[3]);
                    swap_rows(p[0], p[1]);
                    swap_rows(p[2], p[3]);
                    if (row[i].there) *reinterpret_cast<u32x4 *>(dst + row[i].at * o.ldd + (nw >> 1) + 8 * lk) = u32x4{p[0], p[1], p[2], p[3]};
                }
                return;
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    uint32_t p[2][2];
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        f32x4 v = acc[i][j + u];
                        if (o.act == CQ_DENSE_ACT_RELU2) {
#pragma unroll
                            for (int e = 0; e < 4; e++) v[e] = fmaxf(v[e], 0.0f) * fmaxf(v[e], 0.0f);
                        }
                        if (o.row_scale) v *= row[i].scale;
                        p[u][0] = pair_bf16(v.x, v.y);
                        p[u][1] = pair_bf16(v.z, v.w);
                    }
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        swap_halves(p[0][e], p[1][e]);
                        swap_rows(p[0][e], p[1][e]);
                    }
                    if (row[i].there) *reinterpret_cast<u32x4 *>(dst + row[i].at * o.ldd + nw + 16 * j + 8 * lk) = u32x4{p[0][0], p[0][1], p[1][0], p[1][1]};
                }
            return;
        }
    }
    // Sums off 16 bytes, or in the last columns: the next row's in front of this one's stores here too (1125 x 4114 x 832 added to what is there 33.7 -> 26.6 us, 1103 x 960 x 5824 with rows an
    // odd number of floats apart 42.6 -> 40.6).  (bf16 first: the others are arguments that nobody has asked for yet, and a trip to memory that results in
    // bfloat16 need not wait for: half a microsecond.)
    if (!o.bf16 && (o.accumulate || o.add)) {
        f32x4 old[2][TN], more[2][TN];
        auto ask = [&](int i) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if (!row[i].there || column(j) >= N) continue;
                if (o.accumulate) old[i & 1][j] = some4(reinterpret_cast<const float *>(o.dst) + row[i].at * o.ldd + column(j), column(j), N);
                if (o.add) more[i & 1][j] = some4(o.add + row[i].at * o.ld_add + column(j), column(j), N);
            }
        };
        ask(0);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (i + 1 < TM) ask(i + 1);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if (!row[i].there || column(j) >= N) continue;
                f32x4 v = acc[i][j];
                if (o.row_scale) v *= row[i].scale;
                if (o.accumulate) v += old[i & 1][j];
                if (o.add) v += more[i & 1][j];
                store4(reinterpret_cast<float *>(o.dst) + row[i].at * o.ldd + column(j), v, column(j), N);
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        if (!row[i].there) continue;
#pragma unroll
        for (int j = 0; j < TN; j++)
            if (column(j) < N) emit4(o, acc[i][j], row[i], column(j), N);
    }
}

// Tile t of the order that a run follows: GROUP row tiles wide, column by column, so that the workgroups running side by side on an XCD need
// few distinct rows of either operand (f32 rows are twice the bytes of weight rows: a group narrower than it is long).  GROUP 4 / 6 / 8 / 16 at
// 4096 rows: 705 / 686-732 / 683-702 / 634-663 TFLOP/s, all row tiles first 449-474.
constexpr int TILE_GROUP = 6;
__device__ __forceinline__ void tile_at(int t, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int grp = t / (TILE_GROUP * tiles_n), wide = min(TILE_GROUP, tiles_m - TILE_GROUP * grp), in = t - TILE_GROUP * grp * tiles_n;
    tm = TILE_GROUP * grp + in % wide;
    tn = in / wide;
}

// Tile t of a grouped product's order: all tiles of a group (of those in the same sixteen of the table) side by side, column by column, so that its weights are
// read once, and then the next group.  (By a fixed number of row tiles, as above, tiles of one group fall to two runs of workgroups: 1500 tokens, 64 experts of which the largest have three
// times the mean, 1.05 GB come from behind the L2 for 740 MB of weights, and 0.87 so: 264 -> 247 us.)
__device__ __forceinline__ void group_tile_at(const Src &s, int t, int tiles_m, int tiles_n, int lane, int &tm, int &tn) {
    const int at = t / tiles_n, base = at & ~15, x = base + (lane & 15);
    const int group = s.tiles[at].group;
    const uint32_t same = (uint32_t)__ballot(x < tiles_m && s.tiles[min(x, tiles_m - 1)].group == group) & 0xffffu;
    const int me = at - base, below = __builtin_clz(~(same << (31 - me))) - 1, above = __builtin_ctz(~(same >> me)) - 1;      // of the same group in a row before and after
    const int first = at - below, wide = below + above + 1, in = t - first * tiles_n;
    tm = first + in % wide;
    tn = in / wide;
}

// ---- bf16 tiles: BM activation rows x BN weight rows, k in steps of 64, LDS double-buffered -----------------------------
// The weights are the A operand, so a lane ends with four consecutive output columns of one row.  LDS rows are 128 bytes in
// eight 16-byte chunks, chunk c of row r at c ^ (r / 2) % 8, without bank conflicts; c ^ r % 8, with two lanes to a bank, for the large tile of f32 activations,
// where it is all the same 2 % faster (1500 x 5632 x 2048: 75.7 us against 77.2).
// Three stages are on their way for the large tile of bf16 activations (the cold weights of a model's experts and layers: 1500 tokens of Kudurax 2347 -> 2270 us;
// on warm operands 1500 x 5632 x 2048 66 -> 63), one for the others: f32 activations and small tiles gain nothing from more (40 x 4096 x 4096: 13.3 -> 14.2), and
// workgroups of up to 12 stages (a split of k, short rows) lose by it: the three past the end are brought all the same (700 x 2048 x 2048 in six splits 26.4 us
// with one, 28.1 with three; 4 - 11 stages 4 % slower on average, 13 - 16 none, from 18 on faster).
// Rows go by sixteens to the WGM waves that share the tile's rows.  PARTS: the main loop exists once per number of fragments that a wave then has: rows that are not there are neither brought
// nor multiplied (an expert's last tile: a layer of 64 experts of 2048 x 1408, tiles of 128, 120 / 150 / 220 pairs each 380 465 571 -> 377 448 534 us; a Kudurax prompt of 1500, whose
// experts are loaded unevenly, 1 %, which is what two runs differ by).
// XB: the activations are bfloat16; PF: stages on their way.  With a table of tiles (grouped products) the rows of a tile share the weights of one group.
template <int BM, int BN, int WGM, int WGN, bool XB, int PF = 1, bool PARTS = false>
__global__ __launch_bounds__(256, 2) void dense_bf16_kernel(Src src, Out out, int64_t M, int N, int K, int tiles_m, int tiles_n, int k_split) {
    constexpr int XV = XB ? 1 : 2;                         // 16-byte loads per eight activations
    constexpr int TM = BM / WGM / 16, TN = BN / WGN / 16, CA = BM * 8 / 256, CB = BN * 8 / 256;
    constexpr int SW = BM == 128 && !XB ? 0 : 1;
    __shared__ bf16x8 lds[2][(BM + BN) * 8];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (src.tiles) {
        tiles_m = min(src.n_tiles[0], tiles_m);
        if ((int)blockIdx.x >= tiles_m * tiles_n) return;
    }
    int tm, tn;
    if (src.tiles) group_tile_at(src, xcd_tile(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, lane, tm, tn);
    else tile_at(xcd_tile(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    int64_t m0 = (int64_t)tm * BM;
    const uint16_t *w = src.w + blockIdx.z * src.w_batch;
    if (src.tiles) {
        const cq_dense_tile t = src.tiles[tm];
        m0 = t.first;
        M = t.first + t.rows;
        w += t.group * src.w_batch;
    }
    out.dst = out.bf16 ? (void *)(reinterpret_cast<uint16_t *>(out.dst) + blockIdx.z * out.batch) : (void *)(reinterpret_cast<float *>(out.dst) + blockIdx.z * out.batch);
    const int n0 = tn * BN;
    const int k_lo = blockIdx.y * k_split, k_hi = min(K, k_lo + k_split);
    const int wm = 16 * (wv / WGN), wn = (wv % WGN) * (BN / WGN);       // (sixteen rows to each of the WGM waves by turns)

    const uint8_t *xp[CA];                                 // row starts, in bytes
    const uint16_t *wp[CB];
#pragma unroll
    for (int i = 0; i < CA; i++) {
        const int c = tid + 256 * i;
        int64_t r = min(m0 + (c >> 3), M - 1);
        if (src.rows) r = src.rows[r];
        xp[i] = reinterpret_cast<const uint8_t *>(src.x) + (blockIdx.z * src.x_batch + r * src.ldx + (c & 7) * 8) * (XB ? 2 : 4);
    }
#pragma unroll
    for (int i = 0; i < CB; i++) {
        const int c = tid + 256 * i;
        wp[i] = w + (int64_t)min(n0 + (c >> 3), N - 1) * src.ldw + (c & 7) * 8;
    }
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int lr = lane & 15, lk = lane >> 4;
    auto run = [&](auto live) {                            // of each wave's fragments of sixteen rows the first `live` hold any
        constexpr int LM = decltype(live)::value, LA = CA == TM ? LM : CA;
        u32x4 ra[PF][LA][XV];
        u32x4 rb[PF][CB];
        auto fetch = [&](int k, auto set) {                    // (past the end: the last stage again, for nobody)
            k = min(k, k_hi - 64);
#pragma unroll
            for (int i = 0; i < CB; i++) rb[set][i] = *reinterpret_cast<const u32x4 *>(wp[i] + k);
#pragma unroll
            for (int i = 0; i < LA; i++) {
#pragma unroll
                for (int j = 0; j < XV; j++) ra[set][i][j] = *reinterpret_cast<const u32x4 *>(xp[i] + (int64_t)k * (XB ? 2 : 4) + 16 * j);
            }
        };
        auto stage = [&](int b, auto set) {
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int c = tid + 256 * i, r = c >> 3;
                lds[b][BM * 8 + r * 8 + ((c & 7) ^ ((r >> SW) & 7))] = __builtin_bit_cast(bf16x8, rb[set][i]);
            }
#pragma unroll
            for (int i = 0; i < LA; i++) {
                const int c = tid + 256 * i, r = c >> 3;
                lds[b][r * 8 + ((c & 7) ^ ((r >> SW) & 7))] =
                    XB ? __builtin_bit_cast(bf16x8, ra[set][i][0]) : round_bf16(__builtin_bit_cast(f32x4, ra[set][i][0]), __builtin_bit_cast(f32x4, ra[set][i][XV - 1]));
            }
        };
        constexpr std::integral_constant<int, 0> first{};
        constexpr std::integral_constant<int, PF == 3 ? 1 : 0> second{};
        constexpr std::integral_constant<int, PF == 3 ? 2 : 0> third{};
        fetch(k_lo, first);
        if (PF == 3) {
            fetch(k_lo + 64, second);
            fetch(k_lo + 128, third);
        }
        stage(0, first);
        if (PF > 1) {
            __builtin_amdgcn_s_waitcnt(0xc07f);                // (one that the compiler sees: see dense_ring_kernel)
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else __syncthreads();
        int cur = 0;
        auto step = [&](int k, auto set, auto next) {          // the stage at k, which came through `set`
            const bool more = PF > 1 || k + 64 < k_hi;
            if (more) fetch(k + 64 * PF, set);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                bf16x8 fa[LM], fb[TN];
#pragma unroll
                for (int i = 0; i < LM; i++) {
                    const int r = wm + 16 * WGM * i + lr;
                    fa[i] = lds[cur][r * 8 + ((4 * s + lk) ^ ((r >> SW) & 7))];
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int r = wn + 16 * j + lr;
                    fb[j] = lds[cur][BM * 8 + r * 8 + ((4 * s + lk) ^ ((r >> SW) & 7))];
                }
#pragma unroll
                for (int i = 0; i < LM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
            }
            if (!more) return;
            stage(cur ^ 1, next);
            // (__syncthreads would wait for the stages on their way)
            if (PF > 1) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else __syncthreads();
            cur ^= 1;
        };
        int k = k_lo;
        if constexpr (PF == 3) {                               // (not left in the middle: the compiler would keep its sets in memory)
            for (; k + 128 < k_hi; k += 192) {
                step(k, first, second);
                step(k + 64, second, third);
                step(k + 128, third, first);
            }
            if (k < k_hi) step(k, first, second);
            if (k + 64 < k_hi) step(k + 64, second, third);
        } else {
            for (; k < k_hi; k += 64) step(k, first, second);
        }
    };
    // (the smaller tiles in one form: what two cost is more than what is left out, prompts of 20 to 100 through layers 1024 wide 1.012x - 1.028x slower)
    static_assert(!PARTS || TM == 4, "a form for each number of fragments");
    const int frags = PARTS ? (int)((min(M - m0, (int64_t)BM) + 16 * WGM - 1) / (16 * WGM)) : TM;
    if (!PARTS || frags >= TM) run(std::integral_constant<int, TM>{});
    else if constexpr (PARTS) {
        if (frags == 3) run(std::integral_constant<int, 3>{});
        else if (frags == 2) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 1>{});
    }
    put_sums(out, acc, [&](int i) { return m0 + wm + 16 * WGM * i + lr; }, n0 + wn, lk, M, N, blockIdx.y);
}

// ---- bf16 tiles of 256 activation rows x 256 weight rows, for products that fill the chip with them ------------------------------
// The 128 x 128 tile reads a byte of LDS for every 64 multiply-adds and one of L2 for every 128: both are as slow as the matrix cores at 60 % of their rate.  Here
// eight waves, 2 x 4, of 128 x 64 results each need two thirds and half of that.  LDS holds two stages of 64 of k: weights and bf16 activations go there by
// copies that no register sees, f32 activations through registers, rounded on the way.  One barrier a stage, taken between the third and the last quarter of
// its products: their operands are in registers by then, and those of the next stage's first quarter arrive under them.
// LDS rows are 128 bytes in eight 16-byte chunks, chunk c of row r at c ^ (r / 2) % 8: 16 rows of a chunk lie in all 64 banks (c ^ r % 8 takes twice as long).
// 2048 x 7168 x 2048: bf16 activations 80 -> 59 us (1020 TFLOP/s), f32 90 -> 72; 4096 x 4096 x 4096: 154 -> 113 (1220) and 176 -> 138.  Of the 59 about 11 are
// the way to the first products and the stores; with f32 activations the loads that are to be rounded wait behind those of the stage before.
// The copies are buffer loads: beside copies by address the compiler waits for all LDS reads at once.
constexpr int DT_B = 256, DT_A = DT_B * 128, DT_STAGE = 2 * DT_A;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void dt_lds;

template <bool XB>
__global__ __launch_bounds__(512, 2) void dense_tile_kernel(Src src, Out out, int64_t M, int N, int K, int tiles_m, int tiles_n) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler does not know the buffer accesses)
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    tile_at(xcd_tile(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * DT_B;
    const int n0 = tn * DT_B, nst = K >> 6, wm = (wv >> 2) * 128, wn = (wv & 3) * 64, lr = lane & 31, kg = lane >> 5;

    // ---- instruction i of a wave brings the eight rows 8 (wv + 8 i) .. of a stage, one 16-byte chunk (of bf16) a lane; rows past the end repeat the last ----
    const uint8_t *const xbase = reinterpret_cast<const uint8_t *>(src.x) + m0 * src.ldx * (XB ? 2 : 4);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *)(src.w + (int64_t)n0 * src.ldw), 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void *)xbase, 0, -1, 0x00020000);
    uint32_t w_off[4], x_off[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        w_off[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)(2 * src.ldw) + 16 * c;
        // (f32 activations: chunk lane % 8, swizzled when it is written)
        x_off[i] = (uint32_t)min((int64_t)row, M - 1 - m0) * (uint32_t)((XB ? 2 : 4) * src.ldx) + (XB ? 16 * c : 32 * (lane & 7));
    }
    auto copy = [&](int st) {                              // what goes by copies, of stage st (past the last one: that one again, into a place nobody reads)
        uint8_t *const to = lds + (st & 1) * DT_STAGE + 1024 * wv;
        const int at = 128 * min(st, nst - 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (XB) __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (dt_lds *)(to + 8192 * i), 16, x_off[i], at, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (dt_lds *)(to + DT_A + 8192 * i), 16, w_off[i], at, 0, 0);
        }
        asm volatile("" ::: "memory");
    };
    f32x4 xr[4][2];                                        // f32 activations of the stage after the next
    auto fetch = [&](int st) {
        if constexpr (!XB) {
            const uint8_t *const from = xbase + 256 * min(st, nst - 1);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) xr[i][j] = *reinterpret_cast<const f32x4 *>(from + x_off[i] + 16 * j);
        }
    };
    auto put_x = [&](int st) {
        if constexpr (!XB) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 8 * (wv + 8 * i) + (lane >> 3);
                *reinterpret_cast<bf16x8 *>(lds + (st & 1) * DT_STAGE + row * 128 + 16 * ((lane & 7) ^ ((row >> 1) & 7))) = round_bf16(xr[i][0], xr[i][1]);
            }
        }
    };
    // Barrier b: stage b is there for everybody, and nobody reads stage b - 1 any more: stage b + 1 may take its place.
    auto sync = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto request = [&](int b) {
        put_x(b + 1);
        fetch(b + 2);
        copy(b + 1);
    };
    f32x16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
    const uint32_t a_at = (wm + lr) * 128 + 16 * (kg ^ ((lr >> 1) & 7)), b_at = DT_A + (wn + lr) * 128 + 16 * (kg ^ ((lr >> 1) & 7));
    bf16x8 fa[2][4], fb[2][2];
    auto operands = [&](int st, int s) {                   // of quarter s of the stage, into set s % 2
        const uint8_t *const from = lds + (st & 1) * DT_STAGE;
#pragma unroll
        for (int i = 0; i < 2; i++) fb[s & 1][i] = *reinterpret_cast<const bf16x8 *>(from + ((b_at + 4096 * i) ^ (32 * s)));
#pragma unroll
        for (int i = 0; i < 4; i++) fa[s & 1][i] = *reinterpret_cast<const bf16x8 *>(from + ((a_at + 4096 * i) ^ (32 * s)));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s & 1][j], fa[s & 1][i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch(0);
    copy(0);
    put_x(0);
    fetch(1);
    sync();
    operands(0, 0);
    request(0);
    for (int st = 0; st < nst; st++) {
#pragma unroll
        for (int s = 0; s < 3; s++) {
            operands(st, s + 1);
            multiply(s);
        }
        sync();
        operands(st + 1, 0);
        request(st + 1);
        multiply(3);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (copies may not outlive the workgroup)
    Row row[4];
#pragma unroll
    for (int i = 0; i < 4; i++) row[i] = row_of(out, m0 + wm + 32 * i + lr, M);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (!row[i].there) continue;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int n = n0 + wn + 32 * j + 8 * v + 4 * kg;
                if (n < N) emit4(out, f32x4{acc[i][j][4 * v], acc[i][j][4 * v + 1], acc[i][j][4 * v + 2], acc[i][j][4 * v + 3]}, row[i], n, N);
            }
    }
#endif
}

// ---- bf16 tiles of BM (64, 96, 128, 192) activation rows x 128 weight rows, bfloat16 activations, one workgroup on a unit --------------------------------------
// The 128 x 128 tile above, two workgroups to a unit, wants 512 of them: products of a few hundred tiles are cut along k instead, write their sums to memory and have
// another launch add them, and each workgroup waits for stages that it has asked for one or three of its own short steps ago.  Here one workgroup has a unit's LDS.
// Results are those of that tile to the last bit, so that no choice made from them (of a token's experts, say) depends on which of the two a call takes: the same
// instructions in the order of k, and for a product that would be cut along k (PARTS) one sum per part of k_split, added in order.
// 2048 x 2048 x 2048, cold weights: 39.5 -> 27.2 us, of which about 7 are the way to the first products and the last sums.  A stage takes 0.62 us.  Of a unit's busy cycles
// the matrix cores have 40 % (x 7168), reads of LDS 30, and waves wait for 36 % of theirs: for stages, of which 256 units bring 13.4 TB/s out of the L2s and 2.6 from behind.
// Tiles of 64 and 96 rows, 2 x 4 waves of BM / 2 x 32 results, for products that larger ones leave units without (1500 x 2048 x 2048 in 256 workgroups instead of 192 25.4 -> 23.6 us, 1000 x
// 2048 x 2048 in 256 instead of four parts of 128 22.7 -> 16.3).
// Eight waves, 4 x 2, of BM / 4 x 64 results each: four of BM / 2 x 64 read a third less from LDS, but have a matrix core to themselves and wait more (2048 x 2048 x 2048:
// 31.0 us; 192 rows: 52 where eight take 33).  LDS holds four stages of 64 of k; copies that no register sees bring them, four ahead of the products, and the operands of
// half a stage are read while those of the half before are multiplied: one barrier a stage, which waits for nothing that was asked for less than three stages ago.  Rows
// in LDS as above.
template <int BM, bool PARTS>
__global__ __launch_bounds__(512, 2) void dense_ring_kernel(Src src, Out out, int64_t M, int N, int K, int tiles_m, int tiles_n, int k_split) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler does not know the buffer accesses)
    constexpr int WN = BM < 128 ? 4 : 2, STAGE = (BM + 128) * 128, TM = BM / (128 / WN), TN = 8 / WN, NX = (BM + 63) / 64, NW = 2;      // 16-row blocks of a wave; copies of a wave and stage
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    int tm, tn;
    tile_at(xcd_tile(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * BM;
    const int n0 = tn * 128, nst = K >> 6, part = k_split >> 6, wm = wv / WN * (16 * TM), wn = wv % WN * (16 * TN);
    const bool fewer = BM % 64 && wv >= 4;                 // (the last copy of activations is one of the first four waves')

    // ---- copy i of a wave brings eight rows of a stage, one 16-byte chunk a lane; rows past the end repeat the last ----
    const uint8_t *const xbase = reinterpret_cast<const uint8_t *>(src.x) + m0 * src.ldx * 2;
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *)(src.w + (int64_t)n0 * src.ldw), 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void *)xbase, 0, -1, 0x00020000);
    uint32_t x_off[NX], w_off[NW];
#pragma unroll
    for (int i = 0; i < NX; i++) {
        const int row = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        x_off[i] = (uint32_t)min((int64_t)row, M - 1 - m0) * (uint32_t)(2 * src.ldx) + 16 * c;
    }
#pragma unroll
    for (int i = 0; i < NW; i++) {
        const int row = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        w_off[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)(2 * src.ldw) + 16 * c;
    }
    auto copy = [&](int st) {                              // (past the last stage: that one again, into a place nobody reads)
        uint8_t *const to = lds + (st & 3) * STAGE + 1024 * wv;
        const int at = 128 * min(st, nst - 1);
#pragma unroll
        for (int i = 0; i < NW; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (dt_lds *)(to + BM * 128 + 8192 * i), 16, w_off[i], at, 0, 0);
#pragma unroll
        for (int i = 0; i < NX; i++)
            if (i + 1 < NX || !fewer) __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (dt_lds *)(to + 8192 * i), 16, x_off[i], at, 0, 0);
        asm volatile("" ::: "memory");
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 acc[TM][TN], sum[TM][TN];                        // sum: of the parts before
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = zero;
    bf16x8 fa[2][TM], fb[2][TN];
    const uint32_t sw = (lr >> 1) & 7, a_at = (wm + lr) * 128, b_at = (BM + wn + lr) * 128;
    auto operands = [&](int st, auto half) {
        const uint8_t *const from = lds + (st & 3) * STAGE + 16 * ((4 * half + lk) ^ sw);
#pragma unroll
        for (int j = 0; j < TN; j++) fb[half][j] = *reinterpret_cast<const bf16x8 *>(from + b_at + 2048 * j);
#pragma unroll
        for (int i = 0; i < TM; i++) fa[half][i] = *reinterpret_cast<const bf16x8 *>(from + a_at + 2048 * i);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](auto half) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[half][j], fa[half][i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int PER = NX + NW;
    copy(0);
    copy(1);
    copy(2);
    copy(3);
    if (fewer) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PER - 3) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PER) : "memory");
    asm volatile("s_barrier" ::: "memory");
    constexpr std::integral_constant<int, 0> low{};
    constexpr std::integral_constant<int, 1> high{};
    __builtin_amdgcn_s_waitcnt(0xc07f);                    // scalar loads that only the results want: on their way into the loop they would turn its waits for single operands into waits for all
    operands(0, low);
    int left = part;                                       // stages to the end of the part
    bool first = true;
    for (int st = 0; st < nst; st++) {
        operands(st, high);
        multiply(low);
        // stage st + 1 is there for everybody, and everybody has the operands of stage st: stage st + 4 may take its place
        if (fewer) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * PER - 2) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * PER) : "memory");
        asm volatile("s_barrier" ::: "memory");
        copy(st + 4);
        operands(st + 1, low);
        multiply(high);
        if (PARTS && --left == 0 && st + 1 < nst) {
            left = part;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    sum[i][j] = first ? acc[i][j] : sum[i][j] + acc[i][j];
                    acc[i][j] = zero;
                }
            first = false;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (copies may not outlive the workgroup)
    if (PARTS)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = sum[i][j] + acc[i][j];
    put_sums(out, acc, [&](int i) { return m0 + wm + 16 * i + lr; }, n0 + wn, lk, M, N, 0);
#endif
}

// ---- f32 tiles: 64 x 64, k in steps of 32, weights widened on the way into LDS; a lane's float4 along k feeds four steps of
// v_mfma_f32_16x16x4 (both operands use the same k order) ------------------------------------------------------------------
constexpr int DF_ROW = 36;               // floats per LDS row: 32 + 4, 16 rows of a 16-byte read fall on distinct banks
__global__ __launch_bounds__(256) void dense_f32_kernel(Src src, Out out, int64_t M, int N, int K, int tiles_m, int tiles_n, int k_split) {
    __shared__ float lds[2][128 * DF_ROW];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (src.tiles) {
        tiles_m = min(src.n_tiles[0], tiles_m);
        if ((int)blockIdx.x >= tiles_m * tiles_n) return;
    }
    int tm, tn;
    tile_at(xcd_tile(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    int64_t m0 = (int64_t)tm * 64;
    const uint16_t *w = src.w + blockIdx.z * src.w_batch;
    if (src.tiles) {
        const cq_dense_tile t = src.tiles[tm];
        m0 = t.first;
        M = t.first + t.rows;
        w += t.group * src.w_batch;
    }
    out.dst = out.bf16 ? (void *)(reinterpret_cast<uint16_t *>(out.dst) + blockIdx.z * out.batch) : (void *)(reinterpret_cast<float *>(out.dst) + blockIdx.z * out.batch);
    const int n0 = tn * 64;
    const int k_lo = blockIdx.y * k_split, k_hi = min(K, k_lo + k_split);
    const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;
    f32x4 ra[2];
    u32x4 rb;
    const float *xp[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int c = tid + 256 * i;
        int64_t r = min(m0 + (c >> 3), M - 1);
        if (src.rows) r = src.rows[r];
        xp[i] = reinterpret_cast<const float *>(src.x) + blockIdx.z * src.x_batch + r * src.ldx + (c & 7) * 4;
    }
    const uint16_t *wp = w + (int64_t)min(n0 + (tid >> 2), N - 1) * src.ldw + (tid & 3) * 8;
    auto fetch = [&](int k) {
        rb = *reinterpret_cast<const u32x4 *>(wp + k);
#pragma unroll
        for (int i = 0; i < 2; i++) ra[i] = *reinterpret_cast<const f32x4 *>(xp[i] + k);
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int c = tid + 256 * i;
            *reinterpret_cast<f32x4 *>(&lds[b][(c >> 3) * DF_ROW + (c & 7) * 4]) = ra[i];
        }
        float *d = &lds[b][(64 + (tid >> 2)) * DF_ROW + (tid & 3) * 8];
        *reinterpret_cast<f32x4 *>(d) = f32x4{bf_lo(rb.x), bf_hi(rb.x), bf_lo(rb.y), bf_hi(rb.y)};
        *reinterpret_cast<f32x4 *>(d + 4) = f32x4{bf_lo(rb.z), bf_hi(rb.z), bf_lo(rb.w), bf_hi(rb.w)};
    };
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(k_lo);
    stage(0);
    __syncthreads();
    int cur = 0;
    const int lr = lane & 15, lk = lane >> 4;
    for (int k = k_lo; k < k_hi; k += 32) {
        const bool more = k + 32 < k_hi;
        if (more) fetch(k + 32);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            f32x4 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                fa[i] = *reinterpret_cast<const f32x4 *>(&lds[cur][(wm + 16 * i + lr) * DF_ROW + 16 * s + 4 * lk]);
                fb[i] = *reinterpret_cast<const f32x4 *>(&lds[cur][(64 + wn + 16 * i + lr) * DF_ROW + 16 * s + 4 * lk]);
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][e], fa[i][e], acc[i][j], 0, 0, 0);
        }
        if (more) {
            stage(cur ^ 1);
            __syncthreads();
            cur ^= 1;
        }
    }
    put_sums(out, acc, [&](int i) { return m0 + wm + 16 * i + lr; }, n0 + wn, lk, M, N, blockIdx.y);
}

// the planes of a k split, added in order
__global__ __launch_bounds__(256) void dense_planes_kernel(Out out, int64_t M, int N, int splits) {
    const int64_t groups = out.n4 >> 2;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= M * groups) return;
    const int64_t m = i / groups;
    const int n = (int)(i - m * groups) * 4;
    f32x4 v = *reinterpret_cast<const f32x4 *>(out.planes + m * out.n4 + n);
    for (int s = 1; s < splits; s++) v += *reinterpret_cast<const f32x4 *>(out.planes + ((int64_t)s * M + m) * out.n4 + n);
    emit4(out, v, row_of(out, m, M), n, N);
}

struct Plan {
    int bm, bn, tiles_m, tiles_n, splits, k_split;
};

Plan plan(int precision, int64_t m, int64_t n, int64_t k) {
    Plan p;
    auto tiles = [&](int bm, int bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    if (precision == CQ_DENSE_F32) {
        p.bm = p.bn = 64;
    } else if (m > 64 && tiles(128, 128) * (k / 512) >= 256) {      // the large tile where splitting k can still fill the chip
        p.bm = p.bn = 128;
    } else if (m > 32) {
        p.bm = p.bn = 64;
    } else {
        p.bm = 32;
        p.bn = 64;
    }
    p.tiles_m = (int)((m + p.bm - 1) / p.bm);
    p.tiles_n = (int)((n + p.bn - 1) / p.bn);
    // enough workgroups for two per CU, each with at least 256 of k
    const int64_t t = (int64_t)p.tiles_m * p.tiles_n;
    int64_t s = t >= 384 ? 1 : (512 + t - 1) / t;
    s = s < k / 256 ? s : k / 256;
    s = s < 1 ? 1 : (s > 16 ? 16 : s);
    p.k_split = (int)((k / 64 + s - 1) / s) * 64;
    p.splits = (int)((k + p.k_split - 1) / p.k_split);
    return p;
}

// Where the 256 x 256 tile takes the place of the 128 x 128 one: from 1024 of k on (1500 x 8192 x 512: 30.1 us against 28.6), where one round of workgroups
// fills five eighths of the chip (1500 x 7168 x 2048, 168 tiles: 52 against 65) or several fill three quarters (4096 x 7168 x 2048, 448 tiles: 114 against
// 142; 2048 x 10368 x 2048 of f32, 328 tiles: 136 against 131).
bool large_tile(int64_t m, int64_t n, int64_t k, int64_t ldw, int64_t ldx) {
    if (k < 1024 || ldw > (1 << 20) || ldx > (1 << 20)) return false;      // (its offsets have 32 bits: 256 rows of up to 4-byte elements)
    const int64_t t = ((m + DT_B - 1) / DT_B) * ((n + DT_B - 1) / DT_B), rounds = (t + 255) / 256;
    return rounds == 1 ? t >= 160 : 4 * t >= 3 * 256 * rounds;
}

// Where one workgroup to a unit with a ring of stages (64, 96, 128 or 192 rows; 0: none of them) takes the place of two workgroups of 128 x 128 (products of bfloat16 rows; the large
// tile first where it would take the call).  At k = 2048, cold weights, one round of 256 tiles takes 23 - 27 us with 128 rows and 32 - 34 with 192; 512 tiles two to a
// unit take 49 - 53, and fewer tiles 26 - 54 in parts of k and their sum.
//   up to 256 tiles of 128 in up to three parts (2048 x 2048 x 2048: 39.5 -> 27.2 us, 1500 x 2048 x 7168: 86.5 -> 69.3), or four of a short k (1200 x 2048 x 2048: 37.4 ->
//     24.5, 1000 x 2304 x 3072: 45.4 -> 33.9; 128 tiles in four parts just fill the chip, 1000 x 2048 x 2304: 28.2 -> 27.1, x 2560: 30.1 against 31.4, x 7168: 54.1
//     against 66.3); more parts bring more workgroups to a long k (700 x 2048 x 7168: 53.2 against 60.4);
//   one round of 192 where 128 takes two (1500 x 3500 x 2048: 53.5 -> 34.2), else two rounds of 128 up to 384 tiles (1000 x 5632 x 2048: 57.2 -> 49.1; 448: 51.1 against 51.3);
//   beyond one round of two to a unit, rounds of 192 that are two thirds full (1200 x 7168 x 2048: 68.4 -> 63.8, 2048 x 10368 x 2048: 130.5 -> 122.9).
//   64 rows where they are one round, of a k that is no longer than their number pays for, since each brings its 128 weight rows of all of k by itself where parts of k share that: 350 .. 1000 x
//     2048 x 2048 21 - 29 -> 15 - 16, 850 x 2048 x 7168 55.5 -> 39.  220 drawn products of up to 128 tiles, time with 64 rows by the time in parts: up to 112 tiles and k of 2816 0.80, of 3072 to
//     4096 0.95 on average and up to 1.17 (241 x 3200 x 3776 24.2 against 28.4); 113 - 128 tiles 0.86 up to k of 4096; 129 - 136 tiles 0.85 up to 4992, 1.08 - 1.09 beyond (1084 x 960 x 6272 38.4
//     against 42); more 0.79.  Else 96 (1500 x 2048 x 2048: 25.4 -> 23.6, x 7168 65.5 -> 57.6, 1200 x 2048 x 7168 68.3 -> 52).  Silu results want waves of four columns of 16 (small).
int ring_rows(const Plan &p, int64_t m, int64_t n, int64_t k, int64_t ldw, int64_t ldx, bool small) {
    if (p.bm != 128 || ldw > (1 << 20) || ldx > (1 << 20)) return 0;       // (its offsets have 32 bits)
    const int64_t t64 = (m + 63) / 64 * p.tiles_n, t96 = (m + 95) / 96 * p.tiles_n, t128 = (int64_t)p.tiles_m * p.tiles_n, t192 = (m + 191) / 192 * p.tiles_n, rounds = (t192 + 255) / 256;
    if (p.splits == 1 && large_tile(m, n, k, ldw, ldx)) return 0;
    if (t64 <= 256 && small && (t64 > 136 || k <= (t64 > 128 ? 4992 : t64 > 112 ? 4096 : 2816))) return 64;
    if (t96 <= 256 && t64 > 256 && small) return 96;
    if (t128 <= 256) return p.splits <= 3 || (p.splits == 4 && k <= (t128 > 128 ? 3072 : 2304)) ? 128 : 0;
    if (t192 <= 256) return 192;
    if (t128 <= 384) return 128;
    return t128 > 512 && 3 * t192 >= 2 * 256 * rounds ? 192 : 0;
}

// ---- one row --------------------------------------------------------------------------------------------------------------
// 8 waves; a wave takes one weight row at a time and walks it in blocks of 64 lanes x 8 elements x 4, one block ahead; the first
// block is requested before the prologue.  Weights are read once per step: non-temporal loads (33.3 -> 27.1 us on 4096 x 14336).  At most two
// workgroups per CU, which then walk the rows together.  The input row sits in LDS as f32, zero beyond `dim` and up to a whole block.
constexpr int MV_U = 4, MV_BLOCK = 512 * MV_U;
template <int PRO>
__global__ __launch_bounds__(512) void dense_matvec_kernel(const uint16_t *__restrict__ w, int64_t ldw, const float *__restrict__ x,
                                                           const float *__restrict__ vec, float eps, int dim, float *dst, const float *add, int accumulate,
                                                           int n, int k) {
    constexpr int U = MV_U, BLOCK = MV_BLOCK;
    extern __shared__ __attribute__((aligned(16))) float xs[];           // k rounded up to BLOCK
    __shared__ float red[8];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int step = gridDim.x * 8, kb_n = (k + BLOCK - 1) / BLOCK;
    int r = blockIdx.x * 8 + wv;
    u32x4 cur[U], nxt[U];
    auto load = [&](int row, int kb, u32x4 (&d)[U]) {
        const uint16_t *p = w + (int64_t)row * ldw;
#pragma unroll
        for (int u = 0; u < U; u++) d[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p + min(kb * BLOCK + u * 512 + lane * 8, k - 8)));
    };
    if (r < n) load(r, 0, cur);

    // the input row into LDS, several 16-byte loads per thread in flight (it comes from another kernel's hands, far away)
    constexpr int PF = PRO == CQ_DENSE_POLY || PRO == CQ_DENSE_RELU2 ? 8 : 4;
    const int n4 = kb_n * BLOCK / 4;
    f32x4 *xs4 = reinterpret_cast<f32x4 *>(xs);
    float s2 = 0.0f, s4 = 0.0f, s6 = 0.0f;
    for (int i0 = tid; i0 < n4; i0 += 512 * PF) {
        f32x4 v[PF];
#pragma unroll
        for (int j = 0; j < PF; j++) v[j] = *reinterpret_cast<const f32x4 *>(x + min(4 * (i0 + 512 * j), k - 4));
#pragma unroll
        for (int j = 0; j < PF; j++) {
            const int i = i0 + 512 * j;
            if (i >= n4) break;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float z = 4 * i + e < dim ? v[j][e] : 0.0f, q = z * z;
                v[j][e] = PRO == CQ_DENSE_RELU2 ? (z > 0.0f ? q : 0.0f) : z;
                if (PRO == CQ_DENSE_LAYER_NORM) s2 += z;
                else if (PRO != CQ_DENSE_PLAIN) s2 += q;
                if (PRO == CQ_DENSE_POLY) {
                    s4 = fmaf(q, q, s4);
                    s6 = fmaf(q * q, q, s6);
                }
            }
            xs4[i] = v[j];
        }
    }
    if (PRO == CQ_DENSE_NORM) {
        const float m = sqrtf(block_sum_512(s2, red) / (float)dim + eps);
        for (int i = tid; i < dim; i += 512) xs[i] = xs[i] / m * vec[i];
    } else if (PRO == CQ_DENSE_LAYER_NORM) {
        layer_norm_lds_512(xs, dim, s2, vec, eps, red);
    } else if (PRO == CQ_DENSE_POLY) {
        const float inv = 1.0f / (float)dim;
        const float i1 = vec[0] / sqrtf(block_sum_512(s2, red) * inv + eps);
        const float i2 = vec[1] / sqrtf(block_sum_512(s4, red) * inv + eps);
        const float i3 = vec[2] / sqrtf(block_sum_512(s6, red) * inv + eps);
        const float e = vec[3];
        for (int i = tid; i < n4; i += 512) {
            f32x4 v = xs4[i];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float q = v[j] * v[j];
                v[j] = 4 * i + j < dim ? fmaf(i1, v[j], fmaf(i2, q, fmaf(i3, q * v[j], e))) : 0.0f;
            }
            xs4[i] = v;
        }
    }
    __syncthreads();

    for (; r < n; r += step) {
        float acc[2] = {0.0f, 0.0f};
        for (int kb = 0; kb < kb_n; kb++) {
            const bool last = kb + 1 == kb_n;
            const int next = last ? r + step : r;
            if (next < n) load(next, last ? 0 : kb + 1, nxt);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const f32x4 *xv = reinterpret_cast<const f32x4 *>(xs + kb * BLOCK + u * 512 + lane * 8);
                const f32x4 a = xv[0], b = xv[1];
                dot8(cur[u], a, b, acc);
            }
#pragma unroll
            for (int u = 0; u < U; u++) cur[u] = nxt[u];
        }
        const float s = wave_sum(acc[0] + acc[1]);
        if (lane == 0) dst[r] = s + (accumulate ? dst[r] : 0.0f) + (add ? add[r] : 0.0f);
    }
}

// Whether tiles of 128 rows have a form for each number of fragments (dense_bf16_kernel, PARTS).  Not where all of them are full, which lose 0.5 - 1 % by the longer code and eight
// registers more (119 x 13184 x 4096 of bf16 rows 42 -> 46 us), nor where row tiles are many: the one that ends early saves little then, and no longer reads an operand when its neighbours do.
// 2900 drawn products, last tile part-filled, forms for each against one: up to 6 row tiles, 10 of more than 12 stages, 0.967 of the time on average (two of them 0.957), more 1.000 and now and then
// 1.05 - 1.11 (2241 x 3048 x 4736 of f32 rows 95 -> 106 us, 2329 x 676 x 6400 of bf16 rows 49 -> 53).  A few of the former lose as well (135 x 8272 x 7168 58 -> 62).
bool part_tiles(const cq_dense_args &a, int64_t m, const Plan &p) { return a.tiles_dev || (p.tiles_m <= (p.k_split > 12 * 64 ? 10 : 6) && (m - 1) % 128 < 96); }

template <int PRO>
int matvec_launch(const uint16_t *w, int64_t ldw, const float *x, const float *vec, float eps, int dim, float *dst, const float *add, int accumulate, int n,
                  int k, hipStream_t s) {
    const size_t lds = (size_t)((k + MV_BLOCK - 1) / MV_BLOCK) * MV_BLOCK * sizeof(float);
    const int blocks = (n + 7) / 8 < 512 ? (n + 7) / 8 : 512;
    if (lds > 64 * 1024) {
        const int e = (int)hipFuncSetAttribute(reinterpret_cast<const void *>(dense_matvec_kernel<PRO>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 64);
        if (e) return e;
    }
    hipLaunchKernelGGL(dense_matvec_kernel<PRO>, dim3(blocks), dim3(512), lds, s, w, ldw, x, vec, eps, dim, dst, add, accumulate, n, k);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" {

int64_t cq_dense_matmul_workspace_bytes(int precision, int64_t m, int64_t n, int64_t k) {
    if (m <= 0 || n <= 0 || k <= 0 || k % 64) return 0;
    const Plan p = plan(precision, m, n, k);
    return p.splits > 1 ? (int64_t)p.splits * m * ((n + 3) / 4 * 4) * 4 : 0;
}

int cq_dense_product(int precision, const cq_dense_args *args, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    if (!args) return CQ_ERR_NULL;
    const cq_dense_args &a = *args;
    if (precision != CQ_DENSE_BF16 && precision != CQ_DENSE_F32) return CQ_ERR_DTYPE;
    if (precision == CQ_DENSE_F32 && (a.x_bf16 || a.dst_bf16)) return CQ_ERR_DTYPE;
    if (a.act < CQ_DENSE_ACT_NONE || a.act > CQ_DENSE_ACT_SWIGLU) return CQ_ERR_DTYPE;
    const int64_t m = a.m, n = a.n, k = a.k, cols = a.act == CQ_DENSE_ACT_SWIGLU ? n / 2 : n;
    if (m < 0 || n < 0 || k <= 0 || k % 64 || a.ldw % 64 || a.ldw < k || a.ldx % (a.x_bf16 ? 8 : 4) || a.ldx < k || a.ldd < cols || (a.add_dev && a.ld_add < cols) ||
        a.batch < 1)
        return CQ_ERR_SHAPE;
    if ((a.act == CQ_DENSE_ACT_SWIGLU && n % 2) || ((a.act || a.dst_bf16) && (a.accumulate || a.add_dev))) return CQ_ERR_SHAPE;
    if (a.batch > 1 && (a.accumulate || a.add_dev || a.row_scale_dev || a.tiles_dev || a.w_batch % 8 || a.x_batch % (a.x_bf16 ? 8 : 4))) return CQ_ERR_SHAPE;
    if (a.tiles_dev && (a.max_tiles < 1 || a.accumulate || a.add_dev || a.w_batch % 8 || (a.tile_rows != 32 && a.tile_rows != 64 && a.tile_rows != 128) ||
                        (precision == CQ_DENSE_F32 && a.tile_rows != 64)))
        return CQ_ERR_SHAPE;
    if (m == 0 || n == 0) return CQ_OK;
    if (!a.w_dev || !a.x_dev || !a.dst_dev || (a.tiles_dev && !a.n_tiles_dev)) return CQ_ERR_NULL;
    if (misaligned(a.w_dev, 16) || misaligned(a.x_dev, 16) || misaligned(a.dst_dev, a.dst_bf16 ? 2 : 4) || misaligned(a.add_dev, 4) || misaligned(workspace_dev, 16) ||
        misaligned(a.row_scale_dev, 4))
        return CQ_ERR_ALIGN;
    if (m > (1 << 24) || n > (1 << 24) || k > (1 << 24) || a.batch > 65535) return CQ_ERR_RANGE;
    Plan p = plan(precision, m, n, k);
    if (a.batch > 1 || a.tiles_dev) {
        if (a.tiles_dev) {
            p.bm = (int)a.tile_rows;
            p.bn = p.bm == 128 ? 128 : 64;
            p.tiles_m = (int)a.max_tiles;
        }
        p.tiles_n = (int)((n + p.bn - 1) / p.bn);
        p.splits = 1;
        p.k_split = (int)k;
    }
    if ((int64_t)p.tiles_m * p.tiles_n > 0x7fffffffLL) return CQ_ERR_RANGE;
    if (p.splits > 1 && (!workspace_dev || workspace_bytes < cq_dense_matmul_workspace_bytes(precision, m, n, k))) return CQ_ERR_WORKSPACE;
    Out o;
    o.dst = a.dst_dev;
    o.add = a.add_dev;
    o.ldd = a.ldd;
    o.ld_add = a.ld_add;
    o.accumulate = a.accumulate;
    o.planes = p.splits > 1 ? (float *)workspace_dev : nullptr;
    o.n4 = (n + 3) / 4 * 4;
    o.act = a.act;
    o.bf16 = a.dst_bf16;
    o.row_scale = a.row_scale_dev;
    o.rows = a.dst_rows_dev;
    o.batch = a.batch > 1 ? a.dst_batch : 0;
    Src src;
    src.w = (const uint16_t *)a.w_dev;
    src.x = a.x_dev;
    src.ldw = a.ldw;
    src.ldx = a.ldx;
    src.w_batch = a.w_batch;
    src.x_batch = a.x_batch;
    src.rows = a.src_rows_dev;
    src.tiles = a.tiles_dev;
    src.n_tiles = a.n_tiles_dev;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.splits, (unsigned)a.batch);
#define CQ_DM(K_) hipLaunchKernelGGL(K_, grid, dim3(256), 0, s, src, o, m, (int)n, (int)k, p.tiles_m, p.tiles_n, p.k_split)
    const int ring = a.x_bf16 && a.batch == 1 && !a.tiles_dev && !a.src_rows_dev ? ring_rows(p, m, n, k, a.ldw, a.ldx, a.act != CQ_DENSE_ACT_SWIGLU) : 0;
    if (ring) {
        o.planes = nullptr;
        auto *const fn = ring == 192 ? (p.splits > 1 ? dense_ring_kernel<192, true> : dense_ring_kernel<192, false>)
                         : ring == 64 ? (p.splits > 1 ? dense_ring_kernel<64, true> : dense_ring_kernel<64, false>)
                         : ring == 96 ? (p.splits > 1 ? dense_ring_kernel<96, true> : dense_ring_kernel<96, false>)
                                     : (p.splits > 1 ? dense_ring_kernel<128, true> : dense_ring_kernel<128, false>);
        const int lds = 4 * (ring + 128) * 128;
        const hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
        const int tm = (int)((m + ring - 1) / ring), tn = (int)((n + 127) / 128);
        hipLaunchKernelGGL(fn, dim3((unsigned)(tm * tn)), dim3(512), lds, s, src, o, m, (int)n, (int)k, tm, tn, p.k_split);
        return (int)hipGetLastError();
    }
    if (precision == CQ_DENSE_F32) CQ_DM(dense_f32_kernel);
    else if (p.bm == 128 && p.splits == 1 && a.batch == 1 && !a.tiles_dev && !a.src_rows_dev && large_tile(m, n, k, a.ldw, a.ldx)) {
        auto *const fn = a.x_bf16 ? dense_tile_kernel<true> : dense_tile_kernel<false>;
        const hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * DT_STAGE);
        if (e != hipSuccess) return (int)e;
        const int tm = (int)((m + DT_B - 1) / DT_B), tn = (int)((n + DT_B - 1) / DT_B);
        hipLaunchKernelGGL(fn, dim3((unsigned)(tm * tn)), dim3(512), 2 * DT_STAGE, s, src, o, m, (int)n, (int)k, tm, tn);
    }
    else if (p.bm == 128) {
        const bool deep = p.k_split > 12 * 64;
        auto *const fn = !a.x_bf16 ? (part_tiles(a, m, p) ? dense_bf16_kernel<128, 128, 2, 2, false, 1, true> : dense_bf16_kernel<128, 128, 2, 2, false, 1, false>)
                         : deep    ? (part_tiles(a, m, p) ? dense_bf16_kernel<128, 128, 2, 2, true, 3, true> : dense_bf16_kernel<128, 128, 2, 2, true, 3, false>)
                                   : (part_tiles(a, m, p) ? dense_bf16_kernel<128, 128, 2, 2, true, 1, true> : dense_bf16_kernel<128, 128, 2, 2, true, 1, false>);
        CQ_DM(fn);
    }
    else if (p.bm == 64 && a.x_bf16) CQ_DM((dense_bf16_kernel<64, 64, 2, 2, true>));
    else if (p.bm == 64) CQ_DM((dense_bf16_kernel<64, 64, 2, 2, false>));
    else if (a.x_bf16) CQ_DM((dense_bf16_kernel<32, 64, 1, 4, true>));
    else CQ_DM((dense_bf16_kernel<32, 64, 1, 4, false>));
#undef CQ_DM
    if (p.splits > 1)
        hipLaunchKernelGGL(dense_planes_kernel, dim3((unsigned)((m * (o.n4 / 4) + 255) / 256)), dim3(256), 0, s, o, m, (int)n, p.splits);
    return (int)hipGetLastError();
}

int cq_dense_matmul(int precision, const void *w_dev, int64_t ldw, const float *x_dev, int64_t ldx, float *dst_dev, int64_t ldd, const float *add_dev,
                    int64_t ld_add, int accumulate, int64_t m, int64_t n, int64_t k, void *workspace_dev, int64_t workspace_bytes, void *stream) {
    cq_dense_args a = {};
    a.w_dev = w_dev;
    a.ldw = ldw;
    a.x_dev = x_dev;
    a.ldx = ldx;
    a.dst_dev = dst_dev;
    a.ldd = ldd;
    a.add_dev = add_dev;
    a.ld_add = ld_add;
    a.accumulate = accumulate;
    a.m = m;
    a.n = n;
    a.k = k;
    a.batch = 1;
    return cq_dense_product(precision, &a, workspace_dev, workspace_bytes, stream);
}

int cq_dense_matvec(const void *w_dev, int64_t ldw, const float *x_dev, int prologue, const float *vec_dev, float eps, int64_t dim, float *dst_dev,
                    const float *add_dev, int accumulate, int64_t n, int64_t k, void *stream) {
    if (n < 0 || k <= 0 || k % 64 || ldw % 64 || ldw < k || dim <= 0 || dim > k) return CQ_ERR_SHAPE;
    if (prologue < CQ_DENSE_PLAIN || prologue > CQ_DENSE_RELU2) return CQ_ERR_DTYPE;
    if (n == 0) return CQ_OK;
    if (!w_dev || !x_dev || !dst_dev || (prologue != CQ_DENSE_PLAIN && prologue != CQ_DENSE_RELU2 && !vec_dev)) return CQ_ERR_NULL;
    if (misaligned(w_dev, 16) || misaligned(x_dev, 16) || misaligned(vec_dev, 4) || misaligned(dst_dev, 4) || misaligned(add_dev, 4)) return CQ_ERR_ALIGN;
    if (k > CQ_DENSE_MATVEC_MAX_K || n > (1 << 24)) return CQ_ERR_RANGE;
    const uint16_t *w = (const uint16_t *)w_dev;
    hipStream_t s = (hipStream_t)stream;
#define CQ_MV(P_) case P_: return matvec_launch<P_>(w, ldw, x_dev, vec_dev, eps, (int)dim, dst_dev, add_dev, accumulate, (int)n, (int)k, s)
    switch (prologue) {
        CQ_MV(CQ_DENSE_NORM);
        CQ_MV(CQ_DENSE_POLY);
        CQ_MV(CQ_DENSE_LAYER_NORM);
        CQ_MV(CQ_DENSE_RELU2);
        default: return matvec_launch<CQ_DENSE_PLAIN>(w, ldw, x_dev, vec_dev, eps, (int)dim, dst_dev, add_dev, accumulate, (int)n, (int)k, s);
    }
#undef CQ_MV
}

}  // extern "C"
