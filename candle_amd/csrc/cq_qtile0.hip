// Prefill matmul of Q4_0 and Q8_0 over pre-quantized activations (Q8_0 blocks) on the int8 matrix cores of gfx950:
//   dst[m, n] = sum over blocks b of (sum of 32 q8[m, k] * q[n, k]) * d[n, b] * d8[m, b]
//
// Both operands carry a scale per 32 elements, so one v_mfma_i32_32x32x32_i8 is one block of 32 x 32 results, each of which the vector units scale and
// add: they are the bound (two instructions per result and block, against one matrix instruction per 1024).  The usual three are convert, times d[n], fma with
// d8[m].  Here the sums start from 0x4b400000 instead of zero: read as f32 that is F = 12582912 + S exactly (|S| < 2^22), and
// fma(F, d, -12582912 d) rounds S * d once, like the product of the converted sum: 12582912 = 3 * 2^22 and d has 11 bits, so the offset is exact.  The
// results are those of the CPU's order of operations (k_quants.rs:294-311, 720-738).
//
// A workgroup's eight waves lie side by side along n and share 32 MI rows of activations in LDS (two super-blocks of 256, swizzled so that fragments are read
// without bank conflicts); a wave owns 32 weight rows, brings their blocks for itself by copies to LDS, half a super-block at a time, and converts each
// weight once for 32 MI rows.  The products of the next tile run on the matrix cores while those of one are scaled.  WF: the weights are the matrix instructions' first
// operand, so that a lane has sixteen weight rows' results of one activation row: the sixteen scales of the weights, put into LDS as f32 by the wave itself, are read once per
// block for all tiles and one scale of the activations per tile.  (The other way round four reads of 16 bytes per tile and block bring the activations' scales, right in front of
// their use, but a weight row's scale comes with its weights: the better way for some tiles of 32 rows, see launch_mi.)  Results then go out four columns at a time, whatever n
// is a multiple of.  K is split over grid.z where that fills the chip better; see qtile_plan.
//
// The main loop exists for each number of 32-row tiles that hold rows, which makes that known where registers are given out.  The product that follows a tile's goes into the registers of the
// sums that have just been scaled, a block ahead; or (TWO) only the sums of two tiles are there at a time, those of the one that is scaled and of the next: 16 registers a tile less, so that Q4_0
// has tiles of 160 rows, whose weights are converted once where two tiles of 96 did it twice and left a sixth of the work to one of them (131 rows of [13824 x 5120] 59.5 -> 51.6 us with f16
// results), and faster for two tiles of Q8_0 (700 rows of [11008 x 4096] 138 -> 133, a block ahead 136), slower for the others.  us, one loop for any number of tiles / two tiles' sums / now:
//   Q4_0   2048 rows of [14336 x 4096] in tiles of 128 388 387 364   512 of [4096 x 14336] 105.9 103.7 99.6   700 of [11008 x 4096] in tiles of 64 128.3 130.6 129.4
//   Q8_0   2048 rows of [14336 x 4096]                 409 396 393   512 of [4096 x 14336] 110.4 107.5 106.6
// 600 drawn calls, time by that of the one loop, two tiles' sums / now: Q4_0 in tiles of 64 1.013 1.004, of 96 0.993 0.962, of 128 1.004 0.958; Q8_0 0.973 0.973, 0.985 0.979, 0.976 0.965.
//
// us on one card, the activations first in all tiles / the weights first from 64 rows on, quantizing the activations included:      17 rows   131 rows   512 rows   2048 rows
//   Q4_0 [14336 x 4096]                                                                              23.5 23.7  57.6 53.7  108 103    412 393
//   Q8_0 [14336 x 4096]                                                                              27.3 27.3  62.6 56.1  121 111    464 420
// 2048 rows of Q4_0 are 680 TOP/s.  What a block of 32 x 32 results takes beyond its 32 fmas and a matrix instruction (138 cycles of a SIMD): the conversion of the weights from LDS places
// on 2 bytes, the scales and the fragments.
#include "cq_qtile.h"

#include <type_traits>

namespace {

// PPR: 16-byte pieces that cover four blocks of a row (128 elements, half a super-block) and the 8 bytes behind the first half, before the second
template <int DT> struct Q0Tile;
template <> struct Q0Tile<CQ_Q4_0> { static constexpr int BB = 18, PPR = 5; };
template <> struct Q0Tile<CQ_Q8_0> { static constexpr int BB = 34, PPR = 9; };

typedef u32x4 u32x4_at2 __attribute__((aligned(2)));       // (LDS reads on 2 bytes)
typedef f32x4 f32x4_at4 __attribute__((aligned(4)));       // (rows of results begin on an element)
typedef u32x2 u32x2_at2 __attribute__((aligned(2)));

constexpr uint32_t Q0_MAGIC = 0x4b400000u;                 // 12582912.0f
template <int DT, int MI, bool WF> struct Q0Lds {
    static constexpr int NI = (32 * Q0Tile<DT>::PPR + 63) / 64;          // copy instructions per wave and half of weights
    static constexpr int A = MI * 8192, B = NI * 1024, D8 = 8 * 32 * MI * 4, DW = WF ? 8 * 32 * 4 : 0;
    static constexpr int A_OFF = 0, B_OFF = 2 * A, D8_OFF = B_OFF + 2 * QT_NW * B, DW_OFF = D8_OFF + 2 * D8, BYTES = DW_OFF + QT_NW * DW;
};

// Results of a wave: row m0 + 32 t + nr of each tile, columns n0 + 8 e4 + 4 kg .. + 3: four at a time.  MOE: rows of the expert-sorted list, scattered to their pairs' rows and
// scaled.  Splits of K after the first write f32 planes [rows, qt_plane_ld(n)].
template <int MI, bool MOE>
__device__ __forceinline__ void q0_store(const f32x16 (&acc)[MI], void *dst, int dst_dtype, int m0, int rows, int nr, int n0, int n, int kg, int64_t stride_dst, float *planes,
                                         const MoeChunks &mc) {
    const bool plane = !MOE && blockIdx.z > 0;
    if (plane) dst = planes + (int64_t)(blockIdx.z - 1) * rows * qt_plane_ld(n);
    const int64_t ld = plane ? qt_plane_ld(n) : stride_dst;
    int row[MI];                                           // (all of them in front of the stores, which they would be waited for behind)
    float by[MI];
    if constexpr (MOE) {
#pragma unroll
        for (int t = 0; t < MI; t++) {
            row[t] = mc.pair_out[min(m0 + 32 * t + nr, rows - 1)];
            by[t] = mc.pair_scale[min(m0 + 32 * t + nr, rows - 1)];
        }
    }
#pragma unroll
    for (int t = 0; t < MI; t++) {
        const int mm = m0 + 32 * t + nr;
        if (mm >= rows) break;
        const int64_t at = (MOE ? row[t] : mm) * ld;
#pragma unroll
        for (int e4 = 0; e4 < 4; e4++) {
            const int nn = n0 + 8 * e4 + 4 * kg;
            f32x4 v = {acc[t][4 * e4], acc[t][4 * e4 + 1], acc[t][4 * e4 + 2], acc[t][4 * e4 + 3]};
            if (MOE) v *= by[t];
            if (MOE || plane || dst_dtype == CQ_F32) {
                float *const out = (float *)dst + at + nn;
                if (nn + 4 <= n) *reinterpret_cast<f32x4_at4 *>(out) = v;
                else
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (nn + i < n) out[i] = v[i];
            } else {
                uint16_t *const out = (uint16_t *)dst + at + nn;
                uint16_t h[4];
#pragma unroll
                for (int i = 0; i < 4; i++) h[i] = dst_dtype == CQ_F16 ? f2h_bits(v[i]) : f2bf_bits(v[i]);
                if (nn + 4 <= n) *reinterpret_cast<u32x2_at2 *>(out) = u32x2{(uint32_t)h[0] | (uint32_t)h[1] << 16, (uint32_t)h[2] | (uint32_t)h[3] << 16};
                else
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (nn + i < n) out[i] = h[i];
            }
        }
    }
}

// WF: the weights are the first operand
template <int DT, int MI, bool MOE, bool WF>
__global__ __launch_bounds__(QT_NW * 64, 2) void qtile0_kernel(const uint8_t *__restrict__ w, ActView av, void *__restrict__ dst, int dst_dtype, int k, int n,
                                                               int rows, int64_t stride_dst, MoeChunks mc, int64_t expert_bytes, float *__restrict__ planes) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler has no use for the body, and does not know its buffer accesses)
    typedef Q0Tile<DT> T;
    typedef Q0Lds<DT, MI, WF> LD;
    static_assert(WF || MI == 1, "the other order is for tiles of 32 rows");
    constexpr int BB = T::BB, NI = LD::NI, RS = 16 * T::PPR, BM = 32 * MI, BN = 32 * QT_NW, NA = MI, ND = (8 * MI * 32 / 64 + QT_NW - 1) / QT_NW;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nr = lane & 31, kg = lane >> 5;
    int m0 = blockIdx.x * BM, block = blockIdx.y;
    if (MOE) {
        int tile;
        qt_moe_tile(tile, block);
        if (tile >= mc.n_chunks[0]) return;
        m0 = mc.first[tile];
        rows = m0 + mc.count[tile];
        w += (int64_t)mc.expert[tile] * expert_bytes;
        if constexpr (!WF) QtPairs<BM>::request(mc, m0, rows, lds + LD::BYTES, wv, lane);
    }
    const int n0 = block * BN + 32 * wv;
    const int nsb_all = k >> 8;
    const int kb0 = (uint32_t)nsb_all * blockIdx.z / gridDim.z, kb1 = (uint32_t)nsb_all * (blockIdx.z + 1) / gridDim.z;
    const int64_t row_bytes = (int64_t)nsb_all * (8 * BB);

    // ---- weights: piece p of a half is 16-byte piece p % PPR of row p / PPR; rows past the end repeat the last one, pieces past the end the last piece.
    // The first half's pieces begin where the super-block begins, the second's end where it ends: nothing outside it is read ----
    const int wbase = min(n0, n - 1), wrows = min(32, n - wbase);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *)(w + wbase * row_bytes), 0, -1, 0x00020000);
    uint32_t w_off[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int p = min(64 * i + lane, 32 * T::PPR - 1), r = p / T::PPR;
        w_off[i] = (uint32_t)(min(r, wrows - 1) * row_bytes) + 16 * (p - r * T::PPR);
    }
    uint8_t *const myB = lds + LD::B_OFF + wv * (2 * LD::B);
    // (where this lane's row begins, with nothing known of its alignment: pieces at multiples of four bytes would be read as pairs of dwords)
    uint32_t my_row = LD::B_OFF + wv * (2 * LD::B) + nr * RS;
    asm volatile("" : "+v"(my_row));
    auto issue_w = [&](int kb, int h) {
        kb = min(kb, kb1 - 1);
#pragma unroll
        for (int i = 0; i < NI; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + h * LD::B + 1024 * i), 16, w_off[i], kb * (8 * BB) + h * (4 * BB - 8), 0, 0);
    };
    // ---- activations: [4 stages][32 MI rows][64 bytes], piece p of row r in slot p ^ (r / 4) % 4 of its 64 bytes ----
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc((void *)(av.qs + (int64_t)m0 * k), 0, -1, 0x00020000);
    uint32_t a_off[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int blk = wv + QT_NW * i, st = blk / (2 * MI), r = 16 * (blk - st * 2 * MI) + (lane >> 2), p = (lane & 3) ^ ((r >> 2) & 3);
        a_off[i] = (uint32_t)min(r, rows - 1 - m0) * (uint32_t)k + 64 * st + 16 * p;
    }
    // ---- their scales: [8 blocks][32 MI rows], instruction i of a wave brings 64 of them ----
    const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc((void *)(av.d + (int64_t)m0 * (16 * nsb_all)), 0, -1, 0x00020000);
    uint32_t d_off[ND];
    int d_dst[ND];
#pragma unroll
    for (int i = 0; i < ND; i++) {
        const int first = 64 * min(wv + QT_NW * i, 8 * BM / 64 - 1), at = first + lane, b = at / BM, r = at - b * BM;
        d_off[i] = (uint32_t)min(r, rows - 1 - m0) * (uint32_t)(64 * nsb_all) + 8 * b;
        d_dst[i] = 4 * first;
    }
    auto request = [&](int j) {
        const int kb = min(kb0 + j, kb1 - 1), slot = j & 1;
#pragma unroll
        for (int i = 0; i < NA; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (cq_lds_void *)(lds + LD::A_OFF + slot * LD::A + 1024 * (wv + QT_NW * i)), 16, a_off[i], kb * 256, 0, 0);
#pragma unroll
        for (int i = 0; i < ND; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(drs, (cq_lds_void *)(lds + LD::D8_OFF + slot * LD::D8 + d_dst[i]), 4, d_off[i], kb * 64, 0, 0);
        asm volatile("" ::: "memory");
    };

    f32x16 acc[MI];
    i32x16 magic;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) magic[e] = (int)Q0_MAGIC;
    asm volatile("" : "+v"(magic));                       // (in registers, not rebuilt for every block)

    request(0);
    issue_w(kb0, 0);
    const int nsb = kb1 - kb0;
    bool wild = false;
    const int live = (min(rows - m0, BM) + 31) / 32;       // 32-row tiles that hold rows
    const uint32_t nib = 4 - 4 * kg;                       // Q4_0: the lower lanes take the low nibbles
    // this lane's 16 weights of block b, and a block's fragment of the activations
    auto operand = [&](int b, i32x4 &op) {
        const uint8_t *const blk = lds + my_row + ((b >> 2) * (LD::B + 8) + (b & 3) * BB);
        if constexpr (DT == CQ_Q4_0) {
            // nibbles as 16 (q - 8): the high ones where they are, the low ones moved up
            const u32x4 q = *reinterpret_cast<const u32x4_at2 *>(blk + 2);
#pragma unroll
            for (int i = 0; i < 4; i++) op[i] = (int)(((q[i] << nib) ^ 0x80808080u) & 0xf0f0f0f0u);
        } else {
            op = __builtin_bit_cast(i32x4, (u32x4)*reinterpret_cast<const u32x4_at2 *>(blk + 2 + 16 * kg));
        }
    };
    auto a_frag = [&](int slot, int b, int t) {
        return *reinterpret_cast<const i32x4 *>(lds + LD::A_OFF + slot * LD::A + nr * 64 + (b >> 1) * (MI * 2048) + t * 2048 + 16 * ((2 * (b & 1) + kg) ^ ((nr >> 2) & 3)));
    };
    if constexpr (!WF) {
        // ---- a lane has results of one weight row, whose scale comes with its weights ----
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        for (int j = 0; j < nsb; j++) {
            const int kb = kb0 + j, slot = j & 1;
            if (j > 0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            issue_w(kb, 1);
            request(j + 1);
            const uint8_t *const Dj = lds + LD::D8_OFF + slot * LD::D8 + 16 * kg;
            auto row_scale = [&](int b) {
                const float v = h2f(*reinterpret_cast<const uint16_t *>(lds + my_row + ((b >> 2) * (LD::B + 8) + (b & 3) * BB)));
                return DT == CQ_Q4_0 ? v * 0.0625f : v;
            };
            i32x4 op;
            float dw = row_scale(0);
            operand(0, op);
            i32x16 S = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_frag(slot, 0, 0), op, magic, 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                // the second half has landed (behind it only the next super-block's activations were asked for); the first one's place is free
                if (b == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA + ND) : "memory");
                if (b == 4) issue_w(kb + 1, 0);
                const float c = -12582912.0f * dw;
                wild |= !(__builtin_fabsf(dw) < __builtin_inff());
                i32x4 op_n;
                float dw_n = 0.0f;
                if (b < 7) {
                    dw_n = row_scale(b + 1);
                    operand(b + 1, op_n);
                }
                f32x4 d8[4];
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++) d8[e4] = *reinterpret_cast<const f32x4 *>(Dj + 4 * (b * BM + 8 * e4));
                i32x4 af;
                if (b < 7) af = a_frag(slot, b + 1, 0);
#pragma unroll
                for (int e = 0; e < 16; e++) acc[0][e] = fmaf(fmaf(__int_as_float(S[e]), dw, c), d8[e >> 2][e & 3], acc[0][e]);
                qt_pin(acc[0]);
                if (b < 7) S = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, op_n, magic, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                dw = dw_n;
            }
        }
    } else {
        // ---- scales of the weights: [8 blocks][32 rows] of f32 in LDS, since a lane has results of sixteen rows ----
        uint8_t *const my_dw = lds + LD::DW_OFF + wv * LD::DW;
        auto row_scales = [&](int h) {                     // of the half that has landed: blocks 4 h + 2 kg and the one behind it
#pragma unroll
            for (int i = 0; i < 2; i++) {
                float v = h2f(*reinterpret_cast<const uint16_t *>(lds + my_row + (h * (LD::B + 8) + i * BB) + 2 * kg * BB));
                if (DT == CQ_Q4_0) v *= 0.0625f;
                wild |= !(__builtin_fabsf(v) < __builtin_inff());
                *reinterpret_cast<float *>(my_dw + 128 * (4 * h + i) + 256 * kg + 4 * nr) = v;
            }
            asm volatile("" ::: "memory");                 // (other lanes read them; a wave's LDS accesses keep their order)
        };
        auto scales_of = [&](int b, f32x4 (&d)[4]) {
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) d[e4] = *reinterpret_cast<const f32x4 *>(my_dw + 128 * b + 32 * e4 + 16 * kg);
        };
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        row_scales(0);
        f32x4 dw[4];
        scales_of(0, dw);
        // the main loop, for each number of tiles that hold rows
        auto run = [&](auto tiles) {
            constexpr int LIVE = decltype(tiles)::value;
            constexpr bool TWO = LIVE > 1 && (MI == 5 || (DT == CQ_Q8_0 && LIVE == 2));
            constexpr int NS = TWO ? 2 : LIVE, LEAD = TWO ? 1 : NS;
            for (int j = 0; j < nsb; j++) {
                const int kb = kb0 + j, slot = j & 1;
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                issue_w(kb, 1);
                request(j + 1);
                const uint8_t *const Dj = lds + LD::D8_OFF + slot * LD::D8 + 4 * nr;
                auto d8_of = [&](int b, float (&d)[LIVE]) {
#pragma unroll
                    for (int t = 0; t < LIVE; t++) d[t] = *reinterpret_cast<const float *>(Dj + 4 * (b * BM + t * 32));
                };
                // The product LEAD tiles ahead, in this block or the next, is on its way in the matrix cores while the sums of a tile are scaled; its fragment was asked for another tile before.
                i32x4 op, af;
                i32x16 S[NS];
                float d8[LIVE];
                auto ahead = [&](int u) { if (u < 8 * LIVE) af = a_frag(slot, u / LIVE, u % LIVE); };
                operand(0, op);
                d8_of(0, d8);
                ahead(0);
#pragma unroll
                for (int u = 0; u < LEAD; u++) {
                    S[u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(op, af, magic, 0, 0, 0);
                    ahead(u + 1);
                }
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    // the second half has landed (behind it only the next super-block's activations were asked for); the first one's place is free
                    if (b == 3) {
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA + ND) : "memory");
                        row_scales(1);
                    }
                    if (b == 4) issue_w(kb + 1, 0);
                    if (b == 7) {                              // the next super-block's first half
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                        row_scales(0);
                    }
                    f32x4 c[4], dw_n[4];
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) c[e4] = -12582912.0f * dw[e4];
                    scales_of(b == 7 ? 0 : b + 1, dw_n);
                    i32x4 op_n;
                    float d8_n[LIVE];
                    if (b < 7) {
                        operand(b + 1, op_n);
                        d8_of(b + 1, d8_n);
                    }
#pragma unroll
                    for (int t = 0; t < LIVE; t++) {
                        const int u = b * LIVE + t, v = u + LEAD;
                        auto next = [&]() {
                            if (v < 8 * LIVE) S[v % NS] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v / LIVE == b ? op : op_n, af, magic, 0, 0, 0);
                            ahead(v + 1);
                        };
                        if (TWO) next();
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[t][e] = fmaf(fmaf(__int_as_float(S[u % NS][e]), dw[e >> 2][e & 3], c[e >> 2][e & 3]), d8[t], acc[t][e]);
                        qt_pin(acc[t]);
                        if (!TWO) next();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    op = op_n;
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) dw[e4] = dw_n[e4];
#pragma unroll
                    for (int t = 0; t < LIVE; t++) d8[t] = d8_n[t];
                }
            }
        };
        if (live == MI) run(std::integral_constant<int, MI>{});
        else if constexpr (MI > 1) {
            if (live == 1) run(std::integral_constant<int, 1>{});
            else if constexpr (MI > 2) {
                if (live == 2) run(std::integral_constant<int, 2>{});
                else if constexpr (MI > 3) {
                    if (live == 3) run(std::integral_constant<int, 3>{});
                    else if constexpr (MI > 4) run(std::integral_constant<int, 4>{});
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // A scale that is not finite (a file's: no quantizer of finite values writes one) spoils the offset: once more, with the sums themselves, which may be
    // zero or negative.
    if (__builtin_amdgcn_ballot_w64(wild) != 0) {
        const uint8_t *const wr = w + (int64_t)min(n0 + nr, n - 1) * row_bytes;
#pragma unroll 1
        for (int t = 0; t < live; t++) {
            f32x16 a[1];
#pragma unroll
            for (int e = 0; e < 16; e++) a[0][e] = 0.0f;
            const int64_t mm = min(m0 + 32 * t + nr, rows - 1);
#pragma unroll 1
            for (int g = 8 * kb0; g < 8 * kb1; g++) {
                const uint8_t *const blk = wr + (int64_t)g * BB;
                u32x4 q = ld_u<u32x4>(blk + 2 + (DT == CQ_Q4_0 ? 0 : 16 * kg));
                if (DT == CQ_Q4_0) {
#pragma unroll
                    for (int i = 0; i < 4; i++) q[i] = ((q[i] << nib) ^ 0x80808080u) & 0xf0f0f0f0u;
                }
                const i32x4 af = *reinterpret_cast<const i32x4 *>(av.qs + mm * k + 32 * g + 16 * kg);
                const float d8 = av.d[2 * (mm * (8 * nsb_all) + g)];
                i32x16 S;
#pragma unroll
                for (int e = 0; e < 16; e++) S[e] = 0;
                S = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, q), af, S, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int64_t nn = min(n0 + 8 * (e >> 2) + 4 * kg + (e & 3), n - 1);
                    const float dg = h2f(ld_u<uint16_t>(w + nn * row_bytes + (int64_t)g * BB)) * (DT == CQ_Q4_0 ? 0.0625f : 1.0f);
                    a[0][e] = fmaf((float)S[e] * dg, d8, a[0][e]);
                }
            }
            q0_store<1, MOE>(a, dst, dst_dtype, m0 + 32 * t, rows, nr, n0, n, kg, stride_dst, planes, mc);
        }
        return;
    }
    if constexpr (!WF) qt_store<1, MOE>(acc, dst, dst_dtype, m0, rows, n0 + nr, n, kg, stride_dst, planes, lds + LD::BYTES, lds + LD::BYTES + QtPairs<BM>::SCALES);
    else q0_store<MI, MOE>(acc, dst, dst_dtype, m0, rows, nr, n0, n, kg, stride_dst, planes, mc);
#endif
}

}  // namespace

// Which operand comes first in tiles of 32 rows (larger ones: the weights, see above).  us, activations / weights first:
//  - Q4_0, activations: their form leaves room for two workgroups to a unit, the other for one (20 rows of [13824 x 5120] 28.0 / 31.4, of [4096 x 14336] 24.1 / 24.2).  Experts, whose
//    grid has workgroups without rows between those with, by the number that is expected to have rows (3900 drawn calls; the time with the weights first by the other, mean): up to 256
//    0.79, since two come to lie on one unit while others have none (606 pairs on 16 experts of 1536 x 1024 36.9 / 26.5); 257 - 500 1.06; 501 - 640, about two full rounds, 1.00, with more
//    to win than to lose where they are full (600 on 32 of 4096 x 2048 84.6 / 68.7, on 48 of 3072 x 1024 56.9 / 53.8); more 1.10 (2000 on 128 of 2048 x 768 60.8 / 65.9, 2400 on 256 of
//    2048 x 512 74.8 / 89.6).
//  - Q8_0, weights, whose results are stored four columns at a time (900 pairs on 64 experts of 1024 x 1024 30.8 / 29.1), but for weights so large that a model's next call finds them in
//    memory: the scales of a super-block's first half are put into LDS at the end of the one before, when what comes from memory is not there yet.  3500 drawn calls of 9 - 32 rows, the time
//    with the weights first by the other, weights out of a cache and out of memory: up to 8 MB 0.993 and 0.996, 16 - 24 MB 0.987 and 1.007, 48 MB and more 0.993 and 1.015 (24 rows of
//    [4096 x 14336] from memory 27.9 / 28.4).
static constexpr int64_t Q0_ONE_ROUND = 256, Q0_TWO_ROUNDS[2] = {500, 640}, Q0_CACHED = 44 << 20;
template <int DT>
static int launch_mi(int mi, bool moe, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows, int64_t stride_dst,
                     const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s) {
#define Q0_GO(M, E, F) return qtile_go(qtile0_kernel<DT, M, E, F>, QT_NW, Q0Lds<DT, M, F>::BYTES + (E && !F ? QtPairs<32 * M>::BYTES : 0), grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s)
    if (moe) {
        if (mi != 1) Q0_GO(4, true, true);
        if constexpr (DT == CQ_Q4_0)
            if (const int64_t t = rows * grid.y; t > Q0_ONE_ROUND && (t <= Q0_TWO_ROUNDS[0] || t > Q0_TWO_ROUNDS[1])) Q0_GO(1, true, false);
        Q0_GO(1, true, true);
    }
    if (mi == 1) {
        if constexpr (DT == CQ_Q8_0)
            if (n * k <= Q0_CACHED) Q0_GO(1, false, true);
        Q0_GO(1, false, false);
    }
    switch (mi) {
        case 2: Q0_GO(2, false, true);
        case 3: Q0_GO(3, false, true);
        case 4: Q0_GO(4, false, true);
        case 5: if constexpr (DT == CQ_Q4_0) Q0_GO(5, false, true);
        default: return CQ_ERR_RANGE;
    }
#undef Q0_GO
}

int cq_qtile0_launch(int w_dtype, int mi, bool moe, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows,
                     int64_t stride_dst, const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s) {
    return w_dtype == CQ_Q4_0 ? launch_mi<CQ_Q4_0>(mi, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s)
                              : launch_mi<CQ_Q8_0>(mi, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s);
}
