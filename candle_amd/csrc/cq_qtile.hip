// Prefill matmul of Q4_K, Q5_K and Q6_K over pre-quantized activations (Q8_K blocks) on the int8 matrix cores of gfx950, and the choice of tile and split
// that Q4_0 and Q8_0 (cq_qtile0.hip) share:   dst[m, n] = sum_k x^[m, k] * W^[n, k]
//
// Per super-block of 256 elements the exact integer S[m,n] = sum_k q8[m,k] * (scale[n, sub(k)] * q[n,k]) of the CPU's dot products (k_quants.rs:1460-1540,
// 1714-1801, 2035-2092), then acc += d8 * (d * S - dmin * M), M the products of the 16-element sums with the mins (one f16 MFMA, exact).  scale * q has up to
// 13 bits, so it goes through the int8 cores as two operands in two chains: Q4_K as scale % 8 * q and scale / 8 * q (S = lo + 8 hi), Q5_K and Q6_K as the
// low byte less 128 and the high byte of scale * q + 128 (S = lo + 256 hi).
//
// A workgroup is eight waves (or four: qtile_plan) side by side along n that share 32 MI rows of activations: each weight is converted once, by the one wave that
// multiplies it, straight into its operand registers.  Weights go by copies to LDS, into a ring of the wave's own, with counted waits; activations into a ring
// shared by the workgroup, one barrier per super-block.  Two kernels: qtile_kernel interleaves the conversion of one step with the products of the step before and scales the sums of
// all tiles at the end of a super-block (Q4_K, Q5_K, tiles of up to 64 rows); qtile_wide_kernel converts a whole super-block and then multiplies it tile by tile.
//
// What bounds it: at many rows, first the power limit's clock: 2048 rows of Q4_K [4096 x 14336], one workgroup to a unit, take 482 k cycles at 1.93 GHz (249 us), the same workgroups
// on an eighth of the units 468 k at 2.46 (190 us).  Then what the two waves of a SIMD overlap: of a unit's 7960 busy cycles per super-block the matrix cores work 4350 (55 %; Q5_K and Q6_K 43 %)
// and the vector units issue in 61 % (69, 68), waves wait in 30 % of theirs.  A matrix instruction also keeps the vector unit from issuing for ten cycles, whatever its shape, so that half as
// many of 32 x 32 x 32 leave it more room than of 16 x 16 x 64 (282 us for 262).  At few rows the weights' way from memory, and in unsplit small products the chain of one wave a SIMD.
// f16 / bf16 results are written by the product; the f32 copy and its conversion went (12 us of 154 for 512 rows of Q5_K).
//
// [4096 x 14336], us on one card, with Q4_K and Q5_K of 96- and 128-row tiles and Q6_K in qtile_kernel / now, quantizing the activations included:
//              17 rows   131 rows   512 rows   2048 rows
//   Q4_K     19.6 19.5  46.5 43.5  96.7 90.3   307 283
//   Q5_K     22.7 22.7  51.1 49.1   104 99.1   336 317
//   Q6_K     30.7 27.9  57.8 49.2   115 99.9   374 318
// 2048 rows of Q4_K are 930 TOP/s of products asked for and 1860 done.
#include "cq_qtile.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t qt_pk_add(uint32_t a, uint32_t b) {
    half2v r = __builtin_bit_cast(half2v, a) + __builtin_bit_cast(half2v, b);
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t qt_pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t qt_pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}

// the high bytes of both halves
__device__ __forceinline__ uint32_t qt_pk_high(uint32_t a) { return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) >> 8)); }

// The lane's number, worked out where it is asked for (what follows from threadIdx.x is kept in registers over the whole main loop, which needs all of them).
__device__ __forceinline__ int qt_lane() {
    int l = 0;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
#endif
    return l;
}

// A wave's weights: 32 rows, lane (row = lane % 32, kg = lane / 32) holds elements 16 kg .. 16 kg + 15 of every 32-element sub-block.
// EXTRA: 16-byte pieces per lane and super-block beside the four of the quants.  HI: factor of the hi chain.
template <int DT> struct QTile;
template <> struct QTile<CQ_Q4K> {
    static constexpr int EXTRA = 1, HI = 8, QS = 16;
};
template <> struct QTile<CQ_Q5K> {
    static constexpr int EXTRA = 2, HI = 256, QS = 48;
};

// Weights: three stages of 64 elements ahead; activations: three super-blocks.  Waves 4 - 7 (the second on each SIMD) run half a super-block behind, so that the vector work at the
// end of a super-block lies under the other wave's matrix work.  Fragments, conversions and products of one step are interleaved by hand, the sums of a tile pinned before the
// next one's: left to itself the scheduler spills.
constexpr int QT_R = 4, QT_L = QT_R - 1;                 // stages (64 elements) in a wave's ring of weights, stages requested ahead
// RA: super-blocks in the ring of activations
template <int DT, int MI, int NW> struct QtLds {
    static constexpr int RA = 3, A = MI * 8192, B = 1024 * (QT_R + QTile<DT>::EXTRA), AM = MI * 1024, D8 = (MI + 1) / 2 * 256;
    static constexpr int A_OFF = 0, B_OFF = RA * A, AM_OFF = B_OFF + NW * B, D8_OFF = AM_OFF + RA * AM, BYTES = D8_OFF + RA * D8;
};

template <int DT, int MI, bool MOE, int NW>
__global__ __launch_bounds__(NW * 64, 2) void qtile_kernel(const uint8_t *__restrict__ w, ActView av, void *__restrict__ dst, int dst_dtype, int k, int n,
                                                              int rows, int64_t stride_dst, MoeChunks mc, int64_t expert_bytes, float *__restrict__ planes) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler has no use for the body, and does not know its buffer accesses)
    typedef QTile<DT> T;
    typedef QtLds<DT, MI, NW> LD;
    static_assert(NW == 8 || (NW == 4 && MI <= 2), "two waves bring the sums and two the scales of 64 rows at most");
    constexpr int BB = BlockInfo<DT>::bytes, EX = T::EXTRA, BM = 32 * MI, BN = 32 * NW;
    constexpr int NA = 8 * MI / NW;                                 // copy instructions per wave and super-block of activations
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
        QtPairs<BM>::request(mc, m0, rows, lds + LD::BYTES, wv, lane);
    }
    const int n0 = block * BN + 32 * wv;
    const int nsb_all = k >> 8;
    const int kb0 = (uint32_t)nsb_all * blockIdx.z / gridDim.z, kb1 = (uint32_t)nsb_all * (blockIdx.z + 1) / gridDim.z;
    const int64_t row_bytes = (int64_t)nsb_all * BB;

    // ---- weights: rows past the end repeat the last one (their results are not stored) ----
    const int wbase = min(n0, n - 1);
    const uint8_t *const wrow = w + wbase * row_bytes;
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *)wrow, 0, -1, 0x00020000);
    const uint32_t w_off = (uint32_t)(min(nr, n - 1 - wbase) * row_bytes) + 16 * kg;
    // ---- activations: 64 bytes of 16 rows per instruction, piece p of row r in slot p ^ (r / 4) % 4 of its 64 bytes ----
    // (a super-block is [4 stages][32 MI rows][64 bytes]; instruction i of a wave brings block wv + NW i of its 8 MI KB)
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc((void *)(av.qs + (int64_t)m0 * k), 0, -1, 0x00020000);
    constexpr int NAO = NW == 2 * MI ? 1 : NA;             // (as many waves as row blocks: the instructions of a wave are whole stages apart)
    uint32_t a_off[NAO];
#pragma unroll
    for (int i = 0; i < NAO; i++) {
        const int blk = wv + NW * i, st = blk / (2 * MI), r = 16 * (blk - st * 2 * MI) + (lane >> 2), p = (lane & 3) ^ ((r >> 2) & 3);
        a_off[i] = (uint32_t)min(r, rows - 1 - m0) * (uint32_t)k + 64 * st + 16 * p;
    }
    uint8_t *const myB = lds + LD::B_OFF + wv * LD::B;
    // ---- scales and 16-element sums of the activations: the first half of the waves brings the sums of 32 rows each, the others the scales of 64 ----
    const bool x_sums = wv < NW / 2;
    const int x_blk = x_sums ? min(wv, MI - 1) : min(wv & 1, (MI - 1) / 2), x_r = min(x_sums ? 32 * x_blk + (lane >> 1) : 64 * x_blk + lane, rows - 1 - m0);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        x_sums ? (void *)(av.bsums + (int64_t)m0 * (k >> 4)) : (void *)(av.d + (int64_t)m0 * nsb_all), 0, -1, 0x00020000);
    const uint32_t x_off = x_sums ? (uint32_t)x_r * (uint32_t)(32 * nsb_all) + 16 * (lane & 1) : (uint32_t)x_r * (uint32_t)(4 * nsb_all);
    // weights of stage u = 4 (kb - kb0) + q into slot q of this wave's ring; past the end the last super-block again, into slots nobody reads
    auto issue_w = [&](int kb, int q) {
        kb = min(kb, kb1 - 1);
        if (q == 0) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + 1024 * QT_R), 16, w_off, kb * BB, 0, 0);      // (the upper lanes bring the 16 bytes behind it)
            if constexpr (EX == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + 1024 * (QT_R + 1)), 16, w_off, kb * BB + 16, 0, 0);
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + 1024 * q), 16, w_off, kb * BB + T::QS + 32 * q, 0, 0);
    };
    // this wave's part of the activations of super-block j of this workgroup's range
    auto issue_a = [&](int j, int slot) {
        const int kb = min(kb0 + j, kb1 - 1);
#pragma unroll
        for (int i = 0; i < NA; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (cq_lds_void *)(lds + LD::A_OFF + slot * LD::A + 1024 * (wv + NW * i)), 16, a_off[NAO == 1 ? 0 : i], kb * 256 + (NAO == 1 ? 64 * i : 0), 0, 0);
    };
    auto issue_x = [&](int j, int slot) {
        const int kb = min(kb0 + j, kb1 - 1);
        if (x_sums) __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (cq_lds_void *)(lds + LD::AM_OFF + slot * LD::AM + 1024 * x_blk), 16, x_off, 32 * kb, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (cq_lds_void *)(lds + LD::D8_OFF + slot * LD::D8 + 256 * x_blk), 4, x_off, 4 * kb, 0, 0);
    };

    f32x16 acc[MI];
    i32x16 sl[MI], sh[MI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;

    issue_a(0, 0);
    issue_x(0, 0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < QT_L; t++) issue_w(kb0, t);
    const int nsb = kb1 - kb0;
    const int live = MOE ? (rows - m0 + 31) / 32 : MI;     // 32-row tiles that hold rows: an expert rarely fills its last ones

    constexpr bool STAGGER = NW == 8;      // (four waves have a SIMD each)
    auto body = [&](auto late) {
    constexpr bool LATE = decltype(late)::value;
    int slot = 0, slot1 = 1;                               // ring slots of super-blocks j and j + 1
    auto request = [&](int j1, int sl1) {                  // behind barrier j1 - 1: what super-block j1 needs of the activations
        issue_a(j1, sl1);
        issue_x(j1, sl1);
        asm volatile("" ::: "memory");
    };
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(QT_L + EX) : "memory");
    if constexpr (LATE) request(1, 1);
    u32x4 hdr = u32x4{0, 0, 0, 0}, qh = u32x4{0, 0, 0, 0}, raw;
    i32x4 af[MI], bl, bh;
    // operands of step s = 2 q + ks (32 elements): dword i of this lane's weights, tile t of the activations
    uint32_t m_lo, m_hi;
    auto scales = [&](int s) {
        // 6-bit scale of sub-block s (utils.rs:50-60)
        const int sft = 8 * (s & 3);
        const uint32_t sc = s < 4 ? (hdr.y >> sft) & 63u : ((hdr.w >> sft) & 0xFu) | (((hdr.y >> sft) >> 2) & 0x30u);
        if constexpr (DT == CQ_Q4K) { m_lo = (sc & 7u) * 0x00010001u; m_hi = (sc >> 3) * 0x00010001u; }
        else m_lo = sc * 0x00010001u;
    };
    auto convert = [&](int s, int i, i32x4 &lo, i32x4 &hi) {
        uint32_t v = (s & 1 ? raw[i] >> 4 : raw[i]) & 0x0f0f0f0fu;
        if constexpr (DT == CQ_Q4K) {
            lo[i] = (int)qt_pk_mul(v, m_lo);
            hi[i] = (int)qt_pk_mul(v, m_hi);
        } else {
            v |= ((qh[i] >> s) & 0x01010101u) << 4;
            const uint32_t e = qt_pk_mad(v & 0x00ff00ffu, m_lo, 0x00800080u), o = qt_pk_mad((v >> 8) & 0x00ff00ffu, m_lo, 0x00800080u);
            lo[i] = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
            hi[i] = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
        }
    };
    const uint8_t *const a_lane = lds + LD::A_OFF + nr * 64;
    const int a_x0 = 16 * (kg ^ ((nr >> 2) & 3)), a_x1 = a_x0 ^ 32;
    auto a_frag = [&](int s, int t) { return *reinterpret_cast<const i32x4 *>(a_lane + slot * LD::A + (s >> 1) * (MI * 2048) + t * 2048 + (s & 1 ? a_x1 : a_x0)); };
    auto weights = [&](int q) { return *reinterpret_cast<const u32x4 *>(myB + 1024 * q + 16 * lane); };
    // what this wave has requested behind its weights of stage q when it asks for them
    constexpr int NX = NA + 1, W0[4] = {2, 2 + NX, 2 + NX + EX, 2 + EX}, W1[4] = {2 + NX, 2, 2 + EX, 2 + EX + NX};
    for (int j = 0; j < nsb; j++) {
        const int kb = kb0 + j;
        // ---- first step of a super-block: nothing of it is in registers yet ----
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LATE ? W1[0] : W0[0]) : "memory");
        if constexpr (!LATE) {
            if (j > 0) asm volatile("s_barrier" ::: "memory");
            request(j + 1, slot1);
        }
        issue_w(kb, 3);
        hdr = *reinterpret_cast<const u32x4 *>(myB + 1024 * QT_R + 16 * (qt_lane() & 31));
        if constexpr (EX == 2) qh = *reinterpret_cast<const u32x4 *>(myB + 1024 * (QT_R + 1) + 16 * lane);
        raw = weights(0);
#pragma unroll
        for (int t = 0; t < MI; t++) af[t] = a_frag(0, t);
        scales(0);
#pragma unroll
        for (int i = 0; i < 4; i++) convert(0, i, bl, bh);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int q = s >> 1, ns = s + 1;
            i32x4 nl, nh;
            if (s & 1) {
                if (q < 3) {
                    // the weights of the next stage, and a request for those three stages on
                    if (q == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATE ? W1[1] : W0[1]) : "memory");
                    if (q == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATE ? W1[2] : W0[2]) : "memory");
                    if (q == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATE ? W1[3] : W0[3]) : "memory");
                    raw = weights(q + 1);
                }
            } else if (q > 0) {
                if (LATE && q == 2) {
                    asm volatile("s_barrier" ::: "memory");
                    request(j + 2, slot1 == 2 ? 0 : slot1 + 1);
                }
                issue_w(kb + 1, q - 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < MI; t++) {
                if (!MOE || t < live) {
                if (s == 0) {
                    i32x16 z;
#pragma unroll
                    for (int e = 0; e < 16; e++) z[e] = 0;
                    sl[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[t], bl, z, 0, 0, 0);
                    sh[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[t], bh, z, 0, 0, 0);
                } else {
                    sl[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[t], bl, sl[t], 0, 0, 0);
                    sh[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[t], bh, sh[t], 0, 0, 0);
                }
                if (ns < 8) af[t] = a_frag(ns, t);
                }
                if (ns < 8) {
                    if (t == 0) scales(ns);
#pragma unroll
                    for (int i = 4 * t / MI; i < 4 * (t + 1) / MI; i++) convert(ns, i, nl, nh);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (ns < 8) { bl = nl; bh = nh; }
            if (s == 7) {
                const float d = h2f(hdr.x), dmin = h2f(hdr.x >> 16);
                const uint32_t mlo = hdr.z & 0x3f3f3f3fu, mhi = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
                const uint32_t kmask = 0u - (uint32_t)(qt_lane() >> 5), mine = (mhi & kmask) | (mlo & ~kmask);
                u32x4 mv;
#pragma unroll
                for (int i = 0; i < 4; i++) mv[i] = qt_pk_add((0x6400u | ((mine >> (8 * i)) & 0xffu)) * 0x00010001u, 0xe400e400u);
                const half8 bm = __builtin_bit_cast(half8, mv);
#pragma unroll
                for (int t = 0; t < MI; t++) {
                    if (MOE && t >= live) break;
                    __builtin_amdgcn_sched_barrier(0);
                    const s16x8 ai = *reinterpret_cast<const s16x8 *>(lds + LD::AM_OFF + slot * LD::AM + (t * 32 + nr) * 32 + 16 * kg);
                    const half8 am = __builtin_convertvector(ai, half8);           // sums of 16 int8: exact
                    f32x16 z;
#pragma unroll
                    for (int e = 0; e < 16; e++) z[e] = 0.0f;
                    const f32x16 mt = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bm, z, 0, 0, 0);
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) {
                        const f32x4 d8 = *reinterpret_cast<const f32x4 *>(lds + LD::D8_OFF + slot * LD::D8 + 4 * (t * 32 + 8 * e4 + 4 * kg));
#pragma unroll
                        for (int e1 = 0; e1 < 4; e1++) {
                            const int e = 4 * e4 + e1;
                            const float v = fmaf(-dmin, mt[e], d * (float)(T::HI * sh[t][e] + sl[t][e]));
                            acc[t][e] = fmaf(d8[e1], v, acc[t][e]);
                        }
                    }
                    qt_pin(acc[t]);
                }
            }
        }
        slot = slot1;
        slot1 = slot1 == LD::RA - 1 ? 0 : slot1 + 1;
    }
    if constexpr (!LATE && STAGGER) asm volatile("s_barrier" ::: "memory");       // the others' last one
    };
    if constexpr (!STAGGER) body(std::false_type{});
    else if (wv < NW / 2) body(std::false_type{});
    else body(std::true_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    const int lane_out = qt_lane();
    qt_store<MI, MOE>(acc, dst, dst_dtype, m0, rows, n0 + (lane_out & 31), n, lane_out >> 5, stride_dst, planes, lds + LD::BYTES, lds + LD::BYTES + QtPairs<BM>::SCALES);
#endif
}

// ---- the kernel of tiles of 96 and 128 rows (Q6_K: of all) ----------------------------------------------------------------------------------
// A wave converts all weights of a super-block into registers, then multiplies 32 rows at a time: sixteen matrix instructions on two chains, under which the sums of the 32 rows before are
// scaled and added.  Per tile only 32 registers of int32 sums and 32 of scaled ones are alive instead of 32 MI, which is what makes room for the operands.  The second wave of a SIMD
// meets at the barrier before its conversion, the first behind it: one converts while the other multiplies.  (All of the conversion interleaved with the products of the last and first
// tile instead, whichever wave: Q6_K 327 us for 271 of 2048 rows, since the vector work of a wave then waits behind matrix instructions that wait for the other wave's.  Products without any
// vector work between them, and a raised priority for the wave that is among them: no difference.)
// Tiles without rows are left out, of experts and of the end of a prompt.  Integers, and the order of the f32 sums, are those of qtile_kernel: the same bits.
//
// Blocks of a row as they lie in memory: PIECES 16-byte pieces, the quants from piece QS on (Q6_K: 13 pieces and the dword behind them, from the dword that the block
// begins in).  HI: factor of the hi chain.
template <int DT> struct QWide;
template <> struct QWide<CQ_Q4K> {
    static constexpr int PIECES = 9, QS = 1, HI = 8;
    static constexpr bool HAS_MIN = true;
};
template <> struct QWide<CQ_Q5K> {
    static constexpr int PIECES = 11, QS = 3, HI = 256;
    static constexpr bool HAS_MIN = true;
};
template <> struct QWide<CQ_Q6K> {
    static constexpr int PIECES = 13, QS = 0, HI = 256;
    static constexpr bool HAS_MIN = false;
};

// AHEAD: super-blocks requested ahead, as many as the 160 KB of a unit hold (half of that for workgroups of four waves, of which two share a unit): the ring of
// activations has one slot more, a wave's ring of weights as many
template <int DT, int MI, int NW> struct QwLds {
    static constexpr int A = MI * 8192, AM = QWide<DT>::HAS_MIN ? MI * 1024 : 0, D8 = (MI + 1) / 2 * 256;
    static constexpr int NB = (32 * QWide<DT>::PIECES + 63) / 64, B = 1024 * NB + (DT == CQ_Q6K ? 256 : 0);
    static constexpr int bytes(int ahead) { return (ahead + 1) * (A + AM + D8) + ahead * NW * B; }
    static constexpr int ROOM = 20 * 1024 * NW, AHEAD = bytes(3) <= ROOM ? 3 : bytes(2) <= ROOM ? 2 : 1;
    static constexpr int A_OFF = 0, AM_OFF = (AHEAD + 1) * A, D8_OFF = AM_OFF + (AHEAD + 1) * AM, B_OFF = D8_OFF + (AHEAD + 1) * D8, BYTES = bytes(AHEAD);
};

// PAIR: rows of two tensors, the second expert_bytes (of experts: mc.up) behind the first: waves 0 .. 3 multiply by 128 rows of the first, waves 4 .. 7 by the same rows of the second, and the
// results are silu(first) * second (Mlp::forward, quantized_llama.rs:56-63).  At the end the two waves of a SIMD, which have the same rows and columns of both, hand each other
// half of their tiles through LDS, so that both compute and store.  What it saves is a write and a read of both products where one result does, and what it costs is
// that the silu of a workgroup's results has no other workgroup to hide behind (1000 rows of two Q4_K [14336 x 4096]: 309 us and 30.5 of the quantizer that took both products,
// 311 and 17.2 now; a llama's prompt of 150 / 700 / 1000 / 2000 tokens 1.003x / 1.011x / 1.010x / 1.013x).
template <int DT, int MI, bool MOE, int NW, bool PAIR = false>
__global__ __launch_bounds__(NW * 64, 2) void qtile_wide_kernel(const uint8_t *__restrict__ w, ActView av, void *__restrict__ dst, int dst_dtype, int k, int n,
                                                              int rows, int64_t stride_dst, MoeChunks mc, int64_t expert_bytes, float *__restrict__ planes) {
#ifdef __HIP_DEVICE_COMPILE__                             // (the host compiler has no use for the body, and does not know its buffer accesses)
    typedef QWide<DT> T;
    typedef QwLds<DT, MI, NW> LD;
    static_assert(NW == 8 || (NW == 4 && MI <= 2), "two waves bring the sums and two the scales of 64 rows at most");
    static_assert(!PAIR || (NW == 8 && MI > 2), "tiles of four pairs of waves");
    constexpr int BB = BlockInfo<DT>::bytes, BM = 32 * MI, BN = PAIR ? 16 * NW : 32 * NW, AHEAD = LD::AHEAD, ROW = 16 * T::PIECES;
    constexpr int NA = 8 * MI / NW, NX = NA + 1, NB = LD::NB + (DT == CQ_Q6K ? 1 : 0);      // copies per wave and super-block: activations, with scales or sums, weights
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nr = lane & 31, kg = lane >> 5;
    int m0 = blockIdx.x * BM, block = blockIdx.y;
    if (PAIR && wv >= 4) w += MOE ? mc.up : expert_bytes;
    if (MOE) {
        int tile;
        qt_moe_tile(tile, block);
        if (tile >= mc.n_chunks[0]) return;
        m0 = mc.first[tile];
        rows = m0 + mc.count[tile];
        w += (int64_t)mc.expert[tile] * expert_bytes;
        QtPairs<BM>::request(mc, m0, rows, lds + LD::BYTES, wv, lane);
    }
    const int n0 = block * BN + 32 * (PAIR ? wv & 3 : wv);
    const int nsb_all = k >> 8;
    const int kb0 = (uint32_t)nsb_all * blockIdx.z / gridDim.z, kb1 = (uint32_t)nsb_all * (blockIdx.z + 1) / gridDim.z;
    const int64_t row_bytes = (int64_t)nsb_all * BB;

    // ---- weights: piece p of a super-block is piece p % PIECES of row p / PIECES; rows past the end repeat the last one (their results are not stored),
    // pieces past the end the last piece ----
    const int wbase = min(n0, n - 1), wlast = min(31, n - 1 - wbase);
    const uint8_t *const wrow = w + wbase * row_bytes;
    const uint32_t w_odd = DT == CQ_Q6K ? (uint32_t)(uintptr_t)wrow & 2u : 0u;       // (the descriptor begins on a dword)
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *)(wrow - w_odd), 0, -1, 0x00020000);
    uint32_t w_off[NB];
#pragma unroll
    for (int i = 0; i < LD::NB; i++) {
        const int p = min(64 * i + lane, 32 * T::PIECES - 1), r = p / T::PIECES;
        w_off[i] = (uint32_t)(min(r, wlast) * row_bytes) + 16 * (p - r * T::PIECES) + w_odd;
    }
    if constexpr (DT == CQ_Q6K) w_off[NB - 1] = (uint32_t)(min(lane & 31, wlast) * row_bytes) + 208 + w_odd;
    // ---- activations: 64 bytes of 16 rows per instruction, piece p of row r in slot p ^ (r / 4) % 4 of its 64 bytes ----
    // (a super-block is [4 stages][32 MI rows][64 bytes]; instruction i of a wave brings block wv + NW i of its 8 MI KB)
    // (experts' gate and up: of the tokens' rows, each of which several pairs share, those that the tile's pairs name)
    constexpr bool NAMED = MOE && PAIR;
    const int64_t a_first = NAMED ? 0 : m0;
    auto a_row = [&](int r) { return NAMED ? (uint32_t)mc.src[m0 + min(r, rows - 1 - m0)] : (uint32_t)min(r, rows - 1 - m0); };
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc((void *)(av.qs + a_first * k), 0, -1, 0x00020000);
    constexpr int NAO = NW == 2 * MI ? 1 : NA;             // (as many waves as row blocks: the instructions of a wave are whole stages apart)
    uint32_t a_off[NAO];
#pragma unroll
    for (int i = 0; i < NAO; i++) {
        const int blk = wv + NW * i, st = blk / (2 * MI), r = 16 * (blk - st * 2 * MI) + (lane >> 2), p = (lane & 3) ^ ((r >> 2) & 3);
        a_off[i] = a_row(r) * (uint32_t)k + 64 * st + 16 * p;
    }
    uint8_t *const myB = lds + LD::B_OFF + wv * (AHEAD * LD::B);
    // ---- scales and 16-element sums of the activations: the first half of the waves brings the sums of 32 rows each, the others the scales of 64 ----
    const bool x_sums = T::HAS_MIN && wv < NW / 2;
    const int x_blk = x_sums ? min(wv, MI - 1) : min(wv & 1, (MI - 1) / 2), x_r = x_sums ? 32 * x_blk + (lane >> 1) : 64 * x_blk + lane;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        x_sums ? (void *)(av.bsums + a_first * (k >> 4)) : (void *)(av.d + a_first * nsb_all), 0, -1, 0x00020000);
    const uint32_t x_off = x_sums ? a_row(x_r) * (uint32_t)(32 * nsb_all) + 16 * (lane & 1) : a_row(x_r) * (uint32_t)(4 * nsb_all);
    // Super-block kb0 + j of this workgroup's range into slot `slot`; past the end the last one again, into slots nobody reads.
    auto issue_w = [&](int j, int slot) {
        const int at = min(kb0 + j, kb1 - 1) * BB, odd = DT == CQ_Q6K ? at & 2 : 0;      // (210 kb is 2 past a dword for odd kb, and so are odd rows of an odd number of blocks)
#pragma unroll
        for (int i = 0; i < LD::NB; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + slot * LD::B + 1024 * i), 16, DT == CQ_Q6K ? (w_off[i] + odd) & ~2u : w_off[i], at - odd, 0, 0);
        if constexpr (DT == CQ_Q6K)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (cq_lds_void *)(myB + slot * LD::B + 1024 * LD::NB), 4, (w_off[NB - 1] + odd) & ~2u, at - odd, 0, 0);
        asm volatile("" ::: "memory");
    };
    auto issue_a = [&](int j, int slot) {
        const int kb = min(kb0 + j, kb1 - 1);
#pragma unroll
        for (int i = 0; i < NA; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (cq_lds_void *)(lds + LD::A_OFF + slot * LD::A + 1024 * (wv + NW * i)), 16, a_off[NAO == 1 ? 0 : i], kb * 256 + (NAO == 1 ? 64 * i : 0), 0, 0);
        if (x_sums) __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (cq_lds_void *)(lds + LD::AM_OFF + slot * LD::AM + 1024 * x_blk), 16, x_off, 32 * kb, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (cq_lds_void *)(lds + LD::D8_OFF + slot * LD::D8 + 256 * x_blk), 4, x_off, 4 * kb, 0, 0);
        asm volatile("" ::: "memory");
    };

    f32x16 acc[MI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;
    const int live = (min(rows - m0, BM) + 31) / 32;       // 32-row tiles that hold rows: an expert, or the end of a prompt, rarely fills its last ones

    // ---- the weights of a super-block, as operands: lane (nr, kg) has elements 16 kg .. 16 kg + 15 of every 32-element sub-block s of row nr ----
    i32x4 wl[8], wh[8];
    float d;
    uint32_t dm = 0;                                       // d and dmin as they are in the block
    u32x4 bm;                                              // the mins of four sub-blocks as f16, each twice
    const uint8_t *const b_lane = myB + nr * ROW;
    auto convert = [&](int j, int slot) {
        const uint8_t *const blk = b_lane + slot * LD::B, *const quants = blk + 16 * (T::QS + kg);
        if constexpr (DT == CQ_Q6K) {
            const uint32_t shift = (uint32_t)(min(nr, wlast) * row_bytes + w_odd + (kb0 + j) * BB) & 2u;      // bytes by which this super-block is off its dword
            auto piece = [&](const uint8_t *at, uint32_t behind) {
                u32x4 v = *reinterpret_cast<const u32x4 *>(at);
#pragma unroll
                for (int i = 0; i < 3; i++) v[i] = __builtin_amdgcn_alignbyte(v[i + 1], v[i], shift);
                v[3] = __builtin_amdgcn_alignbyte(behind, v[3], shift);
                return v;
            };
            const uint32_t last = *reinterpret_cast<const uint32_t *>(myB + slot * LD::B + 1024 * LD::NB + 4 * nr);
            const u32x4 hdr = piece(blk + 192, last);
            d = h2f(last >> (8 * shift));
#pragma unroll
            for (int h = 0; h < 2; h++) {
                u32x4 qa = piece(quants + 128 + 32 * h, *reinterpret_cast<const uint32_t *>(quants + 144 + 32 * h)), qb;
#pragma unroll
                for (int i = 0; i < 4; i++) {              // high bits of sub-blocks 4 h (low nibbles) and 4 h + 2, and of 4 h + 1 and 4 h + 3
                    qb[i] = (qa[i] >> 2) & 0x33333333u;
                    qa[i] &= 0x33333333u;
                }
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const u32x4 raw = piece(quants + 64 * h + 32 * g, *reinterpret_cast<const uint32_t *>(quants + 64 * h + 32 * g + 16));
                    const u32x4 qh = g ? qb : qa;
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const int s = 4 * h + g + 2 * u;
                        // int8 scale of 16 elements; scale (q - 32) + 128 in 16 bits: high byte, and low byte less 128
                        const int sc = (int)(hdr[s >> 1] << (24 - 16 * (s & 1) - 8 * kg)) >> 24;
                        const uint32_t mul = __builtin_amdgcn_perm(0, (uint32_t)sc, 0x01000100u), add = __builtin_amdgcn_perm(0, (uint32_t)(128 - 32 * sc), 0x01000100u);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const uint32_t v = u ? ((raw[i] >> 4) & 0x0f0f0f0fu) | (qh[i] & ~0x0f0f0f0fu) : (raw[i] & 0x0f0f0f0fu) | ((qh[i] << 4) & ~0x0f0f0f0fu);
                            const uint32_t e = qt_pk_mad(v & 0x00ff00ffu, mul, add), o = qt_pk_mad(qt_pk_high(v), mul, add);
                            wl[s][i] = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
                            wh[s][i] = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
                        }
                    }
                }
            }
        } else {
            const u32x4 hdr = *reinterpret_cast<const u32x4 *>(blk);
            dm = hdr.x;
            d = h2f(hdr.x);
            // 6-bit scales and mins of four sub-blocks each (utils.rs:50-60)
            const uint32_t sc[2] = {hdr.y & 0x3f3f3f3fu, (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u)};
            const uint32_t m = kg ? ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u) : hdr.z & 0x3f3f3f3fu;
#pragma unroll
            for (int i = 0; i < 4; i++) bm[i] = qt_pk_add((0x6400u | ((m >> (8 * i)) & 0xffu)) * 0x00010001u, 0xe400e400u);
            u32x4 qh = u32x4{0, 0, 0, 0};
            if constexpr (DT == CQ_Q5K) qh = *reinterpret_cast<const u32x4 *>(blk + 16 + 16 * kg);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const u32x4 raw = *reinterpret_cast<const u32x4 *>(quants + 32 * q);
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int s = 2 * q + u;
                    const uint32_t twice = 0x0c000c00u + 0x00010001u * (s & 3), scs = sc[s >> 2];       // byte s % 4 of four scales in both halves
                    if constexpr (DT == CQ_Q4K) {
                        const uint32_t lo = __builtin_amdgcn_perm(0, scs & 0x07070707u, twice), hi = __builtin_amdgcn_perm(0, (scs >> 3) & 0x07070707u, twice);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const uint32_t v = (u ? raw[i] >> 4 : raw[i]) & 0x0f0f0f0fu;
                            wl[s][i] = (int)qt_pk_mul(v, lo);
                            wh[s][i] = (int)qt_pk_mul(v, hi);
                        }
                    } else {
                        const uint32_t mul = __builtin_amdgcn_perm(0, scs, twice);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const uint32_t q1 = (qh[i] >> (s & 3)) & 0x11111111u;              // fifth bits of sub-blocks s % 4 (in the low nibbles) and s % 4 + 4
                            const uint32_t v = ((u ? raw[i] >> 4 : raw[i]) & 0x0f0f0f0fu) | ((s < 4 ? q1 << 4 : q1) & ~0x0f0f0f0fu);
                            const uint32_t e = qt_pk_mad(v & 0x00ff00ffu, mul, 0x00800080u), o = qt_pk_mad(qt_pk_high(v), mul, 0x00800080u);
                            wl[s][i] = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
                            wh[s][i] = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
                        }
                    }
                }
            }
        }
    };

    // ---- products of a super-block, 32 rows at a time; the sums of the 32 rows before are scaled and added meanwhile ----
    const uint8_t *const a_lane = lds + LD::A_OFF + nr * 64;
    const int a_x0 = 16 * (kg ^ ((nr >> 2) & 3)), a_x1 = a_x0 ^ 32;
    auto multiply = [&](int slot) {
        const uint8_t *const a0 = a_lane + slot * LD::A + a_x0, *const a1 = a_lane + slot * LD::A + a_x1;
        const uint8_t *const d8_lane = lds + LD::D8_OFF + slot * LD::D8 + 16 * kg, *const am_lane = lds + LD::AM_OFF + slot * LD::AM + nr * 32 + 16 * kg;
        auto a_frag = [&](int t, int s) { return *reinterpret_cast<const i32x4 *>((s & 1 ? a1 : a0) + (s >> 1) * (MI * 2048) + t * 2048); };
        i32x4 af[4];
        i32x16 sl, sh, zero;
        f32x16 sum, mt, none;
        f32x4 d8;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            zero[e] = 0;
            none[e] = 0.0f;
        }
        // results 2 s, 2 s + 1 of the sixteen that a lane has of tile t
        auto scale = [&](int t, int s) {
            if (s % 2 == 0) d8 = *reinterpret_cast<const f32x4 *>(d8_lane + 4 * (32 * t + 4 * s));
#pragma unroll
            for (int e = 2 * s; e < 2 * s + 2; e++) {
                float v = d * sum[e];
                if (T::HAS_MIN) v = fmaf(-h2f(dm >> 16), mt[e], v);
                acc[t][e] = fmaf(d8[e & 3], v, acc[t][e]);
            }
        };
#pragma unroll
        for (int u = 0; u < 4; u++) af[u] = a_frag(0, u);
#pragma unroll
        for (int t = 0; t < MI; t++) {
            if (t < live) {
                s16x8 ai;
                if (T::HAS_MIN) ai = *reinterpret_cast<const s16x8 *>(am_lane + 1024 * t);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    __builtin_amdgcn_sched_barrier(0);
                    sl = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[s & 3], wl[s], s ? sl : zero, 0, 0, 0);
                    sh = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[s & 3], wh[s], s ? sh : zero, 0, 0, 0);
                    if (s < 4) af[s & 3] = a_frag(t, s + 4);
                    else if (t + 1 < MI) af[s & 3] = a_frag(t + 1, s - 4);
                    if (t > 0) scale(t - 1, s);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (T::HAS_MIN) {
                    const half8 am = __builtin_convertvector(ai, half8);               // sums of 16 int8: exact
                    mt = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, __builtin_bit_cast(half8, bm), none, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 16; e++) sum[e] = (float)(T::HI * sh[e] + sl[e]);
                __builtin_amdgcn_sched_barrier(0);
            } else if (t == live) {
#pragma unroll
                for (int s = 0; s < 8; s++) scale(t - 1, s);
            }
        }
        if (live == MI) {
#pragma unroll
            for (int s = 0; s < 8; s++) scale(MI - 1, s);
        }
    };

    const bool late = NW == 8 && wv >= 4;
    // (in the order of the main loop: the waits count what was asked for behind)
#pragma unroll
    for (int j = 0; j < AHEAD; j++) {
        if (late) issue_a(j, j);
        issue_w(j, j);
        if (!late) issue_a(j, j);
    }
    const int nsb = kb1 - kb0;
    int slot_a = 0, slot_w = 0;
    for (int j = 0; j < nsb; j++) {
        // Barrier j: the activations of super-block j are there for everybody, and nobody reads those of j - 1 any more.
        auto meet = [&]() {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AHEAD * NB + (AHEAD - 1) * NX) : "memory");
        };
        const int next_a = slot_a == 0 ? AHEAD : slot_a - 1;
        if (late) {
            meet();
            issue_a(j + AHEAD, next_a);
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD * NX + (AHEAD - 1) * NB) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        convert(j, slot_w);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue_w(j + AHEAD, slot_w);
        if (!late) {
            meet();
            issue_a(j + AHEAD, next_a);
        }
        multiply(slot_a);
        slot_a = slot_a == AHEAD ? 0 : slot_a + 1;
        slot_w = slot_w == AHEAD - 1 ? 0 : slot_w + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (copies may not outlive the workgroup)

    const int lane_out = qt_lane();
    if constexpr (PAIR) {
        static_assert(LD::BYTES >= 8 * 2 * 4096, "two tiles of every wave");
        __syncthreads();                                   // nobody reads operands any more
        float *const mine = (float *)lds + 2048 * wv + lane_out, *const other = (float *)lds + 2048 * (wv ^ 4) + lane_out;
        f32x16 half[2];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) {                 // tiles 0 and 1 are the first four waves', 2 and 3 the others'
                const float hi = u + 2 < MI ? acc[u + 2 < MI ? u + 2 : 0][e] : 0.0f;
                half[u][e] = late ? hi : acc[u][e];
                mine[64 * (16 * u + e)] = late ? acc[u][e] : hi;
            }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float o = other[64 * (16 * u + e)], g = late ? o : half[u][e];
                half[u][e] = g / (1.0f + expf(-g)) * (late ? half[u][e] : o);
            }
        const uint8_t *const to = lds + LD::BYTES + (late ? 256 : 0);
        qt_store<2, MOE>(half, dst, CQ_F32, m0 + (late ? 64 : 0), min(rows, m0 + BM), n0 + (lane_out & 31), n, lane_out >> 5, stride_dst, planes, to, to + QtPairs<BM>::SCALES);
    } else {
        qt_store<MI, MOE>(acc, dst, dst_dtype, m0, rows, n0 + (lane_out & 31), n, lane_out >> 5, stride_dst, planes, lds + LD::BYTES, lds + LD::BYTES + QtPairs<BM>::SCALES);
    }
#endif
}

// The sum of the splits of K in a fixed order, in pairs and pairs of pairs: sixteen sums added one after the other round more than the chain of super-blocks
// that they were cut from (Q6_K rows of 4096: 8.5e-8 of the results' norm against 6.2e-8 in four splits; in pairs 6.2e-8).  The first split comes from
// `first` (dst itself or a plane), the others from planes, whose rows are qt_plane_ld(n) long.  Bound by the latency of the reads at the sizes that are split: four planes are on their way at
// a time, and a workgroup is small enough that 32 x 4096 results fill the chip.  RAGGED: n is no multiple of four (with its bounds in every case the others took 0.2 - 0.5 us more, 2 - 4 %).
constexpr int QT_RT = 128, QT_MAX_SPLITS = 16;
template <int ODT, bool RAGGED>
__global__ __launch_bounds__(QT_RT) void qtile_reduce_kernel(const float *first, int64_t ld_first, const float *__restrict__ planes, void *dst, int splits, int64_t n,
                                                             int64_t stride_dst, int64_t count) {
    const int64_t i = ((int64_t)blockIdx.x * QT_RT + threadIdx.x) * 4;
    if (i >= count) return;
    const int64_t ld_plane = RAGGED ? qt_plane_ld(n) : n;
    const int64_t r = i / ld_plane, c0 = i - r * ld_plane, o = r * stride_dst + c0;
    const int here = RAGGED ? (int)min((int64_t)4, n - c0) : 4;      // columns behind n are not there
    const float none = -0.0f;                              // (x + -0 is x)
    f32x4 sum[QT_MAX_SPLITS / 4];
#pragma unroll
    for (int g = 0; g < QT_MAX_SPLITS / 4; g++) {
        sum[g] = f32x4{none, none, none, none};
        if (4 * g >= splits) continue;
        f32x4 b[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (4 * g + u == 0) {
#pragma unroll
                for (int c = 0; c < 4; c++) b[u][c] = c < here ? first[r * ld_first + c0 + c] : 0.0f;
            } else b[u] = *reinterpret_cast<const f32x4 *>(planes + (min(4 * g + u, splits - 1) - 1) * count + i);
        }
#pragma unroll
        for (int u = 1; u < 4; u++)
            if (4 * g + u >= splits) b[u] = f32x4{none, none, none, none};
#pragma unroll
        for (int c = 0; c < 4; c++) sum[g][c] = (b[0][c] + b[1][c]) + (b[2][c] + b[3][c]);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if (c >= here) break;
        const float a = (sum[0][c] + sum[1][c]) + (sum[2][c] + sum[3][c]);
        if (ODT == CQ_F32) ((float *)dst)[o + c] = a;
        else ((uint16_t *)dst)[o + c] = ODT == CQ_F16 ? f2h_bits(a) : f2bf_bits(a);
    }
}

// Q6_K always, Q4_K and Q5_K in tiles of 96 and 128 rows take qtile_wide_kernel, which converts a super-block's weights first and multiplies then; tiles of 32 and 64 rows, whose
// conversions are not much shorter than their products, are faster with both interleaved (qtile_kernel; Q4_K [4096 x 4096], 200 / 300 / 1000 rows 26.6 / 31.8 / 57.8 us against 28.1 / 33.5 / 60.6)
template <int DT>
int qtile_mi(int mi, int nw, bool moe, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows, int64_t stride_dst,
             const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s) {
#define QT_GO(M, E, NW)                                                                                                                                          \
    if constexpr (DT == CQ_Q6K || M > 2) {                                                                                                                       \
        constexpr int bytes = QwLds<DT, M, NW>::BYTES + (E ? QtPairs<32 * M>::BYTES : 0);                                                                        \
        static_assert(bytes <= 160 * 1024, "LDS of a CU");                                                                                                       \
        return qtile_go(qtile_wide_kernel<DT, M, E, NW>, NW, bytes, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s); \
    } else {                                                                                                                                                     \
        constexpr int bytes = QtLds<DT, M, NW>::BYTES + (E ? QtPairs<32 * M>::BYTES : 0);                                                                        \
        static_assert(bytes <= 160 * 1024, "LDS of a CU");                                                                                                       \
        return qtile_go(qtile_kernel<DT, M, E, NW>, NW, bytes, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s); \
    }
    if (moe) {
        if (mi == 1) { QT_GO(1, true, QT_NW); }
        QT_GO(4, true, QT_NW);
    }
    if (nw == QT_NW_NARROW) {
        if (mi == 1) { QT_GO(1, false, QT_NW_NARROW); }
        QT_GO(2, false, QT_NW_NARROW);
    }
    switch (mi) {
        case 1: { QT_GO(1, false, QT_NW); }
        case 2: { QT_GO(2, false, QT_NW); }
        case 3: { QT_GO(3, false, QT_NW); }
        default: { QT_GO(4, false, QT_NW); }
    }
#undef QT_GO
}

// rows: of grouped products the tiles to be expected (their kernels have the rows from mc)
int qtile_any(int w_dtype, int mi, int nw, bool moe, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows,
              int64_t stride_dst, const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s) {
    switch (w_dtype) {
        case CQ_Q4K: return qtile_mi<CQ_Q4K>(mi, nw, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s);
        case CQ_Q5K: return qtile_mi<CQ_Q5K>(mi, nw, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s);
        case CQ_Q6K: return qtile_mi<CQ_Q6K>(mi, nw, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s);
    }
    return cq_qtile0_launch(w_dtype, mi, moe, grid, w, av, dst, dst_dtype, k, n, rows, stride_dst, mc, expert_bytes, planes, s);
}

}  // namespace

static constexpr int64_t QT_Q6K_MIN_K = 1536;
bool cq_qtile_takes(int w_dtype, const void *w, int64_t k, int64_t rows_of_w) {
    if (w_dtype == CQ_Q4K || w_dtype == CQ_Q5K) return k % 256 == 0;
    if (w_dtype == CQ_Q4_0 || w_dtype == CQ_Q8_0) return k % 256 == 0 && ((uintptr_t)w & 15) == 0;      // (rows are multiples of 16 bytes)
    // Q6_K pieces are read by whole dwords: the tensor has to begin and end on one.  The limit of k is from a kernel with two half super-blocks in flight, which short rows did not pay; from
    // 1536 on it was the faster one whatever the rows.  qtile_wide_kernel is faster below it too (k of 256 - 1280 by 1024 - 8192, 9 - 2048 rows: 0.57 - 0.85 of the general kernel's time,
    // 131 rows of [4096 x 768] 12.2 us for 16.6); the limit has not been moved.
    return w_dtype == CQ_Q6K && k % 256 == 0 && k >= QT_Q6K_MIN_K && ((uintptr_t)w & 3) == 0 && (rows_of_w * (k / 256)) % 2 == 0;
}

// Bytes of split planes that a call may use, not falling with the rows.
static constexpr int64_t QT_PLANE_FLOATS = 12 << 20;
int64_t cq_qtile_plane_bytes(int w_dtype, int64_t k, int64_t n, int64_t rows) {
    if ((w_dtype != CQ_Q4K && w_dtype != CQ_Q5K && w_dtype != CQ_Q6K && w_dtype != CQ_Q4_0 && w_dtype != CQ_Q8_0) || k < (w_dtype == CQ_Q6K ? QT_Q6K_MIN_K : 512) || k % 256) return 0;
    return cq_align256(std::min<int64_t>(16 * rows * qt_plane_ld(n), QT_PLANE_FLOATS) * 4);
}

// Rows of the tile (32 mi), waves of a workgroup and K splits: the choice for which the model
//   rounds * super-blocks per split * (a + b mi) us,  + split + planes / rate where K is split
// is least.  A round is 256 workgroups, a the conversion of the weights, b the products and sums of 32 rows.  Workgroups of the K formats may have four waves
// instead of eight if their rows are at most 64: each SIMD then converts and multiplies for one wave, and a small product takes up twice as many
// compute units (131 rows of Q6_K [4096 x 4096] unsplit: 56 us in eight waves, 41 in four; 65 rows of Q4_K [4096 x 4096] 20.6 -> 17.5).
// Costs: fitted to earlier kernels (qtile_kernel for all tiles of K formats; the activations first in all of Q4_0 and Q8_0; rounds that leave compute units idle run at a higher clock
// there, and a workgroup has 1.3 us of its own), which multiplied 32-row parts without rows as well: a part-filled tile still counts as a full one.  Tiles of 160 rows (Q4_0) have these costs as well,
// but are only taken where that makes a tenth less: those of 96 and 128 rows are 4 % faster by now than the costs say, and 160 rows in several splits slower.  180 drawn calls for which they would
// be the least, time by that of the best other choice: predicted below 0.9 0.79 - 1.01, mean 0.90 (131 rows of [13824 x 5120] in four splits 0.95, 2048 of [14336 x 4096] 0.96); 0.9 - 1 unsplit
// 0.95 - 1.04, in splits 0.98 - 1.27 (139 rows of [4032 x 2816] 22.5 us, 28.6 in eleven splits of 160).  With the kernels before those the choice is
// slower than the best by 1.0 % on average for Q4_K, 0.6 for Q5_K, 1.0 for Q6_K, 1.3 for Q4_0 and 1.1 for Q8_0, by more than 5 % in 3 - 9 % of the calls, by 18 % at most (28 rows of Q6_K
// [3667 x 3072] 16.7 us in twelve splits of eight waves, 14.1 in six of four): 1800 forwards of drawn sizes, 17 (Q4_K, Q5_K: 65) - 1600 rows, 1024 - 16384 by 1536 - 14336, cold weights, every choice timed.
// Only splits whose sums round no more than those of the general kernels (qt_roundings).
// Any number of columns: while those that are no multiple of four were not split, their few workgroups walked all of k (26 rows of Q4_0 [2986 x 9984] 112 us, 19 in splits; 10 rows of
// Q8_0 [1299 x 9728] 113 -> 18, 65 of Q6_K [1970 x 13568] 126 -> 28, 239 of Q8_0 [2818 x 13056] 152 -> 58; 1494 rows of Q8_0 [3987 x 6144] 154 -> 140).
struct QtPlan { int mi, nw, splits; };
// What the f32 sums of one result round, as twice a variance in units of one term's: a chain of c terms takes c fma's, which round partial sums of 1 .. c terms
// (the first one, a product alone, like one and a half), and every addition of two splits rounds a sum of as many terms as both have.  in_pairs: as
// qtile_reduce_kernel adds them, else one after the other like the general kernels (cq_qmm_splits).  More splits shorten the chains, but each begins with a
// rounding that a longer chain does not have.  Q6_K, of the results' norm: rows of 2048 in eight splits 5.95e-8, in two 5.47e-8; rows of 4096 in 16 splits
// 6.55e-8, in eight 6.22e-8, in the four of the general kernel 6.26e-8; 131 rows of Q8_0 [11008 x 4096] unsplit 2.05e-7, in the general kernel's two 1.49e-7.
static int64_t qt_roundings(int64_t nsb, int terms, int splits, bool in_pairs) {
    int64_t total = 0, sum[QT_MAX_SPLITS];
    for (int z = 0; z < splits; z++) {
        const int64_t c = terms * (nsb * (z + 1) / splits - nsb * z / splits);
        total += c * (c + 1) + 1;
        sum[z] = c;
    }
    for (int step = 1; in_pairs && step < splits; step *= 2)
        for (int z = 0; z + step < splits; z += 2 * step) total += 2 * (sum[z] += sum[z + step]);
    for (int z = 1; !in_pairs && z < splits; z++) total += 2 * (sum[z] += sum[z - 1]);
    return total;
}
static QtPlan qtile_plan(int w_dtype, int64_t k, int64_t n, int64_t rows, int64_t most_splits) {
    const int64_t nsb = k / 256;
    struct Cost { double a, b, a_narrow, b_narrow, start, split, rate; };                   // us, bytes per us
    static constexpr Cost q4k{1.25, 0.88, 0.69, 0.39, 0, 2.71, 1.90e6}, q5k{1.80, 0.99, 0.99, 0.53, 0, 3.31, 2.42e6}, q6k{3.12, 1.00, 1.83, 0.65, 0, 5.15, 3.94e6},
        q0{1.6, 1.23, 0, 0, 1.3, 6.8, 4.5e6};
    const bool kq = cq_is_kquant(w_dtype);
    const Cost &c = w_dtype == CQ_Q4K ? q4k : w_dtype == CQ_Q5K ? q5k : w_dtype == CQ_Q6K ? q6k : q0;
    const double plane = (double)rows * n * 4;
    const int most = (int)std::max<int64_t>(1, std::min<int64_t>({QT_MAX_SPLITS, nsb, most_splits}));
    const int terms = kq ? 1 : 8;
    const int general = std::min(most, cq_qmm_splits(k, n, rows));
    bool rounds_less[QT_MAX_SPLITS + 1];
    for (int sp = 1; sp <= most; sp++)
        rounds_less[sp] = sp == general || qt_roundings(nsb, terms, sp, true) < qt_roundings(nsb, terms, general, false);
    QtPlan best{4, QT_NW, general};
    double least = 1e30;
    const int tallest = w_dtype == CQ_Q4_0 ? 5 : 4;           // (160 rows of Q8_0 do not fit LDS, of K formats the registers)
    for (int nw : {QT_NW, QT_NW_NARROW})
        for (int mi = 1; mi <= (nw == QT_NW ? tallest : 2); mi++)
            for (int sp = 1; sp <= most; sp++) {
                const int64_t wgs = (rows + 32 * mi - 1) / (32 * mi) * ((n + 32 * nw - 1) / (32 * nw)) * sp, rounds = (wgs + 255) / 256;
                const bool narrow = nw == QT_NW_NARROW;
                if (!rounds_less[sp] || (narrow && (!kq || (n + 32 * nw - 1) / (32 * nw) > 65535))) continue;
                const double load = kq ? (double)rounds : 1.1 * (rounds - 1) + 1.0 + 0.1 * (double)(wgs - 256 * (rounds - 1)) / 256;
                const double block = narrow ? c.a_narrow + c.b_narrow * mi : c.a + c.b * mi;
                const double t = load * ((double)((nsb + sp - 1) / sp) * block + c.start) + (sp > 1 ? c.split + (sp + 1) * plane / c.rate : 0.0);
                const double as = mi == 5 ? t / 0.9 : t;
                if (as < least) { least = as; best = {mi, nw, sp}; }
            }
    return best;
}

int cq_qtile_launch(int w_dtype, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows, int64_t stride_dst, void *planes,
                    int64_t plane_bytes, hipStream_t s) {
    // an f32 dst takes the first split itself
    const bool f32 = dst_dtype == CQ_F32;
    const QtPlan plan = qtile_plan(w_dtype, k, n, rows, planes ? (f32 ? 1 : 0) + plane_bytes / (4 * rows * qt_plane_ld(n)) : 1);
    const int splits = plan.splits;
    const dim3 grid((unsigned)((rows + 32 * plan.mi - 1) / (32 * plan.mi)), (unsigned)((n + 32 * plan.nw - 1) / (32 * plan.nw)), (unsigned)splits);
    if (grid.y > 65535) return CQ_ERR_RANGE;
    const int64_t ld_plane = qt_plane_ld(n), count = rows * ld_plane;
    const bool direct = splits == 1 || f32;
    void *const first = direct ? dst : planes;
    const int64_t ld = direct ? stride_dst : ld_plane;
    float *const others = direct ? (float *)planes : (float *)planes + count;
    const MoeChunks none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0};
    const int rc = qtile_any(w_dtype, plan.mi, plan.nw, false, grid, w, av, first, direct ? dst_dtype : CQ_F32, k, n, rows, ld, none, 0, others, s);
    if (rc || splits == 1) return rc;
    const dim3 rg((unsigned)((count / 4 + QT_RT - 1) / QT_RT));
    auto *const add_up = n % 4 ? (f32 ? qtile_reduce_kernel<CQ_F32, true> : dst_dtype == CQ_F16 ? qtile_reduce_kernel<CQ_F16, true> : qtile_reduce_kernel<CQ_BF16, true>)
                               : (f32 ? qtile_reduce_kernel<CQ_F32, false> : dst_dtype == CQ_F16 ? qtile_reduce_kernel<CQ_F16, false> : qtile_reduce_kernel<CQ_BF16, false>);
    hipLaunchKernelGGL(add_up, rg, dim3(QT_RT), 0, s, (const float *)first, ld, others, dst, splits, n, stride_dst, count);
    return (int)hipGetLastError();
}

// silu(x w_gate^T) * x w_up^T.  Where the product by the rows of both tensors in one launch, which has as many workgroups, would take the wide kernel unsplit, its
// tiles hold both factors; elsewhere CQ_ERR_RANGE.  (Tensors that do not follow each other would be two launches, which must not be split either: a result is
// the same chain of super-blocks in all of them, bit for bit.)
template <int DT>
static int swiglu_go(int mi, dim3 grid, const void *w, const ActView &av, float *dst, int64_t k, int64_t n, int64_t rows, int64_t up, hipStream_t s) {
    const MoeChunks none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0};
    if (mi == 3) return qtile_go(qtile_wide_kernel<DT, 3, false, QT_NW, true>, QT_NW, QwLds<DT, 3, QT_NW>::BYTES, grid, w, av, dst, CQ_F32, k, n, rows, n, none, up, nullptr, s);
    return qtile_go(qtile_wide_kernel<DT, 4, false, QT_NW, true>, QT_NW, QwLds<DT, 4, QT_NW>::BYTES, grid, w, av, dst, CQ_F32, k, n, rows, n, none, up, nullptr, s);
}
static bool swiglu_plan(int w_dtype, const void *w_gate, const void *w_up, int64_t k, int64_t n, int64_t rows, int64_t plane_bytes, QtPlan &plan) {
    if (!cq_is_kquant(w_dtype) || !cq_qtile_takes(w_dtype, w_gate, k, n) || !cq_qtile_takes(w_dtype, w_up, k, n) || (n + 16 * QT_NW - 1) / (16 * QT_NW) > 65535) return false;
    plan = qtile_plan(w_dtype, k, 2 * n, rows, 1 + plane_bytes / (4 * rows * qt_plane_ld(2 * n)));
    if (plan.splits > 1 || plan.mi < 3 || plan.nw != QT_NW) return false;
    const bool adjacent = (const uint8_t *)w_up - (const uint8_t *)w_gate == n * (k / 256) * cq_type_size(w_dtype);
    return adjacent || qtile_plan(w_dtype, k, n, rows, 1 + plane_bytes / (4 * rows * qt_plane_ld(n))).splits == 1;
}
bool cq_qtile_takes_swiglu(int w_dtype, const void *w_gate, const void *w_up, int64_t k, int64_t n, int64_t rows, int64_t plane_bytes) {
    QtPlan plan;
    return swiglu_plan(w_dtype, w_gate, w_up, k, n, rows, plane_bytes, plan);
}
int cq_qtile_swiglu_launch(int w_dtype, const void *w_gate, const void *w_up, const ActView &av, float *dst, int64_t k, int64_t n, int64_t rows, int64_t plane_bytes,
                           hipStream_t s) {
    QtPlan plan;
    if (!swiglu_plan(w_dtype, w_gate, w_up, k, n, rows, plane_bytes, plan)) return CQ_ERR_RANGE;
    const dim3 grid((unsigned)((rows + 32 * plan.mi - 1) / (32 * plan.mi)), (unsigned)((n + 16 * QT_NW - 1) / (16 * QT_NW)));
    const int64_t up = (const uint8_t *)w_up - (const uint8_t *)w_gate;
    switch (w_dtype) {
        case CQ_Q4K: return swiglu_go<CQ_Q4K>(plan.mi, grid, w_gate, av, dst, k, n, rows, up, s);
        case CQ_Q5K: return swiglu_go<CQ_Q5K>(plan.mi, grid, w_gate, av, dst, k, n, rows, up, s);
        case CQ_Q6K: return swiglu_go<CQ_Q6K>(plan.mi, grid, w_gate, av, dst, k, n, rows, up, s);
    }
    return CQ_ERR_RANGE;
}

// tile_rows: rows of one chunk of the table, 32 or 128
int cq_qtile_moe_launch(int w_dtype, const void *w, const ActView &av, float *out, const MoeChunks &mc, int64_t num_experts, int64_t pairs, int64_t k, int64_t n, int tile_rows,
                        hipStream_t s) {
    const dim3 grid(cq_moe_grid(mc, num_experts, pairs, tile_rows), (unsigned)((n + 32 * QT_NW - 1) / (32 * QT_NW)));
    if (grid.y > 65535) return CQ_ERR_RANGE;
    // tiles to be expected: every expert's last one is half full, and few experts have none
    const int64_t tiles = std::max(std::min(num_experts, pairs), pairs / tile_rows + num_experts / 2);
    return qtile_any(w_dtype, tile_rows / 32, QT_NW, true, grid, w, av, out, CQ_F32, k, n, tiles, n, mc, n * (k / cq_block_size(w_dtype)) * cq_type_size(w_dtype), nullptr, s);
}

// silu(gate) * up of experts in tiles of 128 rows, K formats.  1500 tokens, 128 Q4_K experts of 2048 x 768, 8 each: 131 us, and 15 of the quantizer behind; a launch of 1.5 rounds for
// each of the two took 79 and 79, and the quantizer that multiplied them 22.
bool cq_qtile_moe_takes_swiglu(int w_dtype, const void *w_gate, const void *w_up, int64_t num_experts, int64_t k, int64_t n) {
    return (w_dtype == CQ_Q4K || w_dtype == CQ_Q5K || w_dtype == CQ_Q6K) && cq_qtile_takes(w_dtype, w_gate, k, num_experts * n) &&
           cq_qtile_takes(w_dtype, w_up, k, num_experts * n) && (n + 16 * QT_NW - 1) / (16 * QT_NW) <= 65535;
}
template <int DT>
static int moe_swiglu_go(dim3 grid, const void *w, const ActView &av, float *out, int64_t k, int64_t n, const MoeChunks &mc, hipStream_t s) {
    constexpr int bytes = QwLds<DT, 4, QT_NW>::BYTES + QtPairs<128>::BYTES;
    return qtile_go(qtile_wide_kernel<DT, 4, true, QT_NW, true>, QT_NW, bytes, grid, w, av, out, CQ_F32, k, n, 0, n, mc, n * (k / 256) * cq_type_size(DT), nullptr, s);
}
int cq_qtile_moe_swiglu_launch(int w_dtype, const void *w_gate, const void *w_up, const ActView &av, float *out, const MoeChunks &mc, int64_t num_experts, int64_t pairs, int64_t k,
                               int64_t n, hipStream_t s) {
    if (!cq_qtile_moe_takes_swiglu(w_dtype, w_gate, w_up, num_experts, k, n)) return CQ_ERR_RANGE;
    MoeChunks both = mc;
    both.up = (const uint8_t *)w_up - (const uint8_t *)w_gate;
    const dim3 grid(cq_moe_grid(mc, num_experts, pairs, CQ_MOE_TILE_LARGE), (unsigned)((n + 16 * QT_NW - 1) / (16 * QT_NW)));
    switch (w_dtype) {
        case CQ_Q4K: return moe_swiglu_go<CQ_Q4K>(grid, w_gate, av, out, k, n, both, s);
        case CQ_Q5K: return moe_swiglu_go<CQ_Q5K>(grid, w_gate, av, out, k, n, both, s);
        case CQ_Q6K: return moe_swiglu_go<CQ_Q6K>(grid, w_gate, av, out, k, n, both, s);
    }
    return CQ_ERR_RANGE;
}
