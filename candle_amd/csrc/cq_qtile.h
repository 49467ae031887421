// What the prefill kernels over quantized weights share (cq_qtile.hip: K-quants, cq_qtile0.hip: Q4_0 and Q8_0): the workgroup's shape, the way results go out, the launch.
#pragma once
#include "cq_device.h"
#include "cq_fmt.h"
#include "cq_launch.h"
#include "cq_stream.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int QT_NW = 8;                                 // waves of a workgroup, side by side along n
constexpr int QT_NW_NARROW = 4;                          // of a narrow one

// Floats from one row of a plane of split sums to the next: rows begin on 16 bytes whatever n is, so that four columns at a time are added up.
__host__ __device__ constexpr int64_t qt_plane_ld(int64_t n) { return (n + 3) & ~(int64_t)3; }

// everything that goes into these sums is worked out before what follows (the scheduler would rather work on all tiles at once, out of
// registers that are not there)
__device__ __forceinline__ void qt_pin(f32x16 &v) {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(v) :: "memory");
#endif
}

// Grouped products: which tile of the table, and which columns, a workgroup takes.  The grid (a multiple of eight wide) has room for more tiles than there are; taken along x first, the
// workgroups without a tile would lie between those of one block of columns and of the next, and each of them waits for a whole unit's LDS.  Here they come last, and all column blocks of a
// tile run on one XCD, so that its rows come to one L2.
__device__ __forceinline__ void qt_moe_tile(int &tile, int &block) {
    const uint32_t id = blockIdx.x + gridDim.x * blockIdx.y, at = id >> 3;
    tile = 8 * (at / gridDim.y) + (id & 7);
    block = at % gridDim.y;
}
// ... and where the rows of its tile go, with their factors, brought to LDS in front of everything else: read from memory where they are used they would be
// waited for behind the stores, four rows at a time.
template <int BM> struct QtPairs {
    static constexpr int PARTS = (BM + 63) / 64, SCALES = 256 * PARTS, BYTES = 2 * SCALES;
    static __device__ __forceinline__ void request(const MoeChunks &mc, int m0, int rows, uint8_t *to, int wv, int lane) {
#ifdef __HIP_DEVICE_COMPILE__
        if (wv >= 2 * PARTS) return;
        const int part = wv % PARTS;
        const bool scales = wv >= PARTS;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(scales ? (void *)(mc.pair_scale + m0) : (void *)(mc.pair_out + m0), 0, -1, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (cq_lds_void *)(to + 256 * wv), 4, 4 * min(64 * part + lane, rows - 1 - m0), 0, 0, 0);
        asm volatile("" ::: "memory");
#endif
    }
};

// Results of a wave: column nn of rows m0 .., in the layout of the 32 x 32 matrix instructions (row 8 (e / 4) + 4 kg + e % 4 of each tile).
// MOE: rows of the expert-sorted list, scattered to their pairs' rows and scaled; `to` and `by`: these rows' places and factors, in LDS.
// Splits of K after the first write f32 planes [rows, qt_plane_ld(n)].
template <int MI, bool MOE>
__device__ __forceinline__ void qt_store(const f32x16 (&acc)[MI], void *dst, int dst_dtype, int m0, int rows, int nn, int n, int kg, int64_t stride_dst, float *planes,
                                         const uint8_t *to = nullptr, const uint8_t *by = nullptr) {
    auto store = [&](auto put) {
#pragma unroll
        for (int t = 0; t < MI; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int mm = m0 + t * 32 + 8 * (e >> 2) + 4 * kg + (e & 3);
                if (mm < rows && nn < n) put(mm, acc[t][e]);
                if ((e & 3) == 3) __builtin_amdgcn_sched_barrier(0);
            }
    };
    if constexpr (MOE) {
#pragma unroll
        for (int t = 0; t < MI; t++)
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const int r = t * 32 + 8 * e4 + 4 * kg;
                const i32x4 row = *reinterpret_cast<const i32x4 *>(to + 4 * r);
                const f32x4 f = *reinterpret_cast<const f32x4 *>(by + 4 * r);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (m0 + r + i < rows && nn < n) ((float *)dst)[(int64_t)row[i] * stride_dst + nn] = acc[t][4 * e4 + i] * f[i];
                __builtin_amdgcn_sched_barrier(0);
            }
    } else {
        if (dst_dtype == CQ_F32 || blockIdx.z > 0) {
            float *const out = (blockIdx.z > 0 ? planes + (int64_t)(blockIdx.z - 1) * rows * qt_plane_ld(n) : (float *)dst) + nn;
            const int64_t ld = blockIdx.z > 0 ? qt_plane_ld(n) : stride_dst;
            store([&](int mm, float v) { out[mm * ld] = v; });
        } else if (dst_dtype == CQ_F16) store([&](int mm, float v) { ((uint16_t *)dst)[nn + mm * stride_dst] = f2h_bits(v); });
        else store([&](int mm, float v) { ((uint16_t *)dst)[nn + mm * stride_dst] = f2bf_bits(v); });
    }
}

typedef void (*QtFn)(const uint8_t *, ActView, void *, int, int, int, int, int64_t, MoeChunks, int64_t, float *);

inline int qtile_go(QtFn fn, int nw, int lds_bytes, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows, int64_t stride_dst,
                    const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s) {
    hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(fn, grid, dim3(nw * 64), lds_bytes, s, (const uint8_t *)w, av, dst, dst_dtype, (int)k, (int)n, (int)rows, stride_dst, mc, expert_bytes, planes);
    return (int)hipGetLastError();
}

}  // namespace

// Q4_0 and Q8_0 (cq_qtile0.hip): one launch with tiles of 32 mi rows, K split over grid.z
int cq_qtile0_launch(int w_dtype, int mi, bool moe, dim3 grid, const void *w, const ActView &av, void *dst, int dst_dtype, int64_t k, int64_t n, int64_t rows,
                     int64_t stride_dst, const MoeChunks &mc, int64_t expert_bytes, float *planes, hipStream_t s);
