// The router's logits: out fp32 [m, ne] = x [m, d] @ w^T with w bf16 [ne, d], the reduction over d cut into eight
// slices of kw = d / 8 that are summed in slice order (ops.zig:131-136: router_part native_ops.cu:1405-1460, then
// router_sum native_ops.cu:335-362).
//
// The summation order inside a slice is this build's own (the reference sums a slice inside tensor-core MMAs, an order
// no document fixes): a wave takes one slice of one (row, expert) dot product; lane l sums the 4-value chunks
// c = l, l + 64, l + 128, .. of the slice (c < kw / 4) in ascending order, each chunk's values in order, by fp32 fma;
// then the 64 lane sums are added by a butterfly over lane distances 32, 16, 8, 4, 2, 1. Products of 16-bit operands
// are exact in fp32, so an fma and a multiply-then-add give the same bits. A block holds the eight slices of its
// expert and rows (a wave a slice) and adds them in slice order, so the logits need no second launch.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ea_device.hpp"
#include "ea_gemm.hpp"
#include "ea_host.hpp"

namespace ea {

constexpr int RT_SLICES = 8;  // ops.zig:133

// The lane sums of a wave added by the butterfly, for N (a power of two, at most 32) values: in the first steps a lane keeps
// half of its values and hands its partner the others, so that each value is summed once (the two halves' sum has the same
// bits on either side). v[0] ends as the total of value wave_sums() of the lane, the same in 64 / N neighbouring lanes.
template <int N>
__device__ __forceinline__ int wave_sums(float (&v)[N], int lane) {
    int mine = 0;
    auto step = [&](auto dist_, auto half_) __attribute__((always_inline)) {
        constexpr int D = decltype(dist_)::value, H = decltype(half_)::value;
        if constexpr (H > 0) {
            const bool up = (lane & D) != 0;
#pragma unroll
            for (int i = 0; i < H; ++i) {
                const float keep = up ? v[i + H] : v[i], give = up ? v[i] : v[i + H];
                v[i] = keep + lane_xor<D>(give);
            }
            mine += up ? H : 0;
        } else {
            v[0] = v[0] + lane_xor<D>(v[0]);
        }
    };
#define EA_STEP(D_, H_) step(std::integral_constant<int, D_>{}, std::integral_constant<int, H_>{})
    EA_STEP(32, N / 2);
    EA_STEP(16, N / 4);
    EA_STEP(8, N / 8);
    EA_STEP(4, N / 16);
    EA_STEP(2, N / 32);
    EA_STEP(1, 0);
#undef EA_STEP
    return mine;
}

__device__ __forceinline__ void act4(uint2 u, bool bf, float (&v)[4]) {
    const uint16_t h[4] = {(uint16_t)(u.x & 0xffffu), (uint16_t)(u.x >> 16), (uint16_t)(u.y & 0xffffu),
                           (uint16_t)(u.y >> 16)};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = bf ? bf2f(h[i]) : h2f(h[i]);
}

// Block (expert, row group of ROWS), wave s: slice s of the expert and the group's rows. What bounds it at few rows is round
// trips (3.1 MB of weights at 256 x 6144 are 0.5 us of HBM, a block's rows come from L2), with more the rows' unpacking and
// products. So the loads of RT_BATCH chunks of the weight and of every row are issued before the first product (a row past
// m re-reads the last one, a chunk past the slice the slice's last, and is not added; RT_BATCH follows from d, so that hardly
// a chunk lies past the slice: router_batch), the type is fixed at compile time, and the rows' lane sums share their steps (wave_sums). The form before read each row under a condition of its own, which
// waited for its load, and took four experts a block above 16 rows. 256 x 6144, distinct weights: 1 row 3.5 -> 2.9 us, 2 rows
// 6.6 -> 3.2, 5 rows 8.6 -> 4.5, 16 rows 16.2 -> 6.7, 37 rows 19.6 -> 12.7, 128 rows 38 -> 26.5, 512 rows 190 -> 94.
template <int ROWS, bool BF, int RT_BATCH>
__global__ void __launch_bounds__(64 * RT_SLICES) router_kernel(const uint16_t* __restrict__ x, int x_stride,
                                                                    const uint16_t* __restrict__ w,
                                                                    float* __restrict__ part, float* __restrict__ out,
                                                                    int m, int d, int ne) {
    __shared__ float sums[RT_SLICES][ROWS];
    const int lane = threadIdx.x & 63, s = threadIdx.x >> 6, e = blockIdx.x, m0 = (int)blockIdx.y * ROWS;
    const int rows = min(ROWS, m - m0);
    const int kw = d / RT_SLICES, nc = kw / 4;
    float acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) acc[r] = 0.0f;
    const uint16_t* wr = w + (size_t)e * d + (size_t)s * kw;
    const uint16_t* xr = x + (size_t)m0 * x_stride + (size_t)s * kw;
    for (int c0 = 0; c0 < nc; c0 += RT_BATCH * 64) {
        uint2 wu[RT_BATCH], xu[RT_BATCH][ROWS];
#pragma unroll
        for (int i = 0; i < RT_BATCH; ++i) {
            const size_t k = 4 * (size_t)min(c0 + i * 64 + lane, nc - 1);
            wu[i] = *reinterpret_cast<const uint2*>(wr + k);
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                xu[i][r] = *reinterpret_cast<const uint2*>(xr + (size_t)min(r, rows - 1) * x_stride + k);
        }
        issued();
#pragma unroll
        for (int i = 0; i < RT_BATCH; ++i) {
            float wv[4];
            act4(wu[i], true, wv);
            const bool in = c0 + i * 64 + lane < nc;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                float xv[4], t = acc[r];
                act4(xu[i][r], BF, xv);
#pragma unroll
                for (int q = 0; q < 4; ++q) t = __builtin_fmaf(xv[q], wv[q], t);
                acc[r] = in ? t : acc[r];
            }
        }
    }
    const int mine = wave_sums<ROWS>(acc, lane);
    if ((lane & (64 / ROWS - 1)) == 0) sums[s][mine] = acc[0];
    __syncthreads();
    const int r = threadIdx.x;
    if (r < rows) {
        float tot = sums[0][r];
        if (part) part[(size_t)(m0 + r) * ne + e] = tot;
#pragma unroll
        for (int q = 1; q < RT_SLICES; ++q) {
            const float p = sums[q][r];
            if (part) part[((size_t)q * m + m0 + r) * ne + e] = p;
            tot = tot + p;
        }
        out[(size_t)(m0 + r) * ne + e] = tot;
    }
}

// Chunks of a lane's slice a batch: as few batches as four hold, and no more chunks in each than it takes. (Always three, as
// d = 6144 takes, multiplied chunks past the slice elsewhere: d = 7168, 384 experts, 33 rows 31.1 us, now 22.5; d = 512, 8
// experts, 4096 rows 26.3, now 10.7; d = 7168, 256 experts, 128 rows 48.1, now 33.7.)
static int router_batch(int chunks) {
    const int n = (chunks + 3) / 4;
    return n > 0 ? (chunks + n - 1) / n : 1;
}

int launch_router(hipStream_t s, const void* x, int x_dtype, uint32_t x_stride, const void* w, float* part, float* out,
                  uint32_t m, uint32_t d, uint32_t ne) {
    EA_REQUIRE_CTX(c);
    if (!x || !w || !out) return EA_BAD_ARGUMENT;
    if (x_dtype != F16 && x_dtype != BF16) return EA_BAD_ARGUMENT;
    // ops.zig:134: the reduction splits into eight slices of whole 64-value steps
    if (d == 0 || d % (RT_SLICES * 64) != 0) return EA_UNEVEN_SPLIT;
    if (x_stride < d || x_stride % 4 != 0) return EA_BAD_ROW_STRIDE;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 7) return EA_BAD_ARGUMENT;
    if (m == 0 || ne == 0) return EA_OK;
    const auto* xs = static_cast<const uint16_t*>(x);
    const auto* ws = static_cast<const uint16_t*>(w);
    // rows a block (the least power of two that holds m, at most 16): a block's rows share one read of its weights
    const int chunks = ((int)(d / RT_SLICES / 4) + 63) / 64;
    const int batch = router_batch(chunks);
#define EA_RB(ROWS_, BATCH_) (x_dtype == BF16 ? router_kernel<ROWS_, true, BATCH_> : router_kernel<ROWS_, false, BATCH_>)
#define EA_RF(ROWS_)                                                                                                   \
    (batch == 1 ? EA_RB(ROWS_, 1) : batch == 2 ? EA_RB(ROWS_, 2) : batch == 3 ? EA_RB(ROWS_, 3) : EA_RB(ROWS_, 4))     \
        <<<dim3(ne, (m + (ROWS_) - 1) / (ROWS_)), 64 * RT_SLICES, 0, s>>>(xs, (int)x_stride, ws, part, out, (int)m,    \
                                                                          (int)d, (int)ne)
    if (m == 1) EA_RF(1);
    else if (m == 2) EA_RF(2);
    else if (m <= 4) EA_RF(4);
    else if (m <= 8) EA_RF(8);
    else EA_RF(16);
#undef EA_RF
#undef EA_RB
    return launched();
}

}  // namespace ea

extern "C" int ea_router(ea_stream_t stream, const void* x, int x_dtype, uint32_t x_stride, const void* w, float* part,
                         float* out, uint32_t m, uint32_t d, uint32_t ne) {
    return ea::launch_router(ea::as_stream(stream), x, x_dtype, x_stride, w, part, out, m, d, ne);
}
