// EXL3 linear for up to 128 rows at once: each trellis tile is decoded once into MFMA operands for all the row tiles of a
// block (exl3_linear.cu:231-484 for the arithmetic). A K-split job is two launches (or three with the rotation on its
// own): the products, whose blocks write their split's sums to Z, and a finish that adds the splits in order; a job with
// one split finishes inside its block.
//
// What bounds it: at 6144 x 2048 and 128 rows the decode is 1.4 us of the GPU's VALU and the products 1.3 us of its MFMA
// units, so the call is its launches' and round trips' latency: 24.0 us (16 rows 10.4, 64 rows 17.3). The form before took
// the rows in passes of 8 on the one-row kernel and decoded every tile once a pass: 127 us (16 rows 19.6, 64 rows 66.5).
#include <hip/hip_runtime.h>

#include "ea_device.hpp"
#include "ea_gemm.hpp"
#include "ea_host.hpp"
#include "ea_linear.hpp"

namespace ea {

// 16 bytes that are only 4-byte aligned (a caller's xh), and two fp16 that are only 2-byte aligned (svh, bias)
typedef u4v u4v_a4 __attribute__((aligned(4)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef const __attribute__((address_space(1))) u4v_a4* gptr_u4;

constexpr int LR_WAVES = 8;
constexpr int LR_KT = 4;  // k tiles a wave multiplies of each chunk

// Block (job, group g of 32 CW columns, split; rows m0 = 16 MT blockIdx.y .. + 16 MT - 1) of eight waves: CW column waves
// of two column tiles each times KW = 8 / CW k waves. The split's k range is walked in chunks of 64 KW: the rows' chunk
// staged in LDS for all waves (row tiles past the call's rows are skipped, rows past it repeat the last row and are not
// stored; k past the range is zero), each wave's trellis in its own LDS region, both loaded a chunk ahead. The k waves'
// sums are then added in LDS. CW 4: one split, the block holds whole 128-column blocks and finishes them; CW 2: 64-column
// blocks, twice as many, the sums to Z[split]. ROT: the block rotates its chunk itself while staging it (16 lanes a
// Hadamard block, fwht128_x8), column group 0 also writing xh; worth it while the rows are few (a block repeats the
// rotation that every column group needs). FAR: 64-bit trellis offsets, for a caller's k stride (ea_exl3_linear) that 32 bits
// do not hold or that is negative; 4 % slower, so a build of its own.
template <int CB, int K2, int MT, int CW, bool ROT, bool FAR>
__global__ void __launch_bounds__(LR_WAVES * 64) lin_rows_kernel(ea_jobs jobs, ea_rot_jobs rj, int M, int K,
                                                                 const void* __restrict__ x, int x_bf16) {
    constexpr int KW = LR_WAVES / CW, CK = 64 * KW, XS = CK + 8, ROWS = 16 * MT, COLS = 32 * CW;
    constexpr int TW = 4 * K2, SW = LR_KT * 2 * TW, NL = stage_loads_k<LR_KT, K2>();
    constexpr int PR = CK / 8, PIECES = ROWS * PR, NP = (PIECES + LR_WAVES * 64 - 1) / (LR_WAVES * 64);
    constexpr int ES = COLS + 4;  // row stride of the sums in LDS, floats (rows 4 apart on other banks)
    constexpr size_t A_BYTES = (size_t)ROWS * XS * 2, ST_BYTES = (size_t)LR_WAVES * SW * 4;
    constexpr size_t RED_BYTES = (size_t)(KW / 2) * ROWS * ES * 4;
    constexpr size_t LDS = A_BYTES + ST_BYTES > RED_BYTES ? A_BYTES + ST_BYTES : RED_BYTES;
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];
    uint16_t* xa = reinterpret_cast<uint16_t*>(lds);
    float* red = reinterpret_cast<float*>(lds);  // after the products

    int ji = 0;
#pragma unroll
    for (int q = 1; q < EA_MAX_JOBS; ++q)
        if (q < jobs.n && (int)blockIdx.x >= jobs.j[q].start) ji = q;
    const ea_job& J = jobs.j[ji];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / CW, cw = wave - kw * CW;
    const int N = J.N, SK = J.SK, G = N / COLS;
    const int local = (int)blockIdx.x - J.start, g = local % G, split = local / G;
    const int m0 = (int)blockIdx.y * ROWS, rows = min(ROWS, M - m0), mts = (rows + 15) >> 4;
    const int kt = (K >> 4) / SK, lo = split * kt * 16, kn = kt * 16;  // the split's k tiles, its first k, its k
    const int nch = (kn + CK - 1) / CK;
    uint32_t* st = reinterpret_cast<uint32_t*>(lds + A_BYTES) + wave * SW;

    // the block's trellis: k tiles 0 .. kt - 1 of the split, column tiles of the group (adjacent: a group lies in one
    // 128-column block); this wave's loads take 16 bytes a lane, tile rows past the split re-reading its last row
    const int nt0 = g * 2 * CW;
    const uint32_t* tb = dptr<const uint32_t>(J.T) + (int64_t)(lo >> 4) * J.stride_k + (int64_t)(nt0 >> 3) * J.stride_nb +
                         (nt0 & 7) * TW;
    const __amdgpu_buffer_rsrc_t trs = buffer_rsrc(tb, (uint32_t)(((int64_t)(kt - 1) * J.stride_k + 2 * CW * TW) * 4));
    const int kstride = (int)(J.stride_k * 4);
    auto issue_t = [&](int c, u4v (&tv)[NL]) __attribute__((always_inline)) {
        const int t0 = (c < nch ? c : nch - 1) * KW * LR_KT + kw * LR_KT;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            constexpr int cpr = 2 * K2, last = LR_KT * cpr - 1;
            const int q = min(64 * i + lane, last), t = q / cpr, col = q - t * cpr;
            if constexpr (FAR)
                tv[i] = *(gptr_u4)(tb + min(t0 + t, kt - 1) * J.stride_k + cw * 2 * TW + col * 4);
            else
                tv[i] = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(
                                                    trs, min(t0 + t, kt - 1) * kstride + cw * 2 * TW * 4 + col * 16, 0, 0));
        }
    };

    // this thread's pieces of every chunk: piece i is row prow, columns 8 pq .. + 7; 16 consecutive lanes hold a 128-k
    // block of a row, lane l its group h8_group(l)
    const uint16_t* xsrc = ROT ? static_cast<const uint16_t*>(x) : dptr<const uint16_t>(J.xh);
    const uint16_t* suh = ROT ? dptr<const uint16_t>(rj.suh[ji]) : nullptr;
    uint16_t* xh = ROT ? dptr<uint16_t>(rj.xh[ji]) : nullptr;
    auto piece = [&](int i, int& prow, int& pq) __attribute__((always_inline)) {
        const int idx = i * LR_WAVES * 64 + tid;
        prow = idx / PR;
        pq = (idx % PR & ~15) + h8_group(lane);
    };
    u4v av[NP], sv = u4v{0u, 0u, 0u, 0u};
    auto issue_a = [&](int c) __attribute__((always_inline)) {
        const int k0 = (c < nch ? c : nch - 1) * CK;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            int prow, pq;
            piece(i, prow, pq);
            const int kk = k0 + 8 * pq < kn ? k0 + 8 * pq : 0;
            av[i] = *reinterpret_cast<const u4v_a4*>(xsrc + (size_t)(m0 + min(prow, rows - 1)) * K + lo + kk);
        }
        if constexpr (ROT) {  // pieces of one thread share their column (512 threads cover whole rows)
            int prow, pq;
            piece(0, prow, pq);
            const int kk = k0 + 8 * pq < kn ? k0 + 8 * pq : 0;
            sv = *reinterpret_cast<const u4v*>(suh + lo + kk);
        }
    };
    auto put_all = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            int prow, pq;
            piece(i, prow, pq);
            const int kk = c * CK + 8 * pq;
            u4v v = av[i];
            if constexpr (ROT) {
                v = rot8(v, sv, x_bf16, lane);
                if (g == 0 && xh && kk < kn && prow < rows)
                    *reinterpret_cast<u4v*>(xh + (size_t)(m0 + prow) * K + lo + kk) = v;
            }
            if (kk >= kn) v = u4v{0u, 0u, 0u, 0u};
            if (PIECES % (LR_WAVES * 64) == 0 || prow < ROWS) put_a(xa + prow * XS, pq, v);
        }
    };

    const TileLane<K2, CB> tl(lane);
    constexpr int NWD = TileLane<K2, CB>::NW;
    f4v acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = f4v{0.f, 0.f, 0.f, 0.f};
    const uint16_t* xr = xa + (lane & 15) * XS + kw * 64 + 8 * ((lane >> 4) & 3);
    u4v ta[NL], tn[NL];
    issue_t(0, ta);
    issue_a(0);
    issue_t(1, tn);
    auto step = [&](int c, u4v (&tv)[NL]) __attribute__((always_inline)) {
        __syncthreads();  // the chunk before is read
        stage_store_k<LR_KT, K2>(st, lane, tv);
        put_all(c);
        issue_a(c + 1);
        issue_t(c + 2, tv);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < LR_KT / 2; ++ks) {
            h8v bb[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t w[2][NWD];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t* tw = st + (2 * (2 * ks + h) + j) * TW;
                    w[h][0] = tw[tl.w0];
                    w[h][1] = tw[tl.w1];
                    if constexpr (NWD == 3) w[h][2] = tw[tl.w2];
                }
                bb[j] = __builtin_bit_cast(h8v, tl.decode2(w[0], w[1]));
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if (mt >= mts) break;  // uniform
                const h8v a = *reinterpret_cast<const h8v*>(xr + mt * 16 * XS + ks * 32);
                acc[mt][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bb[0], acc[mt][0], 0, 0, 0);
                acc[mt][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bb[1], acc[mt][1], 0, 0, 0);
            }
        }
    };
    int c = 0;
    for (; c + 1 < nch; c += 2) {  // two steps an iteration with no exit between them
        step(c, ta);
        step(c + 1, tn);
    }
    if (c < nch) step(c, ta);  // uniform

    // the k waves' sums: odd k waves into LDS, even ones add theirs and write the sum back in place
    auto at = [&](int mt, int j, int i) __attribute__((always_inline)) {
        return ((kw >> 1) * ROWS + mt * 16 + 4 * (lane >> 4) + i) * ES + cw * 32 + j * 16 + (lane & 15);
    };
    __syncthreads();  // xa and the staged trellis are read
    if (kw & 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[at(mt, j, i)] = acc[mt][j][i];
    }
    __syncthreads();
    if (!(kw & 1)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[at(mt, j, i)] = acc[mt][j][i] + red[at(mt, j, i)];
    }
    __syncthreads();
    if constexpr (CW == 4) {  // one split: a wave a row
        const uint16_t* svh = dptr<const uint16_t>(J.svh);
        const uint16_t* bias = dptr<const uint16_t>(J.bias);
        const int col = g * 128 + 2 * lane;
        const uint32_t sw = *reinterpret_cast<const u32_a2*>(svh + col);
        const uint32_t bw = *reinterpret_cast<const u32_a2*>((bias ? bias : svh) + col);
        for (int r = wave; r < rows; r += LR_WAVES)
            finish_store_pre(red[r * ES + 2 * lane], red[r * ES + 2 * lane + 1], lane, sw, bias != nullptr, bw,
                             dptr<void>(J.y), J.y_dtype, (size_t)(m0 + r) * N + col);
    } else {
        float* Z = dptr<float>(J.Z) + ((size_t)split * M + m0) * N + g * COLS;
        for (int i = tid; i < rows * COLS; i += LR_WAVES * 64) {
            const int r = i / COLS, cc = i % COLS;
            Z[(size_t)r * N + cc] = red[r * ES + cc] + red[(ROWS + r) * ES + cc];
        }
    }
}

// The splits of Z [SK, M, N] added in order and finished: a wave a (row, 128-column block), eight splits' loads in flight.
// jobs.j[i].start: the job's first column block.
__global__ void __launch_bounds__(256) lin_finish_kernel(ea_jobs jobs, int M) {
    int ji = 0;
#pragma unroll
    for (int q = 1; q < EA_MAX_JOBS; ++q)
        if (q < jobs.n && (int)blockIdx.x >= jobs.j[q].start) ji = q;
    const ea_job& J = jobs.j[ji];
    const int lane = threadIdx.x & 63, m = (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6);
    if (m >= M) return;
    const int N = J.N, SK = J.SK, col = ((int)blockIdx.x - J.start) * 128 + 2 * lane;
    const uint16_t* svh = dptr<const uint16_t>(J.svh);
    const uint16_t* bias = dptr<const uint16_t>(J.bias);
    const float* Z = dptr<const float>(J.Z) + (size_t)m * N + col;
    const size_t zs = (size_t)M * N;
    const uint32_t sw = *reinterpret_cast<const u32_a2*>(svh + col);
    const uint32_t bw = *reinterpret_cast<const u32_a2*>((bias ? bias : svh) + col);
    float v0 = 0.f, v1 = 0.f;
    for (int q0 = 0; q0 < SK; q0 += 8) {
        float z[8][2];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const size_t o = (size_t)min(q0 + q, SK - 1) * zs;
            z[q][0] = Z[o];
            z[q][1] = Z[o + 1];
        }
        issued();
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (q0 + q < SK) {  // uniform
                v0 += z[q][0];
                v1 += z[q][1];
            }
    }
    finish_store_pre(v0, v1, lane, sw, bias != nullptr, bw, dptr<void>(J.y), J.y_dtype, (size_t)m * N + col);
}

// The jobs of one kind (one split, or several) as one launch of the products: columns a block COLS = 32 CW.
template <int CB, int K2, int CW>
static void launch_rows_k2(hipStream_t s, ea_jobs jobs, const ea_rot_jobs& rj, bool rot, bool far, int M, int K, const void* x,
                           int x_bf16, int cus) {
    int nb = 0;
    for (int i = 0; i < jobs.n; ++i) {
        jobs.j[i].start = nb;
        nb += jobs.j[i].N / (32 * CW) * jobs.j[i].SK;
    }
    // row tiles a block (each more is one decode less of every tile). Rotating, one while that many blocks fit the GPU at
    // once, else two. Otherwise as many as leave 7 / 4 blocks a CU: 2048 x 6144 at 128 rows 29.4 us with eight tiles on
    // 1.5 blocks a CU, 25.8 with four on three; shapes with fewer blocks measured the same from 2 / 4 to 8 / 4.
    const int tiles = (M + 15) / 16;
    int mt = rot ? tiles == 1 || nb * tiles <= cus ? 1 : 2 : CW == 4 ? 4 : 8;
    while (!rot && mt > 1 && (mt / 2 >= tiles || nb * ((tiles + mt - 1) / mt) < cus * 7 / 4)) mt /= 2;
    const auto grid = [&](int t) { return dim3((unsigned)nb, (unsigned)((tiles + t - 1) / t)); };
#define EA_LR(MT_, ROT_, FAR_) \
    lin_rows_kernel<CB, K2, MT_, CW, ROT_, FAR_><<<grid(MT_), LR_WAVES * 64, 0, s>>>(jobs, rj, M, K, x, x_bf16)
    if (far) {  // not with rot (launch_linear_rows)
        EA_LR(2, false, true);
    } else if (rot) {
        if (mt == 1) EA_LR(1, true, false);
        else EA_LR(2, true, false);
    } else if (mt <= 2) {
        EA_LR(2, false, false);
    } else if (CW == 4 || mt == 4) {
        EA_LR(4, false, false);
    } else {
        if constexpr (CW == 2) EA_LR(8, false, false);
    }
#undef EA_LR
}

constexpr int LR_ROT_ROWS = 32;  // rows a rotating block takes at most

static bool overlap(uint64_t a, size_t an, uint64_t b, size_t bn) { return a < b + bn && b < a + an; }

int launch_linear_rows(hipStream_t s, const ea_jobs& jobs, const ea_rot_jobs* rot, int M, int K, uint32_t k2,
                       uint32_t cb, const void* x, int x_dtype) {
    EA_REQUIRE_CTX(c);
    bool far = false;
    for (int i = 0; i < jobs.n; ++i) far = far || jobs.j[i].stride_k < 0 || (K >> 4) * jobs.j[i].stride_k >= (1ll << 29);
    // the rotation inside the products while its blocks fit the GPU at once (or the rows one block), a launch of its own
    // above: the shared expert's gate|up (6144 x 256, two jobs) at 64 rows 14.5 -> 11.3 us, 6144 x 2048 at 64 rows 17.2
    // with the launch and 17.8 without
    int blocks = 0;
    for (int i = 0; i < jobs.n; ++i) blocks += jobs.j[i].SK > 1 ? jobs.j[i].N / 64 * jobs.j[i].SK : jobs.j[i].N / 128;
    bool fuse = rot && !far && (M <= LR_ROT_ROWS || blocks * ((M + LR_ROT_ROWS - 1) / LR_ROT_ROWS) <= c->cus) && (x_dtype == F16 || x_dtype == BF16) &&
                (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    // and x is left alone meanwhile (an output, or xh, in its place: the rotation is done before the products start then)
    const uint64_t xa = reinterpret_cast<uintptr_t>(x);
    for (int i = 0; fuse && i < jobs.n; ++i) {
        const ea_job& j = jobs.j[i];
        const size_t xb = (size_t)M * K * 2, yb = (size_t)M * j.N * (j.y_dtype == F32 ? 4 : 2);
        fuse = K / j.SK % 128 == 0 && (rot->suh[i] & 15) == 0 && (rot->xh[i] & 15) == 0 && !overlap(xa, xb, j.y, yb) &&
               !overlap(xa, xb, rot->xh[i], xb);
    }
    if (rot && !fuse) {
        const int r = launch_lin_rot_in(s, x, x_dtype, rot, (uint32_t)jobs.n, (uint32_t)M, (uint32_t)K);
        if (r) return r;
    }
    // jobs of one split finish in their blocks; the others' sums meet in Z
    for (int split = 0; split < 2; ++split) {
        ea_jobs sj{};
        ea_rot_jobs rj{};
        for (int i = 0; i < jobs.n; ++i)
            if ((jobs.j[i].SK > 1) == (split == 1)) {
                if (fuse) {
                    rj.suh[sj.n] = rot->suh[i];
                    rj.xh[sj.n] = rot->xh[i];
                }
                sj.j[sj.n++] = jobs.j[i];
            }
        if (sj.n == 0) continue;
#define EA_LV(K2_, CB_)                                                                               \
    if (k2 == K2_ && cb == CB_) {                                                                     \
        if (split) launch_rows_k2<CB_, K2_, 2>(s, sj, rj, fuse, far, M, K, x, x_dtype == BF16, c->cus);    \
        else launch_rows_k2<CB_, K2_, 4>(s, sj, rj, fuse, far, M, K, x, x_dtype == BF16, c->cus);          \
    }
        EA_LV(10, 2) EA_LV(12, 2) EA_LV(8, 1) EA_LV(8, 2) EA_LV(6, 1) EA_LV(4, 1)
#undef EA_LV
        int r = launched();
        if (r) return r;
        if (split) {
            int nb = 0;
            for (int i = 0; i < sj.n; ++i) {
                sj.j[i].start = nb;
                nb += sj.j[i].N >> 7;
            }
            lin_finish_kernel<<<dim3((unsigned)nb, (unsigned)((M + 3) / 4)), 256, 0, s>>>(sj, M);
            r = launched();
            if (r) return r;
        }
    }
    return EA_OK;
}

}  // namespace ea
