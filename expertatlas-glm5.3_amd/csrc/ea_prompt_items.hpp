// The item lists of a prompt pass (ea_prompt.hip): the gate|up and down products of items of one expert's routed pairs,
// and one list's launches. Included by the sources that instantiate it for widths up to 10 and up to 16.
#pragma once

#include <hip/hip_runtime.h>

#include "ea_device.hpp"
#include "ea_experts.hpp"
#include "ea_gemm.hpp"
#include "ea_host.hpp"

namespace ea {

// Routed pairs an item at most: five row tiles. The reference's items hold up to 112 (prompt_experts.cu:55-58,
// TF_PE_GPM). 80 against 48: the same at 512 rows and 3-4 % faster at 2048 (a heavy expert decoded in fewer items);
// against 112 (seven row tiles, more accumulators) faster at both; 64 and 96 measured between. A pair's sums do not
// depend on its item.
constexpr int IPM = 80;
constexpr int IPM_TILES = IPM / 16;

constexpr int SMALL_ROWS = 16;     // items of at most this many pairs: the kernels holding one row tile

// Item i of list `big` (0: items of at most SMALL_ROWS pairs, from the front of items[]; 1: the others, from its
// back), or false past the list's count.
__device__ __forceinline__ bool item_at(const int* __restrict__ items, const int* __restrict__ count, int big,
                                        int max_items, int i, int& e, int& first, int& cnt) {
    if (i >= count[big]) return false;
    const int at = big ? max_items - 1 - i : i;
    e = items[3 * at];
    first = items[3 * at + 1];
    cnt = items[3 * at + 2];
    return true;
}

// ---- the pair plane -----------------------------------------------------------------------------------------------

// Where the down products go: fp32 [pairs, D] rows of one plane, or (a scratch without a plane) each pair's row split in
// two halves of D / 2 columns over the pair's own rotated inputs, which the pair's gate|up product has read by then: the
// lower columns in its xg row, the upper in its xu row (D fp16 = D / 2 fp32 each). The item lists run side by side, but a
// pair's rows belong to one list, whose gate|up precedes its down product on one stream. Column col of pair p is at
// base(col)[p * stride + col].
struct PairPlane {
    float *lo, *hi;  // hi already moved back by half columns
    int half, stride;
    __host__ __device__ float* base(int col) const { return col < half ? lo : hi; }
};

// ---- the staged item GEMM --------------------------------------------------------------------------------------
// Every kernel is built for widths up to MK: 10 (two trellis words a lane a tile), or 16 (three words above 10, larger
// staging regions) for layers that hold a wider expert.

constexpr int PK = 8;                             // k tiles a chunk: 128 k
constexpr int PXS = PK * 16 + 8;                  // LDS row stride of a staged activation chunk, halves (272 bytes)
constexpr int PW = 4;                             // waves a block: 8 column tiles, 128 columns
constexpr int pstage(int mk) { return PK * 2 * 4 * mk; }  // a wave's staged trellis words a chunk
constexpr int DNG = 16;  // down matrix: column blocks of 128 a block, small items (8, 24 and 48 measured slower at 512 rows)
// the same in a decode window, whose items are too few to fill the GPU with blocks that long (37 rows, 112 experts: 336
// blocks of 16 column blocks took 71 us, 1,344 of 4 take 39; passes of 129 to 511 rows were not measured with 4)
constexpr int DNG_WINDOW = 4;
constexpr int WINDOW_ROWS_MAX = 128;  // the widest decode window (forward.zig:21)
constexpr int DNG_BIG = 2;  // the same for the larger items: more blocks for fewer items (4: 1 % slower at 512 rows)
constexpr int DNG_BIG_LONG = 4;   // passes of more than LONG_ROWS rows: 1.5 % faster at 2048 rows
constexpr int LONG_ROWS = 1024;
// Up to these rows a pass, and this much work (pairs x intermediate width, which follows the blocks there are), the larger
// items' gate|up stages its activations in two buffers (two blocks a CU), above either in one (three or four). 300 rows of 8
// slots over 256 experts of width 256: 254 us with two and 282 with one, 512 rows 306 and 315, 640 rows 351 and 347, 1024 rows
// 447 and 423: few blocks wait on each chunk's round trip, many on each other for a place. Width 512: 129 rows 394 and 416,
// 200 rows 432 and 430, 300 rows 471 and 456, 512 rows 528 and 514. (Picks that spread evenly make more of the items large:
// 512 rows of width 256 then take 333 and 310 us.)
constexpr int MID_ROWS = 600;
constexpr int64_t MID_WORK = 512 * 8 * 256;
// Above this work the one-buffer kernel gives up its reads ahead for a fourth wave a SIMD: 640 rows of width 256 354 us without
// and 366 with it, 1024 rows 435 and 440; width 512, 800 rows 650 and 619, 4096 rows 1,836 and 1,772.
constexpr int64_t DENSE_WORK = 1024 * 8 * 256;
static bool two_buffers(int rows, int pairs, int width) { return rows <= MID_ROWS && (int64_t)pairs * width <= MID_WORK; }
constexpr int GU_SPLIT = 2;                       // K splits of a larger item's gate|up (4 and 8 measured slower)
// The number of K splits of an item's gate|up over K (at most one a chunk). A layer that holds a width above 10 keeps one sum
// over all of K in ascending order, the order of the sums it has always had; two splits would round its outputs differently
// (2e-4 of them, after the bf16 rounding). 5, 6 and 8 bits with one / two: windows of 37 / 128 rows 172 / 146 and 206 / 192 us,
// prompts of 512, 777 and 2048 rows 368 / 375, 428 / 430 and 752 / 721.
static int gu_splits(int K, bool wide = false) {
    return wide ? 1 : K / (PK * 16) < GU_SPLIT ? K / (PK * 16) : GU_SPLIT;
}
constexpr int DXS = 2 * PK * 16 + 8;              // down matrix: LDS row stride of the activations (K up to 256)

// One chunk (PK k tiles) of a wave: its two column tiles times the item's first mts (<= MT) row tiles. The trellis
// words are staged in st (tile (t, j) at word (2 t + j) * 4 K2), the activations in xa (row stride xs halves, laid
// out by put_a); each tile pair decodes once and feeds all row tiles.
template <int CB, int K2, int MT>
__device__ __forceinline__ void item_chunk(const uint32_t* st, const TileLane<K2, CB>& tl, const uint16_t* xa, int mts,
                                           int lane, f4v (&acc)[MT][2], int xs) {
    constexpr int TW = 4 * K2, NWD = TileLane<K2, CB>::NW;
    const uint16_t* xr = xa + (lane & 15) * xs + 8 * ((lane >> 4) & 3);
#pragma unroll
    for (int t = 0; t < PK; t += 2) {
        h8v bb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t w[2][NWD], s[8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                tl.staged(st + (2 * (t + h) + j) * TW, w[h]);
                tl.states(w[h], s + 4 * h);
            }
            // pair by pair: with the accumulators of several row tiles, eight states at once cost registers
            bb[j] = __builtin_bit_cast(h8v, (u4v{cb_pair<CB>(s[0], s[1]), cb_pair<CB>(s[2], s[3]),
                                                 cb_pair<CB>(s[4], s[5]), cb_pair<CB>(s[6], s[7])}));
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt >= mts) break;  // the item's occupied row tiles only (uniform)
            const h8v a = *reinterpret_cast<const h8v*>(xr + mt * 16 * xs + t * 16);
            acc[mt][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bb[0], acc[mt][0], 0, 0, 0);
            acc[mt][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bb[1], acc[mt][1], 0, 0, 0);
        }
    }
}

// One chunk for a single row tile with the LDS reads one k step ahead: the trellis words and the activation operand
// of k step t + 1 are read before k step t decodes, so each read's latency overlaps a step of decoding.
template <int CB, int K2>
__device__ __forceinline__ void item_chunk1(const uint32_t* st, const TileLane<K2, CB>& tl, const uint16_t* xa, int lane,
                                            f4v (&acc)[1][2], int xs) {
    constexpr int TW = 4 * K2, NWD = TileLane<K2, CB>::NW;
    const uint16_t* xr = xa + (lane & 15) * xs + 8 * ((lane >> 4) & 3);
    uint32_t w[2][4][NWD];  // [buffer][tile: (t, j0), (t + 1, j0), (t, j1), (t + 1, j1)][word]
    h8v a[2];
    auto read = [&](int t, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) tl.staged(st + (2 * (t + h) + j) * TW, w[b][2 * j + h]);
        a[b] = *reinterpret_cast<const h8v*>(xr + t * 16);
    };
    read(0, 0);
#pragma unroll
    for (int t = 0; t < PK; t += 2) {
        const int b = (t >> 1) & 1;
        if (t + 2 < PK) read(t + 2, b ^ 1);
        issued();
        h8v bb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            bb[j] = __builtin_bit_cast(h8v, tl.decode2(w[b][2 * j], w[b][2 * j + 1]));
        }
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b], bb[0], acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b], bb[1], acc[0][1], 0, 0, 0);
    }
}

// The same with the LDS reads ahead: the next k step's trellis words are read before this step decodes, and a row tile's
// activations before the products of the one before. Costs registers that the rotating kernel does not have.
template <int CB, int K2, int MT>
__device__ __forceinline__ void item_chunk_ahead(const uint32_t* st, const TileLane<K2, CB>& tl, const uint16_t* xa,
                                                 int mts, int lane, f4v (&acc)[MT][2]) {
    constexpr int TW = 4 * K2, NWD = TileLane<K2, CB>::NW;
    const uint16_t* xr = xa + (lane & 15) * PXS + 8 * ((lane >> 4) & 3);
    uint32_t w[2][2][2][NWD];  // [buffer][column tile][k tile][word]
    auto read = [&](int t, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) tl.staged(st + (2 * (t + h) + j) * TW, w[b][j][h]);
    };
    read(0, 0);
#pragma unroll
    for (int t = 0; t < PK; t += 2) {
        const int b = (t >> 1) & 1;
        h8v a = *reinterpret_cast<const h8v*>(xr + t * 16);
        if (t + 2 < PK) read(t + 2, b ^ 1);
        issued();
        h8v bb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) bb[j] = __builtin_bit_cast(h8v, tl.decode2(w[b][j][0], w[b][j][1]));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt >= mts) break;  // the item's occupied row tiles only (uniform)
            const h8v an = *reinterpret_cast<const h8v*>(xr + (mt + 1 < MT ? mt + 1 : mt) * 16 * PXS + t * 16);
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bb[j], acc[mt][j], 0, 0, 0);
            a = an;
        }
    }
}

// Where a gate|up block's activations come from: rotated already (fp16 [pairs, K], a buffer over them), or the raw rows
// (16-bit, a buffer over them, with the expert's suh row) that the block rotates while staging them.
struct GuSrc {
    __amdgpu_buffer_rsrc_t x, suh;
    int bf16;
};

// The chunk loop of a gate|up block for one width. With TWO activation buffers they are staged for the block's waves a
// chunk ahead: a step stores (ROT: rotates and stores) the next chunk's and issues the loads of the one after, computes
// its own, and meets the other waves once. With one, two barriers a chunk (MID_ROWS says which; above width 10, whose
// staging regions are larger, always one: 777 rows 428 us, with two 437). The trellis is loaded two chunks ahead into the wave's own region. Loads
// complete in issue order and every load is issued (a chunk past the last re-reads the last), so the waits stay exact.
// Thread tid's piece i of a chunk is row (i NT + tid) / 16; aoff: its byte offset in the source.
template <int CB, int K2, int MT, int NT, bool ROT, bool TWO, bool DENSE>
__device__ __forceinline__ void gu_loop(const GuSrc& src, const uint32_t (&aoff)[(MT * 256 + NT - 1) / NT],
                                        const TileSpan& sp, uint16_t* xa, uint32_t* st, int lane, int rows, int mts,
                                        int c0, int nch, f4v (&acc)[MT][2]) {
        constexpr int NL = stage_loads_k<PK, K2>(), NP = (MT * 256 + NT - 1) / NT, BUF = MT * 16 * PXS;
    const TileLane<K2, CB> tl(lane);
    const int row0 = (int)threadIdx.x >> 4, q8 = ROT ? h8_group(lane) : lane & 15;
    u4v av[NP], sv = u4v{0u, 0u, 0u, 0u}, ta[NL], tb[NL];
    auto issue_a = [&](int c) __attribute__((always_inline)) {
        c = c0 + (c < nch ? c : nch - 1);
#pragma unroll
        for (int i = 0; i < NP; ++i)
            av[i] = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(src.x, aoff[i], c * PK * 32, 0));
        if constexpr (ROT)
            sv = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(src.suh, q8 * 16, c * PK * 32, 0));
    };
    auto issue_t = [&](int c, u4v (&tv)[NL]) __attribute__((always_inline)) {
        c = c0 + (c < nch ? c : nch - 1);
        TileSpan sc = sp;
        sc.off = sp.off + c * PK * sp.kstride;
        stage_issue_k<PK, K2>(sc, lane, tv);
    };
    auto put = [&](uint16_t* buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int row = i * (NT / 16) + row0;
            if (row >= rows) continue;  // uniform over a wave (rows % 16 == 0)
            u4v v = av[i];
            if constexpr (ROT) v = rot8(v, sv, src.bf16, lane);
            put_a(buf + row * PXS, q8, v);
        }
    };
    auto step = [&](int c, u4v (&tv)[NL], int b) __attribute__((always_inline)) {
        if constexpr (TWO) {
            stage_store_k<PK, K2>(st, lane, tv);  // only this wave reads its region, in order
            put(xa + (b ^ 1) * BUF);              // the chunk before the one in that buffer was read before the barrier
            issue_t(c + 2, tv);
            issue_a(c + 2);
            if constexpr (ROT) item_chunk<CB, K2, MT>(st, tl, xa + b * BUF, mts, lane, acc, PXS);
            else item_chunk_ahead<CB, K2, MT>(st, tl, xa + b * BUF, mts, lane, acc);
            __syncthreads();
        } else {
            __syncthreads();  // the previous chunk's reads of xa are done
            put(xa);
            stage_store_k<PK, K2>(st, lane, tv);
            issue_a(c + 1);
            issue_t(c + 2, tv);
            __syncthreads();
            if constexpr (DENSE) item_chunk<CB, K2, MT>(st, tl, xa, mts, lane, acc, PXS);
            else item_chunk_ahead<CB, K2, MT>(st, tl, xa, mts, lane, acc);
        }
    };
    if constexpr (TWO) {
        issue_a(0);
        issue_t(0, ta);
        put(xa);
        issue_a(1);
        issue_t(1, tb);
        __syncthreads();
    } else {
        issue_t(0, ta);
        issue_t(1, tb);
        issue_a(0);
    }
    // two steps an iteration with no exit between them, so every load's wait is counted the same on each pass
    int c = 0;
    for (; c + 1 < nch; c += 2) {
        step(c, ta, 0);
        step(c + 1, tb, 1);
    }
    if (c < nch) step(c, ta, 0);  // uniform
}

// Block b of a launch over (items, C column blocks, Z slices) in XCD order. Blocks are dispatched to the 8 XCDs in
// turn (block b on XCD b mod 8); group g = item Z + slice takes blocks on XCD g mod 8 for all C of its column blocks
// (the item's activations of the slice come into that XCD's L2 once), and slice z of an expert's consecutive items
// lands on the XCDs (i Z + z) mod 8, 8 / gcd(Z, 8) of them (two for Z = 4 or 12), whose L2s then hold its trellis
// for the expert's later items. 2048 rows: 719 -> 691 us a layer (item order: a slice's blocks on all 8 XCDs, each
// fetching the slice). Blocks: ceil(items Z / 8) 8 C, those past the list's count return at once.
__device__ __forceinline__ void xcd_order(int b, int C, int Z, int& item, int& cb, int& z) {
    const int q = b >> 3;
    cb = q % C;
    const int g = (q / C) * 8 + (b & 7);
    item = g / Z;
    z = g % Z;
}
static unsigned xcd_blocks(int items, int C, int Z) { return (unsigned)((items * Z + 7) / 8 * 8 * C); }

// Block (item of the larger items' list, 32 WB columns, (matrix, K split)), in XCD order: the item's rows (up to IPM_TILES
// row tiles) times its expert's matrix over split s of K's chunks of 128 (splits [s nch / nsplit, (s + 1) nch / nsplit)).
// A chunk's activations go to LDS once for the block's WB waves; each wave's two column tiles of the chunk come in as
// 16-byte loads staged in the wave's own LDS region. Only the item's occupied row tiles are staged and multiplied; rows
// past the item's count repeat the item's first pair and are not stored (MFMA rows do not mix). Split 0 goes to
// Z[mat][pair][n], split s > 0 to Zp[s - 1][mat][pair][n] (fp32), each accumulated from zero (stored as 0 + sum).
// ROT (WB 8, so that one block covers a rank's 256 columns): X0 is x [rows, K] (16-bit, x_stride apart) and suh0 / suh1
// the stacked scales; the block rotates its rows as rot_in_kernel does, same bits. A pass over the larger items is bound
// by memory (2048 rows: 3.8 TB/s of the 5.2 a copy reaches), and the rotated pairs were a quarter of its bytes.
// DENSE (one buffer): no reads ahead, so that four waves fit a SIMD instead of three.
template <int CB, int MK, bool ROT, bool TWO, int WB, bool DENSE>
__global__ void __launch_bounds__(WB * 64) __attribute__((amdgpu_waves_per_eu(ROT || DENSE ? 4 : 2)))
item_gu_kernel(const void* __restrict__ X0, const void* __restrict__ X1, const int64_t* __restrict__ TP0,
               const int64_t* __restrict__ TP1, const int* __restrict__ K2_0, const int* __restrict__ K2_1,
               const int* __restrict__ sorted, const int* __restrict__ items, const int* __restrict__ item_count,
               float* __restrict__ Z, float* __restrict__ Zp, int K, int N, int P, int nsplit, int mats, int max_items,
               int* __restrict__ status, const uint16_t* __restrict__ suh0, const uint16_t* __restrict__ suh1, int x_bf16,
               int x_stride, int slots) {
    constexpr int MT = IPM_TILES, NT = WB * 64, NP = (MT * 256 + NT - 1) / NT;
    int e, first, cnt;
    int item, cb, zs;
    xcd_order((int)blockIdx.x, N / (32 * WB), mats * nsplit, item, cb, zs);
    if (!item_at(items, item_count, 1, max_items, item, e, first, cnt)) return;
    const int mat = zs / nsplit, split = zs % nsplit;
    const uint32_t* T = reinterpret_cast<const uint32_t*>(mat ? TP1[e] : TP0[e]);
    const int k2 = mat ? K2_1[e] : K2_0[e];
    // the wave index in a scalar register: the trellis offsets built from it are then scalar (a buffer load's soffset)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ int pair_sh[MT * 16];
    __shared__ __attribute__((aligned(16))) uint16_t xa[(TWO ? 2 : 1) * MT * 16 * PXS];
    __shared__ __attribute__((aligned(16))) uint32_t st[WB][pstage(MK)];
    if (tid < MT * 16) pair_sh[tid] = tid < cnt ? sorted[first + tid] : -1;
    __syncthreads();
    // a piece past the item's row tiles reads a row of the first one (a cache hit) and is not stored
    const int mts = (cnt + 15) >> 4, rows = mts * 16;
    uint32_t aoff[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int row = (i * NT + tid) >> 4, rr = row < rows ? row : row & 15;
        const int p = pair_sh[rr] >= 0 ? pair_sh[rr] : pair_sh[0];
        aoff[i] = ROT ? ((uint32_t)(p / slots) * (uint32_t)x_stride + 8u * (uint32_t)h8_group(lane)) * 2u
                      : ((uint32_t)p * (uint32_t)K + 8u * (tid & 15)) * 2u;
    }
    GuSrc src;
    src.bf16 = x_bf16;
    if constexpr (ROT) {
        src.x = buffer_rsrc(X0, (uint32_t)(((size_t)(P / slots - 1) * x_stride + K) * 2));
        src.suh = buffer_rsrc((mat ? suh1 : suh0) + (size_t)e * K, (uint32_t)K * 2u);
    } else {
        src.x = src.suh = buffer_rsrc(mat ? X1 : X0, (uint32_t)((size_t)P * K * 2));
    }
    const int nt0 = cb * (2 * WB) + 2 * wave;
    const int ns = N >> 4, TWB = 16 * k2;
    TileSpan sp;
    sp.r = buffer_rsrc(T, (uint32_t)((K >> 4) * ns * TWB));
    sp.off = nt0 * TWB;
    sp.kstride = ns * TWB;
    f4v acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = f4v{0.f, 0.f, 0.f, 0.f};
    const int nch = K / (PK * 16);
    const int c0 = split * nch / nsplit, nc = (split + 1) * nch / nsplit - c0;  // nsplit <= nch: nc >= 1
    const bool ok = EA_K2_SWITCH(
        k2, 2, MK, (gu_loop<CB, K2V, MT, NT, ROT, TWO, DENSE>(src, aoff, sp, xa, st[wave], lane, rows, mts, c0, nc, acc)));
    if (!ok) {
        if (lane == 0) record_error(status, DEV_UNSUPPORTED_WIDTH);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = nan4();
    }
    float* Zm = (split ? Zp + (size_t)(split - 1) * 2 * P * N : Z) + (size_t)mat * P * N;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = pair_sh[mt * 16 + 4 * (lane >> 4) + i];
            if (p < 0) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) Zm[(size_t)p * N + (nt0 + j) * 16 + (lane & 15)] = 0.f + acc[mt][j][i];
        }
}

// Items of at most 16 pairs: a block is NW waves, one a column-tile pair of one matrix, over all of K. The block's
// waves share each chunk of activations through a ring of RING_S chunk slots in LDS, filled and freed with LDS
// counters instead of barriers, so a wave can run up to RING_S - RING_L - 1 chunks ahead of the slowest:
//   filled[s]: pieces stored into slot s, over all the chunks it has held (NW a chunk);
//   done[s]:   waves that have finished a chunk of slot s, over all its chunks (NW a chunk).
// At its step c a wave stores its piece of chunk p = c + RING_L into slot p % RING_S once every wave is done with
// that slot's previous chunk (done >= NW (p / RING_S)), waits until chunk c is complete in its slot
// (filled >= NW (c / RING_S + 1)), computes it, and counts itself done. The slowest wave can always go on (every
// chunk it waits for was stored at a step no later than its own, and every slot it stores into was freed before),
// so every wait ends. Each wave's trellis goes through its own LDS region as in gu_loop; the activation piece of a
// chunk (1/NW of it) and the trellis are loaded two chunks ahead. K is split as the larger items' is, over the same
// chunk ranges and into the same planes, so a pair's sums do not depend on which list its item is in. (Decode windows
// are bound by the waves there are, not by their work: 37 rows touch about 112 experts, and one block an (item, 128
// columns, matrix) over all of K left 1.75 blocks a CU: 118 us, against 67 with the
// two splits. Prompts of 512 and 2048 rows measured the same either way.)
constexpr int RING_S = 6;  // activation chunk slots
constexpr int RING_L = 2;  // a wave stores its piece of chunk c + RING_L at its step c

template <int NW>
struct RingPiece {  // a lane's words of a chunk: 16 rows x 64 words over NW waves
    static constexpr int WORDS = 16 * 64 / (NW * 64);
};

__device__ __forceinline__ int lds_load_acquire(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// One count for the whole wave: only its first lane adds (the wait before the add covers every lane's accesses).
__device__ __forceinline__ void lds_add_release(int* p, int v, int lane) {
    if (lane == 0) __hip_atomic_fetch_add(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Wait until *p >= target. Every count waited for is reached (see above); the wait is still bounded (about 2^20
// sleeps, tens of milliseconds): past the bound it gives up, returns false and the kernel reports EA_SYNC_TIMEOUT.
__device__ __forceinline__ bool lds_wait_geq(const int* p, int target) {
    for (int n = 0; lds_load_acquire(p) < target; ++n) {
        if (n >= (1 << 20)) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

template <int CB, int K2, int NW>
__device__ __forceinline__ void ring_loop(__amdgpu_buffer_rsrc_t xrs, uint32_t aoff, int lofs, const TileSpan& sp,
                                          uint16_t* ring, int* filled, int* done, uint32_t* st, int lane, int c0,
                                          int nch, f4v (&acc)[1][2], bool& synced) {
    constexpr int NL = stage_loads_k<PK, K2>();
    constexpr int W = RingPiece<NW>::WORDS;  // 2 or 4
    constexpr int SLOT = 16 * PXS;
    using pv = uint32_t __attribute__((ext_vector_type(W)));
    const TileLane<K2, CB> tl(lane);
    pv pa, pb;
    u4v ta[NL], tb[NL];
    auto issue_p = [&](int c, pv& v) __attribute__((always_inline)) {
        c = c0 + (c < nch ? c : nch - 1);
        if constexpr (W == 4)
            v = __builtin_bit_cast(pv, __builtin_amdgcn_raw_buffer_load_b128(xrs, aoff, c * PK * 32, 0));
        else
            v = __builtin_bit_cast(pv, __builtin_amdgcn_raw_buffer_load_b64(xrs, aoff, c * PK * 32, 0));
    };
    auto issue_t = [&](int c, u4v (&tv)[NL]) __attribute__((always_inline)) {
        c = c0 + (c < nch ? c : nch - 1);
        TileSpan sc = sp;
        sc.off = sp.off + c * PK * sp.kstride;
        stage_issue_k<PK, K2>(sc, lane, tv);
    };
    // the piece's words d .. d + W - 1 of its row (d = lofs & 63) at their transposed places (see put_a)
    auto put = [&](int p, const pv& v) __attribute__((always_inline)) {
        const int sl = p % RING_S;
        synced = synced && lds_wait_geq(&done[sl], NW * (p / RING_S));  // after a give-up no more waits
        uint32_t* w = reinterpret_cast<uint32_t*>(ring + sl * SLOT + (lofs >> 6) * PXS);
        const int d = lofs & 63;
#pragma unroll
        for (int r = 0; r < W; ++r) {
            const int dd = (d & 15) + r;  // word within its 32-k step
            w[16 * (d >> 4) + 4 * (dd & 3) + (dd >> 2)] = v[r];
        }
        lds_add_release(&filled[sl], 1, lane);
    };
    auto step = [&](int c, u4v (&tv)[NL], pv& v) __attribute__((always_inline)) {
        if (c + RING_L < nch) put(c + RING_L, v);  // uniform
        issue_p(c + RING_L + 2, v);
        stage_store_k<PK, K2>(st, lane, tv);
        issue_t(c + 2, tv);
        const int sl = c % RING_S;
        synced = synced && lds_wait_geq(&filled[sl], NW * (c / RING_S + 1));
        item_chunk1<CB, K2>(st, tl, ring + sl * SLOT, lane, acc, PXS);
        lds_add_release(&done[sl], 1, lane);  // after the chunk's reads of the slot have returned
    };
    // chunks 0 .. RING_L - 1 go in before the loop; pa / pb then carry chunks RING_L and RING_L + 1
    for (int p = 0; p < RING_L && p < nch; ++p) {
        pv v;
        issue_p(p, v);
        put(p, v);
    }
    issue_p(RING_L, pa);
    issue_t(0, ta);
    issue_p(RING_L + 1, pb);
    issue_t(1, tb);
    int c = 0;
    for (; c + 1 < nch; c += 2) {  // two steps an iteration with no exit between them
        step(c, ta, pa);
        step(c + 1, tb, pb);
    }
    if (c < nch) step(c, ta, pa);  // uniform
}

template <int CB, int MK, int NW>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(4)))
item_ring_kernel(const uint16_t* __restrict__ X0, const uint16_t* __restrict__ X1, const int64_t* __restrict__ TP0,
                 const int64_t* __restrict__ TP1, const int* __restrict__ K2_0, const int* __restrict__ K2_1,
                 const int* __restrict__ sorted, const int* __restrict__ items, const int* __restrict__ item_count,
                 float* __restrict__ Z, float* __restrict__ Zp, int K, int N, int P, int nsplit, int max_items,
                 int* __restrict__ status) {
    int e, first, cnt;
    if (!item_at(items, item_count, 0, max_items, blockIdx.x, e, first, cnt)) return;
    const int mat = blockIdx.z / nsplit, split = blockIdx.z % nsplit;
    const uint16_t* X = mat ? X1 : X0;
    const uint32_t* T = reinterpret_cast<const uint32_t*>(mat ? TP1[e] : TP0[e]);
    const int k2 = mat ? K2_1[e] : K2_0[e];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __shared__ int pair_sh[16];
    __shared__ int filled[RING_S], done[RING_S];
    __shared__ __attribute__((aligned(16))) uint16_t ring[RING_S * 16 * PXS];
    __shared__ __attribute__((aligned(16))) uint32_t st[NW][pstage(MK)];
    if (threadIdx.x < 16) pair_sh[threadIdx.x] = (int)threadIdx.x < cnt ? sorted[first + threadIdx.x] : -1;
    if (threadIdx.x < RING_S) filled[threadIdx.x] = done[threadIdx.x] = 0;
    __syncthreads();
    // this lane's piece of every chunk: words [d, d + W) of row r (word index lofs = 64 r + d over the chunk);
    // a row past the count reads the first pair's row
    constexpr int W = RingPiece<NW>::WORDS;
    const int lofs = (wave * 64 + lane) * W;
    const int row = lofs >> 6;
    const int p = pair_sh[row] >= 0 ? pair_sh[row] : pair_sh[0];
    const uint32_t aoff = ((uint32_t)p * (uint32_t)K + 2u * (uint32_t)(lofs & 63)) * 2u;
    const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(X, (uint32_t)((size_t)P * K * 2));
    const int nt0 = blockIdx.y * (2 * NW) + 2 * wave;
    const int ns = N >> 4, TWB = 16 * k2;
    TileSpan sp;
    sp.r = buffer_rsrc(T, (uint32_t)((K >> 4) * ns * TWB));
    sp.off = nt0 * TWB;
    sp.kstride = ns * TWB;
    f4v acc[1][2];
    acc[0][0] = acc[0][1] = f4v{0.f, 0.f, 0.f, 0.f};
    const int nch = K / (PK * 16);
    const int c0 = split * nch / nsplit, nc = (split + 1) * nch / nsplit - c0;  // nsplit <= nch: nc >= 1
    bool synced = true;
    const bool ok = EA_K2_SWITCH(k2, 2, MK,
                                 (ring_loop<CB, K2V, NW>(xrs, aoff, lofs, sp, ring, filled, done, st[wave], lane, c0,
                                                         nc, acc, synced)));
    if (!ok || !synced) {
        if (lane == 0) record_error(status, ok ? DEV_SYNC_TIMEOUT : DEV_UNSUPPORTED_WIDTH);
        acc[0][0] = acc[0][1] = nan4();
    }
    float* Zm = (split ? Zp + (size_t)(split - 1) * 2 * P * N : Z) + (size_t)mat * P * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int pp = pair_sh[4 * (lane >> 4) + i];
        if (pp < 0) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) Zm[(size_t)pp * N + (nt0 + j) * 16 + (lane & 15)] = 0.f + acc[0][j][i];
    }
}

// The small items' pairs rotated for the ring kernel, when the larger items' products rotate their own: block (item,
// matrix, 2048 columns), 16 lanes a 128-block (rot_in_kernel's arithmetic); the expert's suh is read once for the item's
// rows, eight rows' loads in flight. (2048 rows: 601 us a pass, against 617 with rot_in_kernel over all rows, its other
// pairs skipped.)
static __global__ void __launch_bounds__(256) item_rot_kernel(const uint16_t* __restrict__ x, int x_bf16, int x_stride,
                                                       const int* __restrict__ sorted, const int* __restrict__ items,
                                                       const int* __restrict__ item_count,
                                                       const uint16_t* __restrict__ suh0, const uint16_t* __restrict__ suh1,
                                                       uint16_t* __restrict__ out0, uint16_t* __restrict__ out1, int K,
                                                       int slots, int max_items) {
    int e, first, cnt;
    if (!item_at(items, item_count, 0, max_items, blockIdx.x, e, first, cnt)) return;
    const int lane = threadIdx.x & 63, k = blockIdx.z * 2048 + 128 * ((int)threadIdx.x >> 4) + 8 * h8_group(lane);
    if (k >= K) return;  // whole 16-lane groups (K % 128 == 0)
    const u4v sv = *reinterpret_cast<const u4v*>((blockIdx.y ? suh1 : suh0) + (size_t)e * K + k);
    uint16_t* out = blockIdx.y ? out1 : out0;
    constexpr int QB = 8;
    for (int i0 = 0; i0 < cnt; i0 += QB) {
        int p[QB];
        u4v xv[QB];
#pragma unroll
        for (int i = 0; i < QB; ++i) p[i] = sorted[first + (i0 + i < cnt ? i0 + i : i0)];
#pragma unroll
        for (int i = 0; i < QB; ++i) xv[i] = *reinterpret_cast<const u4v*>(x + (size_t)(p[i] / slots) * x_stride + k);
        issued();
#pragma unroll
        for (int i = 0; i < QB; ++i) {
            if (i0 + i >= cnt) break;  // uniform
            *reinterpret_cast<u4v*>(out + (size_t)p[i] * K + k) = rot8(xv[i], sv, x_bf16, lane);
        }
    }
}

// The column blocks of a down block for one width: step s is column block s / nch, chunk s % nch; the trellis two
// steps ahead; each column block's rows are stored when its last chunk is done.
template <int CB, int K2, int MT, int NG>
__device__ __forceinline__ void dn_loop(const TileSpan& sp, const uint16_t* xa, uint32_t* st, int lane, int wave,
                                        int mts, int nch, int nb0, const int* pair_sh, const PairPlane& plane) {
    constexpr int NL = stage_loads_k<PK, K2>();
    constexpr int TWB = 16 * K2;
    const TileLane<K2, CB> tl(lane);
    const int steps = NG * nch;  // even (NG even, or nch = 2: the caller's choice): two steps an iteration
    u4v ta[NL], tb[NL];
    f4v acc[MT][2];
    auto issue_t = [&](int s2, u4v (&tv)[NL]) __attribute__((always_inline)) {
        s2 = s2 < steps ? s2 : steps - 1;
        TileSpan sc = sp;
        sc.off = sp.off + (s2 / nch) * 8 * TWB + (s2 % nch) * PK * sp.kstride;
        stage_issue_k<PK, K2>(sc, lane, tv);
    };
    auto step = [&](int s2, u4v (&tv)[NL]) __attribute__((always_inline)) {
        const int c = s2 % nch;
        if (c == 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = f4v{0.f, 0.f, 0.f, 0.f};
        }
        stage_store_k<PK, K2>(st, lane, tv);  // only this wave reads its region, in order
        issue_t(s2 + 2, tv);
        item_chunk<CB, K2, MT>(st, tl, xa + c * PK * 16, mts, lane, acc, DXS);
        if (c == nch - 1) {
            const int nt0 = (nb0 + s2 / nch) * 8 + 2 * wave;
            float* Z = plane.base(nt0 * 16);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int p = pair_sh[mt * 16 + 4 * (lane >> 4) + i];
                    if (p < 0) continue;
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        Z[(size_t)p * plane.stride + (nt0 + j) * 16 + (lane & 15)] = acc[mt][j][i];
                }
        }
    };
    issue_t(0, ta);
    issue_t(1, tb);
    for (int s2 = 0; s2 < steps; s2 += 2) {  // steps = NG nch is even: two steps an iteration, no exit between
        step(s2, ta);
        step(s2 + 1, tb);
    }
}

// The down matrix (K = I of 128 or 256: one or two chunks): a block (item of list MT > 2, NG column blocks of 128)
// loads the item's activations for all of K into LDS once, then its waves run the column blocks independently. WB = 8
// (the larger items): two groups of four waves, each over NG / 2 of the column blocks, share one copy
// of the activations, so two blocks fit a CU's LDS at four waves a SIMD (four-wave blocks: three at three).
template <int CB, int MK, int MT, int NG, int WB = PW>
__global__ void __launch_bounds__(WB * 64) __attribute__((amdgpu_waves_per_eu(MT > 2 && WB == PW ? 2 : 4)))
item_dn_kernel(const uint16_t* __restrict__ X, const int64_t* __restrict__ TP, const int* __restrict__ K2T,
               const int* __restrict__ sorted, const int* __restrict__ items, const int* __restrict__ item_count,
               PairPlane plane, int K, int N, int P, int max_items, int* __restrict__ status) {
    int e, first, cnt;
    // the larger items' blocks in XCD order (a column group's slice of an expert on the same XCDs for all of the
    // expert's items); the small items' (one item an expert) item by item
    int item = blockIdx.x, grp = blockIdx.y;
    if constexpr (MT > 2) {
        int cb_unused;
        xcd_order((int)blockIdx.x, 1, N / 128 / NG, item, cb_unused, grp);
    }
    if (!item_at(items, item_count, MT > 2, max_items, item, e, first, cnt)) return;
    const uint32_t* T = reinterpret_cast<const uint32_t*>(TP[e]);
    const int k2 = K2T[e];
    // the wave index in a scalar register: the trellis offsets built from it are then scalar (a buffer load's soffset)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ int pair_sh[MT * 16];
    __shared__ __attribute__((aligned(16))) uint16_t xa[MT * 16 * DXS];
    static_assert(WB == PW || (WB == 2 * PW && NG % 2 == 0), "two wave groups: half the column blocks each");
    __shared__ __attribute__((aligned(16))) uint32_t st[WB][pstage(MK)];
    if (tid < MT * 16) pair_sh[tid] = tid < cnt ? sorted[first + tid] : -1;
    __syncthreads();
    const int mts = (cnt + 15) >> 4;
    const int nch = K / (PK * 16);  // 1 or 2
    {
        // 256 threads cover a chunk of a row tile; with eight waves each half of the block loads one chunk
        constexpr int CPT = WB == PW ? 2 : 1;  // chunks a thread loads
        const int lt = tid & 255, c0 = WB == PW ? 0 : tid >> 8;
        const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(X, (uint32_t)((size_t)P * K * 2));
        u4v av[CPT][MT];
#pragma unroll
        for (int q = 0; q < CPT; ++q)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int rr = i < mts ? i * 16 + (lt >> 4) : (lt >> 4);
                const int p = pair_sh[rr] >= 0 ? pair_sh[rr] : pair_sh[0];
                const int cc = c0 + q < nch ? c0 + q : 0;
                av[q][i] = __builtin_bit_cast(
                    u4v, __builtin_amdgcn_raw_buffer_load_b128(
                             xrs, ((uint32_t)p * (uint32_t)K + (uint32_t)(cc * PK * 16 + 8 * (lt & 15))) * 2u, 0, 0));
            }
#pragma unroll
        for (int q = 0; q < CPT; ++q)
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (c0 + q < nch && i < mts)
                    put_a(xa + (i * 16 + (lt >> 4)) * DXS + (c0 + q) * PK * 16, lt & 15, av[q][i]);
    }
    constexpr int NGW = WB == PW ? NG : NG / 2;  // column blocks a wave group runs
    const int ns = N >> 4, TWB = 16 * k2;
    const int w4 = wave & (PW - 1);
    const int nb0 = grp * NG + (wave / PW) * NGW;  // the wave group's first column block
    TileSpan sp;
    sp.r = buffer_rsrc(T, (uint32_t)((K >> 4) * ns * TWB));
    sp.off = (nb0 * 8 + 2 * w4) * TWB;
    sp.kstride = ns * TWB;
    __syncthreads();  // the activations are in LDS
    const bool ok = EA_K2_SWITCH(
        k2, 2, MK, (dn_loop<CB, K2V, MT, NGW>(sp, xa, st[wave], lane, w4, mts, nch, nb0, pair_sh, plane)));
    if (!ok) {  // no product ran: the item's outputs of the block's column blocks are NaN
        if (lane == 0) record_error(status, DEV_UNSUPPORTED_WIDTH);
        for (int g = 0; g < NGW; ++g)
            for (int i = 0; i < MT * 16; ++i) {
                const int p = pair_sh[i];
                if (p < 0) continue;
                const int o = (nb0 + g) * 128 + w4 * 32 + (lane & 31);
                plane.base(o)[(size_t)p * plane.stride + o] = __builtin_nanf("");
            }
    }
}

// What one item list's pass reads and writes: the rotated activations, the three matrices' trellis tables and
// widths, the items, the pair classes and the per-pair planes (z and zp: gate|up partial sums, xd: down inputs,
// plane: down outputs). The two lists' pairs are disjoint, so their passes touch disjoint rows of every plane.
struct ListPass {
    const void* x;  // the pass's rows, and how they lie
    int x_dtype, x_stride;
    bool fuse;      // the larger items' products rotate x themselves (rotate_fits); only the small items' pairs go through xg / xu
    const uint16_t *suh_g, *suh_u;
    uint16_t *xg, *xu;
    const int64_t* tp[3];
    const int* k2[3];
    const int *sorted, *items, *count, *pclass, *pick;
    const uint16_t *svh_g, *svh_u, *suh_d;
    float *z, *zp;
    PairPlane plane;
    uint16_t* xd;
    int D, I, P, rows, slots, E, mi;
    int* status;
};

// Whether the larger items' products can rotate x themselves: 16-bit rows on 16-byte boundaries within 32-bit offsets, and
// one block over all of a matrix's columns (two would rotate twice).
static bool rotate_fits(const void* x, int x_dtype, uint32_t x_stride, const uint16_t* suh_g, const uint16_t* suh_u,
                        uint32_t rows, uint32_t I) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(suh_g) |
                         reinterpret_cast<uintptr_t>(suh_u) | (uintptr_t)x_stride * 2;
    return I == 256 && (x_dtype == F16 || x_dtype == BF16) && (at & 15) == 0 && (uint64_t)rows * x_stride * 2 < (1ull << 32);
}

// One item list from its gate|up product to its down product, in order on q: big = 1 takes the larger items (the
// gate|up K split into zp; the down matrix by blocks of DNG_BIG column blocks), big = 0 the items of at most
// SMALL_ROWS pairs (the ring kernel; DNG column blocks). The down matrix takes the resident-activation kernel when
// its K and N fit, the chunked ones otherwise. The two lists run on two streams: the small items' blocks leave room
// on many CUs, the larger items' blocks are few and long, and each list's down product starts when its own
// epilogue is done.
template <int CB, int MK>
static int list_pass(hipStream_t q, const ListPass& a, int big) {
    const int ns = gu_splits(a.D, MK > 10);
    const bool dense = (int64_t)a.P * a.I > DENSE_WORK;
#define EA_GU(ROT_, TWO_, WB_, DENSE_, X0_, X1_)                                                                                \
    item_gu_kernel<CB, MK, ROT_, TWO_, WB_, DENSE_><<<xcd_blocks(a.mi, a.I / (32 * (WB_)), 2 * ns), (WB_) * 64, 0, q>>>(             \
        X0_, X1_, a.tp[0], a.tp[1], a.k2[0], a.k2[1], a.sorted, a.items, a.count, a.z, a.zp, a.D, a.I, a.P, ns, 2, a.mi, \
        a.status, a.suh_g, a.suh_u, a.x_dtype == BF16, a.x_stride, a.slots)
    if (big && a.fuse) {
        if constexpr (MK <= 10) EA_GU(true, true, 8, false, a.x, a.x);  // fuse is for these widths only (ea_prompt_experts_run)
    } else if (big && (MK > 10 || !two_buffers(a.rows, a.P, a.I))) {
        if (MK <= 10 && dense) EA_GU(false, false, 4, MK <= 10, a.xg, a.xu);
        else EA_GU(false, false, 4, false, a.xg, a.xu);
    } else if (big) {
        if constexpr (MK <= 10) EA_GU(false, true, 4, false, a.xg, a.xu);
    } else {
        if (a.fuse) {  // the small items' pairs, on their own stream
            item_rot_kernel<<<dim3(a.mi, 2, (a.D + 2047) / 2048), 256, 0, q>>>(
                static_cast<const uint16_t*>(a.x), a.x_dtype == BF16, a.x_stride, a.sorted, a.items, a.count, a.suh_g,
                a.suh_u, a.xg, a.xu, a.D, a.slots, a.mi);
            const int r = launched();
            if (r) return r;
        }
        // blocks of 4 waves over 128 columns (8 waves over 256 measured 1 % slower at 512 rows, the same at 2048)
        item_ring_kernel<CB, MK, 4><<<dim3(a.mi, a.I / 128, 2 * ns), 4 * 64, 0, q>>>(
            a.xg, a.xu, a.tp[0], a.tp[1], a.k2[0], a.k2[1], a.sorted, a.items, a.count, a.z, a.zp, a.D, a.I, a.P, ns,
            a.mi, a.status);
    }
#undef EA_GU
    int r = launched();
    if (r) return r;
    r = launch_gateup_epilogue(q, a.z, a.pick, a.svh_g, a.svh_u, a.suh_d, a.xd, (uint32_t)a.rows, (uint32_t)a.P,
                               (uint32_t)a.I, (uint32_t)ns, (uint32_t)a.slots, (uint32_t)a.E, __builtin_inff(), 1, a.zp, a.pclass,
                               big);
    if (r) return r;
    const int nb = a.D / 128;
    if (a.I <= 2 * PK * 16 && nb % 2 == 0) {
#define EA_DN(MT_, NG_, WB_, grid)                                                                                    \
    item_dn_kernel<CB, MK, MT_, NG_, WB_><<<grid, (WB_) * 64, 0, q>>>(a.xd, a.tp[2], a.k2[2], a.sorted, a.items, a.count,  \
                                                                  a.plane, a.I, a.D, a.P, a.mi, a.status)
        if (big && a.rows > LONG_ROWS && nb % DNG_BIG_LONG == 0)
            EA_DN(IPM_TILES, DNG_BIG_LONG, 2 * PW, xcd_blocks(a.mi, 1, nb / DNG_BIG_LONG));
        else if (big && a.I == 2 * PK * 16)  // two chunks of K: a wave group's one column block is an even step count
            EA_DN(IPM_TILES, DNG_BIG, 2 * PW, xcd_blocks(a.mi, 1, nb / DNG_BIG));
        else if (big)
            EA_DN(IPM_TILES, DNG_BIG, PW, xcd_blocks(a.mi, 1, nb / DNG_BIG));
        else if (a.rows <= WINDOW_ROWS_MAX && nb % DNG_WINDOW == 0)
            EA_DN(SMALL_ROWS / 16, DNG_WINDOW, PW, dim3(a.mi, nb / DNG_WINDOW, 1));
        else if (nb % DNG == 0)
            EA_DN(SMALL_ROWS / 16, DNG, PW, dim3(a.mi, nb / DNG, 1));
        else
            EA_DN(SMALL_ROWS / 16, 2, PW, dim3(a.mi, nb / 2, 1));
#undef EA_DN
    } else if (big) {
        auto down = [&](auto kernel) {
            kernel<<<xcd_blocks(a.mi, a.D / 128, 1), 256, 0, q>>>(
                a.xd, a.xd, a.tp[2], a.tp[2], a.k2[2], a.k2[2], a.sorted, a.items, a.count, a.plane.lo, nullptr, a.I, a.D,
                a.P, 1, 1, a.mi, a.status, nullptr, nullptr, 0, 0, 1);
        };
        if (MK <= 10 && dense) down(item_gu_kernel<CB, MK, false, false, 4, MK <= 10>);
        else down(item_gu_kernel<CB, MK, false, false, 4, false>);
    } else {
        item_ring_kernel<CB, MK, 4><<<dim3(a.mi, a.D / 128, 1), 4 * 64, 0, q>>>(
            a.xd, a.xd, a.tp[2], a.tp[2], a.k2[2], a.k2[2], a.sorted, a.items, a.count, a.plane.lo, nullptr, a.I, a.D, a.P,
            1, a.mi, a.status);
    }
    return launched();
}

// The same for a layer with experts above width 10 (ea_prompt_wide.hip).
int list_pass_wide(hipStream_t q, const ListPass& a, int big, uint32_t cb);

}  // namespace ea
