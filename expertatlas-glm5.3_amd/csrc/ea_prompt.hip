// Routed experts of prompt chunks (hundreds to thousands of rows): route the pairs into items of at most IPM pairs
// of one expert, then per item one MFMA GEMM that decodes each trellis tile once for all of the item's rows
// (prompt_experts.cu / prompt_experts.zig of the reference give the interface and the item scheme).
//
// A pass over <= 4096 rows: route -> per-pair input rotation -> item GEMM gate|up -> gate/up epilogue -> item GEMM
// down -> down epilogue + slot-ordered combine (+ bf16 rounding). Every row's arithmetic is independent of which
// item or M-tile it lands in (MFMA rows do not mix), and the combine adds a row's slots in order, so the output is the
// same on every run. The down products go to a pair plane, or, in a scratch without one (planes 0, the reference's
// default), over the pairs' own rotated inputs: see PairPlane. (The reference adds each slot into out with atomics there;
// that form was bound by the atomics' rate, 320 G/s: 737 against 632 us at 2048 rows and 8 slots of 6144.)
#include <hip/hip_runtime.h>

#include "ea_prompt_items.hpp"

namespace ea {

constexpr uint32_t CHUNK_ROWS = 4096;  // rows a pass at most (prompt_experts.zig:17)
constexpr int ROUTE_THREADS = 1024;
constexpr int ROUTE_HELD = 16;  // picks a route thread holds in registers: 16,384 pairs (2,048 rows of 8 slots)

// One block: per-expert counts; exclusive scans over experts of the counts and of both lists' items; items
// (e, first, cnt <= ipm) of an expert in pair order, each into its list; sorted[] = pair ids grouped by expert (order
// within an expert: arrival); pclass[pair] = 1 when the pair's item is in the list of larger items. (prompt_experts.cu:
// 162-244 with by_count off; the two lists are this library's: they let a launch size its registers for its items'
// rows, and the larger items split K.)
__global__ void __launch_bounds__(ROUTE_THREADS) route_kernel(const int* __restrict__ pick, int n, int E,
                                                             int* __restrict__ sorted, int* __restrict__ items,
                                                             int* __restrict__ item_count, int* __restrict__ pclass,
                                                             int max_items, int ipm) {
    extern __shared__ int sh[];
    int* cnt = sh;          // [E]
    int* cur = sh + E;      // [E]
    int* start = sh + 2 * E;  // [E]
    __shared__ int wsum[ROUTE_THREADS / 64][3];
    for (int e = threadIdx.x; e < E; e += ROUTE_THREADS) cnt[e] = 0;
    // the first ROUTE_HELD * ROUTE_THREADS picks are loaded once, all loads in flight together, and held in
    // registers for both passes (a load then an atomic a pair waited for every load in turn); later ones are re-read
    int held[ROUTE_HELD];
#pragma unroll
    for (int j = 0; j < ROUTE_HELD; ++j) {
        const int i = j * ROUTE_THREADS + (int)threadIdx.x;
        held[j] = i < n ? pick[i] : -1;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ROUTE_HELD; ++j)
        if (held[j] >= 0 && held[j] < E) atomicAdd(&cnt[held[j]], 1);
    for (int i = ROUTE_HELD * ROUTE_THREADS + threadIdx.x; i < n; i += ROUTE_THREADS) {
        const int e = pick[i];
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    const int per = (E + ROUTE_THREADS - 1) / ROUTE_THREADS;
    const int e0 = threadIdx.x * per;
    int own[3] = {0, 0, 0};  // pairs, small items, large items of this thread's experts
    for (int q = 0; q < per; ++q) {
        const int e = e0 + q;
        if (e < E) {
            const int c = cnt[e], full = c / ipm, rem = c - full * ipm;
            own[0] += c;
            own[1] += rem > 0 && rem <= SMALL_ROWS;
            own[2] += full + (rem > SMALL_ROWS);
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc[3] = {own[0], own[1], own[2]};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            const int a = __shfl_up(inc[v], o, 64);
            if (lane >= o) inc[v] += a;
        }
    }
    if (lane == 63)
#pragma unroll
        for (int v = 0; v < 3; ++v) wsum[wave][v] = inc[v];
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            const int a = lane < ROUTE_THREADS / 64 ? wsum[lane][v] : 0;
            int sa = a;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int x = __shfl_up(sa, o, 64);
                if (lane >= o) sa += x;
            }
            if (lane < ROUTE_THREADS / 64) wsum[lane][v] = sa - a;
            if (v > 0 && lane == ROUTE_THREADS / 64 - 1) item_count[v - 1] = min(sa, max_items);
        }
    }
    __syncthreads();
    int off = wsum[wave][0] + inc[0] - own[0];
    int si = wsum[wave][1] + inc[1] - own[1], bi = wsum[wave][2] + inc[2] - own[2];
    for (int q = 0; q < per; ++q) {
        const int e = e0 + q;
        if (e >= E) break;
        const int c = cnt[e];
        cur[e] = off;
        start[e] = off;
        for (int f = 0; f < c; f += ipm) {
            const int m = min(ipm, c - f);
            const int at = m <= SMALL_ROWS ? si++ : max_items - 1 - bi++;
            if (at >= 0 && at < max_items) {
                items[3 * at] = e;
                items[3 * at + 1] = off + f;
                items[3 * at + 2] = m;
            }
        }
        off += c;
    }
    __syncthreads();
    auto place = [&](int i, int e) __attribute__((always_inline)) {
        int big = 0;
        if (e >= 0 && e < E) {
            const int at = atomicAdd(&cur[e], 1);
            sorted[at] = i;
            const int f = (at - start[e]) / ipm * ipm;  // the first pair of its item, within the expert
            big = min(ipm, cnt[e] - f) > SMALL_ROWS;
        }
        pclass[i] = big;
    };
#pragma unroll
    for (int j = 0; j < ROUTE_HELD; ++j) {
        const int i = j * ROUTE_THREADS + (int)threadIdx.x;
        if (i < n) place(i, held[j]);
    }
    for (int i = ROUTE_HELD * ROUTE_THREADS + threadIdx.x; i < n; i += ROUTE_THREADS) place(i, pick[i]);
}

// How a pass's sums leave the combine: fp32, fp32 rounded through bf16 (prompt_experts.zig:246), or fp16 (half sums).
enum OutMode : int { OUT_F32 = 0, OUT_BF16R = 1, OUT_F16 = 2 };

// The down epilogue and slot combine of a prompt pass. Block (row r, 2048 columns): a thread holds 8 consecutive
// columns of one 128-block (16 lanes a block, lane l the columns 8 h8_group(l) .. + 7); for each slot in order
// y = FWHT(plane[pair]) * HAD_SCALE * svh_d[e], then out = fma(w, y, out) from zero; a slot without an expert adds w * 0,
// or nothing with skip. These are the operations and the order of down_combine_kernel with one split (the butterflies over
// value-index bits 0..6, three inside a lane and four across lanes: fwht128_x8), so the same bits (a zero y's sign
// does not reach out, which starts at +0). Bound by the plane's bytes: the rounding happens here and not in a launch of
// its own, which read and wrote out again (2048 rows: 24 us).
// (prompt_experts.cu's deterministic combine; exl3_experts.cu:186-214 for the epilogue.)
__global__ void __launch_bounds__(256) prompt_combine_kernel(PairPlane plane, const int* __restrict__ pick,
                                                             const uint16_t* __restrict__ svh_d,
                                                             const float* __restrict__ wts, void* __restrict__ out,
                                                             int D, int E, int slots, int mode, int skip) {
    const int r = blockIdx.x, lane = threadIdx.x & 63;
    const int k = blockIdx.y * 2048 + 128 * ((int)threadIdx.x >> 4) + 8 * h8_group(lane);
    if (k >= D) return;  // whole 16-lane groups (D % 128 == 0)
    const float* __restrict__ Z = plane.base(k);  // 8 columns never straddle the halves (half % 64 == 0)
    float a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = 0.f;
    // four slots at a time: their picks and weights, then all their plane and svh loads in flight before the first
    // slot's rotation (a slot without an expert loads pair 0's row and expert 0's scales)
    constexpr int QB = 4;
    for (int q0 = 0; q0 < slots; q0 += QB) {
        int ev[QB];
        float wv[QB];
        f4v z0[QB], z1[QB];
        u4v sv[QB];
#pragma unroll
        for (int j = 0; j < QB; ++j) {
            const int p = r * slots + (q0 + j < slots ? q0 + j : q0), e = pick[p];
            wv[j] = wts[p];
            ev[j] = e >= 0 && e < E ? p : -1;
            const size_t zo = (size_t)(ev[j] >= 0 ? p : r * slots) * plane.stride + k;
            z0[j] = *reinterpret_cast<const f4v*>(Z + zo);
            z1[j] = *reinterpret_cast<const f4v*>(Z + zo + 4);
            sv[j] = *reinterpret_cast<const u4v*>(svh_d + (size_t)(ev[j] >= 0 ? e : 0) * D + k);
        }
        issued();
#pragma unroll
        for (int j = 0; j < QB; ++j) {
            if (q0 + j >= slots) break;  // uniform
            float o[8];
            if (ev[j] >= 0) {  // uniform over the block
                float v[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = 0.f + z0[j][i];  // the split sum from zero
                    v[4 + i] = 0.f + z1[j][i];
                }
                const float sc = fwht128_x8(v, lane) * HAD_SCALE;  // the values' sign folded into the scale (exact)
#pragma unroll
                for (int i = 0; i < 8; ++i) o[i] = v[i] * sc * h2f((uint16_t)(sv[j][i >> 1] >> (16 * (i & 1))));
            } else {
                if (skip) continue;
#pragma unroll
                for (int i = 0; i < 8; ++i) o[i] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] = __builtin_fmaf(wv[j], o[i], a[i]);
        }
    }
    if (mode == OUT_BF16R)
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = bf16r(a[j]);
    // 16-byte stores where out allows them (D % 128 == 0 keeps every row as aligned as the first), else 4-byte ones
    const bool al = (reinterpret_cast<uintptr_t>(out) & 15) == 0;  // uniform
    if (mode == OUT_F16) {
        uint32_t* o = reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(out) + (size_t)r * D + k);
        const u4v h = {f2h2(a[0], a[1]), f2h2(a[2], a[3]), f2h2(a[4], a[5]), f2h2(a[6], a[7])};
        if (al) *reinterpret_cast<u4v*>(o) = h;
        else
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = h[j];
        return;
    }
    float* o = static_cast<float*>(out) + (size_t)r * D + k;
    if (al) {
        *reinterpret_cast<f4v*>(o) = f4v{a[0], a[1], a[2], a[3]};
        *reinterpret_cast<f4v*>(o + 4) = f4v{a[4], a[5], a[6], a[7]};
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = a[j];
    }
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

struct PromptLayout {
    size_t sorted, items, count, xd, plane, xg, xu, z, zp, pclass, total;
    uint32_t rows, max_items;
    bool has_plane;
};

// Whether a pass without a pair plane covers the layer's shape: halves of whole 128-column blocks (D % 256 == 0) over the
// pairs' rotated inputs, and the down kernel that takes K = I of at most 256. Other shapes keep the plane.
static bool split_plane_fits(const ea_routed* ex) { return ex->width <= 2 * PK * 16 && ex->dims % 256 == 0; }

static PromptLayout prompt_layout(const ea_routed* ex, uint32_t rows, uint32_t slots, int planes) {
    PromptLayout l{};
    l.has_plane = planes || !split_plane_fits(ex);
    const uint32_t r = rows < CHUNK_ROWS ? rows : CHUNK_ROWS;
    const size_t n = (size_t)r * slots, D = ex->dims, I = ex->width;
    l.rows = r;
    l.max_items = (uint32_t)(n / IPM + (n < ex->count ? n : ex->count));
    size_t off = 0;
    auto take = [&](size_t b) {
        const size_t at = off;
        off += align256(b);
        return at;
    };
    l.sorted = take(n * 4);
    l.items = take(3 * (size_t)l.max_items * 4);
    l.count = take(16);
    l.xd = take(n * I * 2);
    l.plane = l.has_plane ? take(n * D * 4) : 0;  // per-pair down outputs (the reference's pair plane)
    l.xg = take(n * D * 2);
    l.xu = take(n * D * 2);
    l.z = take(2 * n * I * 4);
    l.zp = take((size_t)(gu_splits((int)D) - 1) * 2 * n * I * 4);
    l.pclass = take(n * 4);
    l.total = off;
    return l;
}

// Both lists at once, joined once before the combine. The list whose blocks are dispatched first: the larger items
// up to LONG_ROWS rows a pass (512 rows: 339 us a layer against 355 with the small items first), the small items
// above it (2048 rows: 734 against 767 us), where the larger items fill the GPU for most of the pass and the small
// items' chain would otherwise wait for CUs at each of its steps. Launched eagerly, the side stream's list is
// enqueued (and dispatched) first; a captured graph's replay runs the main stream's branch first, so under capture
// the first list goes on the main stream.
static int list_passes(hipStream_t s, uint32_t cb, bool wide, const ListPass& a) {
    auto pass = [&](hipStream_t q, int big) {
        if (wide) return list_pass_wide(q, a, big, cb);
        return cb == 1 ? list_pass<1, 10>(q, a, big) : cb == 2 ? list_pass<2, 10>(q, a, big) : list_pass<0, 10>(q, a, big);
    };
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess) {
        cap = hipStreamCaptureStatusNone;
        (void)hipGetLastError();  // the query's own error is not a launch's
    }
    const int first = a.rows > LONG_ROWS ? 0 : 1;
    const int side = cap == hipStreamCaptureStatusActive ? 1 - first : first;
    return fork_join(
        s, [&](hipStream_t q) { return pass(q, side); }, [&](hipStream_t q) { return pass(q, 1 - side); });
}

// A decode window of more than 16 rows through the prefill path (ea_moe_routed): the moe scratch holds a prompt
// scratch with the pair plane (the slots added in order, so a window's rows get the same bits on every run) in its
// region; both follow from the layer's shape.
size_t prompt_region_bytes(const ea_routed* ex, uint32_t rows, uint32_t slots) {
    return prompt_layout(ex, rows, slots, 1).total;
}

int prompt_region_carve(const ea_routed* ex, uint32_t rows, uint32_t slots, uint64_t base, ea_prompt_scratch* s) {
    const PromptLayout l = prompt_layout(ex, rows, slots, 1);
    s->sorted = base + l.sorted;
    s->items = base + l.items;
    s->count = base + l.count;
    s->xd = base + l.xd;
    s->plane = base + l.plane;
    s->xg = base + l.xg;
    s->xu = base + l.xu;
    s->z = base + l.z;
    s->zp = base + l.zp;
    s->pclass = base + l.pclass;
    s->rows = l.rows;
    s->slots = slots;
    s->max_items = l.max_items;
    return EA_OK;
}

}  // namespace ea

using namespace ea;

extern "C" {

int ea_prompt_experts_supported(const ea_routed* ex, int* ok) {
    EA_REQUIRE_CTX(c);
    if (!ex || !ok) return EA_BAD_ARGUMENT;
    *ok = 0;
    if (ex->cb > 2 || ex->width % 128 || ex->dims % 128 || ex->count == 0) return EA_OK;
    for (int m = 0; m < 3; ++m) {
        int32_t* k2 = new int32_t[ex->count];
        const int r = hip_status(hipMemcpy(k2, dptr<void>(ex->k2[m]), ex->count * 4, hipMemcpyDeviceToHost));
        bool good = r == EA_OK;
        for (uint32_t e = 0; good && e < ex->count; ++e) good = k2[e] >= 2 && k2[e] <= 16;
        delete[] k2;
        if (r) return r;
        if (!good) return EA_OK;
    }
    *ok = 1;
    return EA_OK;
}

size_t ea_prompt_scratch_bytes(const ea_routed* ex, uint32_t rows, uint32_t slots, int planes) {
    if (!ex || rows == 0 || slots == 0) return 0;
    return prompt_layout(ex, rows, slots, planes).total;
}

int ea_prompt_scratch_init(ea_stream_t stream, ea_prompt_scratch* s, void* base, size_t bytes, const ea_routed* ex,
                           uint32_t rows, uint32_t slots, int planes) {
    EA_REQUIRE_CTX(c);
    if (!s || !base || !ex || rows == 0 || slots == 0 || slots > 32) return EA_BAD_ARGUMENT;
    if (reinterpret_cast<uintptr_t>(base) & 255) return EA_BAD_ARGUMENT;
    const PromptLayout l = prompt_layout(ex, rows, slots, planes);
    if (bytes < l.total) return EA_SCRATCH_TOO_SMALL;
    const uint64_t b = reinterpret_cast<uintptr_t>(base);
    s->sorted = b + l.sorted;
    s->items = b + l.items;
    s->count = b + l.count;
    s->xd = b + l.xd;
    s->plane = l.has_plane ? b + l.plane : 0;
    s->xg = b + l.xg;
    s->xu = b + l.xu;
    s->z = b + l.z;
    s->zp = b + l.zp;
    s->pclass = b + l.pclass;
    s->rows = l.rows;
    s->slots = slots;
    s->max_items = l.max_items;
    // only the count word needs a defined start (prompt_experts.zig:109-110)
    return fill_words(as_stream(stream), dptr<void>(s->count), 0u, 4);
}

int ea_prompt_experts_run(ea_stream_t stream, const void* x, int x_dtype, uint32_t xstride, const int32_t* pick,
                          const float* wts, const ea_routed* ex, const ea_prompt_scratch* sc, void* out, uint32_t R,
                          int do_round, int half_sums) {
    EA_REQUIRE_CTX(c);
    if (half_sums && do_round) return EA_INVALID;  // prompt_experts.zig:147
    if (half_sums && sc && sc->plane) return EA_INVALID;  // prompt_experts.zig:155: the pair plane takes fp32 rows only
    if (!x || !pick || !wts || !ex || !sc || !out) return EA_BAD_ARGUMENT;
    if (x_dtype < 0 || x_dtype > 2 || sc->slots == 0) return EA_BAD_ARGUMENT;
    if (ex->width % 128 || ex->dims % 128) return EA_BAD_WIDTH;
    // no pair plane: the pairs' down outputs take the place of their rotated inputs, which a scratch made for this
    // layer's shape allows (split_plane_fits); out 4-byte aligned (half sums are stored in pairs)
    const bool split = sc->plane == 0;
    if (split && (!split_plane_fits(ex) || (reinterpret_cast<uintptr_t>(out) & 3))) return EA_BAD_ARGUMENT;
    hipStream_t s = as_stream(stream);
    const uint32_t D = ex->dims, I = ex->width, E = ex->count, S = sc->slots;
    const size_t xb = x_dtype == 2 ? 4 : 2;
    const size_t ob = half_sums ? 2 : 4;
    const bool wide = ex->k2_gu[1] > 10 || ex->k2_d[1] > 10;
    for (uint32_t r0 = 0; r0 < R; r0 += sc->rows) {
        const uint32_t n = R - r0 < sc->rows ? R - r0 : sc->rows;
        const uint32_t pairs = n * S;
        const uint32_t items_n = (uint32_t)(pairs / IPM + (pairs < E ? pairs : E));
        const uint32_t max_items = items_n < sc->max_items ? items_n : sc->max_items;
        const char* xs = static_cast<const char*>(x) + (size_t)r0 * xstride * xb;
        const int32_t* pk = pick + (size_t)r0 * S;
        const float* wt = wts + (size_t)r0 * S;
        route_kernel<<<1, ROUTE_THREADS, 3 * E * sizeof(int), s>>>(pk, (int)pairs, (int)E, dptr<int>(sc->sorted),
                                                                  dptr<int>(sc->items), dptr<int>(sc->count),
                                                                  dptr<int>(sc->pclass), (int)max_items, IPM);
        int r = launched();
        if (r) return r;
        const uint16_t *suh_g = dptr<const uint16_t>(ex->suh_g), *suh_u = dptr<const uint16_t>(ex->suh_u);
        // Long passes rotate inside the larger items' products (rotate_fits says when they can): 2048 rows 666 -> 601 us,
        // bound by memory; 1024 rows 423 with the launch and 419 without it, 512 rows 306 and 335 (few blocks, each with the
        // rotation on its chain; a pass of as many rows with fewer slots likewise: 16 experts, 2 slots, 2048 rows 61 us with
        // the launch and 67 without). Widths above 10 keep the rotation launch: the one build of their kernel with the rotation
        // inside hung in a test and its cause was not found, so no such kernel is built (list_pass).
        const bool fuse = !wide && n > (uint32_t)LONG_ROWS && pairs > 8u * LONG_ROWS && rotate_fits(xs, x_dtype, xstride, suh_g, suh_u, n, I);
        if (!fuse) {
            r = launch_rot_in(s, xs, x_dtype, xstride, pk, suh_g, suh_u, dptr<uint16_t>(sc->xg), dptr<uint16_t>(sc->xu), n,
                              D, S, E);
            if (r) return r;
        }
        const int dh = (int)(D / 2);
        const PairPlane plane = split ? PairPlane{dptr<float>(sc->xg), dptr<float>(sc->xu) - dh, dh, dh}
                                      : PairPlane{dptr<float>(sc->plane), dptr<float>(sc->plane), dh, (int)D};
        ListPass a{};
        a.x = xs;
        a.x_dtype = x_dtype;
        a.x_stride = (int)xstride;
        a.fuse = fuse;
        a.suh_g = suh_g;
        a.suh_u = suh_u;
        a.xg = dptr<uint16_t>(sc->xg);
        a.xu = dptr<uint16_t>(sc->xu);
        for (int m = 0; m < 3; ++m) {
            a.tp[m] = dptr<const int64_t>(ex->ptr[m]);
            a.k2[m] = dptr<const int>(ex->k2[m]);
        }
        a.sorted = dptr<const int>(sc->sorted);
        a.items = dptr<const int>(sc->items);
        a.count = dptr<const int>(sc->count);
        a.pclass = dptr<const int>(sc->pclass);
        a.pick = pk;
        a.svh_g = dptr<const uint16_t>(ex->svh_g);
        a.svh_u = dptr<const uint16_t>(ex->svh_u);
        a.suh_d = dptr<const uint16_t>(ex->suh_d);
        a.z = dptr<float>(sc->z);
        a.zp = dptr<float>(sc->zp);
        a.plane = plane;
        a.xd = dptr<uint16_t>(sc->xd);
        a.D = (int)D;
        a.I = (int)I;
        a.P = (int)pairs;
        a.rows = (int)n;
        a.slots = (int)S;
        a.E = (int)E;
        a.mi = (int)max_items;
        a.status = c->status;
        r = list_passes(s, ex->cb, wide, a);
        if (r) return r;
        // the pair plane summed in slot order; slots without an expert add nothing (the reference's route skips them)
        prompt_combine_kernel<<<dim3(n, (D + 2047) / 2048), 256, 0, s>>>(
            plane, pk, dptr<const uint16_t>(ex->svh_d), wt, static_cast<char*>(out) + (size_t)r0 * D * ob, (int)D, (int)E,
            (int)S, half_sums ? OUT_F16 : do_round ? OUT_BF16R : OUT_F32, split);
        r = launched();
        if (r) return r;
    }
    return EA_OK;
}

}  // extern "C"
