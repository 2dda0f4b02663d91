// The q8 multiplies of up to 64 rows (decode batches) that the M <= 16 pass kernels do not take: Y = epilogue(X W^T) for
// gpu-q8w, each output's links in a fixed order.
//
// An output is a chain over the groups of K, y = fma(f_g, ws_g [x xs_g], y) with exact int32 group sums f_g, so its bits
// depend on where the chain starts anew. The order is the weight-streaming kernel's (stream_q8_order: runs of gps groups,
// added in order) where that kernel runs by default, and the whole chain, cpu-q8 bit for bit, above 32 rows with N >= 8192,
// where the large-M kernels do. So a run is never split: a block owns WT 16-row weight tiles, one per wave. A wave streams
// its tile's weights straight into registers in MFMA operand order; the block's X goes through a ring of LDS stages by
// direct loads, whole 128-byte lines, read by all its waves; both are requested D - 1 groups ahead, and one barrier per
// group hands a stage over. A block takes all runs of its tiles, one after the other, and ends in the
// epilogue; or, where that would be a long chain on few blocks, one run: the runs' sums then go to the workspace's
// partial zone ([run][T][N] float32), and a second launch adds them in order and runs the epilogue (q8_rows_blocks).
//
// Measured (us a call, graph replays over cold weights; the kernels whose bits these are -> here): gate/up 19456 x 2560 per
// 128 at 17 / 33 / 64 rows 26.5 / 37.5 / 39.7 -> 16.0 / 18.0 / 21.6, down 2560 x 9728 29.4 / 34.9 / 35.4 -> 12.7 / 13.0 /
// 14.8, 12288 x 5120 per token at 48 rows 53 -> 19, 1024 x 4096 47 -> 12. What bounds it: at 19456 x 2560 the stream of the
// weights and the blocks' X (22 bytes a ns and CU); on few blocks the loads' latency, 5 groups of which are in flight
// (0.23 / 0.31 / 0.39 us a group at 32 / 48 / 64 rows). Steps of two groups between barriers were no faster (the chain of a
// step is not the bound), X in registers without the LDS ring 1.2 to 1.8 times slower (every wave fetched all of X).
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "gemm_kernels.hpp"
#include "group_window.hpp"

namespace sepal::hip {
namespace q8s {

// Stages, and groups of a block whose activation scales fit the LDS (per 128). One array per stage and one for the scales: the
// compiler tells up to eight static arrays apart, and before a read from any other it waits for every direct load.
constexpr int D = 6, kMaxGroups = 96;

struct Params {
    const signed char* x;  // [T, ld_x]
    const signed char* w;  // [N, ld_w]
    const float* ws;       // [N, ld_ws]
    const float* xs;       // activation scales [T, ld_xs], one per token or per 128 columns
    unsigned x_bytes, w_bytes, ws_bytes;
    int ld_x, ld_w, ld_ws;
    std::size_t ld_xs;
    void* y;      // [T, ld_y]
    float* part;  // several runs: [run][T][N]
    std::size_t ld_y;
    int y_type, epilogue;
    int t, n, groups, tiles;
    int splits, gps;  // runs of gps groups
    int parts;        // blocks a tile's runs are spread over: 1, or one per run
    int spans;        // column spans of WT tiles
    float first;      // where a run's chain starts: -0 keeps a first product's sign (the chain), +0 as the stream kernel
};

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

__device__ __forceinline__ i32x4 mfma_i(const u32x4 a, const u32x4 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

// s_waitcnt vmcnt(N) lgkmcnt(0)
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// y or y + v (or SwiGLU of a gate and an up value) of one output.
template <bool PER128>
__device__ __forceinline__ void out_h(const Params& p, std::size_t idx, float g, float u) {
    const float h = swiglu_q8<!PER128>(g, u);
    if (p.y_type == SEPAL_HIP_F32) store_out<SEPAL_HIP_F32>(p.y, idx, h);
    else if (p.y_type == SEPAL_HIP_BF16) store_out<SEPAL_HIP_BF16>(p.y, idx, h);
    else store_out<SEPAL_HIP_F16>(p.y, idx, h);
}
__device__ __forceinline__ void out_y(const Params& p, std::size_t idx, float v) {
    float* const y = static_cast<float*>(p.y);
    y[idx] = p.epilogue == SEPAL_HIP_ADD ? __fadd_rn(y[idx], v) : v;
}

// MT: 16-row tiles of X (T <= 16 MT); WT: weight tiles and waves of a block.
template <int MT, bool PER128, int WT>
__global__ void __launch_bounds__(64 * WT) rows_kernel(const Params p) {
    constexpr int STAGE = MT * 2048, XW = (2 * MT + WT - 1) / WT;  // bytes of a stage; a wave's share of its kilobytes
    constexpr int NLD = XW + 3;                                    // a wave's loads per group: X, one scale, two of weights
    __shared__ __align__(1024) unsigned char l0[STAGE], l1[STAGE], l2[STAGE], l3[STAGE], l4[STAGE], l5[STAGE];
    static_assert(D == 6, "one array per stage");
    __shared__ __align__(16) float xs_lds[PER128 ? kMaxGroups * 16 * MT : 4];  // [group of the run][16 MT rows]
    const auto stage = [&](auto it) __attribute__((always_inline)) -> lds_u8* {
        constexpr int i = decltype(it)::value % D;
        if constexpr (i == 0) return (lds_u8*)l0;
        else if constexpr (i == 1) return (lds_u8*)l1;
        else if constexpr (i == 2) return (lds_u8*)l2;
        else if constexpr (i == 3) return (lds_u8*)l3;
        else if constexpr (i == 4) return (lds_u8*)l4;
        else return (lds_u8*)l5;
    };

    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int span = static_cast<int>(blockIdx.x) % p.spans, part = static_cast<int>(blockIdx.x) / p.spans;
    const int g_lo = part * p.gps, nu = p.parts == 1 ? p.groups : min(p.gps, p.groups - g_lo);
    const int my_tile = span * WT + wave;
    const int tile = min(my_tile, p.tiles - 1);  // tiles past the last repeat it and are never stored
    const bool swiglu = p.epilogue == SEPAL_HIP_SWIGLU;

    // 32-bit lane offsets, the group in the scalar offset; a group past the run is loaded through an empty window
    // (group_window), so that every step issues the same loads
    const int c = lane % 16, kq = lane / 16;
    // X load e fills kilobyte e of a stage = rows 8 e + {0..7}; lane l writes slot l % 8 of row 8 e + l / 8, which holds
    // chunk (l % 8) ^ ((row / 2) % 8); rows past T repeat the last
    int xe[XW], xoff[XW];
#pragma unroll
    for (int q = 0; q < XW; ++q) {
        xe[q] = min(wave + WT * q, 2 * MT - 1);  // (a wave without a share repeats the last kilobyte)
        xoff[q] = min(8 * xe[q] + lane / 8, p.t - 1) * p.ld_x + 16 * ((lane % 8) ^ ((4 * xe[q] + lane / 16) & 7));
    }
    // (SwiGLU tiles: 8 gate rows, then the 8 up rows of the same features, 64 packed rows further)
    const int row = (swiglu ? 128 * (tile / 8) + 8 * (tile % 8) : 16 * tile) + (swiglu && c >= 8 ? 56 + c : c);
    const int woff = row * p.ld_w + 16 * kq, soff = row * p.ld_ws * 4;
    const auto uniform = [](int v) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(v); };
    const auto rsrc = [&](const void* ptr, unsigned bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(ptr), 0, uniform(static_cast<int>(bytes)), 0x00020000);
    };
    const auto load_kb = [](const __amdgpu_buffer_rsrc_t r, lds_u8* dst, int off, int so) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, off, so, 0, 0);
    };
    u32x4 wb[D][2];
    float sc[D];
    // a wave's loads of group u (stage and register set it)
    const auto issue = [&](int u, auto it) __attribute__((always_inline)) {
        constexpr int b = decltype(it)::value % D;
        const bool in = u < nu;
        const Window xw = group_window(in, p.x_bytes, (g_lo + u) * 128), ww = group_window(in, p.w_bytes, (g_lo + u) * 128),
                     sw = group_window(in, p.ws_bytes, (g_lo + u) * 4);
        const __amdgpu_buffer_rsrc_t xr = rsrc(p.x, xw.bytes), wr = rsrc(p.w, ww.bytes), sr = rsrc(p.ws, sw.bytes);
        const int so = uniform(xw.scalar), s_so = uniform(sw.scalar);  // (X and W rows advance alike)
        lds_u8* const dst = stage(it);
#pragma unroll
        for (int q = 0; q < XW; ++q) load_kb(xr, dst + xe[q] * 1024, xoff[q], so);
        sc[b] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, soff, s_so, 0));
#pragma unroll
        for (int j = 0; j < 2; ++j)
            wb[b][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, woff + 64 * j, so, 0));
        __builtin_amdgcn_sched_barrier(0);
    };
    using std::integral_constant;

    // per 128: the run's activation scales, a first batch requested before everything else and written after the first
    // loads are out (the barrier of the first step covers them)
    const int total = PER128 ? nu * 16 * MT : 0;
    constexpr int XB = 4;
    float xv0[XB];
    const auto xs_at = [&](int id) __attribute__((always_inline)) {
        return p.xs[static_cast<std::size_t>(min(id % (16 * MT), p.t - 1)) * p.ld_xs + g_lo + id / (16 * MT)];
    };
    if constexpr (PER128) {
#pragma unroll
        for (int e = 0; e < XB; ++e) xv0[e] = xs_at(min(tid + e * 64 * WT, total - 1));
    }
    __builtin_amdgcn_sched_barrier(0);
    issue(0, integral_constant<int, 0>{});
    issue(1, integral_constant<int, 1>{});
    issue(2, integral_constant<int, 2>{});
    issue(3, integral_constant<int, 3>{});
    issue(4, integral_constant<int, 4>{});
    if constexpr (PER128) {
#pragma unroll
        for (int e = 0; e < XB; ++e)
            if (tid + e * 64 * WT < total) xs_lds[tid + e * 64 * WT] = xv0[e];
        for (int id = tid + XB * 64 * WT; id < total; id += 64 * WT) xs_lds[id] = xs_at(id);
    }

    float acc[MT][4], sum_runs[MT][4];  // the run in hand; the runs before it, added in order
    int run_end = p.gps;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = p.first, sum_runs[i][r] = 0.0f;
    // the lane's operand bytes of half h of a row tile: row lane % 16, chunk 4 h + lane / 16
    int rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd[h] = c * 128 + 16 * ((4 * h + kq) ^ (c / 2));
    const auto step = [&](int u, auto it) __attribute__((always_inline)) {
        constexpr int b = decltype(it)::value;
        // this wave's loads of group u have landed (behind them: the D - 2 groups requested since) and its reads of the stage of
        // group u - 1 are complete; after the barrier both hold for every wave
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_lgkm0<(D - 2) * NLD>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(u + D - 1, integral_constant<int, b + D - 1>{});
        const lds_u8* const src = stage(it);
        u32x4 x[MT][2];
        f32x4 xv[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
#pragma unroll
            for (int h = 0; h < 2; ++h) x[i][h] = *reinterpret_cast<const lds_u32x4*>(src + i * 2048 + rd[h]);
            if constexpr (PER128) xv[i] = *reinterpret_cast<const f32x4*>(xs_lds + u * 16 * MT + 16 * i + 4 * kq);
        }
        i32x4 sum[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) sum[i] = mfma_i(x[i][0], wb[b][0], i32x4{0, 0, 0, 0});
#pragma unroll
        for (int i = 0; i < MT; ++i) sum[i] = mfma_i(x[i][1], wb[b][1], sum[i]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float f = PER128 ? __fmul_rn(sc[b], xv[i][r]) : sc[b];
                acc[i][r] = __builtin_fmaf(static_cast<float>(sum[i][r]), f, acc[i][r]);
            }
        if (u + 1 == run_end && run_end < nu) {  // (uniform) a run is complete and another follows
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum_runs[i][r] = run_end == p.gps ? acc[i][r] : __fadd_rn(sum_runs[i][r], acc[i][r]);
                    acc[i][r] = p.first;
                }
            run_end += p.gps;
        }
    };
    // (no exit inside a turn: the compiler joins such exits at the loop's end, and its waits at the head then cover loads
    // that are still wanted in flight)
    int u = 0;
    for (; u + D <= nu; u += D) {
        step(u, integral_constant<int, 0>{});
        step(u + 1, integral_constant<int, 1>{});
        step(u + 2, integral_constant<int, 2>{});
        step(u + 3, integral_constant<int, 3>{});
        step(u + 4, integral_constant<int, 4>{});
        step(u + 5, integral_constant<int, 5>{});
    }
    if (u < nu) step(u, integral_constant<int, 0>{});
    if (u + 1 < nu) step(u + 1, integral_constant<int, 1>{});
    if (u + 2 < nu) step(u + 2, integral_constant<int, 2>{});
    if (u + 3 < nu) step(u + 3, integral_constant<int, 3>{});
    if (u + 4 < nu) step(u + 4, integral_constant<int, 4>{});
    __builtin_amdgcn_sched_barrier(0);
    wait_vm_lgkm0<0>();  // no direct load of this wave may still write the block's LDS when it ends
    __builtin_amdgcn_sched_barrier(0);
    if (my_tile >= p.tiles) return;
    if (run_end > p.gps) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][r] = __fadd_rn(sum_runs[i][r], acc[i][r]);
    }

    // a lane has rows 16 i + 4 (lane / 16) + 0..3 of tile column lane % 16
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r0 = 16 * i + 4 * kq;
        if (p.parts > 1) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r0 + r < p.t) p.part[(static_cast<std::size_t>(part) * p.t + r0 + r) * p.n + row] = acc[i][r];
            continue;
        }
        if constexpr (!PER128) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[i][r] = __fmul_rn(acc[i][r], p.xs[static_cast<std::size_t>(min(r0 + r, p.t - 1)) * p.ld_xs]);
        }
        if (swiglu) {
            // gate in columns 0..7, up of the same features in columns 8..15
            float up[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) up[r] = __shfl(acc[i][r], (lane + 8) % 64, 64);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (c < 8 && r0 + r < p.t)
                    out_h<PER128>(p, static_cast<std::size_t>(r0 + r) * p.ld_y + 64 * (tile / 8) + 8 * (tile % 8) + c, acc[i][r], up[r]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r0 + r < p.t) out_y(p, static_cast<std::size_t>(r0 + r) * p.ld_y + row, acc[i][r]);
        }
    }
}

// Several runs: their sums added in order, then the epilogue. A thread has four consecutive columns (features) of a row.
template <bool PER128>
__global__ void __launch_bounds__(64) runs_kernel(const Params p) {
    const bool swiglu = p.epilogue == SEPAL_HIP_SWIGLU;
    const int per_row = swiglu ? p.n / 8 : p.n / 4;
    const int id = static_cast<int>(blockIdx.x) * 64 + threadIdx.x;
    if (id >= p.t * per_row) return;
    const int r = id / per_row, c = 4 * (id % per_row);
    const std::size_t plane = static_cast<std::size_t>(p.t) * p.n;
    const auto total = [&](int col) __attribute__((always_inline)) {
        const float* const src = p.part + static_cast<std::size_t>(r) * p.n + col;
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int s0 = 0; s0 < p.splits; s0 += 16) {  // sixteen loads in flight, added in order
            f32x4 o[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) o[q] = *reinterpret_cast<const f32x4*>(src + min(s0 + q, p.splits - 1) * plane);
#pragma unroll
            for (int q = 0; q < 16; ++q)
                if (s0 + q < p.splits) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = s0 + q == 0 ? o[q][e] : __fadd_rn(v[e], o[q][e]);
                }
        }
        if constexpr (!PER128) {
            const float xs = p.xs[static_cast<std::size_t>(r) * p.ld_xs];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fmul_rn(v[e], xs);
        }
        return v;
    };
    const std::size_t idx = static_cast<std::size_t>(r) * p.ld_y + c;
    if (swiglu) {
        const int gate = 128 * (c / 64) + c % 64;  // packed columns of features c .. c + 3
        const f32x4 g = total(gate), u = total(gate + 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) out_h<PER128>(p, idx + e, g[e], u[e]);
    } else {
        const f32x4 v = total(c);
#pragma unroll
        for (int e = 0; e < 4; ++e) out_y(p, idx + e, v[e]);
    }
}

// ---- launch ----------------------------------------------------------------------------------------------------------

inline int device_cus() {
    static std::atomic<int> cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) throw LaunchError("small-M q8 multiply: hipGetDevice failed");
    if (dev < 64) {
        const int known = cached[dev].load(std::memory_order_relaxed);
        if (known > 0) return known;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        throw LaunchError("small-M q8 multiply: device query failed");
    if (dev < 64) cached[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

template <int MT, bool PER128, int WT>
void launch(const Params& p, hipStream_t stream) {
    rows_kernel<MT, PER128, WT><<<dim3(static_cast<unsigned>(p.spans) * p.parts), dim3(64 * WT), 0, stream>>>(p);
    check_launch("small-M q8 multiply launch");
    if (p.parts == 1) return;
    const std::size_t items = static_cast<std::size_t>(p.t) * (p.epilogue == SEPAL_HIP_SWIGLU ? p.n / 8 : p.n / 4);
    runs_kernel<PER128><<<dim3(static_cast<unsigned>((items + 63) / 64)), dim3(64), 0, stream>>>(p);
    check_launch("small-M q8 multiply runs launch");
}

template <int MT, bool PER128>
void launch_tiles(const Params& p, int wt, hipStream_t stream) {
    switch (wt) {
    case 2: launch<MT, PER128, 2>(p, stream); break;
    case 3: launch<MT, PER128, 3>(p, stream); break;
    case 4: launch<MT, PER128, 4>(p, stream); break;
    case 5: launch<MT, PER128, 5>(p, stream); break;
    case 6: launch<MT, PER128, 6>(p, stream); break;
    default: launch<MT, PER128, 8>(p, stream); break;
    }
}

template <bool PER128>
void launch_rows(const Params& p, int wt, hipStream_t stream) {
    if (p.t <= 32) launch_tiles<2, PER128>(p, wt, stream);
    else if (p.t <= 48) launch_tiles<3, PER128>(p, wt, stream);
    else launch_tiles<4, PER128>(p, wt, stream);
}

} // namespace q8s

// How a problem's runs are spread: all runs of a tile in one block, or a block per run and the second launch; and the tiles of
// a block, by the fewest tiles and X rows that a CU goes through. The times below (us) are fitted to forced runs of both
// forms at 17 shapes of N 256 .. 20480, K 1024 .. 10240 and 17 .. 64 rows, over cold weights: a group takes a block the
// longer of its loads' latency (which grows with the X rows) and its kilobytes, whose rate falls where all CUs stream; the
// choice is within 1% of the faster form and block on average, 10% at worst. E.g. 33 rows, us: 2560 x 9728 per 128 28.7 in
// one block, 13.0 spread; 7168 x 1024 SwiGLU 7.4 and 11.0. False where a block's scales exceed their LDS array.
bool q8_rows_blocks(int mt, bool per128, int tiles, int groups, int splits, int gps, int cus, Q8RowsPlan& plan) {
    double best = 0.0;
    for (const int parts : {1, splits}) {
        const int block_groups = parts == 1 ? groups : gps;
        if ((parts == 1 && best > 0.0) || (per128 && block_groups > q8s::kMaxGroups)) continue;
        int wt = 0, rounds = 0, blocks = 0;
        for (const int w : {8, 6, 5, 4, 3, 2}) {
            const int b = (tiles + w - 1) / w * parts, r = (b + cus - 1) / cus;
            if (wt == 0 || r * (w + mt) < rounds * (wt + mt)) wt = w, rounds = r, blocks = b;
        }
        const double group_us = std::max(0.07 + 0.08 * mt, 2.0 * (wt + mt) / (5 * blocks > 4 * cus ? 23.0 : 38.0));
        const double us = 3.5 + rounds * block_groups * group_us +
                          (parts > 1 ? 2.3 + 0.5 * ((parts + 15) / 16) + 2.0 * parts * mt * tiles / 6000.0 : 0.0);
        if (best == 0.0 || us < best) {
            best = us;
            plan.parts = parts;
            plan.wt = wt;
        }
    }
    return best > 0.0;
}

bool q8_rows_plan(const GemmArgs& a, Q8RowsPlan& plan) {
    if (a.config >= 0 || a.t > kSmallM || a.w_stream || a.k % 128 != 0) return false;
    const bool swiglu = a.epilogue == SEPAL_HIP_SWIGLU;
    if (swiglu ? a.n % 128 != 0 : (a.n % 16 != 0 || a.y_type != SEPAL_HIP_F32)) return false;
    const std::size_t lim = std::size_t{1} << 31;
    if (a.t * a.ld_x >= lim || a.n * a.ld_w >= lim || a.n * a.ld_s * 4 >= lim) return false;
    plan.whole = !q8_streams(a.t, a.n) || !stream_q8_order(a, plan.splits, plan.gps);
    if (plan.whole) {
        plan.splits = 1;
        plan.gps = static_cast<int>(a.k / 128);
    }
    const bool per128 = a.act_block != a.k || a.k == 128;
    return q8_rows_blocks(a.t <= 32 ? 2 : (a.t <= 48 ? 3 : 4), per128, static_cast<int>(a.n / 16), static_cast<int>(a.k / 128), plan.splits, plan.gps,
                          q8s::device_cus(), plan);
}

void launch_q8_rows(const GemmArgs& a, const Q8RowsPlan& plan, hipStream_t stream) {
    q8s::Params p{};
    p.x = static_cast<const signed char*>(a.x);
    p.x_bytes = static_cast<unsigned>((a.t - 1) * a.ld_x + a.k);
    p.ld_x = static_cast<int>(a.ld_x);
    p.w = reinterpret_cast<const signed char*>(a.w);
    p.w_bytes = static_cast<unsigned>((a.n - 1) * a.ld_w + a.k);
    p.ld_w = static_cast<int>(a.ld_w);
    p.ws = a.s;
    p.ws_bytes = static_cast<unsigned>(((a.n - 1) * a.ld_s + a.k / 128) * 4);
    p.ld_ws = static_cast<int>(a.ld_s);
    p.xs = a.xs;
    p.ld_xs = a.ld_xs;
    p.y = a.y;
    p.ld_y = a.ld_y;
    p.y_type = a.y_type;
    p.epilogue = a.epilogue;
    p.t = static_cast<int>(a.t);
    p.n = static_cast<int>(a.n);
    p.groups = static_cast<int>(a.k / 128);
    p.tiles = static_cast<int>(a.n / 16);
    p.splits = plan.splits;
    p.gps = plan.gps;
    p.parts = plan.parts;
    p.spans = (p.tiles + plan.wt - 1) / plan.wt;
    if (plan.parts > 1) {
        // (stream_q8_order keeps the runs' sums within the zone)
        if (a.scratch == nullptr) throw LaunchError("small-M q8 multiply: scratch missing");
        p.part = reinterpret_cast<float*>(static_cast<char*>(a.scratch) + kCounterBytes);
    }
    p.first = plan.whole ? -0.0f : 0.0f;
    const bool per128 = a.act_block != a.k || a.k == 128;
    if (per128) q8s::launch_rows<true>(p, plan.wt, stream);
    else q8s::launch_rows<false>(p, plan.wt, stream);
}

} // namespace sepal::hip
