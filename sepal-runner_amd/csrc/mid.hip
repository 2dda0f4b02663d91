// The w8g multiplies of up to 64 rows (decode batches) that the M <= 16 pass kernels do not take: Y = epilogue(X W^T) for
// bf16 / binary16 X.
//
// At these sizes the time to beat is one pass over the weights, as at M <= 16, but the X rows no longer fit the LDS
// beside them (64 rows x 2560 bf16 are 320 KB), and a kernel that shares X tiles between waves spends its time on
// barriers. Here nothing is shared while the weights stream: a block owns NT 16-row weight tiles and a range of K, and
// its 8 waves split that range by whole 128-value groups. A wave reads each of its weights and X values once:
//   weights  straight from global memory into the wave's own LDS slots (one 2 KB slot per tile, two 1 KB loads of 8 rows
//            x 128 bytes: whole cache lines), read back in MFMA operand order; a tile's slot is refilled with the next
//            group as soon as its operands are in registers, so a wave keeps NT - 1 to NT slots in flight (80 KB a CU);
//   X        straight into registers in MFMA operand order (every wave has its own groups, so no X value is read twice
//            by a block; the blocks' re-reads are L2 hits), one group ahead.
// The only block barriers are the three of the final sum (the slots are free, waves 4-7 have written, their sums with waves
// 0-3 are written): the waves' partial tiles meet in the slots' LDS, waves 4-7 added to waves 0-3, then the four in wave
// order; then the epilogue. SwiGLU and one-part Store / Add write Y; a Store / Add
// multiply too narrow to fill the chip splits K over blocks too (parts), in the workspace's partial zone, added in part
// order by a second launch. Per group the sum of products is scaled and added in float32 (y += s_g P_g), so results are
// within float32 rounding of the other paths'. (The q8 multiplies, whose order of links is part of their result, have
// a kernel of their own: q8_small.hip.)
//
// Measured (us a call, HIP-graph replays over cold weights; before: the streaming kernel, or the large-M kernels on
// 64-row tiles): gate/up 19456 x 2560 at 32 / 48 rows 23.0 / 24.4 -> 18.7 / 21.5, down 2560 x 9728 25.4 / 24.2 -> 14.1 /
// 16.2. What bounds it (gate/up, 48 rows, ablations): 6.5 us for an empty run of the grid, 6 for the
// weight stream, 6.5 for the widening and the MFMAs (of which a wave overlaps little with its stream: one group of
// NT tiles is in flight), 3 for the final sum and the epilogue; X costs 0.5.
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "gemm_kernels.hpp"
#include "group_window.hpp"

namespace sepal::hip {
namespace mid {

constexpr int kWaves = 8, kThreads = 64 * kWaves;

struct Params {
    const void* x;            // [T, ld_x] bf16 / binary16
    unsigned x_bytes, w_bytes, s_bytes;
    int ld_xb;                // X row stride in bytes
    const signed char* w;     // [N, ld_w]
    int ld_w;
    const float* s;           // [N, ld_s]
    int ld_s;
    void* y;                  // [T, ld_y], or the parts [parts][T][N] float32
    std::size_t ld_y;
    int y_type, epilogue;     // epilogue of a one-part multiply
    bool libm;                // SwiGLU by swiglu_libm
    int t, n, k;
    int tiles, parts, spans;  // 16-row weight tiles; K-parts; column spans of NT tiles
};

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

template <int XT>
__device__ __forceinline__ f32x4 mfma_f(const u32x4 a, const u32x4 b, f32x4 c) {
    if constexpr (XT == SEPAL_HIP_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// s_waitcnt vmcnt(N) with the other counters left at their maximum.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// MT: 16-row tiles of X (T <= 16 MT); NT: weight tiles of a block.
template <int XT, int MT, int NT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) mid_kernel(const Params p) {
    constexpr int XL = 4;                 // 16-byte X loads per lane, row tile and group
    constexpr int SLOT = kWaves * 2048;   // one tile's slots of all waves; the final sum's [4 waves][MT][64 lanes] x 16 B
    static_assert(4 * MT * 1024 <= SLOT, "the final sum reuses a tile's slots");
    // a separate array per tile: the compiler then knows which one a direct load writes
    __shared__ __align__(1024) unsigned char l0[SLOT], l1[NT > 1 ? SLOT : 16], l2[NT > 2 ? SLOT : 16], l3[NT > 3 ? SLOT : 16],
        l4[NT > 4 ? SLOT : 16];
    const auto slot = [&](auto it) -> lds_u8* {
        constexpr int i = decltype(it)::value;
        if constexpr (i == 0) return (lds_u8*)l0;
        else if constexpr (i == 1) return (lds_u8*)l1;
        else if constexpr (i == 2) return (lds_u8*)l2;
        else if constexpr (i == 3) return (lds_u8*)l3;
        else return (lds_u8*)l4;
    };
    const auto each_tile = [&](auto f) __attribute__((always_inline)) {
        f(std::integral_constant<int, 0>{});
        if constexpr (NT > 1) f(std::integral_constant<int, 1>{});
        if constexpr (NT > 2) f(std::integral_constant<int, 2>{});
        if constexpr (NT > 3) f(std::integral_constant<int, 3>{});
        if constexpr (NT > 4) f(std::integral_constant<int, 4>{});
    };

    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int groups = p.k / 128;
    const int part = static_cast<int>(blockIdx.x) / p.spans, span = static_cast<int>(blockIdx.x) % p.spans;
    const int g_lo = part * groups / p.parts, g_hi = (part + 1) * groups / p.parts, gpt = g_hi - g_lo;
    const int tile0 = span * NT;
    const bool swiglu = p.epilogue == SEPAL_HIP_SWIGLU;

    // this wave's groups [u0, u0 + nu): the part's groups dealt in runs, the first gpt mod 8 waves one more
    const int base = gpt / kWaves, rem = gpt % kWaves;
    const int nu = base + (wave < rem ? 1 : 0);
    const int u0 = g_lo + wave * base + min(wave, rem);

    // ---- addresses: 32-bit lane offsets, the group and the tile in the scalar offset; a group past the wave's range is
    // loaded through an empty window (group_window), so every step issues the same loads ----
    const int xrow = lane % 16, kq = lane / 16;
    int xoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) xoff[i] = min(16 * i + xrow, p.t - 1) * p.ld_xb + 32 * kq;
    // weight load e of a tile: rows 8 e + lane / 8 (SwiGLU: 8 gate rows, then the 8 up rows of the same features, 64
    // packed rows further); the lane's slot lane % 8 of its row holds chunk (lane % 8) ^ ((row / 2) % 8)
    int woff[2], wbase[NT];
#pragma unroll
    for (int e = 0; e < 2; ++e)
        woff[e] = (lane / 8 + (swiglu ? 64 : 8) * e) * p.ld_w + 16 * ((lane % 8) ^ ((4 * e + lane / 16) & 7));
    int soff[NT];  // the lane's column's scales
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int tile = min(tile0 + t, p.tiles - 1);  // tiles past the last repeat it and are never stored
        const int row0 = swiglu ? 128 * (tile / 8) + 8 * (tile % 8) : 16 * tile;
        wbase[t] = row0 * p.ld_w;
        const int c = lane % 16, row = row0 + (swiglu && c >= 8 ? 56 + c : c);
        soff[t] = row * p.ld_s * 4;
    }
    const auto uniform = [](int v) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(v); };
    const auto rsrc = [&](const void* ptr, unsigned bytes) __attribute__((always_inline)) {
        // (descriptors and scalar offsets are kept in scalar registers: taken for divergent, each load became a loop over
        // its lanes' values)
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(ptr), 0, uniform(static_cast<int>(bytes)), 0x00020000);
    };

    u32x4 x[2][MT][XL];
    float sc[2][NT];
    // X and the weight scales of unit u into set b
    const auto load_x = [&](int u, int b) __attribute__((always_inline)) {
        const Window win = group_window(u < nu, p.x_bytes, (u0 + u) * 256);
        const __amdgpu_buffer_rsrc_t xr = rsrc(p.x, win.bytes);
        const int so = uniform(win.scalar);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < XL; ++j)
                // k 64 (j / 2) + 16 kq + 8 (j % 2)
                x[b][i][j] = __builtin_bit_cast(
                    u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[i] + 128 * (j / 2) + 16 * (j % 2), so, 0));
    };
    const auto load_sc = [&](int u, int b) __attribute__((always_inline)) {
        const Window win = group_window(u < nu, p.s_bytes, (u0 + u) * 4);
        const __amdgpu_buffer_rsrc_t sr = rsrc(p.s, win.bytes);
        const int so = uniform(win.scalar);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            sc[b][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, soff[t], so, 0));
    };
    const auto load_w = [&](int u, auto it) __attribute__((always_inline)) {
        constexpr int t = decltype(it)::value;
        const Window win = group_window(u < nu, p.w_bytes, wbase[t] + 128 * (u0 + u));
        const __amdgpu_buffer_rsrc_t wr = rsrc(p.w, win.bytes);
        lds_u8* dst = slot(it) + wave * 2048;
        const int so = uniform(win.scalar);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)dst, 16, woff[0], so, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(dst + 1024), 16, woff[1], so, 0, 0);
    };

    load_x(0, 0);
    load_sc(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    each_tile([&](auto it) { load_w(0, it); });
    __builtin_amdgcn_sched_barrier(0);

    float acc[NT][MT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][i][r] = 0.0f;
    // the lane's operand bytes of half h of a slot: weight row lane % 16, chunk 4 h + lane / 16
    int rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd[h] = (lane % 16) * 128 + 16 * ((4 * h + lane / 16) ^ ((lane % 16) / 2));

    // Step u multiplies unit u, tile by tile, with the next tile's operands being read from LDS under this tile's
    // widening and MFMAs; a tile's refill is requested once its operands have arrived. Loads outstanding behind tile t + 1
    // of unit u when it is waited for: the unit's later tiles (2 each), the next unit's X and scales, the next unit's
    // tiles 0 .. t; tile 0 of unit u + 1, read at the end of unit u, has as many behind it.
    constexpr int NX = MT * XL + NT;  // loads of one unit's X and scales
    u32x4 bw[2];
    const auto read = [&](auto it) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        const lds_u8* src = slot(it) + wave * 2048;
        bw[0] = *reinterpret_cast<const lds_u32x4*>(src + rd[0]);
        bw[1] = *reinterpret_cast<const lds_u32x4*>(src + rd[1]);
    };
    const auto refill = [&](int u, auto it) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot is read
        __builtin_amdgcn_sched_barrier(0);
        load_w(u, it);
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto step = [&](int u, auto bt) __attribute__((always_inline)) {
        constexpr int b = decltype(bt)::value;
        load_x(u + 1, b ^ 1);
        load_sc(u + 1, b ^ 1);
        each_tile([&](auto it) __attribute__((always_inline)) {
            constexpr int t = decltype(it)::value;
            const u32x4 b0 = bw[0], b1 = bw[1];
            using Next = std::integral_constant<int, t + 1 < NT ? t + 1 : 0>;
            __builtin_amdgcn_sched_barrier(0);
            wait_vm<2 * (NT - 1) + NX>();
            read(Next{});
            unsigned o[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (XT == SEPAL_HIP_BF16) {
                    s8x4_to_bf16x4(b0[q], o[2 * q], o[2 * q + 1]);
                    s8x4_to_bf16x4(b1[q], o[8 + 2 * q], o[9 + 2 * q]);
                } else {
                    s8x4_to_f16x4(b0[q], o[2 * q], o[2 * q + 1]);
                    s8x4_to_f16x4(b1[q], o[8 + 2 * q], o[9 + 2 * q]);
                }
            }
            f32x4 prt[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) prt[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    prt[i] = mfma_f<XT>(x[b][i][j], u32x4{o[4 * j], o[4 * j + 1], o[4 * j + 2], o[4 * j + 3]}, prt[i]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][i][r] = __builtin_fmaf(prt[i][r], sc[b][t], acc[t][i][r]);
            // (past the last unit the refills and the reads of empty loads are harmless)
            refill(t + 1 < NT ? u + 1 : u + 2, Next{});
        });
    };
    if (nu > 0) {
        wait_vm<2 * (NT - 1)>();  // behind tile 0 of unit 0: its unit's other tiles
        read(std::integral_constant<int, 0>{});
        refill(1, std::integral_constant<int, 0>{});
    }
    for (int u = 0; u < nu;) {
        step(u, std::integral_constant<int, 0>{});
        if (++u >= nu) break;
        step(u, std::integral_constant<int, 1>{});
        ++u;
    }

    // ---- the waves' sum: waves 4-7 hand their tiles to waves 0-3, whose sums are then added in wave order ----
    wait_vm<0>();  // no direct load of this wave may still write a slot
    asm volatile("" ::: "memory");
    __syncthreads();
    if (wave >= 4)
        each_tile([&](auto it) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                const auto& a = acc[decltype(it)::value][i];
                *reinterpret_cast<lds_f32x4*>(slot(it) + (((wave - 4) * MT + i) * 64 + lane) * 16) = f32x4{a[0], a[1], a[2], a[3]};
            }
        });
    __syncthreads();
    if (wave < 4)
        each_tile([&](auto it) __attribute__((always_inline)) {
            constexpr int t = decltype(it)::value;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                lds_f32x4* dst = reinterpret_cast<lds_f32x4*>(slot(it) + ((wave * MT + i) * 64 + lane) * 16);
                f32x4 o = *dst;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = __fadd_rn(acc[t][i][r], o[r]);
                *dst = o;
            }
        });
    __syncthreads();

    // ---- epilogue: an item is (tile, row tile, lane): rows 16 i + 4 (lane / 16) + 0..3 of tile column lane % 16 ----
    const auto total = [&](const lds_u8* s, int i, int l) __attribute__((always_inline)) {
        f32x4 v = *reinterpret_cast<const lds_f32x4*>(s + (i * 64 + l) * 16);
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const f32x4 o = *reinterpret_cast<const lds_f32x4*>(s + ((w * MT + i) * 64 + l) * 16);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = __fadd_rn(v[r], o[r]);
        }
        return v;
    };
    each_tile([&](auto it) __attribute__((always_inline)) {
        constexpr int t = decltype(it)::value;
        const lds_u8* s = slot(it);
        const int tile = tile0 + t;
        if (tile >= p.tiles) return;  // (uniform)
        // the tiles take turns over the waves, so that MT * NT wave-sized items spread over the 8 waves
        const int i = (wave - t * MT % kWaves + kWaves) % kWaves;
        if (i >= MT) return;
        f32x4 v = total(s, i, lane);
        const int r0 = 16 * i + 4 * (lane / 16), c = lane % 16;
        if (swiglu) {
            // gate in columns 0..7, up of the same features in columns 8..15: the lane of a gate column takes rows 0 and 1,
            // the one of its up column rows 2 and 3
            const bool hi = c >= 8;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float own = hi ? v[j + 2] : v[j], other = __shfl_xor(hi ? v[j] : v[j + 2], 8, 64);
                const float gate = hi ? other : own, up = hi ? own : other;
                const int row = r0 + j + (hi ? 2 : 0);
                const float h = p.libm ? swiglu_libm(gate, up) : swiglu_fast(gate, up);
                if (row >= p.t) continue;
                const std::size_t idx = static_cast<std::size_t>(row) * p.ld_y + 64 * (tile / 8) + 8 * (tile % 8) + c % 8;
                if (p.y_type == SEPAL_HIP_F32) store_out<SEPAL_HIP_F32>(p.y, idx, h);
                else if (p.y_type == SEPAL_HIP_BF16) store_out<SEPAL_HIP_BF16>(p.y, idx, h);
                else store_out<SEPAL_HIP_F16>(p.y, idx, h);
            }
            return;
        }
        const int col = 16 * tile + c;
        float* y = static_cast<float*>(p.y);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (r0 + r >= p.t) continue;
            if (p.parts > 1) {
                y[(static_cast<std::size_t>(part) * p.t + r0 + r) * p.n + col] = v[r];
            } else {
                const std::size_t idx = static_cast<std::size_t>(r0 + r) * p.ld_y + col;
                y[idx] = p.epilogue == SEPAL_HIP_ADD ? __fadd_rn(y[idx], v[r]) : v[r];
            }
        }
    });
}

// Weight tiles a block may own: five; three where 64 rows of 16-bit X fill the registers (with five tiles their next
// group's X could only be requested behind its weights: 24.2-25.6 us at 19456 x 2560 against 23.9-24.4 of the large-M
// kernels' plan, and 18.8 against 17.9 at 2560 x 9728).
constexpr int max_nt(int mt) { return mt == 4 ? 3 : 5; }

// ---- launch ----------------------------------------------------------------------------------------------------------

inline int device_cus() {
    static std::atomic<int> cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) throw LaunchError("mid-M multiply: hipGetDevice failed");
    if (dev < 64) {
        const int known = cached[dev].load(std::memory_order_relaxed);
        if (known > 0) return known;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        throw LaunchError("mid-M multiply: device query failed");
    if (dev < 64) cached[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

template <int XT, int MT, int NT>
void launch(const Params& p, hipStream_t stream) {
    mid_kernel<XT, MT, NT><<<dim3(static_cast<unsigned>(p.parts) * p.spans), dim3(kThreads), 0, stream>>>(p);
    check_launch("mid-M multiply launch");
}

template <int XT, int MT>
void launch_nt(const Params& p, int nt, hipStream_t stream) {
    if (nt == 2) {
        launch<XT, MT, 2>(p, stream);
    } else if (nt == 3) {
        launch<XT, MT, 3>(p, stream);
    } else {
        if constexpr (max_nt(MT) >= 5) launch<XT, MT, 5>(p, stream);
        else throw LaunchError("mid-M multiply: no such tile count");
    }
}

template <int XT>
void launch_mt(const Params& p, int nt, hipStream_t stream) {
    if (p.t <= 32) launch_nt<XT, 2>(p, nt, stream);
    else if (p.t <= 48) launch_nt<XT, 3>(p, nt, stream);
    else launch_nt<XT, 4>(p, nt, stream);
}

} // namespace mid

namespace {

bool make_plan(const GemmArgs& a, int max_parts, MidGemmPlan& plan) {
    if (a.config >= 0 || a.t > kSmallM || a.w_stream || a.k % 128 != 0) return false;
    if (a.x_type != SEPAL_HIP_BF16 && a.x_type != SEPAL_HIP_F16) return false;
    const bool swiglu = a.epilogue == SEPAL_HIP_SWIGLU;
    if (swiglu ? a.n % 128 != 0 : (a.n % 16 != 0 || a.y_type != SEPAL_HIP_F32)) return false;
    const std::size_t lim = std::size_t{1} << 31;
    if (a.t * a.ld_x * 2 >= lim || a.n * a.ld_w >= lim || a.n * a.ld_s * 4 >= lim) return false;
    const int cus = mid::device_cus();
    const int tiles = static_cast<int>(a.n / 16), groups = static_cast<int>(a.k / 128);
    const int mt = a.t <= 32 ? 2 : (a.t <= 48 ? 3 : 4);
    const int max_nt = mid::max_nt(mt);
    // With three tiles a block, more than one round of blocks is slower than the large-M kernels' plan (49-64 rows of
    // 16-bit X: 32-36 against 24-25 us at 19456 x 2560, 36-41 against 25 at 20480 x 3072; level at 12288 x 2560, one
    // round).
    if (max_nt == 3 && (tiles + 2) / 3 > cus) return false;
    const double x_kb = mt * 4.0;  // X of one group
    double best = 0.0;
    for (const int nt : {5, 3, 2}) {
        if (nt > max_nt) continue;
        const int spans = (tiles + nt - 1) / nt;
        for (int kp = 1; kp <= max_parts && (kp == 1 || (!swiglu && groups / kp >= 4)); ++kp) {
            if (kp > 1 && static_cast<std::size_t>(kp) * a.t * a.n * sizeof(float) > kPartialBytes) break;
            const int gpt = (groups + kp - 1) / kp;
            // the kilobytes a CU streams (the groups of a part go to a SIMD's two waves, four SIMDs), and the parts' sum
            const int rounds = (kp * spans + cus - 1) / cus;
            const double cost = static_cast<double>(rounds) * 4 * ((gpt + 3) / 4) * (2.0 * nt + x_kb) + 20.0 * rounds +
                                (kp > 1 ? 40.0 + 2.0 * kp * a.t * a.n * 4 / 1024 / cus : 0.0);
            if (best == 0.0 || cost < best) {
                best = cost;
                plan.nt = nt;
                plan.parts = kp;
            }
        }
    }
    return true;
}

// The multiply alone: Y, or its K-parts [plan.parts][t][n] at part.
void launch_multiply(const GemmArgs& a, const MidGemmPlan& plan, float* part, hipStream_t stream) {
    mid::Params p{};
    p.x = a.x;
    p.x_bytes = static_cast<unsigned>(((a.t - 1) * a.ld_x + a.k) * 2);
    p.ld_xb = static_cast<int>(a.ld_x * 2);
    p.w = reinterpret_cast<const signed char*>(a.w);
    p.w_bytes = static_cast<unsigned>((a.n - 1) * a.ld_w + a.k);
    p.ld_w = static_cast<int>(a.ld_w);
    p.s = a.s;
    p.s_bytes = static_cast<unsigned>(((a.n - 1) * a.ld_s + a.k / 128) * 4);
    p.ld_s = static_cast<int>(a.ld_s);
    p.y = part != nullptr ? static_cast<void*>(part) : a.y;
    p.ld_y = part != nullptr ? a.n : a.ld_y;
    p.y_type = a.y_type;
    p.epilogue = a.epilogue;
    // the silu of the kernels that ran, and run what this one refuses, at these sizes: the streaming kernel's up to 32 rows with
    // N < 8192 (closer to silu(g) u by a third in rms, and finite where g u is not), the large-M kernels' elsewhere
    // (the libm form there, on the gate columns' lanes alone, took 19.9 / 25.0 us at 19456 x 2560 and 17 / 48 rows against
    // 17.4 / 21.8; with the lanes shared as now 4096 x 1024 at 17 / 32 rows takes 6.7 / 7.6 with it and 6.3 / 7.1 took the
    // fast form before)
    p.libm = a.t <= 32 && a.n < 8192;
    p.t = static_cast<int>(a.t);
    p.n = static_cast<int>(a.n);
    p.k = static_cast<int>(a.k);
    p.tiles = static_cast<int>(a.n / 16);
    p.parts = plan.parts;
    p.spans = (p.tiles + plan.nt - 1) / plan.nt;
    if (a.x_type == SEPAL_HIP_BF16) mid::launch_mt<SEPAL_HIP_BF16>(p, plan.nt, stream);
    else mid::launch_mt<SEPAL_HIP_F16>(p, plan.nt, stream);
}

float* partial_zone(const GemmArgs& a) {
    if (a.scratch == nullptr) throw LaunchError("mid-M multiply: scratch missing");
    return reinterpret_cast<float*>(static_cast<char*>(a.scratch) + kCounterBytes);
}

// The multiply of the hi and lo rows of a float32 X as one of 2 T bf16 rows.
GemmArgs pairs_args(const GemmArgs& a) {
    GemmArgs b = a;
    b.x_type = SEPAL_HIP_BF16;
    b.ld_x = a.k;
    b.t = 2 * a.t;
    b.epilogue = SEPAL_HIP_STORE;
    return b;
}

} // namespace

bool mid_gemm_plan(const GemmArgs& a, MidGemmPlan& plan) { return make_plan(a, 16, plan); }

void launch_mid_gemm(const GemmArgs& a, const MidGemmPlan& plan, hipStream_t stream) {
    float* const part = plan.parts > 1 ? partial_zone(a) : nullptr;
    launch_multiply(a, plan, part, stream);
    if (part != nullptr)
        launch_parts_add(plan.parts, a.epilogue == SEPAL_HIP_ADD, a.t, a.n, part, static_cast<float*>(a.y), a.ld_y, stream);
}

// A float32 X of up to 24 rows, N < 8192: its hi and lo rows are one multiply of up to 48 rows, which reads the weights
// once, where two multiplies read them twice. Measured (us a call, graph replays over cold weights, the split included):
// 2560 x 9728 at 1 / 16 / 24 rows 28.0 / 30.9 / 29.8 -> 16.2 / 19.0 / 21.3, 2560 x 4096 21.8 / 23.6 / 22.7 -> 11.7 / 13.8 /
// 15.7, 1024 x 4096 19.1 / 20.6 / 16.8 -> 9.2 / 10.7 / 11.9; 1.1 to 2.2 times over N 1024 .. 8176, K 1024 .. 5120. At 25 to 32
// rows (three tiles a block) 6656 x 5120 took 36.2 against 35.0; from N = 8192 the other route is one pass of the large-M
// hi + lo form, and 10496 x 5120 took 36.6 against 30.8 at 17 rows. What bounds it: the split, the multiply and the sum are
// three dependent launches around one pass over the weights. SwiGLU keeps its own route (the sum comes before the silu).
bool mid_pairs_plan(const GemmArgs& a, MidGemmPlan& plan) {
    if (a.x_type != SEPAL_HIP_F32 || a.epilogue == SEPAL_HIP_SWIGLU || a.t > 24 || a.n >= 8192) return false;
    const GemmArgs b = pairs_args(a);
    // (the sum takes 16 parts: hi and lo of up to 8)
    return 2 * a.t * a.n * sizeof(float) <= kPartialBytes && make_plan(b, 8, plan);
}

void launch_mid_pairs(const GemmArgs& a, const MidGemmPlan& plan, const void* pairs, hipStream_t stream) {
    GemmArgs b = pairs_args(a);
    b.x = pairs;
    float* const part = partial_zone(a);
    launch_multiply(b, plan, part, stream);
    // [parts][2 T][n]: each part's hi rows, then its lo rows, are two planes of [T][n]
    launch_parts_add(2 * plan.parts, a.epilogue == SEPAL_HIP_ADD, a.t, a.n, part, static_cast<float*>(a.y), a.ld_y, stream);
}

} // namespace sepal::hip
