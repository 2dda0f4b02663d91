// The C ABI of sepal_mlp_hip (declarations and conventions: include/sepal_mlp_hip.h).
//
// Error handling follows runner/src/capi/c_api.cpp:28-43: every entry point runs its body under one guard that turns
// std::invalid_argument into SEPAL_HIP_EINVAL and any other exception into SEPAL_HIP_ELAUNCH, keeping the message in a
// thread-local string for sepal_hip_last_error(). The argument checks restate the reference's requirement functions
// (gemm_simt_supports, runner/cuda/src/gemm_simt_kernels.cu:303-310; the checks of launch_quantize_rows_s8 and
// launch_gemm_s8, runner/cuda/src/gemm_s8_kernels.cu:472-546) for the shapes this library takes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <cstdlib>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <utility>
#include <vector>

#include "common.hpp"
#include "gemm_kernels.hpp"
#include "stack_glue.hpp"

namespace sepal::hip {

namespace {

thread_local std::string g_error;

template <class F>
int32_t guarded(F&& f) {
    try {
        f();
        return SEPAL_HIP_OK;
    } catch (const std::invalid_argument& e) {
        g_error = e.what();
        return SEPAL_HIP_EINVAL;
    } catch (const std::bad_alloc& e) {
        g_error = std::string("out of memory: ") + e.what();
        return SEPAL_HIP_ENOMEM;
    } catch (const IoError& e) {
        g_error = e.what();
        return SEPAL_HIP_EIO;
    } catch (const StaleError& e) {
        g_error = e.what();
        return SEPAL_HIP_ESTALE;
    } catch (const std::exception& e) {
        g_error = e.what();
        return SEPAL_HIP_ELAUNCH;
    } catch (...) {
        g_error = "unknown error";
        return SEPAL_HIP_ELAUNCH;
    }
}

inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

bool valid_type(int t) { return t == SEPAL_HIP_F32 || t == SEPAL_HIP_BF16 || t == SEPAL_HIP_F16; }

// One workspace per (device, stream). Work that uses a workspace is enqueued only on its own stream, so growing it
// waits for that stream alone before the old buffer is freed, and two streams (or two engines with their own streams)
// never share counters or scratch. A Lease holds the workspace's mutex from the size check to the end of the entry
// point's enqueueing, so a second thread on the same stream cannot free the buffer under a call that is still
// enqueueing work on it.
struct Workspace {
    std::mutex m;
    void* ptr = nullptr;
    std::size_t bytes = 0;
};
__global__ void zero_words_kernel(unsigned* p, std::size_t n) {
    for (std::size_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += static_cast<std::size_t>(gridDim.x) * 256) p[i] = 0u;
}

std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, std::unique_ptr<Workspace>> g_ws;

} // namespace

Lease::Lease(std::size_t bytes, hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) throw LaunchError("hipGetDevice failed");
    Workspace* w;
    {
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        auto& slot = g_ws[{dev, stream}];
        if (!slot) slot = std::make_unique<Workspace>();
        w = slot.get();
    }
    lock_ = std::unique_lock<std::mutex>(w->m);
    if (w->bytes < bytes) {
        // the old buffer may still be read by work queued on this stream: wait for it before freeing
        if (w->ptr != nullptr) {
            if (hipStreamSynchronize(stream) != hipSuccess) throw LaunchError("hipStreamSynchronize failed");
            (void)hipFree(w->ptr);
            w->ptr = nullptr;
            w->bytes = 0;
        }
        const std::size_t grown = bytes < (std::size_t{64} << 20) ? (std::size_t{64} << 20) : bytes;
        if (hipMalloc(&w->ptr, grown) != hipSuccess) throw std::bad_alloc();
        // The split-K counters must be zero before the first kernel that uses them. hipMemset would run on the null
        // stream, which a non-blocking caller stream does not wait for (its first kernel could count in while the
        // zeros are still being written, and a span's last block would never see the full count); a fill kernel on
        // the workspace's own stream is ordered before every later use. (Only the counter zone needs zeros: every
        // partial is written before it is read.)
        zero_words_kernel<<<dim3(64), dim3(256), 0, stream>>>(static_cast<unsigned*>(w->ptr), kCounterBytes / 4);
        if (hipGetLastError() != hipSuccess) throw LaunchError("the workspace's counter fill failed to launch");
        w->bytes = grown;
    }
    base_ = static_cast<char*>(w->ptr);
}

namespace {

void check_gemm_common(const char* who, const void* x, std::size_t ld_x, const void* w, std::size_t ld_w,
                       const void* s, std::size_t ld_s, const void* y, std::size_t ld_y, std::size_t n, std::size_t k,
                       int epilogue) {
    const std::string w_ = who;
    require(x != nullptr && w != nullptr && s != nullptr && y != nullptr, w_ + ": null pointer");
    require(epilogue == SEPAL_HIP_STORE || epilogue == SEPAL_HIP_ADD || epilogue == SEPAL_HIP_SWIGLU, w_ + ": unknown epilogue");
    require(n != 0 && k != 0 && k % 128 == 0, w_ + ": K must be a non-zero multiple of 128 and N non-zero");
    require(ld_x >= k && ld_w >= k && ld_x % 16 == 0 && ld_w % 16 == 0, w_ + ": row strides of X and W must be multiples of 16 and at least K");
    require(ld_s >= k / 128, w_ + ": the scale row stride must hold K/128 scales");
    require(aligned16(x) && aligned16(w) && aligned16(y), w_ + ": X, W and Y must be 16-byte aligned");
    if (epilogue == SEPAL_HIP_SWIGLU) require(n % 128 == 0 && ld_y >= n / 2, w_ + ": SwiGLU needs N a multiple of 128 and ld_y >= N/2");
    else require(n % 16 == 0 && ld_y >= n, w_ + ": N must be a multiple of 16 and ld_y >= N");
    require(ld_y % 4 == 0, w_ + ": ld_y must be a multiple of 4");
    require(n < 0x7FFFFFFFu && k < 0x7FFFFFFFu, w_ + ": dimension beyond 2^31");
}

// gemm_simt_supports for int8-group weights (runner/cuda/src/gemm_simt_kernels.cu:303-310): K a multiple of 128, X rows
// of whole 4-value multiples, W rows of whole 16 bytes, Y rows of 4-value multiples; SwiGLU N a multiple of 128, Store /
// Add any N.
bool w8g_shape_ok(std::size_t n, std::size_t k, std::size_t ld_x, std::size_t ld_w, std::size_t ld_y, int epilogue) {
    if (k == 0 || n == 0 || k % 128 != 0 || ld_x % 4 != 0 || ld_x < k || ld_w < k || ld_y % 4 != 0 || ld_w % 16 != 0) return false;
    if (epilogue == SEPAL_HIP_SWIGLU) return n % 128 == 0 && ld_y >= n / 2;
    return ld_y >= n;
}

inline std::size_t up256(std::size_t b) { return (b + 255) / 256 * 256; }

// Scratch of one launch_gemm_w8g call beyond the counter zone: its split / sum buffers, then the weight image.
std::size_t w8g_call_bytes(const GemmArgs& a) { return up256(gemm_w8g_scratch_bytes(a)) + gemm_w8g_image_bytes(a); }

void w8g_call(GemmArgs a, char* ws, char* zone, hipStream_t st) {
    const std::size_t extra = up256(gemm_w8g_scratch_bytes(a));
    const std::size_t img = gemm_w8g_image_bytes(a);
    a.scratch = ws;
    a.xsplit = zone;
    a.ytmp = reinterpret_cast<float*>(zone + gemm_w8g_split_bytes(a));
    a.wimage = img != 0 ? zone + extra : nullptr;
    a.wimage_bytes = img;
    launch_gemm_w8g(a, st);
}

// One w8g multiply for every shape w8g_shape_ok takes. The kernels read 16-bit X in 16-byte row chunks and write Store
// / Add outputs in 16-column tiles; the rest is staged (edge.hip): a 16-bit X whose rows are not 16-byte multiples (or
// aligned) is copied to a contiguous [t, k] buffer, and the last N mod 16 columns run as one zero-padded 16-row weight
// tile whose float32 outputs are then stored or added into Y. `a` holds the caller's arguments.
struct W8gAnyLayout {
    std::size_t x_bytes = 0, call = 0, wt = 0, st = 0, yt = 0, total = 0;
    std::size_t n16 = 0, rest = 0;
};

W8gAnyLayout w8g_any_layout(const GemmArgs& a) {
    W8gAnyLayout L;
    const bool sixteen = a.x_type != SEPAL_HIP_F32;
    if (sixteen && (a.ld_x % 16 != 0 || !aligned16(a.x))) L.x_bytes = up256(a.t * a.k * 2);
    L.rest = a.epilogue == SEPAL_HIP_SWIGLU ? 0 : a.n % 16;
    L.n16 = a.n - L.rest;
    GemmArgs m = a, tl = a;
    if (L.x_bytes != 0) m.ld_x = tl.ld_x = a.k;
    m.n = L.n16;
    tl.n = 16;
    tl.ld_w = a.k;
    tl.ld_s = a.k / 128;
    tl.y_type = SEPAL_HIP_F32;
    tl.ld_y = 16;
    tl.epilogue = SEPAL_HIP_STORE;
    L.call = std::max(L.n16 != 0 ? w8g_call_bytes(m) : 0, L.rest != 0 ? w8g_call_bytes(tl) : 0);
    if (L.rest != 0) {
        L.wt = up256(16 * a.k);
        L.st = up256(16 * (a.k / 128) * 4);
        L.yt = up256(a.t * 16 * 4);
    }
    L.total = L.x_bytes + L.call + L.wt + L.st + L.yt;
    return L;
}

void w8g_any(GemmArgs a, const W8gAnyLayout& L, char* ws, char* zone, hipStream_t st) {
    char* p = zone;
    if (L.x_bytes != 0) {
        launch_pad_rows(a.x, a.ld_x * 2, p, a.k * 2, a.t, a.k * 2, st);
        a.x = p;
        a.ld_x = a.k;
        p += L.x_bytes;
    }
    char* call = p;
    p += L.call;
    if (L.n16 != 0) {
        GemmArgs m = a;
        m.n = L.n16;
        w8g_call(m, ws, call, st);
    }
    if (L.rest == 0) return;
    auto* wt = reinterpret_cast<std::int8_t*>(p);
    auto* sc = reinterpret_cast<float*>(p + L.wt);
    auto* yt = reinterpret_cast<float*>(p + L.wt + L.st);
    const std::size_t groups = a.k / 128;
    // the last rows of W and their scales, then zero rows up to 16
    launch_pad_rows(a.w + L.n16 * a.ld_w, a.ld_w, wt, a.k, L.rest, a.k, st);
    launch_pad_rows(nullptr, 0, wt + L.rest * a.k, a.k, 16 - L.rest, 0, st);
    launch_pad_rows(a.s + L.n16 * a.ld_s, a.ld_s * 4, sc, groups * 4, L.rest, groups * 4, st);
    launch_pad_rows(nullptr, 0, sc + L.rest * groups, groups * 4, 16 - L.rest, 0, st);
    GemmArgs tl = a;
    tl.w = wt;
    tl.ld_w = a.k;
    tl.s = sc;
    tl.ld_s = groups;
    tl.n = 16;
    tl.y = yt;
    tl.y_type = SEPAL_HIP_F32;
    tl.ld_y = 16;
    tl.epilogue = SEPAL_HIP_STORE;
    w8g_call(tl, ws, call, st);
    const std::size_t eb = a.y_type == SEPAL_HIP_F32 ? 4 : 2;
    launch_put_cols(yt, 16, static_cast<char*>(a.y) + L.n16 * eb, a.y_type, a.ld_y, a.t, L.rest, a.epilogue == SEPAL_HIP_ADD, st);
}

} // namespace
} // namespace sepal::hip

using namespace sepal::hip;

extern "C" {

int32_t sepal_hip_api_version(void) { return SEPAL_HIP_API_VERSION; }

int32_t sepal_hip_release_workspace(void* stream) {
    return guarded([&] {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) throw LaunchError("hipGetDevice failed");
        const hipStream_t st = as_stream(stream);
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        auto it = g_ws.find({dev, st});
        if (it == g_ws.end()) return;
        {
            // (waits for a call that is still enqueueing on this stream, then for the stream's work)
            std::lock_guard<std::mutex> held(it->second->m);
            if (it->second->ptr != nullptr) {
                if (hipStreamSynchronize(st) != hipSuccess) throw LaunchError("release_workspace: hipStreamSynchronize failed");
                if (hipFree(it->second->ptr) != hipSuccess) throw LaunchError("release_workspace: hipFree failed");
                it->second->ptr = nullptr;
                it->second->bytes = 0;
            }
        }
        g_ws.erase(it);
    });
}



const char* sepal_hip_last_error(void) { return g_error.c_str(); }

int32_t sepal_hip_quantize_group_s8(const void* src, int32_t src_type, size_t ld_src, int8_t* q, size_t ld_q, float* s,
                                    size_t ld_s, size_t rows, size_t k, int32_t rule, void* stream) {
    return guarded([&] {
        require(valid_type(src_type), "quantize_group_s8: unknown source type");
        require(rule == SEPAL_HIP_RULE_DIVIDE || rule == SEPAL_HIP_RULE_RECIPROCAL, "quantize_group_s8: unknown rule");
        require(k % 128 == 0, "quantize_group_s8: K must be a multiple of 128");
        if (rows == 0 || k == 0) return;
        require(src != nullptr && q != nullptr && s != nullptr, "quantize_group_s8: null pointer");
        require(ld_src >= k && ld_q >= k && ld_s >= k / 128 && ld_src % 16 == 0 && ld_q % 16 == 0,
                "quantize_group_s8: strides must be at least K (K/128 for scales) and multiples of 16");
        require(aligned16(src) && aligned16(q), "quantize_group_s8: src and q must be 16-byte aligned");
        launch_quantize_group(src, src_type, ld_src, nullptr, q, ld_q, s, ld_s, rows, k, rule, 0, as_stream(stream));
    });
}

int32_t sepal_hip_quantize_gate_up_s8(const void* gate, const void* up, int32_t src_type, size_t ld_src, int8_t* q,
                                      size_t ld_q, float* s, size_t ld_s, size_t inter, size_t k, int32_t rule,
                                      void* stream) {
    return guarded([&] {
        require(valid_type(src_type), "quantize_gate_up_s8: unknown source type");
        require(rule == SEPAL_HIP_RULE_DIVIDE || rule == SEPAL_HIP_RULE_RECIPROCAL, "quantize_gate_up_s8: unknown rule");
        require(k % 128 == 0 && inter % 64 == 0, "quantize_gate_up_s8: K must be a multiple of 128 and inter of 64");
        if (inter == 0 || k == 0) return;
        require(gate != nullptr && up != nullptr && q != nullptr && s != nullptr, "quantize_gate_up_s8: null pointer");
        require(ld_src >= k && ld_q >= k && ld_s >= k / 128 && ld_src % 16 == 0 && ld_q % 16 == 0,
                "quantize_gate_up_s8: strides must be at least K (K/128 for scales) and multiples of 16");
        require(aligned16(gate) && aligned16(up) && aligned16(q), "quantize_gate_up_s8: pointers must be 16-byte aligned");
        launch_quantize_group(gate, src_type, ld_src, up, q, ld_q, s, ld_s, 2 * inter, k, rule, inter, as_stream(stream));
    });
}

int32_t sepal_hip_gemm_w8g_supports(int32_t x_type, size_t n, size_t k, size_t ld_x, size_t ld_w, size_t ld_y,
                                    int32_t epilogue) {
    if (!valid_type(x_type)) return 0;
    if (epilogue != SEPAL_HIP_STORE && epilogue != SEPAL_HIP_ADD && epilogue != SEPAL_HIP_SWIGLU) return 0;
    return w8g_shape_ok(n, k, ld_x, ld_w, ld_y, epilogue) ? 1 : 0;
}

int32_t sepal_hip_gemm_w8g(const void* x, int32_t x_type, size_t ld_x, const int8_t* w, size_t ld_w, const float* s,
                           size_t ld_s, void* y, int32_t y_type, size_t ld_y, size_t t, size_t n, size_t k,
                           int32_t epilogue, int32_t config, void* stream) {
    return guarded([&] {
        require(valid_type(x_type), "gemm_w8g: X must be float32, bf16 or binary16");
        require(valid_type(y_type), "gemm_w8g: unknown output type");
        require(epilogue == SEPAL_HIP_STORE || epilogue == SEPAL_HIP_ADD || epilogue == SEPAL_HIP_SWIGLU, "gemm_w8g: unknown epilogue");
        require(epilogue == SEPAL_HIP_SWIGLU || y_type == SEPAL_HIP_F32, "gemm_w8g: Store and Add write float32");
        require(config >= -1 && config <= 2, "gemm_w8g: config must be -1, 0, 1 or 2");
        require(x != nullptr && w != nullptr && s != nullptr && y != nullptr, "gemm_w8g: null pointer");
        // the message of launch_gemm_simt (runner/cuda/src/gemm_simt_kernels.cu:314-318)
        require(w8g_shape_ok(n, k, ld_x, ld_w, ld_y, epilogue),
                "gemm_w8g: unsupported shape [" + std::to_string(t) + " x " + std::to_string(k) + "] by [" + std::to_string(n) +
                    " x " + std::to_string(k) + "] (K a multiple of 128; strides multiples of 4 values and W rows of 16 "
                    "bytes; SwiGLU needs N a multiple of 128)");
        require(ld_s >= k / 128, "gemm_w8g: the scale row stride must hold K/128 scales");
        require((x_type != SEPAL_HIP_F32 || aligned16(x)) && aligned16(w) && aligned16(y),
                "gemm_w8g: float32 X, W and Y must be 16-byte aligned");
        require(n < 0x7FFFFFFFu && k < 0x7FFFFFFFu, "gemm_w8g: dimension beyond 2^31");
        if (t == 0) return;
        require(t < 0x7FFFFFFFu, "gemm_w8g: dimension beyond 2^31");
        if (config >= 1) require(t <= kSmallM, "gemm_w8g: the small-M path takes at most 64 rows");
        GemmArgs a;
        a.x = x;
        a.x_type = x_type;
        a.ld_x = ld_x;
        a.w = w;
        a.ld_w = ld_w;
        a.s = s;
        a.ld_s = ld_s;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = epilogue;
        a.config = config == 2 ? 1 : config;
        a.force_splits = config == 2 ? 1 : 0;
        const hipStream_t st = as_stream(stream);
        const W8gAnyLayout L = w8g_any_layout(a);
        Lease ws(kScratchOffset + L.total, st);
        w8g_any(a, L, ws.base(), ws.base() + kScratchOffset, st);
    });
}

int32_t sepal_hip_quantize_rows_s8(const void* x, int32_t x_type, size_t ld_x, int8_t* q, size_t ld_q, float* scales,
                                   size_t ld_s, size_t rows, size_t cols, size_t block, void* stream) {
    return guarded([&] {
        require(valid_type(x_type), "quantize_rows_s8: unknown source type");
        require(block == 128 || block == cols, "quantize_rows_s8: block must be 128 or cols");
        if (rows == 0 || cols == 0) return;
        require(x != nullptr && q != nullptr && scales != nullptr, "quantize_rows_s8: null pointer");
        require(ld_x >= cols && ld_q >= cols && ld_s >= cols / block, "quantize_rows_s8: strides must hold the row");
        if (block == 128) {
            // per 128 (pack_acts I8_Z): whole groups of 16-byte chunks
            require(cols % 128 == 0, "quantize_rows_s8: cols must be a multiple of 128");
            require(ld_x % 16 == 0 && ld_q % 16 == 0, "quantize_rows_s8: strides must be multiples of 16");
            require(aligned16(x) && aligned16(q), "quantize_rows_s8: pointers must be 16-byte aligned");
        }
        // (one scale per row takes any length, stride and alignment: kernel_i8_y's packing, runner/src/cpu/gemm.cpp:286-306)
        launch_quantize_rows(x, x_type, ld_x, q, ld_q, scales, ld_s, rows, cols, block, as_stream(stream));
    });
}

int32_t sepal_hip_gemm_q8(const int8_t* xq, size_t ld_x, const float* xs, size_t ld_xs, size_t act_block,
                          const int8_t* w, size_t ld_w, const float* ws, size_t ld_ws, void* y, int32_t y_type,
                          size_t ld_y, size_t t, size_t n, size_t k, int32_t epilogue, int32_t config, void* stream) {
    return guarded([&] {
        require(valid_type(y_type), "gemm_q8: unknown output type");
        require(epilogue == SEPAL_HIP_SWIGLU || y_type == SEPAL_HIP_F32, "gemm_q8: Store and Add write float32");
        require(config >= -1 && config <= 2, "gemm_q8: config must be -1, 0, 1 or 2");
        check_gemm_common("gemm_q8", xq, ld_x, w, ld_w, ws, ld_ws, y, ld_y, n, k, epilogue);
        require(act_block == 128 || act_block == k, "gemm_q8: act_block must be 128 or K");
        require(xs != nullptr && ld_xs >= k / act_block, "gemm_q8: activation scales missing or stride too small");
        if (t == 0) return;
        require(t < 0x7FFFFFFFu, "gemm_q8: dimension beyond 2^31");
        if (config >= 1) require(t <= kSmallM, "gemm_q8: the small-M path takes at most 64 rows");
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.xs = xs;
        a.ld_xs = ld_xs;
        a.act_block = act_block;
        a.w = w;
        a.ld_w = ld_w;
        a.s = ws;
        a.ld_s = ld_ws;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = epilogue;
        a.config = config == 2 ? 1 : config;
        a.force_splits = config == 2 ? 1 : 0;
        Lease ws(kScratchOffset, as_stream(stream));
        a.scratch = ws.base();
        launch_gemm_q8(a, as_stream(stream));
    });
}

int32_t sepal_hip_s8_quantize_rows(const void* x, int32_t x_type, size_t ld_x, const float* smooth, int8_t* q, size_t ld_q,
                                   float* scales, size_t rows, size_t cols, void* stream) {
    return guarded([&] {
        require(x != nullptr && q != nullptr && scales != nullptr, "s8_quantize_rows: null pointer");
        require(valid_type(x_type), "s8_quantize_rows: unknown input type");
        require(cols != 0 && cols % 16 == 0, "s8_quantize_rows: cols must be a non-zero multiple of 16");
        require(ld_x >= cols && ld_q >= cols && ld_x % 16 == 0 && ld_q % 16 == 0,
                "s8_quantize_rows: row strides must be multiples of 16 and at least cols");
        require(aligned16(x) && aligned16(q) && (smooth == nullptr || aligned16(smooth)),
                "s8_quantize_rows: x, q and smooth must be 16-byte aligned");
        if (rows == 0) return;
        require(rows < 0x7FFFFFFFu, "s8_quantize_rows: dimension beyond 2^31");
        launch_s8_quantize_rows(x, x_type, ld_x, smooth, q, ld_q, scales, rows, cols, as_stream(stream));
    });
}

int32_t sepal_hip_column_absmax(const void* x, size_t ld_x, float* out, size_t rows, size_t cols, void* stream) {
    return guarded([&] {
        require(x != nullptr && out != nullptr, "column_absmax: null pointer");
        require(ld_x >= cols && cols < 0x7FFFFFFFu, "column_absmax: stride below the column count");
        if (cols == 0) return;
        launch_column_stats(x, ld_x, rows, cols, out, nullptr, as_stream(stream));
    });
}

int32_t sepal_hip_channel_stats(const void* x, size_t ld_x, size_t rows, size_t cols, float* amax, double* sums,
                                void* stream) {
    return guarded([&] {
        require(x != nullptr && amax != nullptr && sums != nullptr, "channel_stats: null pointer");
        require(ld_x >= cols && cols < 0x7FFFFFFFu, "channel_stats: stride below the column count");
        if (cols == 0) return;
        launch_column_stats(x, ld_x, rows, cols, amax, sums, as_stream(stream));
    });
}

namespace {
// The checks of launch_gemm_s8 (runner/cuda/src/gemm_s8_kernels.cu:522-531), after its T = 0 / N = 0 no-op.
void check_s8(const void* x, size_t ld_x, const float* sx, const void* w, size_t ld_w, const float* sw, const void* y,
              int32_t y_type, size_t ld_y, size_t n, size_t k) {
    require(x != nullptr && w != nullptr && sx != nullptr && sw != nullptr && y != nullptr, "gemm_s8: null pointer");
    require(y_type == SEPAL_HIP_F32 || y_type == SEPAL_HIP_F16, "gemm_s8: the output is float32 or binary16");
    require(k != 0 && k % 16 == 0 && ld_x >= k && ld_w >= k && ld_x % 16 == 0 && ld_w % 16 == 0 && n % 2 == 0 && ld_y % 2 == 0 &&
                ld_y >= n,
            "gemm_s8: K and the row strides of X and W must be multiples of 16 (strides at least K), N and the row stride "
            "of Y even (at least N)");
    require(aligned16(x) && aligned16(w) && aligned8(y) && reinterpret_cast<std::uintptr_t>(sx) % 4 == 0 &&
                reinterpret_cast<std::uintptr_t>(sw) % 4 == 0,
            "gemm_s8: X and W must be 16-byte aligned, Y 8-byte aligned, the scales 4-byte aligned");
}
} // namespace

// gemm_s8_supports (runner/cuda/src/gemm_s8_kernels.hpp:59-61), the same predicate.
int32_t sepal_hip_gemm_s8_supports(size_t n, size_t k, size_t ld_x, size_t ld_w, size_t ld_y) {
    return k != 0 && k % 16 == 0 && ld_x % 16 == 0 && ld_w % 16 == 0 && ld_x >= k && ld_w >= k && n % 2 == 0 && ld_y % 2 == 0 &&
                   ld_y >= n
               ? 1
               : 0;
}

// gemm_w8a16_supports (runner/cuda/src/gemm_s8_kernels.hpp:62-64), the same predicate.
int32_t sepal_hip_gemm_w8a16_supports(size_t n, size_t k, size_t ld_x, size_t ld_w, size_t ld_y) {
    return k != 0 && k % 16 == 0 && ld_x % 8 == 0 && ld_w % 16 == 0 && ld_x >= k && ld_w >= k && n % 2 == 0 && ld_y % 2 == 0 &&
                   ld_y >= n
               ? 1
               : 0;
}

int32_t sepal_hip_gemm_s8(const int8_t* xq, size_t ld_x, const float* sx, const int8_t* wq, size_t ld_w, const float* sw,
                          void* y, int32_t y_type, size_t ld_y, size_t t, size_t n, size_t k, void* stream) {
    return guarded([&] {
        if (t == 0 || n == 0) return;
        check_s8(xq, ld_x, sx, wq, ld_w, sw, y, y_type, ld_y, n, k);
        require(t < 0x7FFFFFFFu && n < 0x7FFFFFFFu, "gemm_s8: dimension beyond 2^31");
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.xs = sx;
        a.ld_xs = 1;
        a.act_block = k;
        a.w = wq;
        a.ld_w = ld_w;
        a.s = sw;
        a.ld_s = 1;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = SEPAL_HIP_STORE;
        launch_gemm_s8(a, as_stream(stream));
    });
}

int32_t sepal_hip_gemm_q8y(const int8_t* xq, size_t ld_x, const float* xs, const int8_t* wq, size_t ld_w, const float* ws,
                           void* y, int32_t y_type, size_t ld_y, size_t t, size_t n, size_t k, int32_t epilogue, void* stream) {
    return guarded([&] {
        require(xq != nullptr && xs != nullptr && wq != nullptr && ws != nullptr && y != nullptr, "gemm_q8y: null pointer");
        require(epilogue == SEPAL_HIP_STORE || epilogue == SEPAL_HIP_ADD || epilogue == SEPAL_HIP_SWIGLU, "gemm_q8y: unknown epilogue");
        require(valid_type(y_type), "gemm_q8y: unknown output type");
        require(epilogue == SEPAL_HIP_SWIGLU || y_type == SEPAL_HIP_F32, "gemm_q8y: Store and Add write float32");
        require(n != 0 && k != 0, "gemm_q8y: K and N must be non-zero");
        require(ld_x >= k && ld_w >= k, "gemm_q8y: row strides of X and W must be at least K");
        if (epilogue == SEPAL_HIP_SWIGLU) require(n % 128 == 0 && ld_y >= n / 2, "gemm_q8y: SwiGLU needs N a multiple of 128 and ld_y >= N/2");
        else require(ld_y >= n, "gemm_q8y: ld_y must be at least N");
        require(reinterpret_cast<std::uintptr_t>(y) % 4 == 0, "gemm_q8y: Y must be 4-byte aligned");
        if (t == 0) return;
        require(t < 0x7FFFFFFFu && n < 0x7FFFFFFFu && k < 0x7FFFFFFFu, "gemm_q8y: dimension beyond 2^31");
        const hipStream_t st = as_stream(stream);
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.xs = xs;
        a.ld_xs = 1;
        a.act_block = k;
        a.w = wq;
        a.ld_w = ld_w;
        a.s = ws;
        a.ld_s = 1;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = epilogue;
        // kernel_i8_y takes any K (runner/src/cpu/gemm_kernels_avx2.cpp:40-76). The kernel reads whole 16-byte chunks,
        // so K off the 16-grid, or rows that are not 16-byte multiples or aligned, run on zero-padded copies: a zero
        // byte adds an exact zero to the int32 sum, so the sums and every output bit are the unpadded ones.
        if (k % 16 != 0 || ld_x % 16 != 0 || ld_w % 16 != 0 || !aligned16(xq) || !aligned16(wq)) {
            const std::size_t kp = (k + 15) / 16 * 16, xb = up256(t * kp);
            Lease lease(kScratchOffset + xb + up256(n * kp), st);
            char* xp = lease.base() + kScratchOffset;
            char* wp = xp + xb;
            launch_pad_rows(xq, ld_x, xp, kp, t, k, st);
            launch_pad_rows(wq, ld_w, wp, kp, n, k, st);
            a.x = xp;
            a.ld_x = kp;
            a.w = reinterpret_cast<const std::int8_t*>(wp);
            a.ld_w = kp;
            a.k = kp;
            a.act_block = kp;
            launch_gemm_q8y(a, st);
            return;
        }
        launch_gemm_q8y(a, st);
    });
}

int32_t sepal_hip_gemm_w8a16(const void* x, size_t ld_x, const int8_t* wq, size_t ld_w, const float* sw, void* y,
                             int32_t y_type, size_t ld_y, size_t t, size_t n, size_t k, void* stream) {
    return guarded([&] {
        // (the order of launch_gemm_w8a16's checks, runner/cuda/src/gemm_s8_kernels.cu:550-557)
        if (t == 0 || n == 0) return;
        require(x != nullptr && wq != nullptr && sw != nullptr && y != nullptr, "gemm_w8a16: null pointer");
        require(y_type == SEPAL_HIP_F32 || y_type == SEPAL_HIP_F16, "gemm_w8a16: the output is float32 or binary16");
        require(sepal_hip_gemm_w8a16_supports(n, k, ld_x, ld_w, ld_y) == 1,
                "gemm_w8a16: unsupported shape (K a multiple of 16, ld_x of 8, ld_w of 16, N and ld_y even, strides at "
                "least K and N)");
        require(aligned16(x) && aligned16(wq) && aligned8(y) && reinterpret_cast<std::uintptr_t>(sw) % 4 == 0,
                "gemm_w8a16: X and W must be 16-byte aligned, Y 8-byte aligned, the scales 4-byte aligned");
        require(t < 0x7FFFFFFFu && n < 0x7FFFFFFFu && k < 0x7FFFFFFFu, "gemm_w8a16: dimension beyond 2^31");
        const hipStream_t st = as_stream(stream);
        // The per-channel scale as per-group scales, then the w8g multiply (binary16 X, Store). K off the 128-grid runs
        // on zero-padded copies of X and W (an exact zero per padded product), X rows that are not 32-byte multiples on
        // a copy of X. Above the small-M size a binary16 output comes straight from the large-M kernels; below it (or
        // for Y rows the kernels cannot store), through float32 row chunks of at most 64 MB and a conversion (the same
        // rounding; a row's bits do not depend on the batch).
        const std::size_t kp = (k + 127) / 128 * 128, groups = kp / 128;
        const bool pad_k = kp != k, stage_x = pad_k || ld_x % 16 != 0;
        const std::size_t s_bytes = up256(n * groups * 4);
        const std::size_t xs_bytes = stage_x ? up256(t * kp * 2) : 0;
        const std::size_t wp_bytes = pad_k ? up256(n * kp) : 0;
        const bool direct = (y_type == SEPAL_HIP_F32 || t > static_cast<std::size_t>(kSmallM)) && ld_y % 4 == 0 && aligned16(y);
        const std::size_t ldt = (n + 3) / 4 * 4;
        const std::size_t chunk = direct ? t : std::max<std::size_t>(1, (std::size_t{64} << 20) / (ldt * 4));
        const std::size_t rows = std::min(t, chunk);
        const std::size_t tmp_bytes = direct ? 0 : up256(rows * ldt * 4);
        const auto args = [&](const void* xs, const std::int8_t* w, const float* s, char* tmp, std::size_t r0, std::size_t tr) {
            GemmArgs a;
            a.x = static_cast<const std::uint16_t*>(xs) + r0 * (stage_x ? kp : ld_x);
            a.x_type = SEPAL_HIP_F16;
            a.ld_x = stage_x ? kp : ld_x;
            a.w = w;
            a.ld_w = pad_k ? kp : ld_w;
            a.s = s;
            a.ld_s = groups;
            a.y = direct ? static_cast<void*>(static_cast<char*>(y) + r0 * ld_y * (y_type == SEPAL_HIP_F32 ? 4 : 2))
                         : static_cast<void*>(tmp);
            a.y_type = direct ? y_type : SEPAL_HIP_F32;
            a.ld_y = direct ? ld_y : ldt;
            a.t = tr;
            a.n = n;
            a.k = kp;
            a.epilogue = SEPAL_HIP_STORE;
            a.config = tr > static_cast<std::size_t>(kSmallM) ? 0 : -1;  // no K split: a row's bits do not depend on the batch
            return a;
        };
        // (the layout of the first, largest chunk bounds every later one)
        const W8gAnyLayout L0 = w8g_any_layout(args(stage_x ? nullptr : x, wq, sw, nullptr, 0, rows));
        Lease lease(kScratchOffset + s_bytes + xs_bytes + wp_bytes + tmp_bytes + L0.total, st);
        char* ws = lease.base();
        char* p = ws + kScratchOffset;
        float* s = reinterpret_cast<float*>(p);
        char* xs = p + s_bytes;
        auto* wp = reinterpret_cast<std::int8_t*>(xs + xs_bytes);
        char* tmp = xs + xs_bytes + wp_bytes;
        char* zone = tmp + tmp_bytes;
        launch_broadcast_scales(sw, s, n, groups, st);
        if (stage_x) launch_pad_rows(x, ld_x * 2, xs, kp * 2, t, k * 2, st);
        if (pad_k) launch_pad_rows(wq, ld_w, wp, kp, n, k, st);
        for (std::size_t r0 = 0; r0 < t; r0 += rows) {
            const std::size_t tr = std::min(rows, t - r0);
            const GemmArgs a = args(stage_x ? static_cast<const void*>(xs) : x, pad_k ? wp : wq, s, tmp, r0, tr);
            w8g_any(a, w8g_any_layout(a), ws, zone, st);
            if (!direct)
                launch_put_cols(reinterpret_cast<const float*>(tmp), ldt,
                                static_cast<char*>(y) + r0 * ld_y * (y_type == SEPAL_HIP_F32 ? 4 : 2), y_type, ld_y, tr, n,
                                false, st);
        }
    });
}

int32_t sepal_hip_gemm_q8_swiglu_quantize(const int8_t* xq, size_t ld_x, const float* xs, size_t ld_xs, size_t act_block,
                                          const int8_t* w, size_t ld_w, const float* ws, size_t ld_ws, int8_t* hq,
                                          size_t ld_hq, float* hs, size_t ld_hs, size_t t, size_t n, size_t k,
                                          int32_t config, void* stream) {
    return guarded([&] {
        require(config >= -1 && config <= 2, "gemm_q8_swiglu_quantize: config must be -1, 0, 1 or 2");
        check_gemm_common("gemm_q8_swiglu_quantize", xq, ld_x, w, ld_w, ws, ld_ws, hq, ld_hq, n, k, SEPAL_HIP_SWIGLU);
        require(n % 256 == 0, "gemm_q8_swiglu_quantize: N must be a multiple of 256 (128-column output blocks)");
        require(act_block == 128 || act_block == k, "gemm_q8_swiglu_quantize: act_block must be 128 or K");
        require(xs != nullptr && ld_xs >= k / act_block, "gemm_q8_swiglu_quantize: activation scales missing or stride too small");
        require(hs != nullptr && ld_hs >= n / 256, "gemm_q8_swiglu_quantize: output scales missing or stride too small");
        require(ld_hq % 16 == 0, "gemm_q8_swiglu_quantize: ld_hq must be a multiple of 16");
        if (t == 0) return;
        require(t < 0x7FFFFFFFu, "gemm_q8_swiglu_quantize: dimension beyond 2^31");
        if (config >= 1) require(t <= kSmallM, "gemm_q8_swiglu_quantize: the small-M path takes at most 64 rows");
        const hipStream_t st = as_stream(stream);
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.xs = xs;
        a.ld_xs = ld_xs;
        a.act_block = act_block;
        a.w = w;
        a.ld_w = ld_w;
        a.s = ws;
        a.ld_s = ld_ws;
        a.t = t;
        a.n = n;
        a.k = k;
        // (33-64 rows with N >= 8192: the same bits either way; the fused form where a graph is being captured, since it needs
        // no workspace that would have to exist by then)
        bool large = config == 0 || (config < 0 && t > kSmallM);
        if (config < 0 && !large && !q8_streams(t, n)) {
            hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(st, &cap) != hipSuccess) throw LaunchError("gemm_q8_swiglu_quantize: hipStreamIsCapturing failed");
            large = cap != hipStreamCaptureStatusNone;
        }
        if (large) {
            a.y = hq;
            a.ld_y = ld_hq;
            a.ys = hs;
            a.ld_ys = ld_hs;
            launch_gemm_q8_swiglu_q8(a, st);
            return;
        }
        // small M: the float32 H through the workspace, then the activation quantizer (the same values and rule)
        const std::size_t cols = n / 2;
        Lease ws(kScratchOffset + t * cols * 4, st);
        float* h = reinterpret_cast<float*>(ws.base() + kScratchOffset);
        a.scratch = ws.base();
        a.y = h;
        a.y_type = SEPAL_HIP_F32;
        a.ld_y = cols;
        a.epilogue = SEPAL_HIP_SWIGLU;
        a.config = config == 2 ? 1 : config;
        a.force_splits = config == 2 ? 1 : 0;
        launch_gemm_q8(a, st);
        launch_quantize_rows(h, SEPAL_HIP_F32, cols, hq, ld_hq, hs, ld_hs, t, cols, 128, st);
    });
}

int32_t sepal_hip_q8_group_sums(const int8_t* xq, size_t ld_x, const int8_t* w, size_t ld_w, int32_t* sums, size_t t,
                                size_t n, size_t k, void* stream) {
    return guarded([&] {
        require(xq != nullptr && w != nullptr && sums != nullptr, "q8_group_sums: null pointer");
        require(k % 128 == 0 && k != 0 && n != 0, "q8_group_sums: K must be a non-zero multiple of 128");
        require(ld_x >= k && ld_w >= k && ld_x % 16 == 0 && ld_w % 16 == 0, "q8_group_sums: strides");
        require(aligned16(xq) && aligned16(w), "q8_group_sums: pointers must be 16-byte aligned");
        if (t == 0) return;
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.w = w;
        a.ld_w = ld_w;
        a.s = nullptr;
        a.t = t;
        a.n = n;
        a.k = k;
        a.sums = sums;
        const hipStream_t st = as_stream(stream);
        Lease ws(kScratchOffset, st);
        a.scratch = ws.base();
        launch_q8_group_sums(a, st);
    });
}

int32_t sepal_hip_rmsnorm_rows(const float* x, size_t ld_x, void* y, int32_t y_type, size_t ld_y, const float* w1,
                               size_t rows, size_t cols, double eps, void* stream) {
    return guarded([&] {
        require(valid_type(y_type), "rmsnorm_rows: unknown output type");
        require(cols % 8 == 0, "rmsnorm_rows: cols must be a multiple of 8");
        if (rows == 0 || cols == 0) return;
        require(x != nullptr && y != nullptr, "rmsnorm_rows: null pointer");
        require(ld_x >= cols && ld_y >= cols, "rmsnorm_rows: strides below cols");
        require(ld_x % 4 == 0 && aligned16(x), "rmsnorm_rows: x must be 16-byte aligned with a stride that is a multiple of 4");
        require(eps > 0.0, "rmsnorm_rows: eps must be positive");
        launch_rmsnorm(x, ld_x, y, y_type, ld_y, w1, rows, cols, eps, as_stream(stream));
    });
}

int32_t sepal_hip_rmsnorm_quantize_rows(const float* x, size_t ld_x, const float* w1, uint16_t* y_bf16, size_t ld_y,
                                        int8_t* q, size_t ld_q, float* scales, size_t ld_s, size_t rows, size_t cols,
                                        size_t block, double eps, void* stream) {
    return guarded([&] {
        require(block == 128 || block == cols, "rmsnorm_quantize_rows: block must be 128 or cols");
        if (rows == 0 || cols == 0) return;
        require(x != nullptr && q != nullptr && scales != nullptr, "rmsnorm_quantize_rows: null pointer");
        require(cols % 128 == 0, "rmsnorm_quantize_rows: cols must be a multiple of 128");
        require(ld_x >= cols && ld_q >= cols && ld_s >= cols / block && (y_bf16 == nullptr || ld_y >= cols),
                "rmsnorm_quantize_rows: strides below the row");
        require(ld_x % 16 == 0 && ld_q % 16 == 0 && aligned16(x) && aligned16(q),
                "rmsnorm_quantize_rows: x and q must be 16-byte aligned with strides that are multiples of 16");
        require(eps > 0.0, "rmsnorm_quantize_rows: eps must be positive");
        launch_rmsnorm_quantize(x, ld_x, y_bf16, ld_y, w1, q, ld_q, scales, ld_s, rows, cols, block, eps, as_stream(stream));
    });
}

int32_t sepal_hip_float_to_bf16(const float* src, uint16_t* dst, size_t count, void* stream) {
    return guarded([&] {
        if (count == 0) return;
        require(src != nullptr && dst != nullptr, "float_to_bf16: null pointer");
        launch_f32_to_bf16(src, dst, count, as_stream(stream));
    });
}

int32_t sepal_hip_weight_fingerprint(const void* data, size_t bytes, uint64_t* out, void* stream) {
    return guarded([&] {
        require(data != nullptr && out != nullptr, "weight_fingerprint: null pointer");
        require(aligned8(data), "weight_fingerprint: data must be 8-byte aligned");
        const hipStream_t st = as_stream(stream);
        Lease ws(kScratchOffset + fingerprint_scratch_bytes(), st);
        launch_fingerprint(data, bytes, out, ws.base() + kScratchOffset, st);
    });
}

namespace {
void check_packed(const char* who, const char* path, const void* q, std::size_t ld_q, const void* s, std::size_t ld_s,
                  std::size_t rows, std::size_t k, int32_t rule, int32_t layout) {
    const std::string w = who;
    require(path != nullptr && q != nullptr && s != nullptr, w + ": null pointer");
    require(rows != 0 && k != 0 && k % 128 == 0, w + ": rows must be non-zero and k a non-zero multiple of 128");
    require(ld_q == k && ld_s == k / 128, w + ": q and s must be contiguous (ld_q = k, ld_s = k / 128)");
    require(rule == SEPAL_HIP_RULE_DIVIDE || rule == SEPAL_HIP_RULE_RECIPROCAL, w + ": unknown quantizer rule");
    require(layout == 0 || (layout == 1 && rows % 128 == 0), w + ": layout must be 0 (plain rows) or 1 (gate/up interleave, rows a multiple of 128)");
    require(aligned8(q) && aligned8(s), w + ": q and s must be 8-byte aligned");
}
} // namespace

int32_t sepal_hip_packed_save(const char* path, const int8_t* q, size_t ld_q, const float* s, size_t ld_s, size_t rows,
                              size_t k, int32_t rule, int32_t layout, uint64_t source_fp, void* stream) {
    return guarded([&] {
        check_packed("packed_save", path, q, ld_q, s, ld_s, rows, k, rule, layout);
        const hipStream_t st = as_stream(stream);
        Lease ws(kScratchOffset + fingerprint_scratch_bytes(), st);
        packed_save(path, q, ld_q, s, ld_s, rows, k, rule, layout, source_fp, ws.base() + kScratchOffset, st);
    });
}

int32_t sepal_hip_packed_load(const char* path, int8_t* q, size_t ld_q, float* s, size_t ld_s, size_t rows, size_t k,
                              int32_t rule, int32_t layout, uint64_t source_fp, void* stream) {
    return guarded([&] {
        check_packed("packed_load", path, q, ld_q, s, ld_s, rows, k, rule, layout);
        const hipStream_t st = as_stream(stream);
        Lease ws(kScratchOffset + fingerprint_scratch_bytes(), st);
        packed_load(path, q, ld_q, s, ld_s, rows, k, rule, layout, source_fp, ws.base() + kScratchOffset, st);
    });
}

} // extern "C"

namespace sepal::hip {

void check_stack_args(int32_t kind, size_t hidden, size_t inter, const void* x, const int8_t* const* w_gate_up,
                      const float* const* s_gate_up, const int8_t* const* w_down, const float* const* s_down, const float* y,
                      size_t act_block) {
    require(kind == 0 || kind == 1 || kind == 2, "mlp_stack: kind must be 0 (w8g), 1 (q8) or 2 (w8g, float32 H)");
    require(hidden % 128 == 0 && inter % 128 == 0 && hidden != 0 && inter != 0, "mlp_stack: hidden and inter must be multiples of 128");
    require(w_gate_up != nullptr && s_gate_up != nullptr && w_down != nullptr && s_down != nullptr && x != nullptr && y != nullptr,
            "mlp_stack: null pointer");
    require(kind != 1 || act_block == 128 || act_block == 0, "mlp_stack: act_block must be 128 or 0 (one scale per token)");
    require(hidden < 0x7FFFFFFFu && inter < 0x7FFFFFFFu, "mlp_stack: dimension beyond 2^31");
}

StackZones stack_zones(int kind, std::size_t t, std::size_t hidden, std::size_t inter, std::size_t act_block, bool fuse_h) {
    StackZones z;
    z.per_token = act_block == 0;
    z.ab_h = z.per_token ? hidden : 128;
    z.ab_i = z.per_token ? inter : 128;
    const auto up256 = [](std::size_t b) { return (b + 255) / 256 * 256; };
    z.off_h = kScratchOffset;
    if (kind == 0 && small_stack_plan(t, hidden, inter, z.plan)) {
        // M <= 16 (stack_small.hip): H binary16, the down pass's K-part sums float32
        z.form = StackZones::SMALL_W8G;
        z.off_p = z.off_h + up256(t * inter * 2);
        z.end = z.off_p + static_cast<std::size_t>(z.plan.parts) * t * hidden * 4;
        return z;
    }
    // (per token, the down pass reads the gate/up grid's partial row maxima: at most 256 blocks)
    if (kind == 1 && small_stack_plan(t, hidden, inter, z.plan) &&
        (!z.per_token || (inter / 8 + z.plan.tiles_per_block - 1) / z.plan.tiles_per_block <= 256)) {
        // M <= 16 gpu-q8w: H float32 with, per token, its partial row maxima; K-part sums; the int8 layer input
        z.form = StackZones::SMALL_Q8;
        z.off_hmax = z.off_h + up256(t * inter * 4);
        z.off_p = z.off_hmax + up256(t * static_cast<std::size_t>(z.plan.blocks) * 4);
        z.off_qx = z.off_p + up256(static_cast<std::size_t>(z.plan.parts) * t * hidden * 4);
        z.off_sx = z.off_qx + up256(t * hidden);
        z.end = z.off_sx + up256(t * (hidden / z.ab_h) * 4);
        return z;
    }
    // general: H [t, inter] (binary16 for w8g and for q8 with one scale per token; float32 for kind 2, and for q8 per
    // 128 unless the gate/up epilogue quantizes it); q8 also the int8 layer input and int8 H with their scales; kind 2
    // the hi + lo pairs of H for the down multiply
    z.fused_h = kind == 1 && z.ab_i == 128 && (t > kSmallM || (fuse_h && !q8_streams(t, 2 * inter)));
    const std::size_t h_bytes = kind == 0 ? t * inter * 2 : (z.fused_h ? 0 : t * inter * 4);
    z.off_qx = z.off_h + up256(h_bytes);
    z.off_sx = z.off_qx + (kind == 1 ? up256(t * hidden) : 0);
    z.off_qh = z.off_sx + (kind == 1 ? up256(t * (hidden / z.ab_h) * 4) : 0);
    z.off_sh = z.off_qh + (kind == 1 ? up256(t * inter) : 0);
    z.off_split = z.off_sh + (kind == 1 ? up256(t * (inter / z.ab_i) * 4) : 0);
    std::size_t split = 0;
    GemmArgs gu, dn;
    gu.t = dn.t = t;
    gu.n = 2 * inter;
    gu.k = dn.n = hidden;
    dn.k = inter;
    gu.epilogue = SEPAL_HIP_SWIGLU;
    gu.ld_s = hidden / 128;
    dn.ld_s = inter / 128;
    if (kind != 1) {
        z.img = gemm_w8g_image_bytes(gu);
        z.img_dn = gemm_w8g_image_bytes(dn);
    }
    if (kind == 2) {
        GemmArgs dn;
        dn.x_type = SEPAL_HIP_F32;
        dn.t = t;
        dn.n = hidden;
        dn.k = inter;
        dn.ld_w = inter;
        dn.epilogue = SEPAL_HIP_STORE;
        split = gemm_w8g_scratch_bytes(dn);
    }
    z.off_img = z.off_split + up256(split);
    z.off_img_dn = z.off_img + z.img;
    z.end = z.off_img_dn + z.img_dn;
    return z;
}

// One call of the stack on the scratch at `ws` (laid out by stack_zones).
void run_stack(const StackZones& z, int kind, std::size_t layers, std::size_t t, std::size_t hidden, std::size_t inter,
               void* x, const int8_t* const* w_gate_up, const float* const* s_gate_up, const int8_t* const* w_down,
               const float* const* s_down, float* y, double eps, char* ws, hipStream_t st, const void* const* img_gate_up,
               const void* const* img_down, bool stream_w) {
    if (z.form == StackZones::SMALL_W8G) {
        // three launches per layer: whole-K gate/up tiles per CU, the down multiply in K-parts, the finish pass
        for (std::size_t l = 0; l < layers; ++l)
            launch_small_layer(z.plan, t, hidden, inter, x, w_gate_up[l], s_gate_up[l], w_down[l], s_down[l], ws + z.off_h,
                               reinterpret_cast<float*>(ws + z.off_p), y, l + 1 < layers ? x : nullptr, eps, st, stream_w);
        return;
    }
    if (z.form == StackZones::SMALL_Q8) {
        // the same three launches on int8 MFMAs; the down pass quantizes H while staging it; the finish pass quantizes
        // the next layer's input
        auto* qx = reinterpret_cast<std::int8_t*>(ws + z.off_qx);
        auto* sx = reinterpret_cast<float*>(ws + z.off_sx);
        launch_quantize_rows(x, SEPAL_HIP_BF16, hidden, qx, hidden, sx, hidden / z.ab_h, t, hidden, z.ab_h, st);
        for (std::size_t l = 0; l < layers; ++l)
            launch_small_layer_q8(z.plan, t, hidden, inter, qx, sx, z.per_token, w_gate_up[l], s_gate_up[l], w_down[l],
                                  s_down[l], reinterpret_cast<float*>(ws + z.off_h), reinterpret_cast<float*>(ws + z.off_hmax),
                                  reinterpret_cast<float*>(ws + z.off_p), y, l + 1 < layers ? qx : nullptr, sx,
                                  l + 1 < layers ? x : nullptr, eps, st, stream_w);
        return;
    }
    void* h = ws + z.off_h;
    auto* qx = reinterpret_cast<std::int8_t*>(ws + z.off_qx);
    auto* sx = reinterpret_cast<float*>(ws + z.off_sx);
    auto* qh = reinterpret_cast<std::int8_t*>(ws + z.off_qh);
    auto* sh = reinterpret_cast<float*>(ws + z.off_sh);
    for (std::size_t l = 0; l < layers; ++l) {
        GemmArgs gu;
        gu.t = t;
        gu.n = 2 * inter;
        gu.k = hidden;
        gu.w = w_gate_up[l];
        gu.ld_w = hidden;
        gu.s = s_gate_up[l];
        gu.ld_s = hidden / 128;
        gu.y = h;
        gu.ld_y = inter;
        gu.epilogue = SEPAL_HIP_SWIGLU;
        gu.scratch = ws;
        GemmArgs dn;
        dn.t = t;
        dn.n = hidden;
        dn.k = inter;
        dn.w = w_down[l];
        dn.ld_w = inter;
        dn.s = s_down[l];
        dn.ld_s = inter / 128;
        dn.y = y;
        dn.ld_y = hidden;
        dn.epilogue = SEPAL_HIP_STORE;
        dn.scratch = ws;
        if (z.img != 0) {
            gu.wimage = ws + z.off_img;
            gu.wimage_bytes = z.img;
        }
        if (z.img_dn != 0) {
            dn.wimage = ws + z.off_img_dn;
            dn.wimage_bytes = z.img_dn;
        }
        if (img_gate_up != nullptr) {
            // load-time images: nothing to widen
            gu.wimage = const_cast<void*>(img_gate_up[l]);
            gu.wimage_bytes = w8g_image_bytes_nk(2 * inter, hidden);
            gu.image_ready = true;
            dn.wimage = const_cast<void*>(img_down[l]);
            dn.wimage_bytes = w8g_image_bytes_nk(hidden, inter);
            dn.image_ready = true;
        }
        if (z.img != 0 && z.img_dn != 0) {
            // both multiplies on images: the gate/up multiply's halves launch widens this layer's down weights, the
            // down multiply's the next layer's gate/up weights (the first layer's gate/up widens its own)
            gu.image_ready = l > 0;
            gu.next_w = w_down[l];
            gu.next_ld_w = inter;
            gu.next_n = hidden;
            gu.next_k = inter;
            gu.next_f16 = kind == 0 ? 1 : 0;  // the down multiply's X: binary16 H (kind 0), or bf16 hi + lo pairs
            gu.next_image = ws + z.off_img_dn;
            dn.image_ready = true;
            if (l + 1 < layers) {
                dn.next_w = w_gate_up[l + 1];
                dn.next_ld_w = hidden;
                dn.next_n = 2 * inter;
                dn.next_k = hidden;
                dn.next_f16 = 0;
                dn.next_image = ws + z.off_img;
            }
        }
        if (kind != 1) {
            // w8g: H binary16 (kind 0) or float32 (kind 2, the down multiply on its bf16 hi + lo pairs)
            gu.x = x;
            gu.x_type = SEPAL_HIP_BF16;
            gu.ld_x = hidden;
            gu.y_type = kind == 0 ? SEPAL_HIP_F16 : SEPAL_HIP_F32;
            if (kind == 2 && gemm_w8g_pairs_chain(gu, dn)) {
                // the gate/up epilogue writes H as the down multiply's bf16 hi + lo pairs (no split pass; the same
                // pairs as the split of float32 H)
                gu.y_type = kYPairs;
                launch_gemm_w8g(gu, st);
                dn.x = h;
                dn.ld_x = 2 * inter;
                dn.y_type = SEPAL_HIP_F32;
                launch_gemm_w8g_pairs(dn, st);
                if (l + 1 < layers) launch_rmsnorm(y, hidden, x, SEPAL_HIP_BF16, hidden, nullptr, t, hidden, eps, st);
                continue;
            }
            launch_gemm_w8g(gu, st);
            dn.x = h;
            dn.x_type = kind == 0 ? SEPAL_HIP_F16 : SEPAL_HIP_F32;
            dn.ld_x = inter;
            dn.y_type = SEPAL_HIP_F32;
            dn.xsplit = ws + z.off_split;
            launch_gemm_w8g(dn, st);
            if (l + 1 < layers) launch_rmsnorm(y, hidden, x, SEPAL_HIP_BF16, hidden, nullptr, t, hidden, eps, st);
            continue;
        }
        // q8: the first layer's input is quantized here; later ones come quantized out of the fused RMSNorm
        if (l == 0) launch_quantize_rows(x, SEPAL_HIP_BF16, hidden, qx, hidden, sx, hidden / z.ab_h, t, hidden, z.ab_h, st);
        gu.x = qx;
        gu.ld_x = hidden;
        gu.xs = sx;
        gu.ld_xs = hidden / z.ab_h;
        gu.act_block = z.ab_h;
        gu.y_type = SEPAL_HIP_F32;
        if (z.fused_h) {
            // SwiGLU and the int8 re-quantization of H in the gate/up epilogue
            gu.y = qh;
            gu.ld_y = inter;
            gu.ys = sh;
            gu.ld_ys = inter / 128;
            launch_gemm_q8_swiglu_q8(gu, st);
        } else {
            // H binary16 when one scale per token follows (the reference's GPU int8 path quantizes its binary16
            // activations per row, runner/cuda/src/cuda_engine.cpp:1098-1102); float32 per 128, as cpu-q8 keeps it
            const int h_type = z.per_token ? SEPAL_HIP_F16 : SEPAL_HIP_F32;
            gu.y_type = h_type;
            launch_gemm_q8(gu, st);
            launch_quantize_rows(h, h_type, inter, qh, inter, sh, inter / z.ab_i, t, inter, z.ab_i, st);
        }
        dn.x = qh;
        dn.ld_x = inter;
        dn.xs = sh;
        dn.ld_xs = inter / z.ab_i;
        dn.act_block = z.ab_i;
        dn.y_type = SEPAL_HIP_F32;
        launch_gemm_q8(dn, st);
        // the next layer's input: RMSNorm, bf16 and the int8 quantization in one pass (x keeps the bf16 input of the
        // last layer)
        if (l + 1 < layers)
            launch_rmsnorm_quantize(y, hidden, l + 2 == layers ? static_cast<std::uint16_t*>(x) : nullptr, hidden, nullptr, qx,
                                    hidden, sx, hidden / z.ab_h, t, hidden, z.ab_h, eps, st);
    }
}

namespace {

// ---- the no-allocation stack ----------------------------------------------------------------------------------------
//
// Scratch in the code object: every device the library runs on holds this array until the process ends. Host code
// uses the per-device address from hipGetSymbolAddress, never the array's name (a host-side stand-in).
constexpr std::size_t kStaticScratchBytes = std::size_t{64} << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_static_mutex;
char* g_static_ptr[kMaxDevices] = {};
// Calls on one device share its array. Each call's work is recorded in the device's event, and a call on another stream
// than the last waits for it on the device, so calls on different streams run one after the other (graph capture
// excepted: there the caller orders the streams). g_static_mutex is held from the wait to the record.
hipEvent_t g_static_done[kMaxDevices] = {};
hipStream_t g_static_last[kMaxDevices] = {};
bool g_static_used[kMaxDevices] = {};

// The current device's static scratch. The first call on a device looks its address up (with that device current)
// and enqueues, on `stream`, the clearing of the split-K counter zone, which is zero at rest from then on.
// The caller holds g_static_mutex.
char* static_scratch(int dev, hipStream_t stream) {
    if (g_static_ptr[dev] == nullptr) {
        if (hipEventCreateWithFlags(&g_static_done[dev], hipEventDisableTiming) != hipSuccess)
            throw LaunchError("mlp_stack_noalloc: hipEventCreateWithFlags failed");
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
            throw LaunchError(std::string("mlp_stack_noalloc: hipGetSymbolAddress of the static scratch failed: ") +
                              hipGetErrorString(e));
        zero_words_kernel<<<dim3(64), dim3(256), 0, stream>>>(static_cast<unsigned*>(ptr), kCounterBytes / 4);
        check_launch("mlp_stack_noalloc counter clearing launch");
        g_static_ptr[dev] = static_cast<char*>(ptr);
    }

    return g_static_ptr[dev];
}

} // namespace
} // namespace sepal::hip

extern "C" {

int32_t sepal_hip_mlp_stack_noalloc(int32_t kind, size_t layers, size_t t, size_t hidden, size_t inter, void* x,
                                    const int8_t* const* w_gate_up, const float* const* s_gate_up,
                                    const int8_t* const* w_down, const float* const* s_down, float* y, size_t act_block,
                                    double eps, void* stream) {
    return guarded([&] {
        check_stack_args(kind, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, act_block);
        if (layers == 0 || t == 0) return;
        const hipStream_t st = as_stream(stream);
        StackZones z = stack_zones(kind, t, hidden, inter, act_block);
        if (z.end > kStaticScratchBytes && z.img != 0) {
            // without the weight images (the kernels widen the weights themselves; the same bits)
            z.img = z.img_dn = 0;
            z.end = z.off_img;
        }
        // (without the float32 H of 33-64 rows per 128: its quantization in the gate/up epilogue, the same bits)
        if (z.end > kStaticScratchBytes && kind == 1) z = stack_zones(kind, t, hidden, inter, act_block, true);
        require(z.end <= kStaticScratchBytes,
                "mlp_stack_noalloc: this shape needs " + std::to_string(z.end) + " bytes of scratch, beyond the " +
                    std::to_string(kStaticScratchBytes) + " of the static scratch (call with fewer rows)");
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) throw LaunchError("hipGetDevice failed");
        if (dev < 0 || dev >= kMaxDevices) throw LaunchError("mlp_stack_noalloc: device index beyond the library's table");
        std::lock_guard<std::mutex> lock(g_static_mutex);
        char* base = static_scratch(dev, st);
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cap) != hipSuccess) throw LaunchError("mlp_stack_noalloc: hipStreamIsCapturing failed");
        const bool eager = cap == hipStreamCaptureStatusNone;
        if (eager && g_static_used[dev] && g_static_last[dev] != st && hipStreamWaitEvent(st, g_static_done[dev], 0) != hipSuccess)
            throw LaunchError("mlp_stack_noalloc: hipStreamWaitEvent failed");
        run_stack(z, kind, layers, t, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, eps, base, st);
        if (eager) {
            if (hipEventRecord(g_static_done[dev], st) != hipSuccess) throw LaunchError("mlp_stack_noalloc: hipEventRecord failed");
            g_static_last[dev] = st;
            g_static_used[dev] = true;
        }
    });
}

size_t sepal_hip_w8g_image_bytes(size_t n, size_t k) { return n == 0 || k == 0 ? 0 : w8g_image_bytes_nk(n, k); }

int32_t sepal_hip_w8g_make_image(const int8_t* w, size_t ld_w, size_t n, size_t k, int32_t x_type, void* img,
                                 size_t img_bytes, void* stream) {
    return guarded([&] {
        require(w != nullptr && img != nullptr, "w8g_make_image: null pointer");
        require(valid_type(x_type), "w8g_make_image: X must be float32, bf16 or binary16");
        require(n != 0 && k != 0 && k % 128 == 0 && ld_w >= k && ld_w % 16 == 0 && aligned16(w),
                "w8g_make_image: K must be a non-zero multiple of 128, W rows of whole 16 bytes (16-byte aligned)");
        const std::size_t need = w8g_image_bytes_nk(n, k);
        require(need != 0, "w8g_make_image: the image of this shape would exceed 2^31 bytes");
        require(img_bytes >= need && aligned16(img), "w8g_make_image: img must hold sepal_hip_w8g_image_bytes(n, k) bytes, 16-byte aligned");
        launch_w8g_image(w, ld_w, n, k, x_type == SEPAL_HIP_F16, img, as_stream(stream));
    });
}

int32_t sepal_hip_mlp_stack_images(int32_t kind, size_t layers, size_t t, size_t hidden, size_t inter, void* x,
                                   const int8_t* const* w_gate_up, const float* const* s_gate_up,
                                   const int8_t* const* w_down, const float* const* s_down, const void* const* img_gate_up,
                                   const void* const* img_down, float* y, double eps, void* stream) {
    return guarded([&] {
        check_stack_args(kind, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, 128);
        require(kind == 0 || kind == 2, "mlp_stack_images: kind must be 0 or 2 (the w8g stacks)");
        require(img_gate_up != nullptr && img_down != nullptr, "mlp_stack_images: null image array");
        require(w8g_image_bytes_nk(2 * inter, hidden) != 0 && w8g_image_bytes_nk(hidden, inter) != 0,
                "mlp_stack_images: the images of this shape would exceed 2^31 bytes");
        if (layers == 0 || t == 0) return;
        for (std::size_t l = 0; l < layers; ++l)
            require(img_gate_up[l] != nullptr && img_down[l] != nullptr && aligned16(img_gate_up[l]) && aligned16(img_down[l]),
                    "mlp_stack_images: null or misaligned image");
        const hipStream_t st = as_stream(stream);
        StackZones z = stack_zones(kind, t, hidden, inter, 128);
        if (z.form == StackZones::GENERAL) {
            z.img = z.img_dn = 0;  // the caller's images replace the workspace's
            z.end = z.off_img;
        }
        Lease ws(z.end, st);
        run_stack(z, kind, layers, t, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, eps, ws.base(), st,
                  z.form == StackZones::GENERAL ? img_gate_up : nullptr, z.form == StackZones::GENERAL ? img_down : nullptr);
    });
}

size_t sepal_hip_w8g_stream_layout_bytes(size_t n, size_t k) {
    return n != 0 && k != 0 && n % 16 == 0 && k % 128 == 0 ? n * k : 0;
}

int32_t sepal_hip_w8g_make_stream_layout(const int8_t* w, size_t ld_w, size_t n, size_t k, int32_t interleave, void* out,
                                         size_t out_bytes, void* stream) {
    return guarded([&] {
        require(w != nullptr && out != nullptr, "w8g_make_stream_layout: null pointer");
        require(n != 0 && k != 0 && n % 16 == 0 && k % 128 == 0, "w8g_make_stream_layout: N must be a multiple of 16 and K of 128");
        require(!interleave || n % 128 == 0, "w8g_make_stream_layout: the gate/up interleave takes N a multiple of 128");
        require(ld_w >= k && ld_w % 16 == 0 && aligned16(w), "w8g_make_stream_layout: W rows of whole 16 bytes (16-byte aligned)");
        require(out_bytes >= n * k && aligned16(out), "w8g_make_stream_layout: out must hold n * k bytes, 16-byte aligned");
        launch_stream_layout(w, ld_w, n, k, interleave != 0, static_cast<int8_t*>(out), as_stream(stream));
    });
}

int32_t sepal_hip_mlp_stack_stream(int32_t kind, size_t layers, size_t t, size_t hidden, size_t inter, void* x,
                                   const int8_t* const* w_gate_up, const float* const* s_gate_up, const int8_t* const* w_down,
                                   const float* const* s_down, float* y, size_t act_block, double eps, void* stream) {
    return guarded([&] {
        require(kind == 0 || kind == 1, "mlp_stack_stream: kind must be 0 (w8g) or 1 (q8w)");
        check_stack_args(kind, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, act_block);
        if (layers == 0 || t == 0) return;
        for (std::size_t l = 0; l < layers; ++l)
            require(aligned16(w_gate_up[l]) && aligned16(w_down[l]), "mlp_stack_stream: weights must be 16-byte aligned");
        const hipStream_t st = as_stream(stream);
        const StackZones z = stack_zones(kind, t, hidden, inter, act_block);
        require(z.form == StackZones::SMALL_W8G || z.form == StackZones::SMALL_Q8,
                "mlp_stack_stream: the stream layout is read by the M <= 16 passes only (T <= 16 at a shape they take)");
        Lease ws(z.end, st);
        run_stack(z, kind, layers, t, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, eps, ws.base(), st, nullptr,
                  nullptr, true);
    });
}

int32_t sepal_hip_gemm_w8g_stream(const void* x, int32_t x_type, size_t ld_x, const int8_t* w, const float* s, size_t ld_s,
                                  void* y, int32_t y_type, size_t ld_y, size_t t, size_t n, size_t k, int32_t epilogue,
                                  void* stream) {
    return guarded([&] {
        require(x_type == SEPAL_HIP_BF16 || x_type == SEPAL_HIP_F16, "gemm_w8g_stream: X must be bf16 or binary16");
        require(valid_type(y_type), "gemm_w8g_stream: unknown output type");
        require(epilogue == SEPAL_HIP_SWIGLU || y_type == SEPAL_HIP_F32, "gemm_w8g_stream: Store and Add write float32");
        check_gemm_common("gemm_w8g_stream", x, ld_x, w, k, s, ld_s, y, ld_y, n, k, epilogue);
        if (t == 0) return;
        require(t <= 16, "gemm_w8g_stream: the stream layout is read by the M <= 16 kernels only (T <= 16)");
        GemmArgs a;
        a.x = x;
        a.x_type = x_type;
        a.ld_x = ld_x;
        a.w = w;
        a.ld_w = k;
        a.w_stream = true;
        a.s = s;
        a.ld_s = ld_s;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = epilogue;
        SmallGemmPlan plan;
        require(small_gemm_plan(a, plan), "gemm_w8g_stream: a shape the M <= 16 kernels do not take");
        const hipStream_t st = as_stream(stream);
        Lease ws(kScratchOffset, st);
        a.scratch = ws.base();
        launch_small_gemm_w8g(a, plan, st);
    });
}

int32_t sepal_hip_gemm_q8_stream(const int8_t* xq, size_t ld_x, const float* xs, size_t ld_xs, size_t act_block,
                                 const int8_t* w, const float* ws, size_t ld_ws, void* y, int32_t y_type, size_t ld_y,
                                 size_t t, size_t n, size_t k, int32_t epilogue, void* stream) {
    return guarded([&] {
        require(y_type == SEPAL_HIP_F32, "gemm_q8_stream: the M <= 16 q8 kernels write float32");
        check_gemm_common("gemm_q8_stream", xq, ld_x, w, k, ws, ld_ws, y, ld_y, n, k, epilogue);
        require(act_block == 128 || act_block == k, "gemm_q8_stream: act_block must be 128 or K");
        require(xs != nullptr && ld_xs >= k / act_block, "gemm_q8_stream: activation scales missing or stride too small");
        if (t == 0) return;
        require(t <= 16, "gemm_q8_stream: the stream layout is read by the M <= 16 kernels only (T <= 16)");
        GemmArgs a;
        a.x = xq;
        a.ld_x = ld_x;
        a.xs = xs;
        a.ld_xs = ld_xs;
        a.act_block = act_block;
        a.w = w;
        a.ld_w = k;
        a.w_stream = true;
        a.s = ws;
        a.ld_s = ld_ws;
        a.y = y;
        a.y_type = y_type;
        a.ld_y = ld_y;
        a.t = t;
        a.n = n;
        a.k = k;
        a.epilogue = epilogue;
        SmallGemmPlan plan;
        const bool swiglu = epilogue == SEPAL_HIP_SWIGLU;
        require(swiglu ? small_gemm_plan_q8(a, plan) : small_gemm_plan_q8_parts(a, plan),
                "gemm_q8_stream: a shape the M <= 16 kernels do not take");
        const hipStream_t st = as_stream(stream);
        Lease lease(kScratchOffset, st);
        a.scratch = lease.base();
        if (swiglu) launch_small_gemm_q8(a, plan, st);
        else launch_small_gemm_q8_parts(a, plan, st);
    });
}

int32_t sepal_hip_mlp_stack(int32_t kind, size_t layers, size_t t, size_t hidden, size_t inter, void* x,
                            const int8_t* const* w_gate_up, const float* const* s_gate_up, const int8_t* const* w_down,
                            const float* const* s_down, float* y, size_t act_block, double eps, void* stream) {
    return guarded([&] {
        check_stack_args(kind, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, act_block);
        if (layers == 0 || t == 0) return;
        const hipStream_t st = as_stream(stream);
        const StackZones z = stack_zones(kind, t, hidden, inter, act_block);
        Lease ws(z.end, st);
        run_stack(z, kind, layers, t, hidden, inter, x, w_gate_up, s_gate_up, w_down, s_down, y, eps, ws.base(), st);
    });
}

} // extern "C"
