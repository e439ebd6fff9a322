// brotensor runtime: ROCm device registration and the one op stream.
#include "brotensor/runtime.h"

#include <hip/hip_runtime_api.h>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <algorithm>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "brolm_hip.h"
#include "brotensor/tensor.h"
#include "hip_util.h"

namespace {

struct RuntimeState {
    bool ready = false;
    int device = 0;
    hipStream_t stream = nullptr;
    void* linear_ws = nullptr;           // the linear entry points' workspace, for the op stream
    std::size_t linear_ws_bytes = 0;
    std::vector<void (*)()> releases;   // on_shutdown hooks, registration order
};

RuntimeState& state() {
    static RuntimeState s;
    return s;
}

std::mutex& init_mutex() {
    static std::mutex m;
    return m;
}

}  // namespace

namespace hipx {

hipStream_t stream() {
    if (!state().ready) throw std::runtime_error("brotensor: init() has not been called");
    return state().stream;
}

void sync() { check(hipStreamSynchronize(stream()), "hipStreamSynchronize"); }

void* linear_ws() {
    if (!state().ready) throw std::runtime_error("brotensor: init() has not been called");
    return state().linear_ws;
}
std::size_t linear_ws_bytes() { return state().linear_ws_bytes; }

void h2d(void* dst, const void* src, std::size_t n) {
    if (n == 0) return;
    check(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, stream()), "hipMemcpyAsync H2D");
    sync();
}

void d2h(void* dst, const void* src, std::size_t n) {
    if (n == 0) return;
    check(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, stream()), "hipMemcpyAsync D2H");
    sync();
}

// ─── logits to the host ─────────────────────────────────────────────────────
//
// A step's logits come back as FP32 values of FP16 device rows: 152 K of them
// a row, 2.4 M for sixteen sequences.  A pageable copy, a scalar conversion on
// one thread into a vector and a copy of that took 0.2 ms a row, 4 ms of a
// 16-row batched step's 5.9.  Here the rows land in pinned memory and are
// converted from there into the caller's buffer, eight at a time (F16C), by up
// to four threads from 512 K values each; each thread's part is copied with an
// event of its own, so the first parts convert while the later ones arrive.

namespace {

constexpr std::size_t kStageMax = std::size_t(4) << 20;   // FP16 values of pinned memory at most (8 MB)
constexpr int kParts = 4;
constexpr std::size_t kPartMin = std::size_t(1) << 19;    // values that pay for a thread

// Pinned staging shared by every download (one op stream orders them anyway);
// grown on demand up to kStageMax, freed by brotensor::shutdown().
struct Staging {
    std::mutex mu;
    std::uint16_t* buf = nullptr;
    std::size_t cap = 0;
    hipEvent_t done[kParts] = {};

    // false: no pinned memory to be had
    bool reserve(std::size_t n) {
        for (hipEvent_t& e : done)
            if (!e) check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        if (cap >= n) return true;
        if (buf) (void)hipHostFree(buf);
        buf = nullptr;
        cap = 0;
        if (hipHostMalloc(reinterpret_cast<void**>(&buf), n * 2, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            buf = nullptr;
            return false;
        }
        cap = n;
        return true;
    }
    static void release();
};
Staging& staging() {
    static Staging* s = new Staging();   // outlives every caller, emptied by release()
    return *s;
}
void Staging::release() {
    Staging& s = staging();
    std::lock_guard<std::mutex> lk(s.mu);
    if (s.buf) (void)hipHostFree(s.buf);
    for (hipEvent_t& e : s.done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    s.buf = nullptr;
    s.cap = 0;
}

void widen_plain(const std::uint16_t* s, float* d, std::size_t n) {
    for (std::size_t i = 0; i < n; ++i) d[i] = brotensor::fp16_bits_to_fp32(s[i]);
}
#if defined(__x86_64__)
__attribute__((target("avx,f16c"))) void widen_f16c(const std::uint16_t* s, float* d, std::size_t n) {
    std::size_t i = 0;
    for (; i + 8 <= n; i += 8)
        _mm256_storeu_ps(d + i, _mm256_cvtph_ps(_mm_loadu_si128(reinterpret_cast<const __m128i*>(s + i))));
    widen_plain(s + i, d + i, n - i);
}
#endif
void widen(const std::uint16_t* s, float* d, std::size_t n) {
#if defined(__x86_64__)
    static const bool f16c = __builtin_cpu_supports("avx") && __builtin_cpu_supports("f16c");
    if (f16c) return widen_f16c(s, d, n);
#endif
    widen_plain(s, d, n);
}

}  // namespace

void d2h_f16_as_f32(float* dst, const void* src, std::size_t n) {
    const auto* from = static_cast<const std::uint16_t*>(src);
    Staging& st = staging();
    std::lock_guard<std::mutex> lk(st.mu);
    brotensor::on_shutdown(Staging::release);
    for (std::size_t at = 0; at < n;) {
        const std::size_t m = std::min(n - at, kStageMax);
        if (!st.reserve(m)) {
            std::vector<std::uint16_t> bits(m);
            d2h(bits.data(), from + at, m * 2);
            widen(bits.data(), dst + at, m);
            at += m;
            continue;
        }
        const int parts = static_cast<int>(std::clamp<std::size_t>(m / kPartMin, 1, kParts));
        auto begin = [&](int p) { return m * static_cast<std::size_t>(p) / static_cast<std::size_t>(parts); };
        for (int p = 0; p < parts; ++p) {
            check(hipMemcpyAsync(st.buf + begin(p), from + at + begin(p), (begin(p + 1) - begin(p)) * 2,
                                 hipMemcpyDeviceToHost, stream()),
                  "hipMemcpyAsync D2H");
            check(hipEventRecord(st.done[p], stream()), "hipEventRecord");
        }
        auto convert = [&](int p) {
            const hipError_t e = hipEventSynchronize(st.done[p]);
            if (e == hipSuccess) widen(st.buf + begin(p), dst + at + begin(p), begin(p + 1) - begin(p));
            return e;
        };
        hipError_t err[kParts] = {};
        std::thread helpers[kParts];
        for (int p = 1; p < parts; ++p) {
            try {
                helpers[p] = std::thread([&, p] { err[p] = convert(p); });
            } catch (...) {   // no thread, or no memory for one: this thread converts
                err[p] = convert(p);
            }
        }
        err[0] = convert(0);
        for (std::thread& t : helpers)
            if (t.joinable()) t.join();
        for (hipError_t e : err) check(e, "hipEventSynchronize");
        at += m;
    }
}

}  // namespace hipx

namespace brotensor {

void init() {
    std::lock_guard<std::mutex> lk(init_mutex());
    RuntimeState& s = state();
    if (s.ready) return;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
        throw std::runtime_error(
            "brotensor::init: no ROCm device found (this build has no CPU compute backend)");
    int chosen = -1;
    for (int d = 0; d < n; ++d) {
        hipDeviceProp_t p;
        if (hipGetDeviceProperties(&p, d) != hipSuccess) continue;
        if (std::strncmp(p.gcnArchName, "gfx950", 6) == 0) {
            chosen = d;
            break;
        }
    }
    if (chosen < 0) throw std::runtime_error("brotensor::init: no gfx950 (MI355X) device found");
    hipx::check(hipSetDevice(chosen), "hipSetDevice");
    hipStream_t st = nullptr;
    hipx::check(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate");
    // the op stream's linear workspace (split-K partials and counters of the
    // decode-batch GEMVs), taken here once so no op allocates under graph
    // capture
    const std::size_t wsb = bx_linear_workspace_bytes();
    void* ws = nullptr;
    hipx::check(hipMalloc(&ws, wsb), "hipMalloc linear workspace");
    hipx::bx(bx_linear_workspace_init(ws, wsb, st), "linear workspace init");
    hipx::check(hipStreamSynchronize(st), "hipStreamSynchronize");
    s.device = chosen;
    s.stream = st;
    s.linear_ws = ws;
    s.linear_ws_bytes = wsb;
    s.ready = true;
}

bool initialized() { return state().ready; }

Device default_device() { return state().ready ? Device::ROCm : Device::CPU; }

Dtype compute_dtype() { return Dtype::FP16; }

void sync_all() {
    if (state().ready) hipx::sync();
}

void* stream() { return hipx::stream(); }

int device_ordinal() { return state().device; }

void on_shutdown(void (*release)()) {
    std::lock_guard<std::mutex> lk(init_mutex());
    std::vector<void (*)()>& r = state().releases;
    for (void (*f)() : r)
        if (f == release) return;
    r.push_back(release);
}

void shutdown() {
    std::vector<void (*)()> hooks;
    {
        std::lock_guard<std::mutex> lk(init_mutex());
        if (!state().ready) return;
        hooks.swap(state().releases);
    }
    (void)hipStreamSynchronize(state().stream);
    for (auto it = hooks.rbegin(); it != hooks.rend(); ++it) (*it)();
    std::lock_guard<std::mutex> lk(init_mutex());
    RuntimeState& s = state();
    (void)hipStreamSynchronize(s.stream);
    if (s.linear_ws) (void)hipFree(s.linear_ws);
    s.linear_ws = nullptr;
    s.linear_ws_bytes = 0;
    (void)hipStreamDestroy(s.stream);
    s.stream = nullptr;
    s.ready = false;
}

}  // namespace brotensor
