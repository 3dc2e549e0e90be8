// The C ABI of include/presk_hip.h: compile (text -> hand-written class or
// generic printed kernel), run (one KernelFn call on a stream), device memory.
#include "presk_hip.h"

#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <sys/stat.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <functional>
#include <mutex>
#include <sstream>
#include <unordered_map>

#include "branches.hpp"
#include "convert.hpp"
#include "probe.hpp"
#include "synth.hpp"
#include "executor.hpp"

namespace presk {

namespace {

thread_local std::string g_error;
int g_device = -1;
std::mutex g_mu;

int fail(int code, const std::string& msg) {
    g_error = msg;
    return code;
}

int hip_fail(hipError_t e, const char* what) {
    return fail(PRESK_HIP_ERR, std::string("E10001: ") + what + ": " + hipGetErrorString(e));
}

const char kDevfmt[] =
#include "_devfmt.inc"
    ;

uint64_t fnv1a(const std::string& s) {
    uint64_t h = 0xcbf29ce484222325ull;
    for (unsigned char c : s) {
        h ^= c;
        h *= 0x100000001b3ull;
    }
    return h;
}

// PRESK_HIP_MODE=exact|fast: every kernel compiled in that mode whatever
// the caller asks (exact: the interpreter's order everywhere, the parity
// switch); -1 when unset or empty, -2 with a message when malformed
int forced_mode(std::string* err) {
    const char* env = std::getenv("PRESK_HIP_MODE");
    if (!env || !*env) return -1;
    if (std::strcmp(env, "exact") == 0) return PRESK_HIP_EXACT;
    if (std::strcmp(env, "fast") == 0) return PRESK_HIP_FAST;
    *err = std::string("PRESK_HIP_MODE=") + env + ": expected exact or fast";
    return -2;
}

std::string cache_dir() {
    const char* env = std::getenv("PRESK_HIP_CACHE");
    if (env && *env) return env;
    const char* home = std::getenv("HOME");
    std::string base = home && *home ? std::string(home) + "/.cache" : "/tmp";
    return base + "/presk-hip";
}

}  // namespace

bool build_code_object(const std::string& src, std::vector<char>* code, std::string* err) {
    static std::unordered_map<uint64_t, std::vector<char>> memo;
    static const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off",
                                 "-fno-gpu-flush-denormals-to-zero", "-fhip-fp32-correctly-rounded-divide-sqrt",
                                 "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    const int nopts = sizeof(opts) / sizeof(opts[0]);
    std::string key_text = src + kDevfmt;
    for (int i = 0; i < nopts; ++i) key_text += opts[i];
    const uint64_t key = fnv1a(key_text);
    {
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = memo.find(key);
        if (it != memo.end()) { *code = it->second; return true; }
    }
    char name[32];
    std::snprintf(name, sizeof name, "%016llx.co", (unsigned long long)key);
    const std::string dir = cache_dir(), path = dir + "/" + name;
    {
        std::ifstream f(path, std::ios::binary);
        if (f) {
            std::vector<char> data((std::istreambuf_iterator<char>(f)), std::istreambuf_iterator<char>());
            if (!data.empty()) {
                std::lock_guard<std::mutex> lock(g_mu);
                memo[key] = data;
                *code = std::move(data);
                return true;
            }
        }
    }
    hiprtcProgram prog;
    const char* headers[] = {kDevfmt};
    const char* names[] = {"devfmt.hpp"};
    if (hiprtcCreateProgram(&prog, src.c_str(), "presk_kernel.hip", 1, headers, names) != HIPRTC_SUCCESS) {
        *err = "E10001: hiprtcCreateProgram failed";
        return false;
    }
    hiprtcResult r = hiprtcCompileProgram(prog, nopts, opts);
    if (r != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(prog, &log[0]);
        hiprtcDestroyProgram(&prog);
        *err = "E10001: hiprtc: " + log.substr(0, 2000);
        return false;
    }
    size_t n = 0;
    hiprtcGetCodeSize(prog, &n);
    std::vector<char> data(n);
    hiprtcGetCode(prog, data.data());
    hiprtcDestroyProgram(&prog);
    // best-effort disk cache, written atomically (by each of two threads that
    // build the same source under a name of its own)
    ::mkdir(dir.c_str(), 0755);
    static std::atomic<unsigned> serial{0};
    std::string tmp = path + ".tmp" + std::to_string(::getpid()) + "." + std::to_string(serial++);
    {
        std::ofstream f(tmp, std::ios::binary);
        if (f) f.write(data.data(), (std::streamsize)data.size());
    }
    std::rename(tmp.c_str(), path.c_str());
    std::lock_guard<std::mutex> lock(g_mu);
    memo[key] = data;
    *code = std::move(data);
    return true;
}

double kernel_bytes(const Kernel& k) {
    double q = 0;
    for (size_t b = 0; b <= k.inputs.size(); ++b) {
        const BufSpec& s = k.buf((int)b);
        q += s.ty == Ty::Q4 ? (double)((s.numel() + 1) / 2) : (double)s.numel() * ty_bytes(s.ty);
        if (ty_quant(s.ty)) q += 4.0 * (double)s.scale_count();
    }
    return q;
}

double kernel_flops(const Kernel& k) {
    // 2 * numel(out) * K, K the summed length: 2*prod(outer)*I*J*K of a
    // contraction nest (crates/presk-kernel/src/lower.rs:695-784)
    const std::string& n = k.name;
    double K = 0;
    auto prod = [](const std::vector<int64_t>& d, size_t from, size_t to) {
        double p = 1;
        for (size_t i = from; i < to && i < d.size(); ++i) p *= (double)d[i];
        return p;
    };
    if ((n == "dot" || n == "dot+add") && k.inputs.size() >= 2 && !k.inputs[0].dims.empty()) {
        K = (double)k.inputs[0].dims.back();
    } else if ((n == "dot_vjp_l" || n == "dot_vjp_l+add") && k.inputs.size() >= 2) {
        K = prod(k.inputs[1].dims, 1, k.inputs[1].dims.size());
    } else if ((n == "dot_vjp_r" || n == "dot_vjp_r+add") && k.inputs.size() >= 2 && !k.inputs[0].dims.empty()) {
        K = prod(k.inputs[0].dims, 0, k.inputs[0].dims.size() - 1);
    } else if (n.compare(0, 4, "ein[") == 0 && k.inputs.size() >= 2) {
        K = 1;
        for (size_t a = 0; a < k.inputs[0].dims.size(); ++a) {
            const std::string& nm = k.inputs[0].names[a];
            bool out_axis = false;
            for (auto& o : k.output.names) out_axis |= (!nm.empty() && o == nm);
            if (!out_axis) K *= (double)k.inputs[0].dims[a];
        }
    }
    return 2.0 * (double)k.output.numel() * K;
}

}  // namespace presk

using namespace presk;

namespace {
int load_module(const presk_hip_kernel* h);

// ---- scratch memory of presk_hip_run_noalloc ------------------------------------
// One array a device, held from the library's load to the process's end: the
// class kernels' workspaces (split-K partials, chunk sums, mask bits) when the
// caller cannot allocate.  In host code `scratch` names a host-side stand-in,
// never device memory: every use goes through the address hipGetSymbolAddress
// gives on each device (g_scratch), taken once per device with it current.
constexpr size_t kScratchBytes = (size_t)64 << 20;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
void* g_scratch[kMaxDevices];
std::mutex g_scratch_mu;

// The current device's scratch address, looked up on its first use.
int scratch_ptr(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(PRESK_HIP_ERR, "E10001: device " + std::to_string(dev) + " past the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress (scratch)");
        if (!p) return fail(PRESK_HIP_ERR, "E10001: hipGetSymbolAddress gave no scratch address");
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return PRESK_HIP_OK;
}
}  // namespace

struct presk_hip_kernel {
    std::unique_ptr<Kernel> k;
    std::unique_ptr<ClassPlan> plan;
    Generated gen;
    std::vector<char> code;
    mutable hipModule_t module = nullptr;
    mutable std::vector<hipFunction_t> fns;
    // a class kernel's scratch for presk_hip_run, allocated on first use
    mutable void* work = nullptr;
    int mode = PRESK_HIP_EXACT;
    // the printed chains of a recorded batch whose first one begins with this
    // kernel, loaded as its own module is and unloaded with it: a graph in
    // flight may still be running their code when its batch is released
    struct Chains {
        std::string src;
        hipModule_t module;
        std::vector<hipFunction_t> fns;
    };
    mutable std::vector<Chains> chains;
};

// The most batches' chains a kernel keeps; a further batch's kernels are
// launched one by one.
constexpr size_t kMaxChains = 16;
std::mutex g_chains_mu;

extern "C" {

const char* presk_hip_last_error(void) { return g_error.c_str(); }

int presk_hip_init(int device) {
    // device -1: PRESK_HIP_DEVICE, else device 0
    if (device < 0) {
        const char* env = std::getenv("PRESK_HIP_DEVICE");
        char* end = nullptr;
        const long d = env && *env ? std::strtol(env, &end, 10) : 0;
        if (env && *env && (*end != '\0' || d < 0 || d > 1 << 16))
            return fail(PRESK_HIP_ERR, std::string("E10001: PRESK_HIP_DEVICE=") + env + ": expected a device ordinal");
        device = (int)d;
    }
    // the environment's switches are checked once, here
    std::string err;
    TileOverride t;
    if (!tile_override(&t, &err)) return fail(PRESK_HIP_ERR, "E10001: " + err);
    if (forced_mode(&err) == -2) return fail(PRESK_HIP_ERR, "E10001: " + err);
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
    g_device = device;
    // the no-allocation entry point's scratch, looked up once per device
    void* p = nullptr;
    return scratch_ptr(&p);
}

int presk_hip_compile(const char* text, const char* dtype, int lanes, int mode, presk_hip_kernel** out) {
    if (!text || !out) return fail(PRESK_HIP_ERR, "E10001: null argument");
    std::string err;
    auto k = parse_kernel(text, dtype ? dtype : "", lanes, &err);
    if (!k) {
        bool refused = err.compare(0, 5, "E7005") == 0;
        return fail(refused ? PRESK_HIP_REFUSED : PRESK_HIP_ERR, (refused ? "" : "E10001: ") + err);
    }
    if (!k->arith.empty())
        return fail(PRESK_HIP_REFUSED, "E7005: the kernel `" + k->name + "` computes in " + k->arith +
                                           ", which only the kernel interpreter emulates");
    if (const int forced = forced_mode(&err); forced >= 0) mode = forced;
    if (mode != PRESK_HIP_EXACT && mode != PRESK_HIP_FAST) return fail(PRESK_HIP_ERR, "E10001: mode is neither EXACT nor FAST");
    auto h = std::make_unique<presk_hip_kernel>();
    h->mode = mode;
    h->plan = classify(*k, mode);
    if (!h->plan) {
        if (!generate_hip(*k, &h->gen, &err, mode == PRESK_HIP_FAST)) return fail(err.compare(0, 5, "E7005") == 0 ? PRESK_HIP_REFUSED : PRESK_HIP_ERR, err);
        // PRESK_HIP_DUMP=<dir>: keep each printed source, for inspection
        if (const char* dump = std::getenv("PRESK_HIP_DUMP")) {
            char name[40];
            std::snprintf(name, sizeof name, "/%016llx.hip", (unsigned long long)fnv1a(h->gen.src));
            std::ofstream(std::string(dump) + name) << "// " << k->name << "\n" << h->gen.src;
        }
        if (!build_code_object(h->gen.src, &h->code, &err)) return fail(PRESK_HIP_ERR, err);
    }
    h->k = std::move(k);
    // on a device (after presk_hip_init) the code object is loaded now, so
    // that presk_hip_run_noalloc never loads one
    if (g_device >= 0)
        if (int rc = load_module(h.get())) return rc;
    *out = h.release();
    return PRESK_HIP_OK;
}

}  // extern "C"

namespace {

// The generic kernel's code object, loaded on the current device.
int load_module(const presk_hip_kernel* h) {
    if (h->plan || h->module) return PRESK_HIP_OK;
    hipModule_t m = nullptr;
    hipError_t e = hipModuleLoadData(&m, h->code.data());
    if (e != hipSuccess) return hip_fail(e, "hipModuleLoadData");
    std::vector<hipFunction_t> fns;
    for (auto& ph : h->gen.phases) {
        hipFunction_t f;
        e = hipModuleGetFunction(&f, m, ph.fn.c_str());
        if (e != hipSuccess) {
            hipModuleUnload(m);
            return hip_fail(e, "hipModuleGetFunction");
        }
        fns.push_back(f);
    }
    h->module = m;
    h->fns = std::move(fns);
    return PRESK_HIP_OK;
}

// What a kernel's first launch by presk_hip_run sets up: the generic
// kernel's module, a class kernel's workspace.
int prepare_kernel(const presk_hip_kernel* h) {
    if (!h->plan) return load_module(h);
    const size_t bytes = h->plan->workspace_bytes();
    if (bytes && !h->work) {
        hipError_t e = hipMalloc(&h->work, bytes);
        if (e != hipSuccess) {
            h->work = nullptr;
            return hip_fail(e, "hipMalloc (workspace)");
        }
    }
    return PRESK_HIP_OK;
}

// The generic kernel's phases over [lo, hi) of the split loop.
int run_generic(const presk_hip_kernel* h, void* const* bufs, int64_t lo, int64_t hi, hipStream_t s) {
    const Kernel& k = *h->k;
    PhaseArgs args{};
    // inputs, output, one scales pointer a Quant input, then the flag
    const int nb = (int)k.inputs.size() + 1 + k.n_quant();
    for (int i = 0; i < nb; ++i) args.buf[i] = bufs[i];
    args.flag = k.guarded() ? (unsigned*)bufs[k.flag_slot()] : nullptr;
    for (size_t p = 0; p < h->gen.phases.size(); ++p) {
        const Phase& ph = h->gen.phases[p];
        long long total = 1;
        args.lo = 0;
        args.hi = 0;
        if (!ph.bounds.empty()) {
            long long n0 = ph.bounds[0];
            if (ph.split) {
                if (lo < 0 || hi > n0 || lo > hi) return fail(PRESK_HIP_ERR, "E10001: split range outside the loop");
                args.lo = lo;
                args.hi = hi;
                n0 = hi - lo;
            }
            total = n0;
            for (size_t d = 1; d < ph.bounds.size(); ++d) total *= ph.bounds[d];
        }
        if (total == 0) continue;
        const unsigned block = ph.bounds.empty() ? 1 : 256;
        const long long grid = (total + block - 1) / block;
        if (grid > 0x7fffffffLL) return fail(PRESK_HIP_ERR, "E10001: launch too large");
        void* params[] = {&args};
        hipError_t e = hipModuleLaunchKernel(h->fns[p], (unsigned)grid, 1, 1, block, 1, 1, 0, s, params, nullptr);
        if (e != hipSuccess) return hip_fail(e, "hipModuleLaunchKernel");
    }
    return PRESK_HIP_OK;
}

}  // namespace

extern "C" {

int presk_hip_run(const presk_hip_kernel* h, void* const* bufs, int64_t lo, int64_t hi, void* stream) {
    if (!h || !bufs) return fail(PRESK_HIP_ERR, "E10001: null argument");
    hipStream_t s = (hipStream_t)stream;
    if (int rc = prepare_kernel(h)) return rc;
    if (h->plan) {
        hipError_t e = h->plan->launch(bufs, lo, hi, h->work, s);
        return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, h->plan->kind());
    }
    return run_generic(h, bufs, lo, hi, s);
}

int presk_hip_run_noalloc(const presk_hip_kernel* h, void* const* bufs, int64_t lo, int64_t hi, void* stream) {
    if (!h || !bufs) return fail(PRESK_HIP_ERR, "E10001: null argument");
    hipStream_t s = (hipStream_t)stream;
    if (h->plan) {
        const size_t need = h->plan->workspace_bytes();
        if (need > kScratchBytes)
            return fail(PRESK_HIP_ERR, "E10001: the kernel `" + h->k->name + "` needs " + std::to_string(need) +
                                           " bytes of scratch, more than the " + std::to_string(kScratchBytes) +
                                           " presk_hip_run_noalloc holds; run it with presk_hip_run");
        void* p = nullptr;
        if (need)
            if (int rc = scratch_ptr(&p)) return rc;
        hipError_t e = h->plan->launch(bufs, lo, hi, p, s);
        return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, h->plan->kind());
    }
    if (!h->module)
        return fail(PRESK_HIP_ERR, "E10001: the kernel `" + h->k->name + "` has no code object loaded: compile it after "
                                   "presk_hip_init, or run it once with presk_hip_run");
    return run_generic(h, bufs, lo, hi, s);
}

int presk_hip_kernel_info(const presk_hip_kernel* h, presk_hip_info* info) {
    if (!h || !info) return fail(PRESK_HIP_ERR, "E10001: null argument");
    std::memset(info, 0, sizeof *info);
    std::snprintf(info->kind, sizeof info->kind, "%s", h->plan ? h->plan->kind() : "generic");
    std::snprintf(info->order, sizeof info->order, "%s",
                  h->plan ? h->plan->order().c_str() : h->gen.fast_fns ? "sequential+fast-exp-erf" : "sequential");
    info->guarded = h->k->guarded();
    info->n_inputs = (int32_t)h->k->inputs.size();
    info->split_bound = h->plan ? h->plan->split : parallel_outer(*h->k);
    info->flops = kernel_flops(*h->k);
    info->bytes = kernel_bytes(*h->k);
    return PRESK_HIP_OK;
}

int64_t presk_hip_kernel_text(const presk_hip_kernel* h, char* buf, size_t cap) {
    if (!h) return fail(PRESK_HIP_ERR, "E10001: null argument");
    std::string t = show_kernel(*h->k);
    if (buf && cap) std::snprintf(buf, cap, "%s", t.c_str());
    return (int64_t)t.size();
}

void presk_hip_release(presk_hip_kernel* h) {
    if (!h) return;
    if (h->module) hipModuleUnload(h->module);
    for (const auto& c : h->chains) hipModuleUnload(c.module);
    if (h->work) hipFree(h->work);
    delete h;
}

int presk_hip_alloc(size_t bytes, void** dev) {
    hipError_t e = hipMalloc(dev, bytes ? bytes : 1);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipMalloc");
}
int presk_hip_free(void* dev) {
    hipError_t e = hipFree(dev);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipFree");
}
int presk_hip_h2d(void* dev, const void* host, size_t bytes, void* stream) {
    hipError_t e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipMemcpy h2d");
}
int presk_hip_d2h(void* host, const void* dev, size_t bytes, void* stream) {
    hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipMemcpy d2h");
}
int presk_hip_memset(void* dev, int value, size_t bytes, void* stream) {
    hipError_t e = hipMemsetAsync(dev, value, bytes, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipMemsetAsync");
}
int presk_hip_sync(void* stream) {
    hipError_t e = hipStreamSynchronize((hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipStreamSynchronize");
}
int presk_hip_stream_create(void** stream) {
    hipError_t e = hipStreamCreate((hipStream_t*)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipStreamCreate");
}
int presk_hip_stream_destroy(void* stream) {
    hipError_t e = hipStreamDestroy((hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipStreamDestroy");
}

int presk_hip_time(const presk_hip_kernel* h, void* const* bufs, int64_t lo, int64_t hi, void* stream, int warmup, int reps,
                   double* ms_per_launch) {
    if (reps <= 0 || !ms_per_launch) return fail(PRESK_HIP_ERR, "E10001: bad timing arguments");
    for (int i = 0; i < warmup; ++i) {
        int rc = presk_hip_run(h, bufs, lo, hi, stream);
        if (rc) return rc;
    }
    hipEvent_t a, b;
    hipEventCreate(&a);
    hipEventCreate(&b);
    hipEventRecord(a, (hipStream_t)stream);
    for (int i = 0; i < reps; ++i) {
        int rc = presk_hip_run(h, bufs, lo, hi, stream);
        if (rc) {
            hipEventDestroy(a);
            hipEventDestroy(b);
            return rc;
        }
    }
    hipEventRecord(b, (hipStream_t)stream);
    hipError_t e = hipEventSynchronize(b);
    float ms = 0;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
    hipEventDestroy(a);
    hipEventDestroy(b);
    if (e != hipSuccess) return hip_fail(e, "hipEvent timing");
    *ms_per_launch = (double)ms / reps;
    return PRESK_HIP_OK;
}

}  // extern "C"

struct presk_hip_batch {
    // a kernel launch, or (k null) an edge conversion, or (k null, rate >= 0)
    // a dropout mask: bufs {key, dst}, type in `to`
    struct Item {
        const presk_hip_kernel* k;
        std::vector<void*> bufs;
        int64_t lo, hi;
        int from = -1, to = -1;
        int64_t n = 0;
        double rate = -1.0;
    };
    std::vector<Item> items;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // the graph's launches: an item, or (`fn` set) a run of `count`
    // elementwise items from `first` in one printed kernel
    struct Unit {
        int first = 0, count = 1;
        hipFunction_t fn = nullptr;
        unsigned grid = 0;
        PhaseArgs args{};
    };
    std::vector<Unit> units;

    void drop_graph() {
        if (exec) hipGraphExecDestroy(exec);
        if (graph) hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
        units.clear();
    }
    int run_units(hipStream_t s) const {
        for (const Unit& u : units) {
            if (!u.fn) {
                if (int rc = run_one(items[u.first], s)) return rc;
                continue;
            }
            PhaseArgs a = u.args;
            void* params[] = {&a};
            hipError_t e = hipModuleLaunchKernel(u.fn, u.grid, 1, 1, 256, 1, 1, 0, s, params, nullptr);
            if (e != hipSuccess) return hip_fail(e, "hipModuleLaunchKernel");
        }
        return PRESK_HIP_OK;
    }
    static int run_one(const Item& it, hipStream_t s) {
        if (!it.k && it.rate >= 0.0) {
            hipError_t e = dropout_launch(it.bufs[0], it.rate, it.to, it.n, it.bufs[1], s);
            return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "dropout mask");
        }
        if (!it.k) {
            hipError_t e = convert_launch(it.bufs[0], it.from, it.bufs[1], it.to, it.n, (unsigned*)it.bufs[2], s);
            return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "edge conversion");
        }
        return presk_hip_run(it.k, it.bufs.data(), it.lo, it.hi, s);
    }
    int run_each(hipStream_t s) const {
        for (const Item& it : items)
            if (int rc = run_one(it, s)) return rc;
        return PRESK_HIP_OK;
    }
    ~presk_hip_batch() { drop_graph(); }
};

namespace {

constexpr int kMaxBranches = 8;
constexpr bool kBranchesOn = false;

// Whether byte ranges [a, a + na) and [b, b + nb) meet.
bool meet(const void* a, int64_t na, const void* b, int64_t nb) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return x < y + (uintptr_t)nb && y < x + (uintptr_t)na;
}

int64_t buffer_bytes(const BufSpec& s) { return s.numel() * ty_bytes(s.ty); }

// The functions of a batch's printed chains (one source, `n` of them), from
// those that the first one's first kernel holds; empty when they cannot be had
// (their kernels are then launched one by one).  Built and loaded outside the
// lock, so that recordings on other threads do not wait for it; of two threads
// that load the same source the first one's is kept.
std::vector<hipFunction_t> chain_functions(const presk_hip_kernel* h, const std::string& src, size_t n) {
    // (with the lock held)
    auto held = [&]() {
        for (const auto& c : h->chains)
            if (c.src == src) return c.fns;
        return std::vector<hipFunction_t>();
    };
    {
        std::lock_guard<std::mutex> lock(g_chains_mu);
        auto fns = held();
        if (!fns.empty() || h->chains.size() >= kMaxChains) return fns;
    }
    std::vector<char> code;
    std::string err;
    presk_hip_kernel::Chains c{src, nullptr, std::vector<hipFunction_t>(n, nullptr)};
    if (!build_code_object(src, &code, &err)) return {};
    hipError_t e = hipModuleLoadData(&c.module, code.data());
    if (e == hipSuccess) {
        for (size_t i = 0; i < n && e == hipSuccess; ++i) e = hipModuleGetFunction(&c.fns[i], c.module, chain_name(i).c_str());
        if (e == hipSuccess) {
            std::lock_guard<std::mutex> lock(g_chains_mu);
            auto fns = held();
            if (fns.empty() && h->chains.size() < kMaxChains) {
                h->chains.push_back(c);
                return c.fns;
            }
            c.fns = fns;
        }
        (void)hipModuleUnload(c.module);
    }
    // the launches that stand in read the last error: a failed load is not theirs
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return {};
    }
    return c.fns;
}

// The batch's launches as the graph takes them: runs of elementwise nests
// over the same elements, each reading one of the run's earlier outputs,
// become one launch that writes every output and takes what it reads of them
// from registers.  Such a run is bound by its bytes and by the ~2 us a launch
// takes to fill and drain the chip: LayerNorm's reverse mode in bf16 at
// 16384 x 384, 20 launches over 12.6 MB matrices 126 -> 101 us; the
// attention gradient's broadcast, sub and mul, div over 100 MB matrices
// saves two of its eight passes, 499 -> 458 us for the whole call.
// A thread reads only what it wrote itself: the later nest reads the earlier
// one's whole output at its own index, and the bytes it writes meet nothing
// that the run reads or writes.  FAST only: the compiler may order a product's
// operands differently in the longer kernel, and the sign of a NaN is that of
// the first one.  A batch's chains are one source and one module (a module
// takes 0.3-0.4 ms to load): recording LayerNorm's four 1.74 ms as modules of
// their own, 0.65 as one (0.19 without chains), and 558 -> 164 ms the first
// time, when they are compiled; the course step 5.9 -> 3.2 ms.
void plan_units(presk_hip_batch& b, bool chains) {
    constexpr size_t kMaxChain = 6;
    b.units.clear();
    std::vector<std::string> sources;                // the chains', each once
    std::vector<std::pair<size_t, size_t>> printed;  // (unit, its source)
    const size_t n = b.items.size();
    auto flat = [&](const presk_hip_batch::Item& it, FlatNest* f) {
        if (!it.k || it.k->mode != PRESK_HIP_FAST || it.k->plan || it.k->gen.phases.size() != 1) return false;
        const int64_t split = parallel_outer(*it.k->k);
        if (it.lo != 0 || it.hi != (split > 0 ? split : 0)) return false;
        return flat_nest(*it.k->k, f);
    };
    for (size_t i = 0; i < n;) {
        presk_hip_batch::Unit u;
        u.first = (int)i;
        FlatNest f0;
        std::vector<std::vector<int>> from;
        size_t count = 1, slots = 0;
        if (chains && flat(b.items[i], &f0)) {
            const Kernel& k0 = *b.items[i].k->k;
            from.push_back(std::vector<int>(k0.inputs.size(), -1));
            slots = k0.inputs.size() + 1;
            for (; count < kMaxChain && i + count < n; ++count) {
                const auto& it = b.items[i + count];
                FlatNest f;
                if (!flat(it, &f) || f.vec != f0.vec || f.numel != f0.numel) break;
                const Kernel& k = *it.k->k;
                if (k.output.ty != k0.output.ty) break;
                const void* out = it.bufs[k.out_buf()];
                const int64_t out_bytes = buffer_bytes(k.output);
                std::vector<int> link(k.inputs.size(), -1);
                bool ok = true, linked = false;
                size_t need = 1;
                for (size_t q = 0; q < k.inputs.size() && ok; ++q) {
                    if (meet(it.bufs[q], buffer_bytes(k.inputs[q]), out, out_bytes)) ok = false;
                    for (size_t e = 0; e < count && ok; ++e) {
                        const auto& pe = b.items[i + e];
                        const Kernel& ke = *pe.k->k;
                        const void* po = pe.bufs[ke.out_buf()];
                        if (!meet(it.bufs[q], buffer_bytes(k.inputs[q]), po, buffer_bytes(ke.output))) continue;
                        if (po != it.bufs[q] || !f.same[q] || k.inputs[q].ty != ke.output.ty) ok = false;
                        link[q] = (int)e;
                        linked = true;
                    }
                    if (link[q] < 0) ++need;
                }
                // nothing of the run reads or writes the bytes this one writes
                for (size_t e = 0; e < count && ok; ++e) {
                    const auto& pe = b.items[i + e];
                    const Kernel& ke = *pe.k->k;
                    for (size_t q = 0; q <= ke.inputs.size(); ++q)
                        if (meet(pe.bufs[q], buffer_bytes(ke.buf((int)q)), out, out_bytes)) ok = false;
                    if (k.guarded() && it.bufs[k.flag_slot()] != pe.bufs[ke.flag_slot()]) ok = false;
                }
                if (!ok || !linked || slots + need > (size_t)kMaxBufs) break;
                slots += need;
                from.push_back(link);
            }
        }
        if (count > 1) {
            std::vector<const Kernel*> ks;
            for (size_t e = 0; e < count; ++e) ks.push_back(b.items[i + e].k->k.get());
            Generated g;
            std::vector<std::pair<int, int>> where;
            std::string err;
            if (generate_chain(ks, from, &g, &where, &err) && (g.phases[0].bounds[0] + 255) / 256 <= 0x7fffffffLL) {
                const size_t at = std::find(sources.begin(), sources.end(), g.src) - sources.begin();
                if (at == sources.size()) sources.push_back(g.src);
                printed.push_back({b.units.size(), at});
                u.count = (int)count;
                u.grid = (unsigned)((g.phases[0].bounds[0] + 255) / 256);
                for (size_t q = 0; q < where.size(); ++q) u.args.buf[q] = b.items[i + where[q].first].bufs[where[q].second];
                const Kernel& k0 = *ks[0];
                u.args.flag = k0.guarded() ? (unsigned*)b.items[i].bufs[k0.flag_slot()] : nullptr;
            }
        }
        i += (size_t)u.count;
        b.units.push_back(u);
    }
    if (printed.empty()) return;
    const auto fns = chain_functions(b.items[b.units[printed[0].first].first].k, chain_source(sources), sources.size());
    if (fns.empty()) {
        b.units.assign(n, presk_hip_batch::Unit());
        for (size_t i = 0; i < n; ++i) b.units[i].first = (int)i;
        return;
    }
    for (const auto& p : printed) b.units[p.first].fn = fns[p.second];
}

// The batch's items as the branch planner (branches.hpp) reads them.
std::vector<BranchStep> branch_steps(const presk_hip_batch& b) {
    std::vector<BranchStep> out;
    out.reserve(b.items.size());
    for (const auto& it : b.items) {
        BranchStep st;
        st.k = it.k ? it.k->k.get() : nullptr;
        st.handle = it.k;
        st.bufs = it.bufs;
        st.from = it.from;
        st.to = it.to;
        st.n = it.n;
        st.rate = it.rate;
        out.push_back(std::move(st));
    }
    return out;
}

}  // namespace

extern "C" {

int presk_hip_batch_create(presk_hip_batch** out) {
    if (!out) return fail(PRESK_HIP_ERR, "E10001: null argument");
    *out = new presk_hip_batch();
    return PRESK_HIP_OK;
}

int presk_hip_batch_add(presk_hip_batch* b, const presk_hip_kernel* k, void* const* bufs, int64_t lo, int64_t hi) {
    if (!b || !k || !bufs) return fail(PRESK_HIP_ERR, "E10001: null argument");
    const size_t n = k->k->flag_slot() + (k->k->guarded() ? 1 : 0);
    b->drop_graph();
    b->items.push_back({k, std::vector<void*>(bufs, bufs + n), lo, hi});
    return PRESK_HIP_OK;
}

int presk_hip_convert(const void* src, const char* from, void* dst, const char* to, int64_t n, uint32_t* flag,
                      void* stream) {
    const int f = convert_type(from), t = convert_type(to);
    if (f < 0 || t < 0) return fail(PRESK_HIP_ERR, "E10001: a conversion between `" + std::string(from ? from : "") +
                                                       "` and `" + std::string(to ? to : "") + "`, not storage types");
    if (n < 0 || (n > 0 && (!src || !dst))) return fail(PRESK_HIP_ERR, "E10001: bad conversion arguments");
    hipError_t e = convert_launch(src, f, dst, t, n, flag, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "edge conversion");
}

int presk_hip_dropout_mask(const void* key, double rate, const char* type, int64_t n, void* dst, void* stream) {
    const int t = convert_type(type);
    if (t < 0) return fail(PRESK_HIP_ERR, "E10001: a dropout mask of type `" + std::string(type ? type : "") + "`");
    if (!(rate >= 0.0 && rate < 1.0)) return fail(PRESK_HIP_ERR, "E7001: dropout: the rate " + std::to_string(rate) + " is not in [0, 1)");
    if (n < 0 || (n > 0 && (!key || !dst)) || (uintptr_t)key % 4) return fail(PRESK_HIP_ERR, "E10001: bad dropout arguments");
    hipError_t e = dropout_launch(key, rate, t, n, dst, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "dropout mask");
}

int presk_hip_batch_add_dropout(presk_hip_batch* b, const void* key, double rate, const char* type, int64_t n, void* dst) {
    if (!b) return fail(PRESK_HIP_ERR, "E10001: null argument");
    const int t = convert_type(type);
    if (t < 0 || !(rate >= 0.0 && rate < 1.0) || n < 0 || (n > 0 && (!key || !dst)) || (uintptr_t)key % 4)
        return fail(PRESK_HIP_ERR, "E10001: bad dropout arguments");
    b->drop_graph();
    presk_hip_batch::Item it{nullptr, {const_cast<void*>(key), dst}, 0, 0};
    it.to = t;
    it.n = n;
    it.rate = rate;
    b->items.push_back(it);
    return PRESK_HIP_OK;
}

int presk_hip_batch_add_convert(presk_hip_batch* b, const void* src, const char* from, void* dst, const char* to,
                                int64_t n, uint32_t* flag) {
    if (!b) return fail(PRESK_HIP_ERR, "E10001: null argument");
    const int f = convert_type(from), t = convert_type(to);
    if (f < 0 || t < 0 || n < 0 || (n > 0 && (!src || !dst))) return fail(PRESK_HIP_ERR, "E10001: bad conversion arguments");
    b->drop_graph();
    presk_hip_batch::Item it{nullptr, {const_cast<void*>(src), dst, flag}, 0, 0};
    it.from = f;
    it.to = t;
    it.n = n;
    b->items.push_back(it);
    return PRESK_HIP_OK;
}

int presk_hip_batch_graph(presk_hip_batch* b) { return presk_hip_batch_graph_branches(b, 1); }

int presk_hip_batch_graph_branches(presk_hip_batch* b, int branches) {
    if (!b) return fail(PRESK_HIP_ERR, "E10001: null argument");
    if (branches < 1 || branches > kMaxBranches)
        return fail(PRESK_HIP_ERR, "E10001: branches " + std::to_string(branches) + " not in 1.." + std::to_string(kMaxBranches));
    // switched off: the one branched capture run on the device (the course
    // step, four branches) ended in a host segmentation fault inside this
    // call whose cause is not found; one branch is the tested sequence
    if (branches > 1 && !kBranchesOn)
        return fail(PRESK_HIP_ERR, "E10001: parallel graph branches are switched off in this build; use 1");
    b->drop_graph();
    for (const auto& it : b->items)
        if (it.k)
            if (int rc = prepare_kernel(it.k)) return rc;
    const int n = (int)b->items.size();
    plan_units(*b, branches == 1);
    std::vector<int> lane;       // each step's capture stream
    std::vector<std::vector<std::pair<int, int>>> waits;   // (stream, step) events each step waits for
    plan_branches(branch_steps(*b), branches, &lane, &waits);
    int used = 1;
    for (int s : lane) used = std::max(used, s + 1);
    std::vector<hipStream_t> cs(used, nullptr);
    std::vector<hipEvent_t> ev;   // one a step when there are branches, then the fork
    hipError_t e = hipSuccess;
    auto cleanup = [&]() {
        for (hipEvent_t x : ev)
            if (x) hipEventDestroy(x);
        for (hipStream_t s : cs)
            if (s) hipStreamDestroy(s);
    };
    for (int s = 0; s < used && e == hipSuccess; ++s) e = hipStreamCreateWithFlags(&cs[s], hipStreamNonBlocking);
    if (used > 1)
        for (int i = 0; i <= n && e == hipSuccess; ++i) {
            ev.push_back(nullptr);
            e = hipEventCreateWithFlags(&ev.back(), hipEventDisableTiming);
        }
    if (e != hipSuccess) {
        cleanup();
        return hip_fail(e, "graph streams and events");
    }
    e = hipStreamBeginCapture(cs[0], hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) {
        cleanup();
        return hip_fail(e, "hipStreamBeginCapture");
    }
    int rc = PRESK_HIP_OK;
    if (used == 1) {
        rc = b->run_units(cs[0]);
    } else {
        // the other streams join the capture from the first one, then each
        // step waits for the last step of every other stream it depends on,
        // runs, and marks its end; the first stream finally waits for all
        e = hipEventRecord(ev[n], cs[0]);
        for (int s = 1; s < used && e == hipSuccess; ++s) e = hipStreamWaitEvent(cs[s], ev[n], 0);
        for (int i = 0; i < n && e == hipSuccess && !rc; ++i) {
            hipStream_t s = cs[lane[i]];
            for (const auto& w : waits[i])
                if (e == hipSuccess) e = hipStreamWaitEvent(s, ev[w.second], 0);
            if (e != hipSuccess) break;
            rc = b->run_one(b->items[i], s);
            if (!rc) e = hipEventRecord(ev[i], s);
        }
        for (int s = 1; s < used && e == hipSuccess && !rc; ++s) {
            e = hipEventRecord(ev[n], cs[s]);
            if (e == hipSuccess) e = hipStreamWaitEvent(cs[0], ev[n], 0);
        }
    }
    hipGraph_t g = nullptr;
    const hipError_t ee = hipStreamEndCapture(cs[0], &g);  // ended whatever the launches returned
    cleanup();
    if (rc || e != hipSuccess) {
        if (g) hipGraphDestroy(g);
        return rc ? rc : hip_fail(e, "branched capture");
    }
    e = ee;
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        hipGraphDestroy(g);
        return hip_fail(e, "hipGraphInstantiate");
    }
    b->graph = g;
    b->exec = x;
    return PRESK_HIP_OK;
}

int presk_hip_batch_run(presk_hip_batch* b, void* stream) {
    if (!b) return fail(PRESK_HIP_ERR, "E10001: null argument");
    if (b->exec) {
        hipError_t e = hipGraphLaunch(b->exec, (hipStream_t)stream);
        return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "hipGraphLaunch");
    }
    return b->run_each((hipStream_t)stream);
}

void presk_hip_batch_release(presk_hip_batch* b) { delete b; }

int presk_hip_fill_normal(void* dst, const char* type, int64_t n, uint64_t seed, double mean, double std, void* stream) {
    const int t = convert_type(type);
    if (t != 1 && t != 2 && t != 4)
        return fail(PRESK_HIP_ERR, "E10001: a fill of type `" + std::string(type ? type : "") + "` (f32, bf16 or f16)");
    if (n < 0 || (n > 0 && !dst)) return fail(PRESK_HIP_ERR, "E10001: bad fill arguments");
    hipError_t e = synth_normal_launch(dst, t, n, seed, (float)mean, (float)std, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "fill");
}

int presk_hip_mfma_probe(const char* type, int64_t iters, void* stream, double* ms, double* flops) {
    const std::string t = type ? type : "";
    if ((t != "bf16" && t != "f32") || iters <= 0 || !ms || !flops)
        return fail(PRESK_HIP_ERR, "E10001: an MFMA probe of type `" + t + "` (bf16 or f32) and iters > 0");
    if (g_device < 0) return fail(PRESK_HIP_ERR, "E10001: no device (presk_hip_init)");
    hipError_t e = mfma_probe(t == "bf16" ? 0 : 1, iters, (hipStream_t)stream, ms, flops);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "MFMA probe");
}

}  // extern "C"

namespace {

// A version 3 header's six bytes as a format (crates/presk-data/src/lib.rs:143-166,
// Enc::of_description), refused unless it is one (presk-format lib.rs:220-240,
// Float::check); "" when it is, else why not.
std::string psk_format(const uint8_t* d, PskFormat* f) {
    const unsigned flags = d[5];
    const int specials = (int)(flags >> 1 & 3), overflow = (int)(flags >> 3 & 3);
    if (specials > 2) return "special values " + std::to_string(specials);
    if (overflow > 2) return "overflow " + std::to_string(overflow);
    if (flags >> 7) return "flags " + std::to_string(flags);
    f->p = d[0];
    f->emin = (int16_t)(d[1] | d[2] << 8);
    f->emax = (int16_t)(d[3] | d[4] << 8);
    f->subnormals = flags & 1;
    f->specials = specials;
    const bool default_nan = flags & 64;
    if (f->p < 2 || f->p > 53) return "a float format has 2 to 53 bits of significand, not " + std::to_string(f->p);
    if (f->emin > f->emax || f->emin < -1022 || f->emax > 1023) return "the exponent range is not inside f64's";
    const unsigned long long codes = (unsigned long long)(f->emax - f->emin + 2) + (specials == 0 ? 1 : 0);
    if (codes & (codes - 1)) return "the exponent range does not fill an exponent field";
    if (default_nan && specials == 2) return "a format with no NaN gives no default NaN";
    // (specials, overflow): IEEE any; NaN only -> NaN or saturation; none -> saturation
    if ((specials == 1 && overflow == 0) || (specials == 2 && overflow != 2)) return "an overflow its special values do not allow";
    f->ebits = __builtin_ctzll(codes);
    f->bits = 1 + f->ebits + f->p - 1;
    f->width = (f->bits + 7) / 8;
    return "";
}

}  // namespace

extern "C" {

int presk_hip_pskd_decode(const void* src, int enc, const uint8_t* desc, int64_t n, void* dst, const char* to, uint32_t* flag,
                          void* stream) {
    const int t = convert_type(to);
    if (t < 0) return fail(PRESK_HIP_ERR, "E10001: a .psk.d leaf decoded into `" + std::string(to ? to : "") + "`, not a storage type");
    if (n < 0 || (n > 0 && (!src || !dst))) return fail(PRESK_HIP_ERR, "E10001: bad decode arguments");
    PskFormat f{};
    if (enc == 3) {
        if (!desc) return fail(PRESK_HIP_ERR, "E10001: encoding 3 needs its format's description");
        const std::string why = psk_format(desc, &f);
        if (!why.empty()) return fail(PRESK_HIP_ERR, "E9002: a format the encoding does not describe (" + why + ")");
    } else if (enc < 0 || enc > 2) {
        return fail(PRESK_HIP_ERR, "E9002: unknown encoding " + std::to_string(enc));
    }
    hipError_t e = pskd_decode_launch(src, enc, f, n, dst, t, flag, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, ".psk.d decode");
}

int presk_hip_pskd_decode_idx(const void* src, uint64_t bound, int64_t n, int64_t* dst, void* stream) {
    if (bound == 0) return fail(PRESK_HIP_ERR, "E9001: an `idx[0]` has no values");
    if (n < 0 || (n > 0 && (!src || !dst))) return fail(PRESK_HIP_ERR, "E10001: bad decode arguments");
    const uint64_t top = bound - 1;
    const int width = top <= 0xffu ? 1 : top <= 0xffffu ? 2 : top <= 0xffffffffu ? 4 : 8;
    hipError_t e = pskd_idx_launch(src, width, n, (long long*)dst, (hipStream_t)stream);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, ".psk.d decode");
}

int presk_hip_scalar_digest(int fn, uint64_t lo, uint64_t hi, uint64_t* digest) {
    hipError_t e = scalar_digest(fn, lo, hi, digest);
    return e == hipSuccess ? PRESK_HIP_OK : hip_fail(e, "scalar digest");
}

}  // extern "C"
