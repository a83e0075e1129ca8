// General step functions: user HIP device code compiled with hipRTC.
//
// Replaces generate_gpu_func + the CuPy JIT of the generated module
// (model.py:2010-2457, :800-865) for models whose step functions are not the
// built-in compartment step: the host side writes one wrapper kernel per
// priority group around the user's __device__ functions, this file compiles
// it for gfx950 (code objects cached by a hash of the source, as the
// reference caches its generated module, model.py:843-865), loads it, and
// runs the per-tick launch schedule followed by the write-back of
// double-buffered arrays (model.py:2368-2408).
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include <sys/stat.h>
#include <unistd.h>

#include <hip/hiprtc.h>

#include "../../include/sagestep.h"
#include "ss_runtime.h"

namespace {

// the device runtime header, embedded at build time from step_rt.h
const char *kStepRtHeader =
#include "step_rt_embed.inc"
    ;

#define SS_MAXP_HOST 64
#define SS_MAXX_HOST 16

struct ProgArgsHost {           // layout of SSProgArgs in step_rt.h
    long long n_agents;
    const long long *row_ptr;
    const int *col_idx;
    const float *agent_ids;
    const float *logical_ids;
    const float *breeds;
    const double *globals;
    void *prop_r[SS_MAXP_HOST];
    void *prop_w[SS_MAXP_HOST];
    int seed;
    const long long *logical_ids64;
    void *extra[SS_MAXX_HOST];
};

// a device array of the program: rows x width elements, double-buffered
// (read and write buffer) or one buffer for both
struct ProgProp {
    int32_t elem_bytes = 0;
    int64_t rows = 0;
    int64_t width = 1;
    bool double_buffered = true;
    void *r = nullptr, *w = nullptr;
    size_t bytes() const { return (size_t)elem_bytes * (size_t)width * (size_t)rows; }
};

struct Launch {
    int32_t kernel;
    int64_t start, count;
    int64_t order_off;          // first entry of this launch in the order array, -1: agents in index order
    int64_t n_long = 0;         // agents at the front of the order that get a block each
    int64_t long_deg = 0;       // entries of the longest of their rows
};

// Whether the one-block kernel still pays, from the time its launches take.  What
// a step does is the user's: one that walks all agents keeps a compute unit busy
// for a millisecond a tick, where the schedule spreads it over several.  A
// schedule's tick takes its launches at least (5 us each), so a tick below that
// (and the 30 us of a launch that is waited for) is left alone; a longer one is set
// against the schedule, two samples of either over ticks that are due anyway, and
// the faster one goes on (asked again once a tick takes twice as long).  us a tick
// of such a step, one block and schedule: 300 agents 70 and 62, 1000 agents 317 and
// 190, 2000 agents 1260 and 376.  The first launch gets 16 ticks, the next ones four
// times as many as the one before, at most 4096 and 20 ms of them.
struct LoopTrial {
    int64_t chunk = 16;         // ticks of the next launch
    int samples = 0;            // taken since a launch took too long: that one, another, two of the schedule
    double bar = 0.0;           // us a tick above which the schedule is tried; 0: what its launches take
    double loop = 0.0, sched = 0.0;

    void add(double us, int64_t n, size_t launches) {
        const double tick = us / (double)n;
        if (samples >= 2) {
            sched = samples == 2 ? tick : std::min(sched, tick);
            ++samples;
            return;
        }
        loop = samples == 0 ? tick : std::min(loop, tick);
        const double limit = bar > 0.0 ? bar : 5.0 * (double)launches;
        if (samples || us > 30.0 + limit * (double)n) ++samples;
        chunk = std::max<int64_t>(1, std::min<int64_t>({4 * chunk, (int64_t)(20000.0 / tick), 4096}));
    }
    bool schedule_wins() {
        if (samples < 4) return false;
        samples = 0;
        bar = 2.0 * loop;
        return sched < loop;
    }
};

struct Extra {
    void *d = nullptr;
    int64_t bytes = 0;
};

uint64_t fnv1a(uint64_t h, const void *p, size_t n) {
    const unsigned char *b = static_cast<const unsigned char *>(p);
    for (size_t i = 0; i < n; ++i) {
        h ^= b[i];
        h *= 1099511628211ull;
    }
    return h;
}

// Loops of unknown trip count (a step function's walk over its neighbour row)
// are unrolled at run time, so one thread has several neighbour loads in
// flight instead of one round trip per neighbour; entries beyond the last whole
// round run one at a time, so the count has to fit the rows
// (ss_prog_set_unroll; 48 by default).  SAGESIM_AMD_RTC_UNROLL overrides the
// count (1 disables it) and SAGESIM_AMD_RTC_UNROLL_THRESHOLD the size the
// unrolled body may reach (LLVM lowers the count of a loop whose body would
// grow past it: a heavy loop body unrolls less).
std::vector<std::string> rtc_options(int unroll) {
    std::vector<std::string> o = {"--offload-arch=gfx950", "-O3", "-std=c++20", "-ffp-contract=off",
                                  "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    std::string threshold = "1200";
    if (const char *u = std::getenv("SAGESIM_AMD_RTC_UNROLL")) unroll = std::atoi(u);
    if (const char *t = std::getenv("SAGESIM_AMD_RTC_UNROLL_THRESHOLD")) threshold = t;
    if (unroll > 1) {
        o.insert(o.end(), {"-mllvm", "-unroll-runtime", "-mllvm", "-unroll-count=" + std::to_string(unroll)});
        if (!threshold.empty()) o.insert(o.end(), {"-mllvm", "-unroll-threshold=" + threshold});
    }
    return o;
}

// code objects by hash of (options, runtime header, source), for the process
std::mutex g_cache_mu;
std::map<uint64_t, std::vector<char>> g_code_cache;

std::string disk_cache_dir() {
    if (const char *d = std::getenv("SAGESIM_AMD_RTC_CACHE")) return d;   // "" disables the disk cache
    const char *home = std::getenv("HOME");
    return home ? std::string(home) + "/.cache/sagesim_amd/rtc" : std::string();
}

bool read_file(const std::string &path, std::vector<char> &out) {
    std::ifstream f(path, std::ios::binary);
    if (!f) return false;
    out.assign(std::istreambuf_iterator<char>(f), std::istreambuf_iterator<char>());
    return !out.empty();
}

void write_file_atomic(const std::string &dir, const std::string &name, const std::vector<char> &data) {
    std::string acc;
    for (size_t i = 0; i <= dir.size(); ++i) {          // mkdir -p
        if (i == dir.size() || dir[i] == '/') {
            if (!acc.empty()) ::mkdir(acc.c_str(), 0755);
        }
        if (i < dir.size()) acc += dir[i];
    }
    const std::string tmp = dir + "/" + name + ".tmp" + std::to_string((long long)::getpid());
    {
        std::ofstream f(tmp, std::ios::binary);
        if (!f) return;
        f.write(data.data(), (std::streamsize)data.size());
        if (!f) return;
    }
    std::rename(tmp.c_str(), (dir + "/" + name).c_str());
}

// Write buffer -> read buffer of every double-buffered array, one launch:
// block row y copies array y.  Bound by the launch at small sizes (2.2 us each,
// a launch per array before) and by the copy at large ones.
struct WriteBack {
    const void *src[SS_MAXP_HOST];
    void *dst[SS_MAXP_HOST];
    int64_t bytes[SS_MAXP_HOST];
};
__global__ __launch_bounds__(256) void writeback_kernel(const WriteBack w) {
    const int64_t nb = w.bytes[blockIdx.y], n16 = nb / 16;
    const uint4 *src = (const uint4 *)w.src[blockIdx.y];
    uint4 *dst = (uint4 *)w.dst[blockIdx.y];
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = g; i < n16; i += stride) dst[i] = src[i];
    for (int64_t i = n16 * 16 + g; i < nb; i += stride) ((unsigned char *)dst)[i] = ((const unsigned char *)src)[i];
}

}  // namespace

struct ss_prog {
    ss_ctx *ctx = nullptr;
    int64_t n = 0;
    int64_t *row_ptr = nullptr;
    int32_t *col_idx = nullptr;
    int64_t nnz = 0;
    uint64_t csr_hash = 0;
    float *agent_ids = nullptr, *logical_ids = nullptr, *breeds = nullptr;
    int64_t *logical_ids64 = nullptr;
    double *globals = nullptr;
    int64_t n_globals = 0;
    std::vector<double> h_globals;
    std::vector<ProgProp> props;
    Extra extras[SS_MAXX_HOST];
    ProgArgsHost host{};
    ProgArgsHost *d_args = nullptr;
    hipModule_t module = nullptr;
    std::vector<hipFunction_t> kernels;
    std::vector<Launch> schedule;
    int32_t loop_kernel = -1;                   // kernel that runs whole ticks on one block, -1: none
    int32_t loop_threads = 0;
    LoopTrial trial;
    std::vector<int64_t> h_row_ptr;             // row bounds, for the long rows' LDS
    int32_t *order = nullptr;                   // agent order of every launch (concatenated)
    std::vector<int32_t> h_order;
    int64_t order_n = 0;
    int32_t seed = 0;
    int32_t unroll = 48;                        // neighbour-loop unroll count of the next compile
    int32_t cache_hit = 0;                      // the last compile came from the code-object cache
    std::string err;
};

static thread_local std::string g_prog_err;

#define P_FAIL(p, code, ...)                                      \
    do {                                                          \
        char _b[1024];                                            \
        std::snprintf(_b, sizeof _b, __VA_ARGS__);                \
        if (p) (p)->err = _b; else g_prog_err = _b;               \
        return code;                                              \
    } while (0)

#define P_HIP(p, expr)                                                                   \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess)                                                            \
            P_FAIL(p, ss_hip_code(_e), "%s: %s", #expr, hipGetErrorString(_e));          \
    } while (0)

#define P_LIVE(p)                                                                                  \
    do {                                                                                           \
        if ((p) && !(p)->ctx) P_FAIL(p, SS_ERR_STATE, "the context of this program has been destroyed"); \
    } while (0)

static void pfree(void *q) {
    if (q) (void)hipFree(q);
}

static int push_args(ss_prog *p) {
    p->host.n_agents = p->n;
    p->host.row_ptr = (const long long *)p->row_ptr;
    p->host.col_idx = p->col_idx;
    p->host.agent_ids = p->agent_ids;
    p->host.logical_ids = p->logical_ids;
    p->host.breeds = p->breeds;
    p->host.globals = p->globals;
    for (size_t i = 0; i < p->props.size(); ++i) {
        p->host.prop_r[i] = p->props[i].r;
        p->host.prop_w[i] = p->props[i].w;
    }
    p->host.seed = p->seed;
    p->host.logical_ids64 = (const long long *)p->logical_ids64;
    for (int i = 0; i < SS_MAXX_HOST; ++i) p->host.extra[i] = p->extras[i].d;
    P_HIP(p, hipMemcpy(p->d_args, &p->host, sizeof p->host, hipMemcpyHostToDevice));
    return SS_OK;
}

// the module globals neighbor_offsets / neighbor_values (step_rt.h) -> the CSR
static int push_csr_globals(ss_prog *p) {
    if (!p->module) return SS_OK;
    const void *vals[2] = {p->row_ptr, p->col_idx};
    const char *names[2] = {"neighbor_offsets", "neighbor_values"};
    for (int k = 0; k < 2; ++k) {
        hipDeviceptr_t dp = nullptr;
        size_t sz = 0;
        P_HIP(p, hipModuleGetGlobal(&dp, &sz, p->module, names[k]));
        if (sz != sizeof(void *)) P_FAIL(p, SS_ERR_RTC, "%s has size %zu", names[k], sz);
        P_HIP(p, hipMemcpy((void *)dp, &vals[k], sizeof(void *), hipMemcpyHostToDevice));
    }
    return SS_OK;
}

static int push_seed(ss_prog *p) {
    if (!p->module) return SS_OK;
    hipDeviceptr_t dp = nullptr;
    size_t sz = 0;
    P_HIP(p, hipModuleGetGlobal(&dp, &sz, p->module, "ss_rt_seed"));
    if (sz != sizeof(int32_t)) P_FAIL(p, SS_ERR_RTC, "ss_rt_seed has size %zu", sz);
    P_HIP(p, hipMemcpy((void *)dp, &p->seed, sizeof(int32_t), hipMemcpyHostToDevice));
    return SS_OK;
}

// copy every double-buffered array's write buffer into its read buffer
static int write_back(ss_prog *p, hipStream_t st) {
    WriteBack w{};
    int n = 0;
    int64_t most = 0;
    for (const ProgProp &q : p->props) {
        if (!q.double_buffered || q.rows == 0) continue;
        w.src[n] = q.w;
        w.dst[n] = q.r;
        w.bytes[n] = (int64_t)q.bytes();
        most = std::max(most, w.bytes[n++]);
    }
    if (n == 0) return SS_OK;
    const int grid = (int)std::min<int64_t>(std::max<int64_t>((most / 16 + 255) / 256, 1), (int64_t)p->ctx->num_cus * 4);
    hipLaunchKernelGGL(writeback_kernel, dim3(grid, n), dim3(256), 0, st, w);
    P_HIP(p, hipGetLastError());
    return SS_OK;
}

// The program's device resources; its context is alive.
static void release(ss_prog *p) {
    (void)hipStreamSynchronize(p->ctx->stream);
    if (p->module) (void)hipModuleUnload(p->module);
    pfree(p->d_args); pfree(p->agent_ids); pfree(p->logical_ids); pfree(p->breeds);
    pfree(p->row_ptr); pfree(p->col_idx); pfree(p->globals); pfree(p->logical_ids64); pfree(p->order);
    for (auto &q : p->props) {
        if (q.w != q.r) pfree(q.w);
        pfree(q.r);
    }
    for (auto &x : p->extras) pfree(x.d);
    p->module = nullptr;
    p->ctx = nullptr;
}

// Programs may be destroyed after their context (a garbage collector picks the
// order): the context's end frees what they hold on its device, and they keep
// no pointer to it.
void ss_release_programs(ss_ctx *ctx) {
    for (ss_prog *p : ctx->progs) release(p);
    ctx->progs.clear();
}

extern "C" {

const char *ss_prog_last_error(const ss_prog *p) { return p ? p->err.c_str() : g_prog_err.c_str(); }

int ss_prog_create(ss_ctx *ctx, int64_t n_agents, ss_prog **out) {
    if (!ctx || !out || n_agents < 0 || n_agents > INT32_MAX) P_FAIL((ss_prog *)nullptr, SS_ERR_INVALID, "bad arguments");
    auto *p = new ss_prog();
    p->ctx = ctx;
    p->n = n_agents;
    const size_t nn = (size_t)std::max<int64_t>(n_agents, 1);
    hipError_t e = hipSetDevice(ctx->device);
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->d_args, sizeof(ProgArgsHost));
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->agent_ids, nn * sizeof(float));
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->logical_ids, nn * sizeof(float));
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->breeds, nn * sizeof(float));
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->logical_ids64, nn * sizeof(int64_t));
    if (e == hipSuccess) e = ss_device_alloc(ctx, (void **)&p->row_ptr, (nn + 1) * sizeof(int64_t));
    // on the context's stream, like the upload that follows (ss_prog_set_csr): a
    // clear on the null stream could land after it and empty every row
    if (e == hipSuccess) e = hipMemsetAsync(p->row_ptr, 0, (nn + 1) * sizeof(int64_t), ctx->stream);
    if (e != hipSuccess) {
        g_prog_err = std::string("ss_prog_create: ") + hipGetErrorString(e);
        pfree(p->d_args); pfree(p->agent_ids); pfree(p->logical_ids); pfree(p->breeds); pfree(p->row_ptr);
        pfree(p->logical_ids64);
        delete p;
        return ss_hip_code(e);
    }
    ctx->progs.push_back(p);
    *out = p;
    return SS_OK;
}

int ss_prog_destroy(ss_prog *p) {
    if (!p) return SS_OK;
    if (p->ctx) {
        auto &v = p->ctx->progs;
        v.erase(std::remove(v.begin(), v.end(), p), v.end());
        release(p);
    }
    delete p;
    return SS_OK;
}

int ss_prog_set_csr(ss_prog *p, const int64_t *row_ptr, const int32_t *col_idx, int64_t nnz) {
    P_LIVE(p);
    if (!p || !row_ptr || (nnz && !col_idx)) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    if (row_ptr[0] != 0 || row_ptr[p->n] != nnz) P_FAIL(p, SS_ERR_INVALID, "row_ptr must start at 0 and end at nnz");
    for (int64_t i = 0; i < p->n; ++i)
        if (row_ptr[i + 1] < row_ptr[i]) P_FAIL(p, SS_ERR_INVALID, "row_ptr decreases at row %lld", (long long)i);
    for (int64_t e = 0; e < nnz; ++e)
        if (col_idx[e] < 0 || col_idx[e] >= p->n)
            P_FAIL(p, SS_ERR_RANGE, "col_idx[%lld] = %d outside [0, %lld)", (long long)e, col_idx[e], (long long)p->n);
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    pfree(p->col_idx);
    p->col_idx = nullptr;
    P_HIP(p, ss_device_alloc(p->ctx, (void **)&p->col_idx, sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1)));
    P_HIP(p, ss_copy_in(p->ctx, p->col_idx, col_idx, sizeof(int32_t) * (size_t)nnz));
    P_HIP(p, ss_copy_in(p->ctx, p->row_ptr, row_ptr, sizeof(int64_t) * (size_t)(p->n + 1)));
    p->nnz = nnz;
    p->h_row_ptr.assign(row_ptr, row_ptr + p->n + 1);
    for (Launch &l : p->schedule) l.n_long = l.long_deg = 0;   // of the rows before
    p->csr_hash = fnv1a(fnv1a(1469598103934665603ull, row_ptr, sizeof(int64_t) * (size_t)(p->n + 1)), col_idx,
                        sizeof(int32_t) * (size_t)nnz);
    int rc = push_csr_globals(p);
    if (rc) return rc;
    return push_args(p);
}

int ss_prog_set_ids(ss_prog *p, const float *agent_ids, const float *logical_ids, const int64_t *logical_ids64,
                    const float *breeds) {
    P_LIVE(p);
    if (!p || (p->n && (!agent_ids || !logical_ids || !logical_ids64 || !breeds)))
        P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    if (p->n) {
        P_HIP(p, hipMemcpy(p->agent_ids, agent_ids, sizeof(float) * p->n, hipMemcpyHostToDevice));
        P_HIP(p, hipMemcpy(p->logical_ids, logical_ids, sizeof(float) * p->n, hipMemcpyHostToDevice));
        P_HIP(p, hipMemcpy(p->logical_ids64, logical_ids64, sizeof(int64_t) * p->n, hipMemcpyHostToDevice));
        P_HIP(p, hipMemcpy(p->breeds, breeds, sizeof(float) * p->n, hipMemcpyHostToDevice));
    }
    return push_args(p);
}

int ss_prog_add_array(ss_prog *p, int32_t elem_bytes, int64_t rows, int64_t width, int32_t double_buffered,
                      const void *init, int32_t *id) {
    P_LIVE(p);
    if (!p || !id) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    if (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4 && elem_bytes != 8)
        P_FAIL(p, SS_ERR_INVALID, "elem_bytes must be 1, 2, 4 or 8");
    if (width < 1 || rows < 0) P_FAIL(p, SS_ERR_INVALID, "width must be >= 1 and rows >= 0");
    if (p->props.size() >= SS_MAXP_HOST) P_FAIL(p, SS_ERR_FULL, "at most %d device arrays", SS_MAXP_HOST);
    ProgProp q;
    q.elem_bytes = elem_bytes;
    q.rows = rows;
    q.width = width;
    q.double_buffered = double_buffered != 0;
    const size_t b = std::max<size_t>(q.bytes(), 16);
    P_HIP(p, ss_device_alloc(p->ctx, &q.r, b));
    if (q.double_buffered) {
        hipError_t e = ss_device_alloc(p->ctx, &q.w, b);
        if (e != hipSuccess) { pfree(q.r); P_HIP(p, e); }
    } else {
        q.w = q.r;
    }
    const size_t nb = q.bytes();
    hipError_t e = hipSuccess;
    if (nb) {
        if (init) e = ss_copy_in(p->ctx, q.r, init, nb);
        else e = hipMemsetAsync(q.r, 0, nb, p->ctx->stream);
        if (e == hipSuccess && q.w != q.r) e = hipMemcpyAsync(q.w, q.r, nb, hipMemcpyDeviceToDevice, p->ctx->stream);
        if (e != hipSuccess) (void)hipStreamSynchronize(p->ctx->stream);
    }
    if (e != hipSuccess) {
        if (q.w != q.r) pfree(q.w);
        pfree(q.r);
        P_HIP(p, e);
    }
    p->props.push_back(q);
    p->loop_kernel = -1;                        // it writes back the arrays it was compiled for
    *id = (int32_t)p->props.size() - 1;
    return push_args(p);
}

int ss_prog_add_prop(ss_prog *p, int32_t elem_bytes, int64_t width, int32_t double_buffered, const void *init,
                     int32_t *id) {
    P_LIVE(p);
    if (!p) P_FAIL(p, SS_ERR_INVALID, "NULL program");
    return ss_prog_add_array(p, elem_bytes, p->n, width, double_buffered, init, id);
}

int ss_prog_prop_upload(ss_prog *p, int32_t id, const void *data) {
    P_LIVE(p);
    if (!p || id < 0 || id >= (int32_t)p->props.size() || !data) P_FAIL(p, SS_ERR_INVALID, "bad array or NULL");
    const ProgProp &q = p->props[id];
    const size_t nb = q.bytes();
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    if (nb) {
        P_HIP(p, ss_copy_in(p->ctx, q.r, data, nb));
        if (q.w != q.r) P_HIP(p, hipMemcpyAsync(q.w, q.r, nb, hipMemcpyDeviceToDevice, p->ctx->stream));
    }
    return SS_OK;
}

int ss_prog_prop_download(ss_prog *p, int32_t id, void *out) {
    P_LIVE(p);
    if (!p || id < 0 || id >= (int32_t)p->props.size() || !out) P_FAIL(p, SS_ERR_INVALID, "bad array or NULL");
    const ProgProp &q = p->props[id];
    P_HIP(p, ss_copy_out(p->ctx, out, q.r, q.bytes()));
    return SS_OK;
}

int ss_prog_set_globals(ss_prog *p, const double *values, int64_t count) {
    P_LIVE(p);
    if (!p || (count && !values) || count < 0) P_FAIL(p, SS_ERR_INVALID, "bad globals");
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    if (count != p->n_globals) {
        pfree(p->globals);
        p->globals = nullptr;
        P_HIP(p, ss_device_alloc(p->ctx, (void **)&p->globals, sizeof(double) * (size_t)std::max<int64_t>(count, 1)));
        p->n_globals = count;
    }
    if (count) P_HIP(p, hipMemcpy(p->globals, values, sizeof(double) * count, hipMemcpyHostToDevice));
    p->h_globals.assign(values, values + count);
    return push_args(p);
}

// The reference keeps the seed as int32 (model.py:1104) and reduces it mod
// 2^32 in the RNG (math_utils.py:108-111); the low 32 bits are what matter.
int ss_prog_set_seed(ss_prog *p, int64_t seed) {
    P_LIVE(p);
    if (!p) P_FAIL(p, SS_ERR_INVALID, "NULL program");
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    p->seed = (int32_t)(uint32_t)(uint64_t)seed;
    int rc = push_args(p);
    if (rc) return rc;
    return push_seed(p);
}

int ss_prog_set_extra(ss_prog *p, int32_t slot, int64_t bytes, const void *data) {
    P_LIVE(p);
    if (!p || slot < 0 || slot >= SS_MAXX_HOST || bytes < 0 || (bytes && !data))
        P_FAIL(p, SS_ERR_INVALID, "bad extra slot, size or NULL data");
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    Extra &x = p->extras[slot];
    if (x.bytes != bytes || !x.d) {
        pfree(x.d);
        x.d = nullptr;
        x.bytes = 0;
        P_HIP(p, ss_device_alloc(p->ctx, &x.d, (size_t)std::max<int64_t>(bytes, 16)));
        x.bytes = bytes;
    }
    P_HIP(p, ss_copy_in(p->ctx, x.d, data, (size_t)bytes));
    return push_args(p);
}

int ss_prog_get_extra(ss_prog *p, int32_t slot, int64_t bytes, void *out) {
    P_LIVE(p);
    if (!p || slot < 0 || slot >= SS_MAXX_HOST || (bytes && !out)) P_FAIL(p, SS_ERR_INVALID, "bad extra slot or NULL");
    const Extra &x = p->extras[slot];
    if (!x.d || bytes != x.bytes) P_FAIL(p, SS_ERR_INVALID, "extra slot %d holds %lld bytes", slot, (long long)x.bytes);
    P_HIP(p, ss_copy_out(p->ctx, out, x.d, (size_t)bytes));
    return SS_OK;
}

int ss_prog_set_unroll(ss_prog *p, int32_t count) {
    if (!p || count < 1 || count > 128) P_FAIL(p, SS_ERR_INVALID, "unroll count must be 1..128");
    P_LIVE(p);
    p->unroll = count;
    return SS_OK;
}

int ss_prog_compile(ss_prog *p, const char *source, const char *kernel_names, char *log, int64_t log_cap) {
    P_LIVE(p);
    if (!p || !source || !kernel_names) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    if (log && log_cap > 0) log[0] = 0;
    const std::vector<std::string> opts_s = rtc_options(p->unroll);
    std::vector<const char *> opts;
    for (const auto &o : opts_s) opts.push_back(o.c_str());
    uint64_t key = 1469598103934665603ull;
    for (const auto &o : opts_s) key = fnv1a(key, o.c_str(), o.size() + 1);
    key = fnv1a(key, kStepRtHeader, std::strlen(kStepRtHeader));
    key = fnv1a(key, source, std::strlen(source));
    char key_hex[32];
    std::snprintf(key_hex, sizeof key_hex, "%016llx.co", (unsigned long long)key);
    std::vector<char> code;
    p->cache_hit = 0;
    {
        std::lock_guard<std::mutex> lk(g_cache_mu);
        auto it = g_code_cache.find(key);
        if (it != g_code_cache.end()) {
            code = it->second;
            p->cache_hit = 1;
        }
    }
    const std::string dir = disk_cache_dir();
    if (code.empty() && !dir.empty() && read_file(dir + "/" + key_hex, code)) p->cache_hit = 2;
    if (code.empty()) {
        hiprtcProgram prog;
        const char *hdrs[] = {kStepRtHeader};
        const char *names[] = {"sagesim_rt.h"};
        if (hiprtcCreateProgram(&prog, source, "step_functions.hip", 1, hdrs, names) != HIPRTC_SUCCESS)
            P_FAIL(p, SS_ERR_RTC, "hiprtcCreateProgram failed");
        // packed-FP32 instructions stay out of the generated code object
        hiprtcResult rc = hiprtcCompileProgram(prog, (int)opts.size(), opts.data());
        size_t ls = 0;
        hiprtcGetProgramLogSize(prog, &ls);
        std::string lg(ls, '\0');
        if (ls) hiprtcGetProgramLog(prog, &lg[0]);
        if (log && log_cap > 0) {
            std::strncpy(log, lg.c_str(), (size_t)log_cap - 1);
            log[log_cap - 1] = 0;
        }
        if (rc != HIPRTC_SUCCESS) {
            hiprtcDestroyProgram(&prog);
            P_FAIL(p, SS_ERR_RTC, "hipRTC compile failed: %s", lg.substr(0, 900).c_str());
        }
        size_t cs = 0;
        hiprtcGetCodeSize(prog, &cs);
        code.resize(cs);
        hiprtcGetCode(prog, code.data());
        hiprtcDestroyProgram(&prog);
        if (!dir.empty()) write_file_atomic(dir, key_hex, code);
    }
    {
        std::lock_guard<std::mutex> lk(g_cache_mu);
        g_code_cache.emplace(key, code);
    }
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    if (p->module) {
        (void)hipModuleUnload(p->module);
        p->module = nullptr;
    }
    p->kernels.clear();
    p->loop_kernel = -1;
    P_HIP(p, hipModuleLoadData(&p->module, code.data()));
    std::string names_s(kernel_names);
    size_t pos = 0;
    while (pos <= names_s.size()) {
        size_t nl = names_s.find('\n', pos);
        std::string nm = names_s.substr(pos, nl == std::string::npos ? std::string::npos : nl - pos);
        if (!nm.empty()) {
            hipFunction_t f = nullptr;
            hipError_t e = hipModuleGetFunction(&f, p->module, nm.c_str());
            if (e != hipSuccess) P_FAIL(p, SS_ERR_RTC, "kernel %s not in the compiled module", nm.c_str());
            p->kernels.push_back(f);
        }
        if (nl == std::string::npos) break;
        pos = nl + 1;
    }
    int rc = push_csr_globals(p);
    if (rc) return rc;
    return push_seed(p);
}

int ss_prog_cache_hit(ss_prog *p, int32_t *hit) {
    P_LIVE(p);
    if (!p || !hit) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    *hit = p->cache_hit;
    return SS_OK;
}

int ss_prog_set_schedule(ss_prog *p, int32_t n, const int32_t *kernel, const int64_t *start, const int64_t *count) {
    P_LIVE(p);
    if (!p || n < 0 || (n && (!kernel || !start || !count))) P_FAIL(p, SS_ERR_INVALID, "bad schedule");
    std::vector<Launch> s;
    for (int32_t i = 0; i < n; ++i) {
        if (kernel[i] < 0 || kernel[i] >= (int32_t)p->kernels.size())
            P_FAIL(p, SS_ERR_RANGE, "launch %d names kernel %d of %zu", i, kernel[i], p->kernels.size());
        if (start[i] < 0 || count[i] < 0 || start[i] + count[i] > p->n)
            P_FAIL(p, SS_ERR_RANGE, "launch %d covers agents outside [0, %lld)", i, (long long)p->n);
        s.push_back({kernel[i], start[i], count[i], -1});
    }
    p->schedule = s;
    p->loop_kernel = -1;                        // it runs the schedule it was compiled for
    pfree(p->order);
    p->order = nullptr;
    p->order_n = 0;
    return SS_OK;
}

int ss_prog_set_order(ss_prog *p, const int32_t *order, int64_t n) {
    P_LIVE(p);
    if (!p || n < 0 || (n && !order)) P_FAIL(p, SS_ERR_INVALID, "bad order");
    int64_t need = 0;
    for (const Launch &l : p->schedule) need += l.count;
    if (n != need) P_FAIL(p, SS_ERR_INVALID, "order has %lld entries, the schedule covers %lld", (long long)n,
                          (long long)need);
    // each launch's segment is a permutation of its range
    int64_t off = 0;
    std::vector<char> seen;
    for (Launch &l : p->schedule) {
        seen.assign((size_t)l.count, 0);
        for (int64_t k = 0; k < l.count; ++k) {
            const int64_t a = (int64_t)order[off + k] - l.start;
            if (a < 0 || a >= l.count || seen[(size_t)a])
                P_FAIL(p, SS_ERR_RANGE, "order of a launch is not a permutation of its agents");
            seen[(size_t)a] = 1;
        }
        l.order_off = off;
        l.n_long = l.long_deg = 0;
        off += l.count;
    }
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    pfree(p->order);
    p->order = nullptr;
    P_HIP(p, ss_device_alloc(p->ctx, (void **)&p->order, sizeof(int32_t) * (size_t)std::max<int64_t>(n, 1)));
    if (n) P_HIP(p, hipMemcpy(p->order, order, sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice));
    p->order_n = n;
    p->h_order.assign(order, order + n);
    return SS_OK;
}

int ss_prog_set_long(ss_prog *p, const int64_t *n_long, int32_t n_launches) {
    P_LIVE(p);
    if (!p || !n_long) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    if (n_launches != (int32_t)p->schedule.size())
        P_FAIL(p, SS_ERR_INVALID, "%d launches, the schedule has %zu", n_launches, p->schedule.size());
    if (p->h_row_ptr.empty()) P_FAIL(p, SS_ERR_STATE, "no CSR");
    std::vector<int64_t> deg(p->schedule.size(), 0);
    for (size_t q = 0; q < p->schedule.size(); ++q) {
        const Launch &l = p->schedule[q];
        if (n_long[q] < 0 || n_long[q] > l.count || (n_long[q] > 0 && (l.order_off < 0 || !p->order)))
            P_FAIL(p, SS_ERR_INVALID, "launch %zu: %lld long rows of %lld agents, or no order", q,
                   (long long)n_long[q], (long long)l.count);
        for (int64_t k = 0; k < n_long[q]; ++k) {
            const int32_t i = p->h_order[(size_t)(l.order_off + k)];
            deg[q] = std::max(deg[q], p->h_row_ptr[i + 1] - p->h_row_ptr[i]);
        }
        if (deg[q] * 4 > 65536) P_FAIL(p, SS_ERR_INVALID, "launch %zu: a row of %lld entries exceeds 64 KB of LDS", q,
                                       (long long)deg[q]);
    }
    for (size_t q = 0; q < p->schedule.size(); ++q) {
        p->schedule[q].n_long = n_long[q];
        p->schedule[q].long_deg = deg[q];
    }
    return SS_OK;
}

int ss_prog_set_loop(ss_prog *p, int32_t kernel, int32_t threads) {
    if (!p) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    P_LIVE(p);
    if (kernel < -1 || kernel >= (int32_t)p->kernels.size() || threads < 64 || threads > 1024 || threads % 64)
        P_FAIL(p, SS_ERR_INVALID, "kernel %d of %zu with %d threads", kernel, p->kernels.size(), threads);
    p->loop_kernel = kernel;
    p->loop_threads = threads;
    p->trial = LoopTrial();
    return SS_OK;
}

int ss_prog_loop(ss_prog *p, int32_t *kernel) {
    if (!p || !kernel) P_FAIL(p, SS_ERR_INVALID, "NULL argument");
    P_LIVE(p);
    *kernel = p->loop_kernel;
    return SS_OK;
}

// Every tick: the launches of the schedule in order (a kernel boundary
// between priority groups is the grid barrier of model.py:2356-2366), then the
// copy of every double-buffered array's write buffer into its read buffer
// (model.py:2378-2406).  Waits.
static int run_schedule(ss_prog *p, int64_t tick0, int64_t ticks) {
    hipStream_t st = p->ctx->stream;
    for (int64_t k = 0; k < ticks; ++k) {
        long long tick = (long long)(tick0 + k);
        for (const Launch &l : p->schedule) {
            if (l.count == 0) continue;
            const ProgArgsHost *a = p->d_args;
            long long start = l.start, count = l.count;
            const int32_t *ord = l.order_off >= 0 && p->order ? p->order + l.order_off : nullptr;
            long long n_long = l.n_long;
            void *args[] = {(void *)&a, (void *)&tick, (void *)&start, (void *)&count, (void *)&ord, (void *)&n_long};
            const unsigned grid = (unsigned)(n_long + (count - n_long + 255) / 256);
            P_HIP(p, hipModuleLaunchKernel(p->kernels[l.kernel], grid, 1, 1, 256, 1, 1, (unsigned)(4 * l.long_deg), st,
                                           args, nullptr));
        }
        int rc = write_back(p, st);
        if (rc) return rc;
    }
    P_HIP(p, hipStreamSynchronize(st));
    return SS_OK;
}

// The same ticks by the one-block kernel.  Waits.
static int run_loop(ss_prog *p, int64_t tick0, int64_t ticks) {
    const ProgArgsHost *a = p->d_args;
    long long tick = (long long)tick0, n_ticks = (long long)ticks;
    void *args[] = {(void *)&a, (void *)&tick, (void *)&n_ticks};
    P_HIP(p, hipModuleLaunchKernel(p->kernels[p->loop_kernel], 1, 1, 1, (unsigned)p->loop_threads, 1, 1, 0,
                                   p->ctx->stream, args, nullptr));
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    return SS_OK;
}

int ss_prog_simulate(ss_prog *p, int64_t tick0, int64_t ticks) {
    P_LIVE(p);
    if (!p || ticks < 0) P_FAIL(p, SS_ERR_INVALID, "bad arguments");
    if (!p->module) P_FAIL(p, SS_ERR_STATE, "no compiled step functions");
    if (p->loop_kernel < 0 || ticks == 0) return run_schedule(p, tick0, ticks);
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));     // what is queued is not the step's time
    LoopTrial &t = p->trial;
    for (int64_t k = 0; k < ticks;) {
        if (p->loop_kernel < 0) return run_schedule(p, tick0 + k, ticks - k);
        const bool loop = t.samples < 2;
        const int64_t n = std::min(ticks - k, t.samples ? std::min<int64_t>(t.chunk, 16) : t.chunk);
        const auto from = std::chrono::steady_clock::now();
        const int rc = loop ? run_loop(p, tick0 + k, n) : run_schedule(p, tick0 + k, n);
        if (rc) return rc;
        const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - from).count();
        k += n;
        t.add(us, n, p->schedule.size() + 1);
        if (t.schedule_wins()) p->loop_kernel = -1;
    }
    return SS_OK;
}

// ---- checkpoint: replaces the pickle of Model.save / Model.load
// (model.py:1289-1310) with the program's device state, bit for bit ----
// layout: magic, version, n, nnz, csr_hash, tick, seed, n_globals, n_arrays,
// globals, then per array (elem_bytes, rows, width, double_buffered) and its
// read buffer (the write buffer equals it between ticks)
static const uint64_t kProgMagic = 0x53534147455052ull;   // "SSAGEPR"

int ss_prog_save(ss_prog *p, int64_t tick, void *buf, int64_t cap, int64_t *size) {
    P_LIVE(p);
    if (!p || !size || cap < 0 || (cap && !buf)) P_FAIL(p, SS_ERR_INVALID, "bad arguments");
    int64_t need = 9 * 8 + 8 * p->n_globals;
    for (const ProgProp &q : p->props) need += 4 * 8 + (int64_t)((q.bytes() + 7) / 8 * 8);
    *size = need;
    if (!buf) return SS_OK;
    if (cap < need) P_FAIL(p, SS_ERR_INVALID, "buffer of %lld bytes, checkpoint needs %lld", (long long)cap,
                           (long long)need);
    P_HIP(p, hipStreamSynchronize(p->ctx->stream));
    std::memset(buf, 0, (size_t)need);
    int64_t *h = static_cast<int64_t *>(buf);
    h[0] = (int64_t)kProgMagic; h[1] = 1; h[2] = p->n; h[3] = p->nnz; h[4] = (int64_t)p->csr_hash;
    h[5] = tick; h[6] = p->seed; h[7] = p->n_globals; h[8] = (int64_t)p->props.size();
    char *c = static_cast<char *>(buf) + 9 * 8;
    if (p->n_globals) std::memcpy(c, p->h_globals.data(), 8 * (size_t)p->n_globals);
    c += 8 * p->n_globals;
    for (const ProgProp &q : p->props) {
        int64_t d[4] = {q.elem_bytes, q.rows, q.width, q.double_buffered ? 1 : 0};
        std::memcpy(c, d, sizeof d);
        c += sizeof d;
        if (q.bytes()) P_HIP(p, hipMemcpy(c, q.r, q.bytes(), hipMemcpyDeviceToHost));
        c += (q.bytes() + 7) / 8 * 8;
    }
    return SS_OK;
}

int ss_prog_restore(ss_prog *p, const void *buf, int64_t size, int64_t *tick) {
    P_LIVE(p);
    if (!p || !buf || size < 9 * 8) P_FAIL(p, SS_ERR_INVALID, "bad arguments");
    const int64_t *h = static_cast<const int64_t *>(buf);
    if (h[0] != (int64_t)kProgMagic || h[1] != 1) P_FAIL(p, SS_ERR_INVALID, "not a program checkpoint");
    if (h[2] != p->n || h[3] != p->nnz || h[4] != (int64_t)p->csr_hash)
        P_FAIL(p, SS_ERR_INVALID, "checkpoint of another network (agents, entries or CSR differ)");
    if (h[7] != p->n_globals || h[8] != (int64_t)p->props.size())
        P_FAIL(p, SS_ERR_INVALID, "checkpoint has %lld globals and %lld arrays, the program %lld and %zu",
               (long long)h[7], (long long)h[8], (long long)p->n_globals, p->props.size());
    int64_t need = 9 * 8 + 8 * p->n_globals;
    for (const ProgProp &q : p->props) need += 4 * 8 + (int64_t)((q.bytes() + 7) / 8 * 8);
    if (size != need) P_FAIL(p, SS_ERR_INVALID, "checkpoint has %lld bytes, expected %lld", (long long)size,
                             (long long)need);
    const char *c = static_cast<const char *>(buf) + 9 * 8 + 8 * p->n_globals;
    for (const ProgProp &q : p->props) {
        int64_t d[4];
        std::memcpy(d, c, sizeof d);
        if (d[0] != q.elem_bytes || d[1] != q.rows || d[2] != q.width || d[3] != (q.double_buffered ? 1 : 0))
            P_FAIL(p, SS_ERR_INVALID, "checkpoint arrays differ in shape or buffering");
        c += sizeof d + (q.bytes() + 7) / 8 * 8;
    }
    int rc = ss_prog_set_globals(p, reinterpret_cast<const double *>(static_cast<const char *>(buf) + 9 * 8), h[7]);
    if (rc) return rc;
    if ((rc = ss_prog_set_seed(p, h[6]))) return rc;
    c = static_cast<const char *>(buf) + 9 * 8 + 8 * p->n_globals;
    for (size_t i = 0; i < p->props.size(); ++i) {
        c += 4 * 8;
        if (p->props[i].bytes() && (rc = ss_prog_prop_upload(p, (int32_t)i, c))) return rc;
        c += (p->props[i].bytes() + 7) / 8 * 8;
    }
    if (tick) *tick = h[5];
    return SS_OK;
}

}  // extern "C"
