// Copies between the caller's ordinary memory and the device, through
// page-locked memory of the context.  A hipMemcpy of ordinary memory stages it
// itself, on one thread: 26 MB go up at 29 GB/s and down at 17, into pages that
// were never touched at 9 (the page faults are on that thread), and 100 KB to
// 1 MB take 0.05 to 0.45 ms.  The bus carries 57 GB/s.  Here a copy goes in
// chunks that overlap with their transfers, and one of several chunks on up to
// SS_STAGE_LANES threads, each with two chunks of its own.  The compute units
// move the chunks: the copy engine takes 4 to 10 us longer for each (10 MB down
// 405 us by it, 320 us so).  Readback of n states, hipMemcpy before and so now:
// 100k 52 and 18 us, 1M 73 to 450 and 66, 10M 615 and 320, 27M 1600 and 690; up,
// with the bitmaps made anew: 100k 150 and 53, 1M 162 and 103, 10M 713 and 450.
#include <hip/hip_runtime.h>
#include <sched.h>
#include <stdint.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "ss_runtime.h"

namespace {

const size_t kChunk = 1u << 20;
const size_t kManyFrom = 4u << 20;         // below this, waking threads costs what they save
// From here on a copy up goes over two streams: a chunk's kernel reads at 38 GB/s
// (27 us) and the next one starts 6 us after it, where two kernels at a time fill
// the gap.  Uploads of 112 and 32 MB for a ghost discovery 6.79 and 6.37 ms, a
// replica of 10M agents and 50M entries 12.2 and 11.1, 26 MB of history down 0.61
// and 0.57; handing over to the second stream and back costs some 20 us, which
// 4 to 16 MB do not win back.  (No gain: six or eight lanes, stores past the
// host's caches.)
const size_t kForkFrom = 16u << 20;

struct Job {
    char *host;
    size_t bytes;
    bool in;                               // host to device
    const ss_stage_issue *issue;
    hipStream_t on[2];                     // the streams of the lanes' slots
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};
};

struct Lane {
    char *mem[2] = {};                     // two chunks, page-locked
    hipEvent_t ev[2] = {};                 // the transfer of chunk s is done
    bool flying[2] = {};                   // ... and may not be yet
};

// A chunk is allocated by the lane that first needs it, and each by itself: 1 MB
// of page-locked memory takes 45 us, 2 MB and more 320 us.
bool open_slot(Lane &l, int s) {
    if (l.mem[s]) return true;
    if ((l.ev[s] || hipEventCreateWithFlags(&l.ev[s], hipEventDisableTiming) == hipSuccess) &&
        hipHostMalloc((void **)&l.mem[s], kChunk, hipHostMallocDefault) == hipSuccess)
        return true;
    l.mem[s] = nullptr;
    (void)hipGetLastError();
    return false;
}

// chunks of the job, claimed one by one, until none is left (or this lane has no
// memory for more)
void run_lane(Lane &l, Job &j) {
    const size_t n = (j.bytes + kChunk - 1) / kChunk;
    auto len = [&](size_t c) { return std::min(kChunk, j.bytes - c * kChunk); };
    auto stop = [&](hipError_t e) {
        int none = hipSuccess;
        j.err.compare_exchange_strong(none, (int)e);
        j.next = n;
    };
    size_t pending = n;                    // down: the chunk on its way into the other slot
    for (int s = 0;; s ^= 1) {
        const size_t c = j.next.load() < n && open_slot(l, s) ? j.next.fetch_add(1) : n;
        char *slot = l.mem[s];
        hipError_t e = hipSuccess;
        if (c < n) {
            if (j.in) {
                if (l.flying[s]) e = hipEventSynchronize(l.ev[s]);
                if (e == hipSuccess) std::memcpy(slot, j.host + c * kChunk, len(c));
            }
            if (e == hipSuccess) e = (*j.issue)(c * kChunk, len(c), slot, j.on[s]);
            if (e == hipSuccess) e = hipEventRecord(l.ev[s], j.on[s]);
            if (e == hipSuccess) l.flying[s] = true;
        }
        if (e == hipSuccess && !j.in && pending < n) {
            e = hipEventSynchronize(l.ev[s ^ 1]);
            l.flying[s ^ 1] = false;
            if (e == hipSuccess) std::memcpy(j.host + pending * kChunk, l.mem[s ^ 1], len(pending));
        }
        if (e != hipSuccess) return stop(e);
        if (c >= n) return;
        pending = c;
    }
}

}  // namespace

struct ss_stager {
    int device;
    hipStream_t stream, second;
    hipEvent_t fork = nullptr, join = nullptr;
    pid_t pid;                             // threads do not survive a fork
    Lane lane[SS_STAGE_LANES];
    std::thread thread[SS_STAGE_LANES];
    int helpers = 0;                       // threads started, for lanes 1 .. helpers
    std::mutex m;
    std::condition_variable go, done;
    Job *job = nullptr;
    uint64_t turn = 0;
    int busy = 0;
    bool quit = false;

    void help(int i) {
        (void)hipSetDevice(device);
        uint64_t seen = 0;
        std::unique_lock<std::mutex> g(m);
        for (;;) {
            go.wait(g, [&] { return quit || (job && turn != seen); });
            if (quit) return;
            seen = turn;
            Job &j = *job;
            ++busy;
            g.unlock();
            run_lane(lane[i], j);
            g.lock();
            if (--busy == 0) done.notify_all();
        }
    }

    // as many threads as there are lanes and processors to run them on
    void hire() {
        cpu_set_t set;
        CPU_ZERO(&set);
        int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
        while (helpers + 1 < std::min(cpus, (int)SS_STAGE_LANES)) {
            const int i = helpers + 1;
            try {
                thread[i] = std::thread([this, i] { help(i); });
            } catch (...) {
                return;                    // goes on with those it has
            }
            helpers = i;
        }
    }

    hipError_t fork_second() {
        hipError_t e = hipSuccess;
        for (hipEvent_t *ev : {&fork, &join})
            if (!*ev && (e = hipEventCreateWithFlags(ev, hipEventDisableTiming)) != hipSuccess) return e;
        if ((e = hipEventRecord(fork, stream)) != hipSuccess) return e;
        return hipStreamWaitEvent(second, fork, 0);
    }
    hipError_t join_second() {
        hipError_t e = hipSuccess;
        if (!join && (e = hipEventCreateWithFlags(&join, hipEventDisableTiming)) != hipSuccess) return e;
        if ((e = hipEventRecord(join, second)) != hipSuccess) return e;
        return hipStreamWaitEvent(stream, join, 0);
    }

    hipError_t run(Job &j) {
        hipError_t e = hipSuccess;
        const bool many = j.bytes >= kManyFrom && getpid() == pid;
        j.on[0] = j.on[1] = stream;
        if (many) {
            hire();
            // what is queued before the copies would hold every lane
            if (!j.in && (e = hipStreamSynchronize(stream)) != hipSuccess) return e;
            // every other chunk goes over the second stream, up after what is
            // queued on the first and before what will be
            if (j.in && j.bytes >= kForkFrom && (e = fork_second()) != hipSuccess) return e;
            if (!j.in || j.bytes >= kForkFrom) j.on[1] = second;
            std::lock_guard<std::mutex> g(m);
            job = &j;
            ++turn;
            go.notify_all();
        }
        run_lane(lane[0], j);
        if (many) {
            std::unique_lock<std::mutex> g(m);
            job = nullptr;                 // a thread that is not awake yet finds nothing to do
            done.wait(g, [&] { return busy == 0; });
        }
        e = (hipError_t)j.err.load();
        // (a copy down has been waited for on both streams, unless it failed)
        if (j.on[1] == second && (j.in || e != hipSuccess)) {
            const hipError_t e2 = join_second();
            if (e == hipSuccess) e = e2;
        }
        const bool all = j.next.load() * kChunk >= j.bytes;
        return e == hipSuccess && !all ? hipErrorOutOfMemory : e;
    }

    ~ss_stager() {
        const bool mine = getpid() == pid;
        if (mine) {
            std::lock_guard<std::mutex> g(m);
            quit = true;
            go.notify_all();
        }
        for (auto &t : thread)
            if (t.joinable()) {
                if (mine) t.join();
                else t.detach();
            }
        for (auto &l : lane) {
            for (auto &m : l.mem)
                if (m) (void)hipHostFree(m);
            for (auto &ev : l.ev)
                if (ev) (void)hipEventDestroy(ev);
        }
        if (fork) (void)hipEventDestroy(fork);
        if (join) (void)hipEventDestroy(join);
    }
};

void ss_stager_close(ss_ctx *ctx) {
    delete ctx->stager;
    ctx->stager = nullptr;
}

static hipError_t stager(ss_ctx *ctx) {
    if (ctx->stager) return hipSuccess;
    auto *s = new (std::nothrow) ss_stager();
    if (!s) return hipErrorOutOfMemory;
    s->device = ctx->device;
    s->stream = ctx->stream;
    s->second = ctx->copy_stream;
    s->pid = getpid();
    ctx->stager = s;
    return hipSuccess;
}

bool ss_known_to_hip(const void *p) {
    hipPointerAttribute_t at;
    const hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) (void)hipGetLastError();       // ordinary memory: not an error here
    return e == hipSuccess && at.type != hipMemoryTypeUnregistered;
}

hipError_t ss_stage_out(ss_ctx *ctx, void *host, size_t bytes, const ss_stage_issue &issue) {
    if (!bytes) return hipSuccess;
    const hipError_t e = stager(ctx);
    if (e != hipSuccess) return e;
    Job j;
    j.host = (char *)host;
    j.bytes = bytes;
    j.in = false;
    j.issue = &issue;
    return ctx->stager->run(j);
}

hipError_t ss_copy_out(ss_ctx *ctx, void *host, const void *dev, size_t bytes) {
    if (!bytes) return hipSuccess;
    if (ss_known_to_hip(host)) {
        const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream);
        return e == hipSuccess ? hipStreamSynchronize(ctx->stream) : e;
    }
    return ss_stage_out(ctx, host, bytes, [&](size_t at, size_t len, void *slot, hipStream_t st) {
        return ss_launch_stage((const char *)dev + at, slot, (int64_t)len, nullptr, nullptr, 0, st);
    });
}

hipError_t ss_copy_in(ss_ctx *ctx, void *dev, const void *host, size_t bytes) {
    if (!bytes) return hipSuccess;
    if (ss_known_to_hip(host)) {
        const hipError_t e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream);
        return e == hipSuccess ? hipStreamSynchronize(ctx->stream) : e;
    }
    const hipError_t e = stager(ctx);
    if (e != hipSuccess) return e;
    const ss_stage_issue issue = [&](size_t at, size_t len, void *slot, hipStream_t st) {
        return ss_launch_stage(slot, (char *)dev + at, (int64_t)len, nullptr, nullptr, 0, st);
    };
    Job j;
    j.host = (char *)const_cast<void *>(host);
    j.bytes = bytes;
    j.in = true;
    j.issue = &issue;
    return ctx->stager->run(j);
}
