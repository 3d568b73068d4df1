// transfer.hip — copies between the caller's (pageable) memory and the device.
//
// The runtime copies pageable memory through a pinned buffer of its own on one host thread: 28 GB/s
// up and 18 GB/s down on a link that carries 57 GB/s of pinned memory either way. Large copies go
// through a ring of pinned slots here instead: a few threads copy between the caller's memory and
// their own two slots each, so host copies (and the page faults of freshly allocated results) of
// one slot run beside the transfers of the others. 537 MB of records (256^3 particles): up 19 -> 11
// ms, up and down again 51 -> 22.5 ms.
#include <atomic>
#include <cstring>
#include <exception>
#include <new>
#include <thread>

#include "lagpm_internal.h"

namespace {

constexpr int MAX_WORKERS = 4;  // eight gave the same
constexpr int SLOTS = 2 * MAX_WORKERS;
// A transfer costs some 10 us beside its bytes, so slots are large (537 MB up: 17.2 ms in 1 MB slots,
// 13.4 in 2 MB, 11.8 in 4 MB, 11.0 in 8 MB), and smaller only as far as a copy needs for its workers.
constexpr size_t SLOT_BYTES = (size_t)8 << 20;
constexpr size_t SLOT_MIN = (size_t)2 << 20;
// below this the runtime's own path is as fast (a thread takes some 30 us to start)
constexpr size_t STAGED_MIN = (size_t)2 << 20;

struct chunk {
    char *dev, *host;
    size_t bytes;
};

int direct_copy(lagpm_ctx* ctx, const lagpm_segment* seg, size_t nseg, bool to_host, hipStream_t st) {
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < nseg && e == hipSuccess; k++) {
        if (!seg[k].bytes) continue;
        e = to_host ? hipMemcpyAsync(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost, st)
                    : hipMemcpyAsync(seg[k].dev, seg[k].host, seg[k].bytes, hipMemcpyHostToDevice, st);
    }
    // the stream is waited for even when queuing failed: no copy may still write to the host later
    const hipError_t w = to_host ? hipStreamSynchronize(st) : hipSuccess;
    if (e != hipSuccess) return lagpm_fail(ctx, LAGPM_E_HIP, std::string("host copy: ") + hipGetErrorString(e));
    if (w != hipSuccess) return lagpm_fail(ctx, LAGPM_E_HIP, std::string("host copy (wait): ") + hipGetErrorString(w));
    return LAGPM_OK;
}

}  // namespace

struct lagpm_stager {
    char* buf = nullptr;
    hipEvent_t ev[SLOTS] = {};
    bool busy[SLOTS] = {};  // a transfer from or to the slot may still be under way
    std::mutex mu;

    ~lagpm_stager() {
        for (int i = 0; i < SLOTS; i++)
            if (ev[i]) {
                if (busy[i]) (void)hipEventSynchronize(ev[i]);
                (void)hipEventDestroy(ev[i]);
            }
        if (buf) (void)hipHostFree(buf);
    }
    bool ready() {
        if (buf) return true;
        for (int i = 0; i < SLOTS; i++)
            if (!ev[i] && hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) != hipSuccess) return false;
        return hipHostMalloc((void**)&buf, SLOTS * SLOT_BYTES, hipHostMallocDefault) == hipSuccess;
    }
    hipError_t wait(int slot) {
        if (!busy[slot]) return hipSuccess;
        const hipError_t e = hipEventSynchronize(ev[slot]);
        busy[slot] = false;
        return e;
    }

    // Worker w takes chunks until none are left or one failed. Upwards: fill a slot, queue its
    // transfer, go on with the other slot. Downwards: queue the next chunk's transfer before
    // emptying the slot of the last one.
    void work(int w, int device, const std::vector<chunk>& chunks, std::atomic<size_t>& next, std::atomic<int>& err, bool to_host,
              hipStream_t st) {
        hipError_t e = hipSetDevice(device);
        int k = 0;
        const chunk* held = nullptr;  // downwards: the chunk whose transfer to the other slot is under way
        while (e == hipSuccess && err.load(std::memory_order_relaxed) == 0) {
            const size_t c = next.fetch_add(1, std::memory_order_relaxed);
            const bool have = c < chunks.size();
            if (!have && !held) break;
            const int slot = 2 * w + k, other = 2 * w + 1 - k;
            if (have) {
                const chunk& q = chunks[c];
                char* s = buf + (size_t)slot * SLOT_BYTES;
                e = wait(slot);
                if (e != hipSuccess) break;
                if (!to_host) std::memcpy(s, q.host, q.bytes);
                e = to_host ? hipMemcpyAsync(s, q.dev, q.bytes, hipMemcpyDeviceToHost, st)
                            : hipMemcpyAsync(q.dev, s, q.bytes, hipMemcpyHostToDevice, st);
                if (e == hipSuccess) e = hipEventRecord(ev[slot], st);
                busy[slot] = true;
            }
            if (to_host) {
                if (held && e == hipSuccess) {
                    e = wait(other);
                    if (e == hipSuccess) std::memcpy(held->host, buf + (size_t)other * SLOT_BYTES, held->bytes);
                }
                held = have ? &chunks[c] : nullptr;
            }
            k ^= 1;
        }
        if (e != hipSuccess) err.store((int)e);
    }
};

int lagpm_copy_segments(lagpm_ctx* ctx, const lagpm_segment* seg, size_t nseg, bool to_host, hipStream_t st) {
    size_t total = 0;
    for (size_t k = 0; k < nseg; k++) total += seg[k].bytes;
    if (total < STAGED_MIN) return direct_copy(ctx, seg, nseg, to_host, st);
    if (!ctx->stager) return direct_copy(ctx, seg, nseg, to_host, st);
    try {
        lagpm_stager& S = *ctx->stager;
        std::lock_guard<std::mutex> lk(S.mu);
        if (!S.ready()) {  // no pinned memory to be had: the runtime's own path
            (void)hipGetLastError();
            return direct_copy(ctx, seg, nseg, to_host, st);
        }
        const size_t step = std::min(SLOT_BYTES, std::max(SLOT_MIN, (total / SLOTS + 4095) / 4096 * 4096));
        std::vector<chunk> chunks;
        for (size_t k = 0; k < nseg; k++)
            for (size_t o = 0; o < seg[k].bytes; o += step)
                chunks.push_back({(char*)seg[k].dev + o, (char*)seg[k].host + o, std::min(step, seg[k].bytes - o)});
        std::atomic<size_t> next{0};
        std::atomic<int> err{0};
        std::thread others[MAX_WORKERS];
        const int workers = (int)std::min<size_t>(MAX_WORKERS, (chunks.size() + 1) / 2);
        for (int w = 1; w < workers; w++) {
            try {
                others[w] = std::thread([&, w] { S.work(w, ctx->device, chunks, next, err, to_host, st); });
            } catch (const std::exception&) {  // no thread or no memory for one: the others take its chunks
                break;
            }
        }
        S.work(0, ctx->device, chunks, next, err, to_host, st);
        for (std::thread& t : others)
            if (t.joinable()) t.join();
        if (err.load())
            return lagpm_fail(ctx, LAGPM_E_HIP, std::string("staged host copy: ") + hipGetErrorString((hipError_t)err.load()));
        return LAGPM_OK;
    } catch (const std::bad_alloc&) {
        return lagpm_fail(ctx, LAGPM_E_NOMEM, "host memory for a staged copy");
    }
}

int lagpm_d2h(lagpm_ctx* ctx, void* dst, const void* src, size_t bytes, hipStream_t s) {
    const lagpm_segment g{const_cast<void*>(src), dst, bytes};
    return lagpm_copy_segments(ctx, &g, 1, true, s);
}
int lagpm_h2d(lagpm_ctx* ctx, void* dst, const void* src, size_t bytes, hipStream_t s) {
    const lagpm_segment g{dst, const_cast<void*>(src), bytes};
    return lagpm_copy_segments(ctx, &g, 1, false, s);
}

// With the context, so that threads whose first copies come at once find the same one (and its lock); the
// slots are pinned by the first large copy.
void lagpm_stager_create(lagpm_ctx* ctx) { ctx->stager = new (std::nothrow) lagpm_stager; }
void lagpm_stager_release(lagpm_ctx* ctx) {
    delete ctx->stager;
    ctx->stager = nullptr;
}
