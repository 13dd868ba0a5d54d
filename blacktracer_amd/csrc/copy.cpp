// copy.cpp -- large copies between a caller's pageable host memory and the
// device.
//
// The runtime moves pageable memory through a staging buffer of its own, one
// thread copying a megabyte at a time: 11 GB/s, and half of that where the
// destination is fresh memory whose pages are first touched (and cleared) by
// that thread.  Exporting a level-10 grid (44 MB) took 5.5 ms that way, more
// than its build.  Here several threads share the pieces of a copy, each with
// two pinned pieces in flight, so that the link (53 GB/s) and the page faults
// of several threads overlap.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

#include "bt_internal.h"

namespace bt {
namespace {

// Copies from kCopyLarge on take this path: below it the threads' start
// (about 100 us) is not won back.  One thread for every kCopyPerThread bytes,
// up to the number from which they wait for each other in the runtime's calls:
// building and exporting a level-10 grid took 9.7 ms with the runtime's
// copies, and 6.6, 6.4 and 6.3 ms with eight threads on pieces of 1 MiB, four
// and six on pieces of 2 MiB.
constexpr size_t kCopyLarge = size_t(4) << 20;
constexpr size_t kCopyPerThread = size_t(2) << 20;
constexpr int kCopyThreads = 6;
constexpr size_t kPiece = size_t(2) << 20;
static_assert(2 * kCopyThreads == Context::kCopySlots, "two pieces per thread");

bool is_pinned(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // plain host memory is unknown to the runtime
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

struct Piece {
    char* dst;
    const char* src;
    size_t bytes;
};

}  // namespace

// The pinned pieces and their events; false where the runtime has none to give.
bool Context::copy_slots() {
    for (int k = 0; k < kCopySlots; k++)
        if (!ev_copy[k] && hipEventCreateWithFlags(&ev_copy[k], hipEventDisableTiming) != hipSuccess) {
            ev_copy[k] = nullptr;
            (void)hipGetLastError();
            return false;
        }
    if (!copy_stage && hipHostMalloc(&copy_stage, kCopySlots * kPiece, 0) != hipSuccess) {
        copy_stage = nullptr;
        (void)hipGetLastError();
        return false;
    }
    return true;
}

void Context::release_copy_slots() {
    for (int k = 0; k < kCopySlots; k++)
        if (ev_copy[k]) (void)hipEventDestroy(ev_copy[k]);
    if (copy_stage) (void)hipHostFree(copy_stage);
    copy_stage = nullptr;
}

int Context::copy(const CopySeg* segs, int nsegs, bool to_device) {
    const hipMemcpyKind kind = to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
    size_t total = 0, npieces = 0;
    bool pageable = true;
    for (int s = 0; s < nsegs; s++) {
        total += segs[s].bytes;
        npieces += (segs[s].bytes + kPiece - 1) / kPiece;
        if (segs[s].bytes && is_pinned(to_device ? segs[s].src : segs[s].dst)) pageable = false;
    }
    // also where there is no pinned memory for the pieces
    if (!pageable || total < kCopyLarge || !copy_slots()) {
        for (int s = 0; s < nsegs; s++)
            if (segs[s].bytes) BT_HIP(hipMemcpyAsync(segs[s].dst, segs[s].src, segs[s].bytes, kind, stream));
        // the runtime has read a pageable source when its call returns, a pinned one it may still read
        if (!to_device || !pageable) BT_HIP(hipStreamSynchronize(stream));
        return BT_OK;
    }
    const auto piece = [&](size_t n) {
        for (int s = 0;; s++) {
            const size_t m = (segs[s].bytes + kPiece - 1) / kPiece, o = n * kPiece;
            if (n < m) return Piece{(char*)segs[s].dst + o, (const char*)segs[s].src + o, std::min(kPiece, segs[s].bytes - o)};
            n -= m;
        }
    };
    std::atomic<size_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    const auto worker = [&](int w) {
        const auto ok = [&](hipError_t e) {
            if (e != hipSuccess) error.store((int)e);
            return e == hipSuccess;
        };
        if (!ok(hipSetDevice(device))) return;
        char* slot[2] = {(char*)copy_stage + (2 * w) * kPiece, (char*)copy_stage + (2 * w + 1) * kPiece};
        hipEvent_t ev[2] = {ev_copy[2 * w], ev_copy[2 * w + 1]};
        Piece open[2] = {};   // device to host: on its way into the slot
        for (int k = 0;; k ^= 1) {
            // the slot's last copy is done (an event never recorded is)
            if (!to_device || next.load() < npieces)
                if (!ok(hipEventSynchronize(ev[k]))) return;
            if (open[k].bytes) std::memcpy(open[k].dst, slot[k], open[k].bytes);
            open[k].bytes = 0;
            const size_t n = error.load() == (int)hipSuccess ? next.fetch_add(1) : npieces;
            if (n < npieces) {
                const Piece p = piece(n);
                if (to_device) {
                    std::memcpy(slot[k], p.src, p.bytes);
                    if (!ok(hipMemcpyAsync(p.dst, slot[k], p.bytes, kind, stream))) return;
                } else {
                    if (!ok(hipMemcpyAsync(slot[k], p.src, p.bytes, kind, stream))) return;
                    open[k] = p;
                }
                if (!ok(hipEventRecord(ev[k], stream))) return;
            } else if (!open[k ^ 1].bytes) {
                return;
            }
        }
    };
    std::thread threads[kCopyThreads];
    const int want = (int)std::min<size_t>(kCopyThreads, total / kCopyPerThread);
    try {
        for (int w = 1; w < want; w++) threads[w] = std::thread(worker, w);
    } catch (const std::exception&) {
        // fewer threads share the pieces then
    }
    worker(0);
    for (std::thread& t : threads)
        if (t.joinable()) t.join();
    if (error.load() != (int)hipSuccess) {
        (void)hipStreamSynchronize(stream);
        return fail(BT_ERR_HIP, std::string("copy: ") + hipGetErrorString((hipError_t)error.load()));
    }
    return BT_OK;
}

}  // namespace bt
