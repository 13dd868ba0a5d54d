// Context::copy (csrc/copy.cpp) on the host alone, over a stand-in for the
// runtime whose copies to and from pinned memory are carried out no earlier
// than somebody waits for them.  Prints what went wrong; exits 0 if nothing did.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>

#include "../blacktracer_amd/csrc/bt_internal.h"

namespace {
std::recursive_mutex mu;
std::map<const char*, size_t> pinned;         // allocations the runtime knows
std::deque<std::function<void()>> work;       // the stream's copies, not yet carried out
size_t done = 0;                              // copies carried out so far
std::map<void*, size_t> events;               // copies that an event waits for
bool no_pinned = false;

bool is_known(const void* p) {
    for (auto& a : pinned)
        if ((const char*)p >= a.first && (const char*)p < a.first + a.second) return true;
    return false;
}
void run_to(size_t n) {
    while (done < n && !work.empty()) {
        work.front()();
        work.pop_front();
        done++;
    }
}
}  // namespace

extern "C" {
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    a->type = is_known(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free((void*)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    events[(void*)e] = done + work.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    run_to(events[(void*)e]);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    run_to(~size_t(0));
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned) return hipErrorOutOfMemory;
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = std::malloc(n);
    pinned[(const char*)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    pinned.erase((const char*)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    work.push_back([=] { std::memcpy(d, s, n); });
    if (!is_known(kind == hipMemcpyHostToDevice ? s : d)) run_to(~size_t(0));   // pageable: at once
    return hipSuccess;
}
}

namespace bt {
int fail(int code, const std::string& msg) {
    std::printf("fail: %s\n", msg.c_str());
    return code;
}
}  // namespace bt

int main() {
    int bad = 0;
    const size_t mib = size_t(1) << 20;
    const size_t sets[][3] = {{1, 0, 0}, {4 * mib - 1, 0, 0}, {4 * mib, 0, 0}, {2 * mib, 2 * mib + 1, 0},
                              {4 * mib + 1, 7, 2 * mib - 1}, {0, 9 * mib + 5, 3}, {30 * mib + 11, 1, 14 * mib}};
    for (int mode = 0; mode < 3; mode++) {   // pageable, no pinned memory to have, the caller's memory pinned
        bt::Context c;
        no_pinned = mode == 1;
        for (const auto& set : sets)
            for (int to_device = 0; to_device < 2; to_device++) {
                bt::CopySeg segs[3];
                unsigned char *src[3], *dst[3];
                for (int s = 0; s < 3; s++) {
                    src[s] = (unsigned char*)std::malloc(set[s] + 1);
                    dst[s] = (unsigned char*)std::calloc(set[s] + 1, 1);
                    for (size_t k = 0; k < set[s]; k++) src[s][k] = (unsigned char)(1 + (k * 2654435761u >> 13) % 255);
                    if (mode == 2) pinned[(const char*)(to_device ? src[s] : dst[s])] = set[s] + 1;
                    segs[s] = {dst[s], src[s], set[s]};
                }
                const int rc = c.copy(segs, 3, to_device != 0);
                bool ok = rc == 0;
                for (int s = 0; s < 3 && ok; s++) {
                    // the caller's memory is its own again; what it gave is on the stream, or there
                    if (to_device) {
                        unsigned char* keep = (unsigned char*)std::malloc(set[s] + 1);
                        std::memcpy(keep, src[s], set[s]);
                        std::memset(src[s], 0, set[s]);
                        (void)hipStreamSynchronize(nullptr);
                        ok = std::memcmp(keep, dst[s], set[s]) == 0;
                        std::free(keep);
                    } else {
                        ok = std::memcmp(src[s], dst[s], set[s]) == 0;
                    }
                    ok = ok && dst[s][set[s]] == 0;
                }
                (void)hipStreamSynchronize(nullptr);
                if (!ok) {
                    std::printf("mode %d, %zu + %zu + %zu bytes, %s: rc %d\n", mode, set[0], set[1], set[2],
                                to_device ? "to the device" : "to the host", rc);
                    bad++;
                }
                for (int s = 0; s < 3; s++) {
                    pinned.erase((const char*)src[s]);
                    pinned.erase((const char*)dst[s]);
                    std::free(src[s]);
                    std::free(dst[s]);
                }
            }
        c.release_copy_slots();
    }
    return bad ? 1 : 0;
}
