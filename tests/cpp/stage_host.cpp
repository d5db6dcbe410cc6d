// The staging and planning memory of stage.cpp on the CPU: the HIP calls are
// replaced by host ones that can be told to fail. Exit code 0 when a failed
// growth leaves what was there, large requests leave the context's buffers alone
// and nothing is freed twice or lost.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "../../quant-iron_amd/csrc/qi_internal.h"

static bool fail_host = false;
static std::map<void *, size_t> live;
static int copies = 0, waits = 0;

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (fail_host) return hipErrorOutOfMemory;
    *p = malloc(n);
    live[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    if (!live.erase(p)) abort();
    free(p);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    copies++;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    waits++;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stub"; }
}

#define CHECK(x)                                          \
    do {                                                  \
        if (!(x)) {                                       \
            printf("line %d: %s\n", __LINE__, #x);        \
            return 1;                                     \
        }                                                 \
    } while (0)

int main() {
    using namespace qi;
    Ctx C;
    CHECK(ensure_stage(C, 1000).ok() && C.stage_bytes >= 1000 && live.size() == 1);
    unsigned char *const first = C.stage;
    memset(first, 7, 1000);
    // a growth that fails: an error, and the buffer is still there
    fail_host = true;
    const Status e = ensure_stage(C, 100000);
    CHECK(!e.ok() && e.code == QI_ERR_OUT_OF_MEMORY);
    CHECK(C.stage == first && C.stage_bytes >= 1000 && live.count(first) && first[999] == 7);
    Staging s;
    CHECK(stage_tables(C, 900, s).ok() && s.p == first);
    CHECK(!stage_tables(C, 100000, s).ok() && C.stage == first);
    fail_host = false;
    CHECK(ensure_stage(C, 100000).ok() && C.stage_bytes >= 100000 && live.size() == 1);
    // tables above the limit: memory of the call's own, sent before it can go
    const size_t kept = C.stage_bytes, big = kStageKept + 1;
    std::vector<unsigned char> dst(big);
    {
        Staging large;
        CHECK(stage_tables(C, big, large).ok() && large.p != C.stage && C.stage_bytes == kept && live.size() == 1);
        large.p[big - 1] = 9;
        CHECK(send_tables(large, dst.data(), big, nullptr).ok() && copies == 1 && waits == 1 && dst[big - 1] == 9);
    }
    Staging small;
    CHECK(stage_tables(C, 64, small).ok() && small.p == C.stage);
    CHECK(send_tables(small, dst.data(), 64, nullptr).ok() && copies == 2 && waits == 1);
    CHECK(send_tables(small, nullptr, 0, nullptr).ok() && copies == 2);
    // planning memory: kept up to its limit, the call's own above
    std::vector<unsigned char> own;
    unsigned char *p = nullptr;
    CHECK(plan_memory(C, 5000, own, &p).ok() && p == C.plan_arena.data() && own.empty() && C.plan_arena.size() >= 5000);
    CHECK(plan_memory(C, kArenaKept + 1, own, &p).ok() && p == own.data() && C.plan_arena.size() <= kArenaKept);
    // no more than the limit is ever pinned
    for (size_t n = 1 << 20; n <= kStageKept; n += 3 << 20) CHECK(ensure_stage(C, n).ok() && C.stage_bytes <= kStageKept);
    CHECK(ensure_stage(C, kStageKept).ok() && C.stage_bytes == kStageKept && live.size() == 1);
    (void)hipHostFree(C.stage);
    return 0;
}
