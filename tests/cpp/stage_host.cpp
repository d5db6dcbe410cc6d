// The staging and planning memory of stage.cpp on the CPU: the HIP calls are
// replaced by host ones that can be told to fail. Exit code 0 when a failed
// growth leaves what was there and nothing is freed twice or lost.
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
    std::vector<unsigned char> dst(64);
    Staging small;
    CHECK(stage_tables(C, 64, small).ok() && small.p == C.stage);
    CHECK(send_tables(small, dst.data(), 64, nullptr).ok() && copies == 1 && waits == 0);
    CHECK(send_tables(small, nullptr, 0, nullptr).ok() && copies == 1);
    (void)hipHostFree(C.stage);
    return 0;
}
