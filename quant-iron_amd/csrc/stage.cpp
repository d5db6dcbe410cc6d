// stage.cpp — host memory in which calls plan and pack the tables they send to
// the device. Host-only (built with g++).
#include <algorithm>
#include <new>

#include "qi_internal.h"

namespace qi {

namespace {
Status host_oom() { return make_err(QI_ERR_OUT_OF_MEMORY, 0, 0, 0, 0, "host memory"); }
bool grow(std::vector<unsigned char> &v, size_t bytes) {
    try {
        if (v.size() < bytes) v.resize(bytes);
    } catch (const std::bad_alloc &) {
        return false;
    }
    return true;
}
}  // namespace

Status plan_memory(Ctx &C, size_t bytes, std::vector<unsigned char> &own, unsigned char **p) {
    std::vector<unsigned char> &v = bytes <= kArenaKept ? C.plan_arena : own;
    if (!grow(v, bytes)) return host_oom();
    *p = v.data();
    return Status{};
}

Status ensure_stage(Ctx &C, size_t bytes) {
    if (C.stage_bytes >= bytes) return Status{};
    // the old buffer goes when the new one is there: what the context could
    // stage before, it can after a failure
    void *p = nullptr;
    size_t want = std::max(bytes, std::min(kStageKept, C.stage_bytes + C.stage_bytes / 2));
    if (hipHostMalloc(&p, want, 0) != hipSuccess) {
        (void)hipGetLastError();
        return host_oom();
    }
    if (C.stage) (void)hipHostFree(C.stage);
    C.stage = (unsigned char *)p;
    C.stage_bytes = want;
    return Status{};
}

Status stage_tables(Ctx &C, size_t bytes, Staging &s) {
    if (bytes <= kStageKept) {
        Status e = ensure_stage(C, bytes);
        s.p = C.stage;
        return e;
    }
    if (!grow(s.own, bytes)) return host_oom();
    s.p = s.own.data();
    return Status{};
}

Status send_tables(const Staging &s, void *dst, size_t bytes, hipStream_t st) {
    if (!bytes) return Status{};
    QI_HIP_TRY(hipMemcpyAsync(dst, s.p, bytes, hipMemcpyHostToDevice, st));
    if (!s.own.empty()) QI_HIP_TRY(hipStreamSynchronize(st));
    return Status{};
}

}  // namespace qi
