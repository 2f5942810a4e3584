// Copies of several contiguous buffers in one launch: the inputs of a recorded forward into the buffers it was recorded on.
// Bound by the launch at the sizes it is for: tokens of 2 MB and one timestep take 4.0 us as two copies, 2.1 as one launch (16 MB 5.9 /
// 5.1), back to back in a recorded graph; traced ahead of the replays of a stack's forward the copies take 4.7 us each, the launch 4.8.
#include "cdm_common.h"

namespace {

constexpr int kMaxRuns = 8;
constexpr int kThreads = 256;

struct CopyParams {
    const char* src[kMaxRuns];
    char* dst[kMaxRuns];
    int64_t bytes[kMaxRuns];
};

// blockIdx.y = run.  16 bytes per thread and iteration where both ends are aligned to that, single bytes otherwise and behind the
// last whole 16.  A run may be copied onto itself: every byte is read by the thread that writes it.
__global__ __launch_bounds__(kThreads) void copy_runs_kernel(const CopyParams p) {
    const int run = blockIdx.y;
    const char* src = p.src[run];
    char* dst = p.dst[run];
    const int64_t bytes = p.bytes[run], stride = (int64_t)gridDim.x * kThreads, first = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const bool wide = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15u) == 0;
    const int64_t n16 = wide ? bytes >> 4 : 0;
    for (int64_t i = first; i < n16; i += stride) reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
    for (int64_t i = n16 * 16 + first; i < bytes; i += stride) dst[i] = src[i];
}

// do [a, a + n) and [b, b + m) share a byte?
inline bool overlap(const void* a, int64_t n, const void* b, int64_t m) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return n > 0 && m > 0 && x < y + (uintptr_t)m && y < x + (uintptr_t)n;
}

}  // namespace

extern "C" int32_t cdm_copy_runs(const void* const* src, void* const* dst, const int64_t* bytes, int32_t n, void* stream) {
    CDM_REQUIRE(n >= 0 && n <= kMaxRuns, CDM_ERR_BAD_ARG, "copy_runs: n=%d must be 0..%d", n, kMaxRuns);
    CDM_REQUIRE(n == 0 || (src && dst && bytes), CDM_ERR_BAD_ARG, "copy_runs: null pointer");
    for (int i = 0; i < n; ++i) {
        CDM_REQUIRE(bytes[i] >= 0, CDM_ERR_BAD_ARG, "copy_runs: negative size");
        CDM_REQUIRE(bytes[i] == 0 || (src[i] && dst[i]), CDM_ERR_BAD_ARG, "copy_runs: null pointer");
        CDM_REQUIRE(src[i] == dst[i] || !overlap(src[i], bytes[i], dst[i], bytes[i]), CDM_ERR_BAD_ARG, "copy_runs: run %d overlaps its target", i);
    }
    if (n == 0) return CDM_OK;
    int32_t rc = cdm_require_device();
    if (rc) return rc;
    // in the order of the runs: one that reads or writes what an earlier one writes, or writes what one reads, starts a new launch
    for (int at = 0; at < n;) {
        int end = at + 1;
        for (bool apart = true; end < n; ++end) {
            for (int i = at; i < end && apart; ++i)
                apart = !overlap(src[end], bytes[end], dst[i], bytes[i]) && !overlap(dst[end], bytes[end], dst[i], bytes[i]) &&
                        !overlap(dst[end], bytes[end], src[i], bytes[i]);
            if (!apart) break;
        }
        CopyParams p{};
        int64_t most = 0;
        for (int i = at; i < end; ++i) {
            p.src[i - at] = (const char*)src[i]; p.dst[i - at] = (char*)dst[i]; p.bytes[i - at] = bytes[i];
            most = bytes[i] > most ? bytes[i] : most;
        }
        int64_t blocks = (most + 16 * kThreads - 1) / (16 * kThreads);
        if (blocks > 8192) blocks = 8192;
        if (blocks > 0) {
            copy_runs_kernel<<<dim3((unsigned)blocks, (unsigned)(end - at)), kThreads, 0, (hipStream_t)stream>>>(p);
            if ((rc = cdm_check_launch("copy_runs"))) return rc;
        }
        at = end;
    }
    return CDM_OK;
}
