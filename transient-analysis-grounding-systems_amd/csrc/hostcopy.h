// Copies between a caller's pageable arrays and the device through pinned
// staging buffers.
#pragma once

#include <cstring>

#include "tags_common.h"

namespace tags {

// Two pinned chunks with the events of the copies that last used them.
struct PinnedStage {
    static constexpr size_t kChunk = (size_t)4 << 20;
    char* p[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    bool used[2] = {false, false};
    int dev = 0;  // the device its events belong to
    int wait(int i)
    {
        if (used[i]) TAGS_HIP(hipEventSynchronize(ev[i]));
        used[i] = false;
        return 0;
    }
};

// A stage held for one copy (from a process-wide pool of at most kStageIdle
// idle ones, safe from several threads; stage_release frees the idle ones).
constexpr int kStageIdle = 4;
PinnedStage* stage_get();
void stage_put(PinnedStage* s);
void stage_release();
struct StageRef {
    PinnedStage* s;
    StageRef() : s(stage_get()) {}
    ~StageRef()
    {
        if (s) stage_put(s);
    }
};

// bytes of `src` (host) to `dst` on st, in stream order; `src` may change once
// it returns. Up to 8 MiB through the stage (a pageable copy of 0.25 MB takes
// 127 us, staged 20), larger ones by the runtime's own pageable path (35 GB/s
// at 17 MB, where one thread's copy into the stage runs at 30), waited for: from
// memory that the caller has pinned the runtime's copy is still under way when it
// returns.
inline int copy_in(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    if (bytes == 0) return 0;
    if (bytes > 2 * PinnedStage::kChunk) {
        TAGS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
        TAGS_HIP(hipStreamSynchronize(st));
        return 0;
    }
    StageRef r;
    if (!r.s) return TAGS_ERR_HIP;
    int k = 0;
    for (size_t o = 0; o < bytes; o += PinnedStage::kChunk, k ^= 1) {
        const size_t len = bytes - o < PinnedStage::kChunk ? bytes - o : PinnedStage::kChunk;
        const int rc = r.s->wait(k);
        if (rc) return rc;
        std::memcpy(r.s->p[k], (const char*)src + o, len);
        TAGS_HIP(hipMemcpyAsync((char*)dst + o, r.s->p[k], len, hipMemcpyHostToDevice, st));
        TAGS_HIP(hipEventRecord(r.s->ev[k], st));
        r.s->used[k] = true;
    }
    return 0;
}

// bytes of device memory after what is queued on st, chunk by chunk, handed to
// take(chunk, offset, length) in order while the next chunk's copy runs (a
// pageable copy out ran at 16 GB/s, 10 into fresh pages; the pinned ones at 55).
// Waits for all of it.
template <typename F>
int copy_out_each(const void* src, size_t bytes, hipStream_t st, F take)
{
    if (bytes == 0) return 0;
    StageRef r;
    if (!r.s) return TAGS_ERR_HIP;
    constexpr size_t C = PinnedStage::kChunk;
    const size_t n = (bytes + C - 1) / C;
    auto issue = [&](size_t i) -> int {
        const int k = (int)(i & 1);
        const int rc = r.s->wait(k);
        if (rc) return rc;
        const size_t len = bytes - i * C < C ? bytes - i * C : C;
        TAGS_HIP(hipMemcpyAsync(r.s->p[k], (const char*)src + i * C, len, hipMemcpyDeviceToHost,
                                st));
        TAGS_HIP(hipEventRecord(r.s->ev[k], st));
        r.s->used[k] = true;
        return 0;
    };
    int rc = issue(0);
    for (size_t i = 0; i < n && !rc; i++) {
        if (i + 1 < n && (rc = issue(i + 1))) break;
        if ((rc = r.s->wait((int)(i & 1)))) break;
        take((const char*)r.s->p[i & 1], i * C, bytes - i * C < C ? bytes - i * C : C);
    }
    return rc;
}
inline int copy_out(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    return copy_out_each(src, bytes, st, [&](const char* c, size_t o, size_t len) {
        std::memcpy((char*)dst + o, c, len);
    });
}

// Upper triangles of m x m row-major arrays, rows packed one after the other
// (entry (i, k >= i) at i m - i (i - 1) / 2 + k - i): calls row(i, k, value
// pointer, count) for the pieces of rows that a chunk holds.
template <typename F>
int copy_out_rows(const c64* packed, long m, hipStream_t st, F row)
{
    long i = 0, k = 0;
    return copy_out_each(packed, sizeof(c64) * (size_t)(m * (m + 1) / 2), st,
                         [&](const char* c, size_t, size_t len) {
                             const c64* v = (const c64*)c;
                             long left = (long)(len / sizeof(c64));
                             while (left > 0) {
                                 const long n = m - k < left ? m - k : left;
                                 row(i, k, v, n);
                                 v += n;
                                 left -= n;
                                 k += n;
                                 if (k == m) k = ++i;
                             }
                         });
}

}  // namespace tags
