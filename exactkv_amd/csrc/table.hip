// Small host values to the device and device words to the host, through kernel arguments and
// mapped host memory: the page table's updates and the overflow check's counters. A copy from
// pageable memory waits for the whole stream before it returns, so each of them drained the
// GPU (and cost a copy and a scatter launch); a launch with the values in its arguments does
// neither. Twelve paged sequences joining, 24 steps and leaving: 4,060 -> 3,000 us.
//
// No counterpart in the reference (its token count and counters are read and written by torch
// calls, cache.py:57-60,149-158; paged KV is in its future work, README.md:121-123).
#include <chrono>

#include "common.hpp"
#include "../../include/exactkv.h"

namespace exkv {

constexpr int kPairs = 448;          // (index, value) pairs per launch (whole wavefronts; 3,584 of the 4,096 argument bytes)
constexpr int kWords = 448;          // word addresses per launch

struct Pairs {
    int32_t at[kPairs];
    int32_t val[kPairs];
};

// Pairs [0, nl) into lens, [nl, n) into table.
__global__ void __launch_bounds__(kPairs) table_write_kernel(int32_t* lens, int32_t* table, int nl, int n, Pairs p) {
    const int i = threadIdx.x;
    if (i < n) (i < nl ? lens : table)[p.at[i]] = p.val[i];
}

struct Words {
    const int32_t* p[kWords];
};
// The words to out, then the tag to *done.
__global__ void __launch_bounds__(kWords) fetch_words_kernel(Words w, int n, int32_t* out, int32_t* done, int32_t tag) {
    const int i = threadIdx.x;
    if (i < n) __hip_atomic_store(out + i, *w.p[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (i == 0) __hip_atomic_store(done, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace exkv

using namespace exkv;

extern "C" int exkv_table_write(int32_t* lens, int64_t lens_size, int32_t* table, int64_t table_size, const int32_t* at,
                                const int32_t* val, int32_t n_lens, int32_t n, hipStream_t stream) {
    EXKV_REQUIRE(n >= 0 && n_lens >= 0 && n_lens <= n, "table_write: bad counts %d of %d", n_lens, n);
    EXKV_REQUIRE(n == 0 || (lens && table && at && val), "table_write: null pointer");
    for (int32_t i = 0; i < n; ++i)
        EXKV_REQUIRE(at[i] >= 0 && at[i] < (i < n_lens ? lens_size : table_size), "table_write: index %d of pair %d", at[i],
                     i);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(stream, &capturing);
    if (e != hipSuccess) return hip_status(e, "table_write");
    // a replay would write this call's values again, over later ones
    EXKV_REQUIRE(capturing == hipStreamCaptureStatusNone, "table_write: the stream is being captured");
    Pairs p;
    for (int32_t i0 = 0; i0 < n; i0 += kPairs) {
        const int32_t m = n - i0 < kPairs ? n - i0 : kPairs;
        for (int32_t i = 0; i < m; ++i) {
            p.at[i] = at[i0 + i];
            p.val[i] = val[i0 + i];
        }
        const int32_t nl = n_lens - i0 < 0 ? 0 : n_lens - i0;
        hipLaunchKernelGGL(table_write_kernel, dim3(1), dim3((m + 63) / 64 * 64), 0, stream, lens, table, nl, m, p);
    }
    return hip_status(hipGetLastError(), "table_write");
}

// The stream's last kernel here says through mapped host memory that everything before it is
// done, and the host polls for that: 6.4 us from the launch to the answer on an idle stream,
// where a launch and hipStreamSynchronize take 11.9. After kPollUs without it (a long queue)
// the stream is waited for instead.
constexpr int kPollUs = 200;

extern "C" int exkv_fetch_words(const int32_t* const* words, int32_t n, int32_t* host, int32_t tag, hipStream_t stream) {
    EXKV_REQUIRE(n >= 0 && host && (n == 0 || words), "fetch_words: null pointer");
    for (int32_t i = 0; i < n; ++i) EXKV_REQUIRE(words[i], "fetch_words: null word %d", i);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(stream, &capturing);
    if (e != hipSuccess) return hip_status(e, "fetch_words");
    EXKV_REQUIRE(capturing == hipStreamCaptureStatusNone, "fetch_words: the stream is being captured");
    Words w;
    int32_t i0 = 0;
    do {
        const int32_t m = n - i0 < kWords ? n - i0 : kWords;
        for (int32_t i = 0; i < m; ++i) w.p[i] = words[i0 + i];
        // only the last launch's tag is the call's
        hipLaunchKernelGGL(fetch_words_kernel, dim3(1), dim3(m < 1 ? 64 : (m + 63) / 64 * 64), 0, stream, w, m,
                           host + 1 + i0, host, i0 + m < n ? ~tag : tag);
        i0 += kWords;
    } while (i0 < n);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_status(e, "fetch_words");
    return wait_for_tag("fetch_words", host, tag, stream);
}

int exkv::wait_for_tag(const char* what, const int32_t* host, int32_t tag, hipStream_t stream) {
    const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(kPollUs);
    do {
        for (int k = 0; k < 64; ++k) {
            if (__atomic_load_n(host, __ATOMIC_ACQUIRE) == tag) return EXKV_OK;
            __builtin_ia32_pause();
        }
    } while (std::chrono::steady_clock::now() < end);
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return hip_status(e, what);
    EXKV_REQUIRE(__atomic_load_n(host, __ATOMIC_ACQUIRE) == tag, "%s: no answer from the GPU", what);
    return EXKV_OK;
}
