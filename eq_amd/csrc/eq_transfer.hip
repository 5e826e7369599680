// eq_transfer.hip -- fields and host arrays in and out of the batch.
//
// A field lies in rows of `pitch` doubles inside its frame; callers hold it in
// natural order.  Between the two one kernel moves the rows, whichever side is
// where: device memory, or a pinned buffer that the GPU reads and writes
// through the bus.  Pageable memory goes through two such buffers in turn, so
// the host's copy of one chunk runs beside the kernel of the next.  A strided
// copy to pageable memory by the runtime goes row by row (7 to 10 us a row):
// 401x201 nodes took 1.90 ms up and 1.41 ms down, now 0.04 and 0.05.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "eq_internal.h"

namespace eqk {

// one pinned buffer; a larger one is no faster (the host's copy bounds both
// directions beyond it) and costs more to pin
constexpr size_t kStageWords = 1 << 17;

// Words [k0, k0 + n) of the natural order of rows of w words, between `flat`
// (its word k0 first) and `rows` (pitch p).  Both sides are walked in order,
// W words a thread in flight: bound by the memory or the bus.  An uploaded
// field is a new state: the kept solutions are no start for it (restart: the
// problem's have_prev and have_prev2).
template <bool TO_ROWS, int W>
__global__ __launch_bounds__(256) void k_rows(double* __restrict__ flat, double* __restrict__ rows, int64_t k0,
                                              int64_t n, uint32_t w, int64_t p, int32_t* restart)
{
    if (restart && blockIdx.x == 0 && threadIdx.x < 2) restart[threadIdx.x] = 0;
    const int64_t first = (int64_t)blockIdx.x * (256 * W) + threadIdx.x;
    double v[W];
    int64_t at[W];
#pragma unroll
    for (int q = 0; q < W; ++q) {
        const int64_t k = first + 256 * q, g = k0 + k;
        // (divisions in 32 bits wherever the field allows)
        const int64_t i = (g >> 32) == 0 ? (int64_t)((uint32_t)g / w) : g / (int64_t)w;
        at[q] = g + i * (p - (int64_t)w);
        if (k < n) v[q] = TO_ROWS ? flat[k] : rows[at[q]];
    }
#pragma unroll
    for (int q = 0; q < W; ++q)
        if (first + 256 * q < n) {
            if (TO_ROWS)
                rows[at[q]] = v[q];
            else
                flat[first + 256 * q] = v[q];
        }
}

template <bool TO_ROWS>
static void launch_rows(eq_batch* b, double* flat, double* rows, int64_t k0, int64_t n, int64_t w, int64_t p,
                        int32_t* restart)
{
    // up to one round of threads on the chip (2^19) a word each: there a launch
    // is latency (0.18 M words 4.0 us with four words a thread, 3.1 with one);
    // beyond, four in flight
    const int words = n <= (1 << 19) ? 1 : 4, per = 256 * words;
    auto kern = words == 1 ? k_rows<TO_ROWS, 1> : k_rows<TO_ROWS, 4>;
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, b->stream, flat, rows, k0, n, (uint32_t)w,
                       p, restart);
}

// Whether the batch's device reads and writes this memory in a kernel, word by
// word; other memory (pageable, another device's, off the words' alignment)
// goes through the runtime's copy.
static bool reachable(const eq_batch* b, const void* p)
{
    if ((uintptr_t)p % sizeof(double)) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        hipGetLastError();
        return false;
    }
    return (a.type == hipMemoryTypeDevice && a.device == b->device) || a.type == hipMemoryTypeManaged;
}

static int ensure_stage(eq_batch* b)
{
    for (int k = 0; k < 2; ++k) {
        if (!b->stage[k] &&
            hipHostMalloc((void**)&b->stage[k], sizeof(double) * kStageWords, hipHostMallocDefault) != hipSuccess)
            return set_error(EQ_ERR_NOMEM, "pinned staging");
        if (!b->stage_ev[k]) EQ_HIP(hipEventCreateWithFlags(&b->stage_ev[k], hipEventDisableTiming));
    }
    return EQ_OK;
}

void free_stage(eq_batch* b)
{
    for (int k = 0; k < 2; ++k) {
        if (b->stage[k]) hipHostFree(b->stage[k]);
        if (b->stage_ev[k]) hipEventDestroy(b->stage_ev[k]);
        b->stage[k] = nullptr;
        b->stage_ev[k] = nullptr;
    }
}

// Host memory to rows of w doubles with pitch p (bytes: the last word may be
// in part).  Returns when the source has been read; the stream has the rest.
int rows_from_host(eq_batch* b, double* rows, int64_t w, int64_t p, const void* src, size_t bytes, int32_t* restart)
{
    int rc = ensure_stage(b);
    if (rc) return rc;
    const int64_t n = (int64_t)((bytes + 7) / 8);
    int at = 0;
    for (int64_t k0 = 0; k0 < n; k0 += kStageWords, at ^= 1) {
        const int64_t m = std::min<int64_t>(kStageWords, n - k0);
        EQ_HIP(hipEventSynchronize(b->stage_ev[at])); // the buffer's last kernel (any call's)
        std::memcpy(b->stage[at], (const char*)src + 8 * k0, std::min<size_t>(8 * (size_t)m, bytes - 8 * (size_t)k0));
        launch_rows<true>(b, b->stage[at], rows, k0, m, w, p, k0 == 0 ? restart : nullptr);
        EQ_HIP(hipEventRecord(b->stage_ev[at], b->stream));
    }
    EQ_HIP(hipGetLastError());
    return EQ_OK;
}

// The reverse; complete when it returns.
int rows_to_host(eq_batch* b, const double* rows, int64_t w, int64_t p, void* dst, size_t bytes)
{
    int rc = ensure_stage(b);
    if (rc) return rc;
    const int64_t n = (int64_t)((bytes + 7) / 8);
    auto put = [&](int64_t k0, int at) {
        launch_rows<false>(b, b->stage[at], const_cast<double*>(rows), k0, std::min<int64_t>(kStageWords, n - k0), w, p,
                           nullptr);
        return hipEventRecord(b->stage_ev[at], b->stream);
    };
    // (the stream orders the first kernel behind an upload's that still reads the buffer)
    if (n > 0) EQ_HIP(put(0, 0));
    int at = 0;
    for (int64_t k0 = 0; k0 < n; k0 += kStageWords, at ^= 1) {
        if (k0 + (int64_t)kStageWords < n) EQ_HIP(put(k0 + kStageWords, at ^ 1));
        EQ_HIP(hipEventSynchronize(b->stage_ev[at]));
        std::memcpy((char*)dst + 8 * k0, b->stage[at],
                    std::min<size_t>(8 * (size_t)std::min<int64_t>(kStageWords, n - k0), bytes - 8 * (size_t)k0));
    }
    EQ_HIP(hipGetLastError());
    return EQ_OK;
}

static int check_field(eq_batch* b, int32_t prob, const void* u, size_t n)
{
    if (!u) return set_error(EQ_ERR_INVALID, "NULL data");
    if (!b) return set_error(EQ_ERR_INVALID, "NULL batch");
    if (prob < 0 || prob >= b->nprob) return set_error(EQ_ERR_INVALID, "problem index out of range");
    const LevelProb& P = b->levels[0].probs[prob];
    if (n != ((size_t)P.nx + 1) * ((size_t)P.ny + 1)) return set_error(EQ_ERR_INVALID, "length must be (nx+1)*(ny+1)");
    hipSetDevice(b->device);
    return EQ_OK;
}

} // namespace eqk

using namespace eqk;

extern "C" {

int eq_batch_upload(eq_batch* b, int32_t prob, const double* u, size_t n)
{
    int rc = check_field(b, prob, u, n);
    if (rc) return rc;
    const LevelProb& P = b->levels[0].probs[prob];
    rc = rows_from_host(b, b->u + P.origin, P.nx + 1, P.pitch, u, sizeof(double) * n, &b->d_state[prob].have_prev);
    if (rc) return rc;
    EQ_HIP(hipStreamSynchronize(b->stream));
    return EQ_OK;
}

int eq_batch_download(eq_batch* b, int32_t prob, double* u, size_t n)
{
    int rc = check_field(b, prob, u, n);
    if (rc) return rc;
    const LevelProb& P = b->levels[0].probs[prob];
    return rows_to_host(b, b->u + P.origin, P.nx + 1, P.pitch, u, sizeof(double) * n);
}

int eq_batch_upload_dev(eq_batch* b, int32_t prob, const double* d_u, size_t n)
{
    int rc = check_field(b, prob, d_u, n);
    if (rc) return rc;
    const LevelProb& P = b->levels[0].probs[prob];
    double* to = b->u + P.origin;
    const size_t w = (size_t)P.nx + 1;
    if (reachable(b, d_u)) {
        launch_rows<true>(b, const_cast<double*>(d_u), to, 0, (int64_t)n, w, P.pitch, &b->d_state[prob].have_prev);
        EQ_HIP(hipGetLastError());
        return EQ_OK;
    }
    EQ_HIP(hipMemsetAsync(&b->d_state[prob].have_prev, 0, 2 * sizeof(int32_t), b->stream)); // and have_prev2
    EQ_HIP(hipMemcpy2DAsync(to, sizeof(double) * P.pitch, d_u, sizeof(double) * w, sizeof(double) * w, n / w,
                            hipMemcpyDeviceToDevice, b->stream));
    return EQ_OK;
}

int eq_batch_download_dev(eq_batch* b, int32_t prob, double* d_u, size_t n)
{
    int rc = check_field(b, prob, d_u, n);
    if (rc) return rc;
    const LevelProb& P = b->levels[0].probs[prob];
    double* from = b->u + P.origin;
    const size_t w = (size_t)P.nx + 1;
    if (reachable(b, d_u)) {
        launch_rows<false>(b, d_u, from, 0, (int64_t)n, w, P.pitch, nullptr);
        EQ_HIP(hipGetLastError());
        return EQ_OK;
    }
    EQ_HIP(hipMemcpy2DAsync(d_u, sizeof(double) * w, from, sizeof(double) * P.pitch, sizeof(double) * w, n / w,
                            hipMemcpyDeviceToDevice, b->stream));
    return EQ_OK;
}

} // extern "C"
