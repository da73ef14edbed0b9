// C ABI of the batched dequant-GEMM (include/wpcg.h). No reference
// counterpart: the reference decodes one token at a time (README.md:174-180).
#include <algorithm>
#include <cstring>
#include <memory>

#include "wpcg_internal.hpp"

namespace wpcg {

void free_gemm(GemmWork& w)
{
    if (w.xf) (void)hipFree(w.xf);
    if (w.xsum) (void)hipFree(w.xsum);
    if (w.part) (void)hipFree(w.part);
    if (w.counters) (void)hipFree(w.counters);
    for (void* p : w.wide)
        if (p) (void)hipFree(p);
    const int req = w.kg_req;
    w = GemmWork{};
    w.kg_req = req;
}

namespace {

// Floats of the K-slices' partials (0: no kernel of this matrix has slices).
uint64_t part_floats(const DeviceMatrix& m, const GemmWork& w)
{
    if (w.kg <= 1 && w.kg_small <= 1) return 0;
    return std::max<uint64_t>((uint64_t)w.kg * GEMM_MAX_M, (uint64_t)w.kg_small * 16) * m.rows_pad;
}

int make_gemm(wpcg_linear* L, hipStream_t s)
{
    const DeviceMatrix& m = L->m;
    GemmWork& w = L->gemm;
    w.kg = gemm_kslices(m.rows, m.nb, w.kg_req);
    w.kg_small = gemm_small_kslices(m.rows, m.nb, w.kg_req);
    const uint64_t part = part_floats(m, w);
    // partial sums are addressed with 32-bit byte offsets
    if (part * 4 >= (1ull << 31))
        return fail(WPCG_E_SHAPE, "batched GEMM: too many rows for the split-K workspace");
    const uint64_t rgs = (uint64_t)std::max(gemm_row_groups(m.rows), gemm_small_row_groups(m.rows));
    hipError_t e = hipMalloc(&w.xf, m.nb * 4 * 4096);
    if (e == hipSuccess) e = hipMalloc(&w.xsum, m.nb * GEMM_MAX_M * sizeof(float));
    if (e == hipSuccess && part) e = hipMalloc(&w.part, part * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&w.counters, std::max<uint64_t>(1, rgs) * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemsetAsync(w.counters, 0, std::max<uint64_t>(1, rgs) * sizeof(uint32_t), s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        free_gemm(w);
        return hip_fail(e, "batched GEMM workspace");
    }
    return WPCG_OK;
}

// Whether the many-row kernel takes a batch of M rows: more than one
// launch_gemm covers, unless the caller set the K-slices (its knob is that
// kernel's).
bool wide(const wpcg_linear* L, int x_mode, uint32_t M)
{
    return L->gemm.kg_req == 0 && M > (uint32_t)(x_mode == GX_SPLIT ? GEMM_MAX_M_SPLIT : GEMM_MAX_M) &&
           L->m.nb * GEMM_WIDE_TILES * 4096 < (1ull << 30);  // the kernel's buffer offsets
}

// Device memory also while this thread captures a stream: an allocation is no
// stream operation, but the capture's default mode refuses (and is ended by)
// calls that could wait for one.
hipError_t malloc_capturing(void** p, uint64_t bytes)
{
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) return e;
    e = hipMalloc(p, bytes);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return e;
}

// The many-row kernel over M rows. Its packed X is made by the first call
// that wants its size (the least of 8, 16, ... GEMM_WIDE_TILES tiles that
// hold the rows, so at most twice what the largest call needs stays held),
// captured or not: passes of 64 rows replayed 1024 in 879 us that one pass
// takes 149 for (15360 x 3840 bf16). Where the memory is not there, the
// largest one made, or the 64-column workspace, serves in smaller passes,
// with the same results.
int run_wide(wpcg_linear* L, const void* x, int x_mode, uint32_t M, float* y, hipStream_t s)
{
    const DeviceMatrix& m = L->m;
    GemmWork& w = L->gemm;
    constexpr int N = sizeof w.wide / sizeof w.wide[0];
    static_assert((8 << (N - 1)) == GEMM_WIDE_TILES, "the steps end at a whole pass");
    int want = 0;
    while (want < N - 1 && (uint32_t)gemm_wide_cols(x_mode, gemm_wide_step(want)) < M) want++;
    int i = want;
    while (i < N && !w.wide[i]) i++;
    if (i == N) {
        i = want;
        if (malloc_capturing(&w.wide[i], m.nb * gemm_wide_step(i) * (4096 + 16 * sizeof(float))) != hipSuccess) {
            (void)hipGetLastError();
            w.wide[i] = nullptr;
        }
        while (i >= 0 && !w.wide[i]) i--;
    }
    const int tiles = i < 0 ? GEMM_MAX_M / 16 : gemm_wide_step(i);
    void* xf = i < 0 ? w.xf : w.wide[i];
    float* xsum = i < 0 ? w.xsum : reinterpret_cast<float*>(static_cast<uint8_t*>(xf) + m.nb * tiles * 4096);
    WPCG_HIP(launch_gemm_wide(m, xf, xsum, tiles, x, x_mode, M, L->bias, y, w.part, part_floats(m, w), s));
    return WPCG_OK;
}

int run_gemm(wpcg_linear* L, const void* x, int x_dtype, uint32_t M, float* y, hipStream_t s)
{
    const DeviceMatrix& m = L->m;
    if (M == 0 || m.rows == 0) return WPCG_OK;
    if (m.nb == 0) {  // no inputs: every row of Y is the bias (or 0)
        for (uint32_t r = 0; r < M; r++)
            if (int rc = wpcg_linear_matvec(L, nullptr, y + (uint64_t)r * m.rows, s)) return rc;
        return WPCG_OK;
    }
    if (x_dtype == WPCG_DTYPE_F32 && M == 1)
        return wpcg_linear_matvec(L, static_cast<const float*>(x), y, s);
    if (!L->gemm.xf) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        WPCG_HIP(hipStreamIsCapturing(s, &st));
        if (st != hipStreamCaptureStatusNone)
            return fail(WPCG_E_ARG, "the first batched call on a linear allocates its workspace: "
                                    "make it before capturing a graph");
        if (int rc = make_gemm(L, s)) return rc;
    }
    if (wide(L, x_dtype, M)) return run_wide(L, x, x_dtype, M, y, s);
    const uint64_t es = x_dtype == WPCG_DTYPE_BF16 ? 2 : 4;
    const uint32_t step = x_dtype == WPCG_DTYPE_F32_SPLIT ? GEMM_MAX_M_SPLIT : GEMM_MAX_M;
    for (uint32_t c = 0; c < M; c += step) {
        const int mc = (int)std::min<uint32_t>(step, M - c);
        WPCG_HIP(launch_gemm(m, L->gemm, static_cast<const uint8_t*>(x) + (uint64_t)c * m.cols * es, x_dtype, mc,
                             L->bias, nullptr, y + (uint64_t)c * m.rows, s));
    }
    return WPCG_OK;
}

}  // namespace

namespace {

int check_gemm_args(wpcg_linear* L, const void* x, int x_dtype, uint32_t M, const float* y)
{
    if (!L) return fail(WPCG_E_ARG, "null linear");
    if (x_dtype != WPCG_DTYPE_F32 && x_dtype != WPCG_DTYPE_BF16 && x_dtype != WPCG_DTYPE_F32_SPLIT)
        return fail(WPCG_E_ARG, "unknown x dtype");
    if (M && L->m.rows && (!y || (!x && L->m.cols))) return fail(WPCG_E_ARG, "null x or y");
    if ((uint64_t)M * L->m.cols > (1ull << 40)) return fail(WPCG_E_SHAPE, "batch too large");
    return check_ctx(L->ctx);
}

}  // namespace
}  // namespace wpcg

using namespace wpcg;

extern "C" {

int wpcg_linear_gemm(wpcg_linear* L, const void* x, int x_dtype, uint32_t M, float* y, wpcg_stream stream)
{
    if (int rc = check_gemm_args(L, x, x_dtype, M, y)) return rc;
    return run_gemm(L, x, x_dtype, M, y, pick(L->ctx, stream));
}

int wpcg_linear_gemm_noalloc(wpcg_linear* L, const void* x, int x_dtype, uint32_t M, float* y,
                             wpcg_stream stream)
{
    if (int rc = check_gemm_args(L, x, x_dtype, M, y)) return rc;
    const DeviceMatrix& m = L->m;
    hipStream_t s = pick(L->ctx, stream);
    if (M == 0 || m.rows == 0) return WPCG_OK;
    // the cases the matvec serves use no batched workspace
    if (m.nb == 0 || (x_dtype == WPCG_DTYPE_F32 && M == 1)) return run_gemm(L, x, x_dtype, M, y, s);
    // the workspace make_gemm would allocate, at 256-byte aligned offsets
    GemmWork w{};
    w.kg_req = L->gemm.kg_req;
    w.kg = gemm_kslices(m.rows, m.nb, w.kg_req);
    w.kg_small = gemm_small_kslices(m.rows, m.nb, w.kg_req);
    const uint64_t ncnt = std::max<uint64_t>(
        1, (uint64_t)std::max(gemm_row_groups(m.rows), gemm_small_row_groups(m.rows)));
    const uint64_t part = part_floats(m, w) * sizeof(float);
    auto up = [](uint64_t b) { return (b + 255) / 256 * 256; };
    const uint64_t o_part = up(ncnt * sizeof(uint32_t));
    const uint64_t o_xsum = o_part + up(part);
    const uint64_t o_xf = o_xsum + up(m.nb * GEMM_MAX_M * sizeof(float));
    const uint64_t need = o_xf + up(m.nb * 4 * 4096);
    if (need > WPCG_NOALLOC_SCRATCH_BYTES)
        return fail(WPCG_E_UNSUPPORTED, "batched GEMM without allocation: this matrix needs " + std::to_string(need) +
                                            " bytes of workspace, the fixed array holds " +
                                            std::to_string(WPCG_NOALLOC_SCRATCH_BYTES));
    uint8_t* base = static_cast<uint8_t*>(scratch_ptr(L->ctx->device));
    if (!base) return fail(WPCG_E_DEVICE, "the no-allocation workspace is not set up on this device");
    w.counters = reinterpret_cast<uint32_t*>(base);
    w.xsum = reinterpret_cast<float*>(base + o_xsum);
    w.xf = base + o_xf;
    w.part = part ? reinterpret_cast<float*>(base + o_part) : nullptr;
    if (wide(L, x_dtype, M)) {  // packed X behind the rest; its sums need half of what xf would take there
        const int tiles = (int)std::min<uint64_t>(GEMM_WIDE_TILES, SCRATCH_PACK_BYTES / (m.nb * 4096) / 4 * 4);
        static_assert(SCRATCH_PACK_BYTES >= 4 * WPCG_NOALLOC_SCRATCH_BYTES && GEMM_WIDE_TILES * 64 <= 4 * 4096,
                      "four tiles at least, and room for the sums of all");
        w.xf = base + WPCG_NOALLOC_SCRATCH_BYTES;
        WPCG_HIP(launch_gemm_wide(m, w.xf, w.xsum, tiles, x, x_dtype, M, L->bias, y, w.part, part_floats(m, w), s));
        return WPCG_OK;
    }
    // the array keeps the last call's contents: the counters must start at 0
    WPCG_HIP(launch_fill_u32(w.counters, (int)ncnt, 0u, s));
    const uint64_t es = x_dtype == WPCG_DTYPE_BF16 ? 2 : 4;
    const uint32_t step = x_dtype == WPCG_DTYPE_F32_SPLIT ? GEMM_MAX_M_SPLIT : GEMM_MAX_M;
    for (uint32_t c = 0; c < M; c += step) {
        const int mc = (int)std::min<uint32_t>(step, M - c);
        WPCG_HIP(launch_gemm(m, w, static_cast<const uint8_t*>(x) + (uint64_t)c * m.cols * es, x_dtype, mc,
                             L->bias, nullptr, y + (uint64_t)c * m.rows, s));
    }
    return WPCG_OK;
}

int wpcg_linear_gemm_host(wpcg_linear* L, const void* x, int x_dtype, uint32_t M, float* y)
{
    if (int rc = check_gemm_args(L, x, x_dtype, M, y)) return rc;
    if (M == 0 || L->m.rows == 0) return WPCG_OK;
    const uint64_t xb = (uint64_t)M * L->m.cols * (x_dtype == WPCG_DTYPE_BF16 ? 2 : 4);
    const uint64_t yb = (uint64_t)M * L->m.rows * sizeof(float);
    std::lock_guard<std::mutex> g(L->host_mu);
    hipStream_t s = L->ctx->stream;
    void *dx = nullptr, *dy = nullptr;
    hipError_t e = hipMalloc(&dx, std::max<uint64_t>(xb, 4));
    if (e == hipSuccess) e = hipMalloc(&dy, yb);
    if (e == hipSuccess && xb) e = hipMemcpyAsync(dx, x, xb, hipMemcpyHostToDevice, s);
    int rc = e == hipSuccess ? run_gemm(L, dx, x_dtype, M, static_cast<float*>(dy), s) : hip_fail(e, "staging");
    if (rc == WPCG_OK) {
        e = hipMemcpyAsync(y, dy, yb, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) rc = hip_fail(e, "batched GEMM copy-back");
    } else {
        (void)hipStreamSynchronize(s);
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    return rc;
}

int wpcg_linear_set_gemm_kslices(wpcg_linear* L, int kslices)
{
    if (!L) return fail(WPCG_E_ARG, "null linear");
    if (kslices < 0) return fail(WPCG_E_ARG, "kslices must be >= 0");
    if (int rc = check_ctx(L->ctx)) return rc;
    WPCG_HIP(hipStreamSynchronize(L->ctx->stream));
    free_gemm(L->gemm);
    L->gemm.kg_req = kslices;
    return WPCG_OK;
}

int wpcg_linear_gemm_kslices(wpcg_linear* L, int* kslices_small, int* kslices)
{
    if (!L || !kslices_small || !kslices) return fail(WPCG_E_ARG, "null argument");
    *kslices_small = L->gemm.xf ? L->gemm.kg_small : gemm_small_kslices(L->m.rows, L->m.nb, L->gemm.kg_req);
    *kslices = L->gemm.xf ? L->gemm.kg : gemm_kslices(L->m.rows, L->m.nb, L->gemm.kg_req);
    return WPCG_OK;
}

}  // extern "C"
