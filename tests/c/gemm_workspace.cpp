// The workspace rules of the batched GEMM (csrc/capi_gemm.cpp) with the HIP
// calls and kernel launchers replaced by counters: how much a call allocates,
// captured or not, what it falls back to when an allocation fails, and that
// what a captured graph may hold stays allocated. Then the rows of the
// prefill's batch buffers (grow_rows).
#include "../../wpc-engine_amd/csrc/capi_gemm.cpp"

#include <cstdio>
#include <cstdlib>
#include <map>

static std::map<void*, size_t> live;
static size_t held, limit = ~size_t(0);
static bool capturing, pending;
static hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
static int broken;  // captures that an allocation ended
struct Launch {
    void* xf;
    float* xsum;
    int tiles;
    uint32_t M;
};
static std::vector<Launch> launched;
static int passes;

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    if (capturing && mode != hipStreamCaptureModeRelaxed) {
        broken++;
        return hipErrorStreamCaptureUnsupported;
    }
    if (held + n > limit) {
        pending = true;
        return hipErrorOutOfMemory;
    }
    *p = std::malloc(1);
    live[*p] = n;
    held += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!live.count(p)) std::abort();
    held -= live[p];
    live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    pending = false;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m)
{
    std::swap(*m, mode);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st)
{
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
int wpcg_linear_matvec(wpcg_linear*, const float*, float*, wpcg_stream) { return WPCG_OK; }
}

namespace wpcg {
int fail(int code, const std::string&) { return code; }
int hip_fail(hipError_t, const char*) { return WPCG_E_DEVICE; }
int check_ctx(wpcg_ctx*) { return WPCG_OK; }
int gemm_row_groups(uint64_t rows) { return (int)((rows + 127) / 128); }
int gemm_small_row_groups(uint64_t rows) { return (int)((rows + 63) / 64); }
int gemm_kslices(uint64_t, uint64_t, int req) { return req ? req : 2; }
int gemm_small_kslices(uint64_t, uint64_t, int req) { return req ? req : 2; }
hipError_t launch_gemm(const DeviceMatrix&, const GemmWork&, const void*, int, int, const float*, const float*, float*,
                       hipStream_t)
{
    passes++;
    return hipSuccess;
}
hipError_t launch_gemm_wide(const DeviceMatrix&, void* xf, float* xsum, int tiles, const void*, int, uint32_t M,
                            const float*, float*, float*, uint64_t, hipStream_t)
{
    launched.push_back({xf, xsum, tiles, M});
    return hipSuccess;
}
hipError_t launch_fill_u32(uint32_t*, int, uint32_t, hipStream_t) { return hipSuccess; }
void* scratch_ptr(int) { return nullptr; }
hipStream_t pick(wpcg_ctx*, wpcg_stream s) { return static_cast<hipStream_t>(s); }
}  // namespace wpcg

#define CHECK(c)                                                              \
    do {                                                                      \
        if (!(c)) {                                                           \
            std::printf("line %d: %s\n", __LINE__, #c);                       \
            return 1;                                                         \
        }                                                                     \
    } while (0)

int main()
{
    using namespace wpcg;
    const uint64_t nb = 120, rows = 3840;
    const auto packed = [&](int tiles) { return nb * tiles * (4096 + 64); };
    float x = 0, y = 0;
    wpcg_ctx ctx{};
    auto linear = [&](wpcg_linear& L) {
        L.ctx = &ctx;
        L.m.scheme = 4;
        L.m.rows = L.m.rows_pad = rows;
        L.m.nb = nb;
        L.m.cols = nb * 128;
    };
    auto gemm = [&](wpcg_linear& L, int dtype, uint32_t M) {
        launched.clear();
        return wpcg_linear_gemm(&L, &x, dtype, M, &y, nullptr);
    };
    const int bf = WPCG_DTYPE_BF16, sp = WPCG_DTYPE_F32_SPLIT;
    {  // sized to the call, grown by what is missing, kept
        wpcg_linear L{};
        linear(L);
        CHECK(gemm(L, bf, 64) == WPCG_OK && launched.empty());
        const size_t base = held;
        CHECK(gemm(L, bf, 65) == WPCG_OK && launched[0].tiles == 8 && held == base + packed(8));
        CHECK((uint8_t*)launched[0].xsum == (uint8_t*)launched[0].xf + nb * 8 * 4096);
        void* first = launched[0].xf;
        CHECK(gemm(L, bf, 128) == WPCG_OK && launched[0].xf == first && held == base + packed(8));
        CHECK(gemm(L, sp, 33) == WPCG_OK && launched[0].xf == first);
        CHECK(gemm(L, sp, 65) == WPCG_OK && launched[0].tiles == 16);
        CHECK(gemm(L, bf, 1024) == WPCG_OK && launched[0].tiles == 64);
        CHECK(held == base + packed(8) + packed(16) + packed(64) && live.count(first));
        CHECK(gemm(L, bf, 300) == WPCG_OK && launched[0].tiles == 64);  // a larger one serves
        CHECK(gemm(L, bf, 100000) == WPCG_OK && launched[0].tiles == 128);
        CHECK(wpcg_linear_set_gemm_kslices(&L, 0) == WPCG_OK && held == 0);
    }
    {  // no memory: the largest one made, else the 64-column workspace
        wpcg_linear L{};
        linear(L);
        CHECK(gemm(L, bf, 2) == WPCG_OK);
        limit = held;
        CHECK(gemm(L, bf, 1000) == WPCG_OK && launched[0].tiles == 4 && launched[0].xf == L.gemm.xf);
        CHECK(launched[0].xsum == L.gemm.xsum && !pending);
        limit = held + packed(8);
        CHECK(gemm(L, bf, 65) == WPCG_OK && launched[0].tiles == 8);
        void* first = launched[0].xf;
        CHECK(gemm(L, sp, 1000) == WPCG_OK && launched[0].xf == first && launched[0].tiles == 8 && !pending);
        limit = ~size_t(0);
        CHECK(gemm(L, sp, 1000) == WPCG_OK && launched[0].tiles == 128);
        free_gemm(L.gemm);
        CHECK(held == 0);
    }
    {  // captured: as outside, with the capture's mode as it was afterwards
        wpcg_linear L{};
        linear(L);
        CHECK(gemm(L, bf, 2) == WPCG_OK);
        capturing = true;
        const size_t base = held;
        CHECK(gemm(L, bf, 500) == WPCG_OK && launched[0].tiles == 32 && held == base + packed(32));
        CHECK(broken == 0 && mode == hipStreamCaptureModeGlobal);
        limit = held;
        CHECK(gemm(L, bf, 600) == WPCG_OK && launched[0].tiles == 32 && broken == 0 && !pending);
        CHECK(mode == hipStreamCaptureModeGlobal);
        limit = ~size_t(0);
        wpcg_linear N{};  // the first batched call on a linear is still refused
        linear(N);
        CHECK(gemm(N, bf, 500) == WPCG_E_ARG && launched.empty() && broken == 0);
        capturing = false;
        free_gemm(L.gemm);
    }
    {  // a caller's K-slices keep the 64-row passes
        wpcg_linear L{};
        linear(L);
        L.gemm.kg_req = 3;
        passes = 0;
        CHECK(gemm(L, bf, 130) == WPCG_OK && launched.empty() && passes == 3);
        CHECK(gemm(L, sp, 70) == WPCG_OK && launched.empty() && passes == 6);
        free_gemm(L.gemm);
    }
    {  // the prefill's rows: as many as wanted, else those there, else the least
        uint32_t have = 0, most = 1024;
        std::vector<uint32_t> asked;
        auto make = [&](uint32_t rows) {
            asked.push_back(rows);
            if (rows > most) return WPCG_E_DEVICE;
            have = rows;
            return WPCG_OK;
        };
        CHECK(grow_rows(have, 256, 256, make) == WPCG_OK && have == 256);
        CHECK(grow_rows(have, 256, 256, make) == WPCG_OK && asked.size() == 1);
        most = 500;
        CHECK(grow_rows(have, 1024, 256, make) == WPCG_OK && have == 256 && asked.size() == 2);
        most = 1024;
        CHECK(grow_rows(have, 1024, 256, make) == WPCG_OK && have == 1024);
        have = 0, most = 300;
        CHECK(grow_rows(have, 1024, 256, make) == WPCG_OK && have == 256);
        have = 0, most = 100;
        CHECK(grow_rows(have, 1024, 256, make) != WPCG_OK && grow_rows(have, 256, 256, make) != WPCG_OK && have == 0);
    }
    std::printf("workspace ok\n");
    return 0;
}
