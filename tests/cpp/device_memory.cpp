// The engine's device memory on a device of a chosen size: the library's own
// objects linked with the HIP calls below in the runtime's place, which count
// the bytes allocated, fail beyond the size, and run nothing.  Prints what the
// scenario named on the command line did as one JSON object;
// tests/test_device_memory.py reads it.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../../include/cfamd.h"

namespace {

size_t g_size = size_t(288) << 30, g_used = 0, g_peak = 0;
long g_launches = 0, g_uploads = 0;
bool g_hide = false;        // hipMemGetInfo reports 288 GiB as free
long g_fail_upload = 0;     // the upload that fails, counted from 1
std::map<void*, size_t> g_blocks;

size_t room() { return g_used < g_size ? g_size - g_used : 0; }

}  // namespace

extern "C" {

hipError_t hipMalloc(void** p, size_t n)
{
    if (n > room()) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    g_blocks[*p] = n;
    g_used += n;
    if (g_used > g_peak) g_peak = g_used;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    g_used -= g_blocks.at(p);
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t)
{
    *f = g_hide ? size_t(288) << 30 : room();
    *t = g_size;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind)
{
    return ++g_uploads == g_fail_upload ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { ++g_launches; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 << 10;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char at[16]; *p = at; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipLaunchHostFunc(hipStream_t, hipHostFn_t f, void* d) { f(d); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* q)
{
    *g = *b = dim3(1);
    *s = 0;
    *q = nullptr;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* at; return &at; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

}  // extern "C"

int main(int argc, char** argv)
{
    const std::string scenario = argc > 1 ? argv[1] : "";
    const int precision = argc > 2 ? std::atoi(argv[2]) : 0, mode = argc > 3 ? std::atoi(argv[3]) : 0;
    const int paths = argc > 4 ? std::atoi(argv[4]) : 1 << 20;

    // the 30 x 36 grid and three years of weekly dates
    std::vector<double> spots(30), times(36), vols(30 * 36, 0.2);
    for (int i = 0; i < 30; ++i) spots[i] = 50.0 + 150.0 * i / 29.0;
    for (int j = 0; j < 36; ++j) times[j] = (j + 1) / 12.0;
    cf_model lv{};
    lv.kind = CF_MODEL_DUPIRE;
    lv.spot = 100.0;
    lv.n_spots = 30;
    lv.n_times = 36;
    lv.spots = spots.data();
    lv.times = times.data();
    lv.vols = vols.data();
    lv.max_dt = 1.0 / 52;
    cf_product uoc{};
    uoc.kind = CF_PRODUCT_BARRIER;
    uoc.strike = 120.0;
    uoc.barrier = 150.0;
    uoc.maturity = 3.0;
    uoc.monitor_freq = 1.0 / 52;
    uoc.smooth = 0.05;
    double mats[4] = {1.0, 2.0, 2.0, 1.0}, ks[4] = {90.0, 100.0, 110.0, 95.0};
    cf_product eus{};
    eus.kind = CF_PRODUCT_EUROPEANS;
    eus.n_options = 3;
    eus.maturities = mats;
    eus.strikes = ks;
    cf_num num{};
    num.use_sobol = 1;
    num.num_path = paths;
    num.precision = precision;
    num.aad_mode = mode;
    const double w[4] = {1.0, 0.0, 0.0, 0.0};
    double means[4], agg = 0.0;
    std::vector<double> risks(4 * (1 + 30 * 36)), per_path;
    auto risk = [&](const cf_num& n) {
        return cf_mc_simul_aad(&lv, &uoc, &n, w, means, &agg, risks.data(), nullptr, nullptr);
    };
    auto itemized = [&](const cf_num& n) { return cf_mc_simul_aad_multi(&lv, &eus, &n, means, risks.data()); };

    long rc0 = 0, rc = -1;
    int64_t footprint = 0;
    size_t before = 0;
    cf_num fp64 = num;
    fp64.num_path = 1 << 20;
    fp64.precision = CF_FP64;
    if (scenario == "footprint") {
        footprint = cf_aad_footprint(&lv, &uoc, &num);
        rc = risk(num);
    } else if (scenario == "tight") {
        // the checkpoints of four slots a wave fit with 256 MiB to spare, but not
        // beside the per-path outputs
        g_size = size_t(1700) << 20;
        per_path.resize(size_t(paths) * 2);
        rc = cf_mc_simul_aad(&lv, &uoc, &num, w, means, &agg, risks.data(), per_path.data(), nullptr);
    } else if (scenario == "short") {
        // the device is fuller than it says
        g_size = size_t(700) << 20;
        g_hide = true;
        rc = risk(fp64);
    } else if (scenario == "held" || scenario == "server" || scenario == "itemized" || scenario == "points") {
        // a risk call first, then one that needs what it left behind
        rc0 = risk(fp64);
        before = g_used;
        g_size = g_used + (size_t(64) << 20);
        g_launches = 0;
        if (scenario == "held") {
            per_path.resize(size_t(paths) * 2);
            rc = cf_mc_simul(&lv, &uoc, &num, means, nullptr, per_path.data());
        } else if (scenario == "server") {
            cf_server* srv = nullptr;
            cf_server_opts opts{2, int64_t(1) << 30, 1, 1};
            rc = cf_server_create(&opts, &srv);
            if (rc == 0) rc = cf_server_destroy(srv);
        } else if (scenario == "itemized") {
            rc = itemized(num);
        } else {
            std::vector<double> z(size_t(1) << 25);
            rc = cf_sobol_points(0, 1 << 18, 128, CF_FP64, 0, nullptr, z.data());
        }
    } else if (scenario == "itemized_calls") {
        eus.n_options = argc > 5 ? std::atoi(argv[5]) : 3;
        rc = itemized(num);
    } else if (scenario == "itemized_short") {
        g_size = size_t(500) << 20;
        g_hide = true;
        rc = itemized(num);
    } else if (scenario == "upload") {
        // one upload of the first call fails
        (void)risk(num);
        g_uploads = 0;
        eus.n_options = 2;
        g_fail_upload = argc > 5 ? std::atol(argv[5]) : 1;
        rc0 = itemized(num);
        g_fail_upload = 0;
        const long done = g_uploads;
        rc = itemized(num);
        before = size_t(done);
    }
    std::printf("{\"rc0\": %ld, \"rc\": %ld, \"footprint\": %lld, \"peak\": %zu, \"used\": %zu, \"before\": %zu, "
                "\"launches\": %ld, \"uploads\": %ld, \"error\": \"%s\"}\n",
                rc0, rc, static_cast<long long>(footprint), g_peak, g_used, before, g_launches, g_uploads,
                cf_last_error());
    return 0;
}
