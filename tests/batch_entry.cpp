// Calls pgf_batch_pcg and pgf_pcg on a context made by hand, with a stand-in for
// the GPU runtime that keeps device memory on the host and runs no kernel: what
// the C entries do when memory runs out or the cooperative launch is refused,
// and what they do again on a repeated call.
//   batch_entry batch SIDE NRHS CALLS FAIL    one system of SIDE x SIDE rows
//   batch_entry single SIDE 1 CALLS FAIL
// FAIL: none | device (every device allocation fails for want of a device) |
//   short K (the K-th device allocation finds no memory) | host BYTES (host
//   blocks of BYTES or more) | refused (cooperative launches)
// Prints, for each call: status, cooperative launches, other launches, host
// bytes allocated, threads per row of the batch's layout.  An exception that
// leaves an entry ends the program.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../include/pgfem.h"
#include "../pigfem_assignment_amd/csrc/kernels/pgf_device.hpp"

static size_t g_limit = ~(size_t)0;
static std::atomic<size_t> g_bytes{0};
void* operator new(size_t n) {
    g_bytes += n;
    void* p = n >= g_limit ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// ---- the stand-in
static bool g_no_device = false, g_refuse = false;
static int g_short = 0, g_mallocs = 0, g_coop = 0, g_plain = 0;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (g_no_device) return hipErrorNoDevice;
    if (++g_mallocs == g_short) return hipErrorOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    return hipSuccess;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    if (d && s) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { ++g_plain; return hipSuccess; }
hipError_t hipLaunchCooperativeKernel(const void*, dim3, dim3, void**, unsigned, hipStream_t) {
    ++g_coop;
    return g_refuse ? hipErrorIllegalState : hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = nullptr; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
}

struct pgf_ctx : public pgfd::Ctx {};

// n x n rows in groups of one, each with its neighbours in the grid
static void grid_pattern(pgf_ctx& c, int n) {
    c.dim = 2;
    c.n_free = c.n_rows = (int64_t)n * n;
    c.n_cu = 256;
    c.h_rowptr.push_back(0);
    for (int r = 0; r < n * n; ++r) {
        const int b = (int)c.h_colidx.size(), y = r / n, x = r % n;
        for (int j = std::max(y - 1, 0); j <= std::min(y + 1, n - 1); ++j)
            for (int i = std::max(x - 1, 0); i <= std::min(x + 1, n - 1); ++i) c.h_colidx.push_back(j * n + i);
        const int len = (int)c.h_colidx.size() - b;
        c.h_rowsplit.push_back(len);
        c.h_rowptr.push_back((int64_t)c.h_colidx.size());
        c.h_grp.push_back(pgft::GroupRec{r, b, len << 2 | 1, len});
    }
    c.n_grp = (int64_t)c.h_grp.size();
    c.h_grp.push_back(pgft::GroupRec{n * n, 0, 0, 0});
    c.nnz = (int64_t)c.h_colidx.size();
}

int main(int argc, char** argv) {
    if (argc < 6) return 2;
    const bool batch = !std::strcmp(argv[1], "batch");
    const int n = std::atoi(argv[2]), nrhs = std::atoi(argv[3]), calls = std::atoi(argv[4]);
    const char* fail = argv[5];
    pgf_ctx* c = new pgf_ctx();
    grid_pattern(*c, n);
    c->h_scal = (double*)std::calloc(64, sizeof(double));
    c->scal = (double*)std::calloc(64, sizeof(double));
    const int64_t sys[2] = {0, c->n_free};
    double* b = (double*)std::calloc((size_t)n * n * nrhs, sizeof(double));
    double* x = (double*)std::calloc((size_t)n * n * nrhs, sizeof(double));
    g_no_device = !std::strcmp(fail, "device");
    g_refuse = !std::strcmp(fail, "refused");
    if (!std::strcmp(fail, "short")) g_short = std::atoi(argv[6]);
    for (int call = 0; call < calls; ++call) {
        if (!std::strcmp(fail, "host")) g_limit = (size_t)std::atoll(argv[6]);
        g_bytes = 0;
        g_coop = g_plain = 0;
        int32_t tune[2] = {0, 0};
        pgf_solve_info info;
        const int rc = batch ? pgf_batch_pcg(c, 1, sys, nrhs, b, x, 1e-8, 10, nullptr, nullptr, nullptr, tune)
                             : pgf_pcg(c, b, x, nullptr, 1e-8, 10, 64, &info);
        const size_t bytes = g_bytes;
        g_limit = ~(size_t)0;
        std::printf("%d %d %d %zu %d\n", rc, g_coop, g_plain, bytes, (int)tune[0]);
        if (rc) std::fprintf(stderr, "%s\n", pgf_last_error(c));
    }
    std::fflush(stdout);
    std::_Exit(0);
}
