// The packed sweep tables with device memory that runs out: the HIP calls the
// tables make are replaced by host ones, and every allocation in turn fails.
// Exit status: the number of checks that failed.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "device.hpp"

using namespace unap_hip;

static std::map<void*, size_t> g_live;
static int g_calls = 0, g_failAt = -1, g_launches = 0;
static hipError_t g_last = hipSuccess;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (g_calls++ == g_failAt) {
        *p = nullptr;
        return g_last = hipErrorOutOfMemory;
    }
    *p = std::calloc(n, 1);
    g_live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p && !g_live.erase(p)) std::abort();
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (!d || !s) return hipErrorInvalidValue;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    ++g_launches;
    return hipSuccess;
}
}

static int g_bad = 0;
#define EXPECT(c)                                             \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);       \
            ++g_bad;                                          \
        }                                                     \
    } while (0)

// A matrix of three levels whose rows are longer than a table's first chunk.
static void fill(DevMatrix<double>& M) {
    M.n = 300;
    M.sweepable = true;
    M.entriesPerRow = 20;
    M.fwdStartH = {0, 100, 200, 300};
    M.bwdStartH = M.fwdStartH;
    M.bwdSliceH.assign(M.n / 32 + 2, 0);
    M.bwdInfoH.assign(M.n, 0);
    M.rowInfo.upload(std::vector<uint32_t>(M.n, 70u | 30u << 16), nullptr);
}

template <class Make>
static void check(Make make) {
    for (int k = 0;; ++k) {
        DevMatrix<double> M;
        fill(M);
        g_calls = 0;
        g_failAt = k;
        const GroupTab* t = make(M);
        const bool reached = g_calls > k;
        g_failAt = -1;
        if (!reached) {  // nothing failed: the table is whole
            EXPECT(t && t->tab.p && t->filled);
            EXPECT(make(M) == t);
            break;
        }
        EXPECT(t == nullptr);
        for (const GroupTab* u : {&M.gsTab, &M.luTab})
            EXPECT(!u->grp.p && !u->grp0.p && !u->grpOvf.p && !u->tab.p && !u->ovf.p);
        EXPECT(g_last == hipSuccess);  // no error is left for the next call to find
        const int launches = g_launches;
        EXPECT(make(M) == nullptr);  // the same route on every later call
        EXPECT(g_launches == launches);
    }
    EXPECT(g_live.empty());
}

int main() {
    check([](DevMatrix<double>& M) { return M.gsTable(nullptr); });
    check([](DevMatrix<double>& M) { return M.luTable(nullptr); });
    // a buffer whose allocation failed has no size
    DBuf<int> b;
    g_calls = 0;
    g_failAt = 0;
    bool threw = false;
    try {
        b.alloc(100);
    } catch (const Error&) {
        threw = true;
    }
    EXPECT(threw && b.n == 0 && !b.p);
    return g_bad;
}
