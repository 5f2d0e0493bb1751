// Host-only trace of the launches behind the C ABI: the HIP runtime calls that
// liblsmx.so makes are answered here (a 256-CU gfx950 that runs nothing), so a
// call records which kernels it would launch, with their grids, without a GPU.
// Reads one command per line and answers each with one line of JSON; built and
// driven by tests/test_launch_routes.py.
//
//   w4 M N K dual ws fmt lda ldw ld_sw   lsmx_gemm_bf16f4_ws (ws: 0 none, 1 as queried)
//   f4 M N K fmt lda ldb                 lsmx_gemm_f4f4
//   f4q M N K lda ldb                    lsmx_gemm_f4f4_quant
//   f8 M N K nc                          lsmx_gemm_f8f8_nb (nc = 1) or lsmx_gemm_f8f8
//   dense M N K dtype mode nc            lsmx_gemm_dense_nb or lsmx_gemm_dense
//   threads M N K n calls                n threads x calls of lsmx_gemm_bf16f4_ws on one stream;
//                                        "split": launches of a call that another thread's interrupted
//   kernels                              the names of all kernels in the library
// A leading dimension of 0 stands for the dense one.
#include <cxxabi.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <iostream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <thread>
#include <vector>

#include "../include/lsmx.h"

namespace {
std::map<const void *, std::string> g_names;
struct Launch {
    std::string name;
    unsigned grid;
    int call;   // which call made it
};
std::mutex g_mu;
std::vector<Launch> g_launches;
thread_local int t_call = 0;
thread_local dim3 t_grid;
int g_pause_us = 0;   // after each launch, so that other threads get their turn
}  // namespace

#define STUB extern "C" __attribute__((visibility("default")))
STUB void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
STUB void __hipUnregisterFatBinary(void **) {}
STUB void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
STUB void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                                void *, int *) {
    int st = 0;
    char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string s = st == 0 ? d : name;
    free(d);
    s = s.substr(0, s.find('('));
    const size_t ns = s.find("lsmx::");
    g_names[host] = ns == std::string::npos ? s : s.substr(ns + 6);
}
STUB hipError_t __hipPushCallConfiguration(dim3 grid, dim3, size_t, hipStream_t) {
    t_grid = grid;
    return hipSuccess;
}
STUB hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = t_grid, *block = dim3(1), *lds = 0, *s = nullptr;
    return hipSuccess;
}
STUB hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        g_launches.push_back(Launch{g_names[f], grid.x * grid.y * grid.z, t_call});
    }
    if (g_pause_us) usleep(g_pause_us);
    return hipSuccess;
}
STUB hipError_t hipGetLastError() { return hipSuccess; }
STUB const char *hipGetErrorString(hipError_t) { return "none"; }
STUB hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
STUB hipError_t hipSetDevice(int) { return hipSuccess; }
STUB hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { return *d = 0, hipSuccess; }
STUB hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
STUB hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {   // hipGetDevicePropertiesR0600
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
STUB hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = reinterpret_cast<void *>(0x10000), hipSuccess; }

namespace {
void *lib;
template <typename F>
F *sym(const char *name, F *) {
    return reinterpret_cast<F *>(dlsym(lib, name));
}
#define L(f) sym(#f, &f)
// stands for a device buffer: never dereferenced
template <typename T = void>
T *P() {
    return reinterpret_cast<T *>(0x100000);
}

std::string answer(int rc, int64_t need = 0, int slices = 1) {
    std::ostringstream o;
    o << "{\"rc\": " << rc << ", \"workspace\": " << need << ", \"slices\": " << slices << ", \"launches\": [";
    for (size_t i = 0; i < g_launches.size(); ++i)
        o << (i ? ", " : "") << "[\"" << g_launches[i].name << "\", " << g_launches[i].grid << "]";
    o << "]}";
    g_launches.clear();
    return o.str();
}
int w4(int64_t M, int64_t N, int64_t K, int dual, int64_t need, int fmt, int64_t lda, int64_t ldw, int64_t lds) {
    return L(lsmx_gemm_bf16f4_ws)(P(), dual ? P() : nullptr, lda, P<uint8_t>(), ldw, P(), lds, fmt, P(),
                                  dual ? P() : nullptr, LSMX_F32, N, M, N, K, need ? P() : nullptr, need, nullptr);
}
}  // namespace

int main(int argc, char **argv) {
    if (argc != 2 || !(lib = dlopen(argv[1], RTLD_NOW))) return fprintf(stderr, "dlopen: %s\n", dlerror()), 2;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string op;
        int64_t M, N, K;
        in >> op >> M >> N >> K;
        auto arg = [&](int64_t zero = 0) {
            int64_t v = 0;
            in >> v;
            return v ? v : zero;
        };
        if (op == "w4") {
            const int dual = (int)arg(), ws = (int)arg(), fmt = (int)arg();
            const int64_t lda = arg(K), ldw = arg(K / 2), lds = arg(K / 32);
            const int64_t need = L(lsmx_gemm_bf16f4_workspace)(M, N, K, dual);
            const int rc = w4(M, N, K, dual, ws ? need : 0, fmt, lda, ldw, lds);
            std::cout << answer(rc, need, L(lsmx_gemm_bf16f4_slices)(M, N, K)) << std::endl;
        } else if (op == "f4") {
            const int fmt = (int)arg();
            const int64_t lda = arg(K / 2), ldb = arg(K / 2);
            const bool km = fmt == LSMX_SCALE_E8M0_KMAJOR;
            const int rc = L(lsmx_gemm_f4f4)(P<uint8_t>(), lda, P(), km ? M : K / 32, P<uint8_t>(), ldb, P(),
                                             km ? N : K / 32, fmt, P(), LSMX_F32, N, M, N, K, nullptr);
            std::cout << answer(rc) << std::endl;
        } else if (op == "f4q") {
            const int64_t lda = arg(K / 2), ldb = arg(K / 2);
            const int rc = L(lsmx_gemm_f4f4_quant)(P<uint8_t>(), lda, P(), M, P<uint8_t>(), ldb, P(), N, P(), N,
                                                   P<uint8_t>(), N / 2, P<uint8_t>(), M, P<uint8_t>(), M / 2,
                                                   P<uint8_t>(), N, M, N, K, nullptr);
            std::cout << answer(rc) << std::endl;
        } else if (op == "f8") {
            const int rc = arg() ? L(lsmx_gemm_f8f8_nb)(P<uint8_t>(), K, P<uint8_t>(), M, P<uint8_t>(), N, P<uint8_t>(), N,
                                                        P(), LSMX_F32, N, M, N, K, nullptr)
                                 : L(lsmx_gemm_f8f8)(P<uint8_t>(), K, P<uint8_t>(), M, P<uint8_t>(), K, P<uint8_t>(), N,
                                                     LSMX_SCALE_E8M0_KMAJOR, P(), LSMX_F32, N, M, N, K, nullptr);
            std::cout << answer(rc) << std::endl;
        } else if (op == "dense") {
            const int dt = (int)arg(), mode = (int)arg();
            const int rc = arg() ? L(lsmx_gemm_dense_nb)(P(), P(), K, P(), P(), N, dt, mode, P<float>(), P<float>(), N, M, N,
                                                         K, nullptr)
                                 : L(lsmx_gemm_dense)(P(), P(), K, P(), P(), K, dt, mode, P<float>(), P<float>(), N, M, N,
                                                      K, 1, nullptr);
            std::cout << answer(rc) << std::endl;
        } else if (op == "threads") {
            const int n = (int)arg(), calls = (int)arg();
            const int64_t need = L(lsmx_gemm_bf16f4_workspace)(M, N, K, 0);
            std::atomic<int> rc{0};
            g_pause_us = 200;
            std::vector<std::thread> ts;
            for (int i = 0; i < n; ++i)
                ts.emplace_back([&, i] {
                    for (int c = 0; c < calls; ++c) {
                        t_call = 1 + i * calls + c;
                        if (w4(M, N, K, 0, need, LSMX_SCALE_E8M0, K, K / 2, K / 32) != 0) rc = 1;
                    }
                });
            for (auto &t : ts) t.join();
            g_pause_us = 0;
            int runs = 0;   // a call's launches in a row are one run
            for (size_t i = 0; i < g_launches.size(); ++i) runs += i == 0 || g_launches[i].call != g_launches[i - 1].call;
            std::cout << "{\"rc\": " << rc << ", \"launches\": " << g_launches.size() << ", \"calls\": " << n * calls
                      << ", \"split\": " << runs - n * calls << "}" << std::endl;
            g_launches.clear();
        } else if (op == "kernels") {
            std::cout << "[";
            const char *sep = "";
            for (auto &k : g_names) std::cout << sep << "\"" << k.second << "\"", sep = ", ";
            std::cout << "]" << std::endl;
        } else {
            return fprintf(stderr, "unknown command %s\n", op.c_str()), 2;
        }
    }
    return 0;
}
