// CPU check of it_launch.h: how often dynamic LDS is asked for, with the runtime's three calls stood in for.
#include "../../inferred-thoughts_amd/csrc/it_launch.h"

#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

static thread_local int device = 0;
static std::mutex mu;
static std::map<std::pair<const void*, int>, int> asked;   // (kernel, device) -> calls
static bool refuse = false;
static int cleared = 0;

extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int) {
    std::lock_guard<std::mutex> g(mu);
    if (a != hipFuncAttributeMaxDynamicSharedMemorySize) return hipErrorInvalidValue;
    asked[{f, device}]++;
    return refuse ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipGetLastError() {
    cleared++;
    return hipSuccess;
}
}

template <int N> void kernel(int) {}   // (two instances: one type)

#define CHECK(x) do { if (!(x)) { printf("failed: %s\n", #x); return 1; } } while (0)

int main() {
    using itk::lds_allowed;
    const auto calls = [](auto f, int dev) { return asked[{(const void*)f, dev}]; };
    // up to 64 KB nothing is asked for
    CHECK(lds_allowed<&kernel<0>>(64 * 1024) && asked.empty());
    // a refusal is an answer for this call only, and leaves no error behind
    refuse = true;
    CHECK(!lds_allowed<&kernel<0>>(100000) && cleared == 1);
    refuse = false;
    for (int i = 0; i < 5; i++) CHECK(lds_allowed<&kernel<0>>(100000));
    CHECK(calls(&kernel<0>, 0) == 2);
    // each kernel for itself, each device for itself
    for (int i = 0; i < 5; i++) CHECK(lds_allowed<&kernel<1>>(100000));
    CHECK(calls(&kernel<1>, 0) == 1);
    for (device = 1; device < 80; device++)
        for (int i = 0; i < 3; i++) CHECK(lds_allowed<&kernel<1>>(100000));
    CHECK(calls(&kernel<1>, 1) == 1 && calls(&kernel<1>, 63) == 1 && calls(&kernel<1>, 64) == 3);
    // threads on several devices at once: every answer is yes, and afterwards nobody asks again
    std::vector<std::thread> t;
    std::vector<int> ok(16);
    for (int i = 0; i < 16; i++)
        t.emplace_back([&, i] {
            device = i % 4;
            ok[i] = 1;
            for (int k = 0; k < 1000; k++) ok[i] &= lds_allowed<&kernel<2>>(100000);
        });
    for (auto& x : t) x.join();
    int before = 0;
    for (int i = 0; i < 16; i++) CHECK(ok[i]);
    for (int d = 0; d < 4; d++) {
        before = calls(&kernel<2>, d);
        CHECK(before >= 1 && before <= 4);
        device = d;
        CHECK(lds_allowed<&kernel<2>>(100000) && calls(&kernel<2>, d) == before);
    }
    printf("ok\n");
    return 0;
}
