"""ggb_ground_state from several threads: one set of teams per device at a time, and threads on different
devices do not wait for each other.

The driver stands in for the HIP calls of the function (host memory, launches that do nothing); its
hipStreamSynchronize waits a while for the other thread, so that it sees whether both were inside their
sweeps at once."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang++")

DRIVER = r"""
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>
#include <hip/hip_runtime_api.h>
#include "ggbtd.h"

static std::mutex mu;
static std::condition_variable cv;
static int inside = 0, together = 0;
static thread_local bool waited = false;

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)8, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return *p = calloc(n, 1), hipSuccess; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    if (waited) return hipSuccess;  // the first one of a thread follows its sweeps
    waited = true;
    std::unique_lock<std::mutex> l(mu);
    if (++inside == 2) together = 1;
    cv.notify_all();
    cv.wait_for(l, std::chrono::milliseconds(1500), [] { return together != 0; });
    --inside;
    return hipSuccess;
}
}

static int run(int device) {
    const int N = 160;
    ggb_gs_problem p = {N, 1, 1, 5, 1, device, 2.0, 0.3, 2.0, 1e-9};
    std::vector<double> r(N, 1.0), T(N * N, 0.0), lam(N, 1.0), u(N), v(N), rho(N);
    const int32_t l = 0;
    const double occ = 2.0;
    double eps;
    int32_t it, conv;
    return ggb_ground_state(&p, &l, &occ, r.data(), r.data(), T.data(), T.data(), lam.data(), u.data(), &eps, v.data(),
                            rho.data(), &it, &conv);
}

int main(int argc, char **argv) {
    const int dev[2] = {atoi(argv[1]), atoi(argv[2])};
    int rc[2];
    std::thread a([&] { rc[0] = run(dev[0]); }), b([&] { rc[1] = run(dev[1]); });
    a.join(), b.join();
    printf("rc %d %d together %d\n", rc[0], rc[1], together);
    return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("ROCm's clang not installed")
    lib = os.path.join(ROOT, "ggbtddft_amd")
    if not os.path.exists(os.path.join(lib, "libggbtd.so")):
        from ggbtddft_amd import build
        build.build()
    d = tmp_path_factory.mktemp("lock")
    (d / "drive.cpp").write_text(DRIVER)
    r = subprocess.run([CLANG, "-std=c++17", "-O1", "-pthread", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                        "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"), str(d / "drive.cpp"),
                        "-L", lib, "-l:libggbtd.so", "-Wl,-rpath," + lib, "-L", os.path.join(ROCM, "lib"),
                        "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-o", str(d / "drive")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    return str(d / "drive")


@pytest.mark.parametrize("devices, together", [((0, 1), 1), ((2, 2), 0)])
def test_one_set_of_teams_per_device(driver, devices, together):
    r = subprocess.run([driver, str(devices[0]), str(devices[1])], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.split() == ["rc", "0", "0", "together", str(together)], r.stdout
