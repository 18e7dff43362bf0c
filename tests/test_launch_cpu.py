"""The launches of ``csrc/ixh_dev.h`` on machines of several GPUs: the runtime's calls are stand-ins that keep count of devices, streams
and errors as the runtime does, so that no GPU is needed."""
import os
import shutil
import subprocess

import pytest

HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ixrun_amd", "csrc")
PROGRAM = r"""
#include "ixh_dev.h"
#include <cstdio>
#include <string>

// two GPUs with two streams each beside the null stream; a kernel's function on GPU d is 0x1000 + d
static int current = 0, lookups = 0;
static hipError_t last = hipSuccess, lookup_gives = hipSuccess, stream_gives = hipSuccess;
static std::string launched;
static hipError_t done(hipError_t e) { return e == hipSuccess ? e : last = e; }
static int device_of(hipStream_t s) { return (uintptr_t)s < 0x10 ? current : (int)((uintptr_t)s >> 8); }
static hipStream_t stream(int device, int n) { return (hipStream_t)((uintptr_t)device << 8 | 0x10u | (unsigned)n); }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { *d = device_of(s); return done(stream_gives); }
hipError_t hipGetFuncBySymbol(hipFunction_t *f, const void *) {
    ++lookups;
    if (lookup_gives == hipSuccess) *f = (hipFunction_t)(uintptr_t)(0x1000 + current);
    return done(lookup_gives);
}
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t s, void **, void **extra) {
    const int of = (int)(uintptr_t)f - 0x1000;
    const uint8_t *block = (const uint8_t *)extra[1];
    launched = of == device_of(s) && *(const size_t *)extra[3] == 16 && *(const int *)block == 7 && *(const double *)(block + 8) == 0.5
                   ? "function of " + std::to_string(of) : "another device's function";
    return done(of == device_of(s) ? hipSuccess : hipErrorInvalidDevice);
}
// (of hipLaunchKernelGGL) the runtime finds the function of the stream's device
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) { launched = "symbol on " + std::to_string(device_of(s)); return hipSuccess; }
}
// (a kernel's address is that of a word which holds the host function's)
static void (*host_function)(int, double) = [](int, double) {};
static void (*const kernel)(int, double) = reinterpret_cast<void (*)(int, double)>(&host_function);

static void expect(const char *what, const std::string &launch, hipError_t error, hipStream_t s, ixh::LaunchHandle &handle) {
    launched = "nothing";
    ixh::launch_packed(handle, kernel, dim3(1), dim3(64), 0, s, 7, 0.5);
    const hipError_t e = hipGetLastError();
    if (launched != launch || e != error) std::printf("%s: %s, error %d, not %s, error %d\n", what, launched.c_str(), (int)e, launch.c_str(), (int)error);
}

int main() {
    ixh::LaunchHandle handle;
    expect("null stream", "function of 0", hipSuccess, nullptr, handle);
    expect("its own stream", "function of 0", hipSuccess, stream(0, 1), handle);
    expect("a stream of another device", "symbol on 1", hipSuccess, stream(1, 1), handle);
    if (lookups != 1) std::printf("%d look-ups\n", lookups);
    current = 1;
    expect("null stream of the other device", "function of 1", hipSuccess, nullptr, handle);
    expect("that device's stream", "function of 1", hipSuccess, stream(1, 2), handle);
    expect("back to a stream of the first", "symbol on 0", hipSuccess, stream(0, 2), handle);
    expect("the null stream by its other name", "function of 1", hipSuccess, hipStreamLegacy, handle);
    expect("the thread's stream", "function of 1", hipSuccess, hipStreamPerThread, handle);
    if (lookups != 2) std::printf("%d look-ups\n", lookups);
    current = 16;
    expect("a device without a handle", "symbol on 16", hipSuccess, nullptr, handle);
    current = 0;
    ixh::LaunchHandle fresh;
    lookup_gives = hipErrorInvalidSymbol;
    expect("a look-up that fails", "symbol on 0", hipSuccess, nullptr, fresh);
    lookup_gives = hipSuccess;
    expect("and is tried again", "function of 0", hipSuccess, nullptr, fresh);
    stream_gives = hipErrorContextIsDestroyed;
    expect("a stream whose device is not told", "symbol on 0", hipSuccess, stream(0, 1), fresh);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
def test_launches_go_to_the_device_of_the_stream(tmp_path):
    """The kept function is the one of the stream's device, else the launch is by symbol, which the runtime resolves; no error of a look-up
    is left for the caller, who asks for the launch's."""
    (tmp_path / "launch.hip").write_text(PROGRAM)
    subprocess.check_call([HIPCC, "-std=c++17", "-O1", "-fPIC", "--offload-host-only", "--offload-arch=gfx950", "-I", CSRC, "-c", str(tmp_path / "launch.hip"), "-o", str(tmp_path / "launch.o")])
    subprocess.check_call(["g++", str(tmp_path / "launch.o"), "-o", str(tmp_path / "launch")])
    assert subprocess.run([str(tmp_path / "launch")], capture_output=True, text=True, check=True).stdout == ""
