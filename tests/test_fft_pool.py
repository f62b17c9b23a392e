"""The pool of FFT plans on the CPU: csrc/fftplan.{h,hip} compiled against a
stand-in FFT library that counts its plans.  A plan belongs to one user at a
time, at most 8 unused ones are kept, an error destroys its plan, work areas go
with their user, and the last context takes every unused plan with it, each on
its own device."""
import os
import shutil
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cosmograph_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstddef>
#include <string>
typedef int hipError_t; typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0;
extern int cur_dev, live_work, fail_malloc;
inline hipError_t hipSetDevice(int d) { cur_dev = d; return 0; }
inline hipError_t hipGetDevice(int* d) { *d = cur_dev; return 0; }
inline hipError_t hipMalloc(void** p, size_t) { if (fail_malloc) return 2; *p = new char; ++live_work; return 0; }
inline hipError_t hipFree(void* p) { delete (char*)p; --live_work; return 0; }
inline const char* hipGetErrorString(hipError_t) { return "error"; }
enum { CG_OK = 0, CG_ERR_HIP = -2 };
struct P { int device, nx, ny, nz; };
struct cg_ctx { P p; std::string err; };
namespace cg {
inline int fail(cg_ctx* c, int code, const std::string& m) { c->err = m; return code; }
}
#define HIPCHK(ctx, expr) do { if ((expr) != hipSuccess) return cg::fail(ctx, CG_ERR_HIP, #expr); } while (0)
"""

HIPFFT = r"""
#pragma once
#include <cstddef>
typedef int hipfftHandle; typedef int hipfftResult; typedef int hipfftType;
constexpr hipfftResult HIPFFT_SUCCESS = 0;
constexpr hipfftType HIPFFT_D2Z = 1, HIPFFT_Z2D = 2;
struct hipfftDoubleComplex { double x, y; };
extern int made, fail_make, plan_dev[1000]; extern bool alive[1000];
extern int live_plans, wrong_dev, cur_dev;
inline hipfftResult hipfftCreate(hipfftHandle* h) { *h = made; plan_dev[made] = cur_dev; alive[made++] = true; ++live_plans; return 0; }
inline hipfftResult hipfftDestroy(hipfftHandle h) { if (!alive[h]) return 1; alive[h] = false; wrong_dev += plan_dev[h] != cur_dev; --live_plans; return 0; }
inline hipfftResult hipfftSetAutoAllocation(hipfftHandle, int) { return 0; }
inline hipfftResult hipfftMakePlan3d(hipfftHandle, int, int, int, hipfftType, size_t* b) { *b = 64; return fail_make; }
inline hipfftResult hipfftSetWorkArea(hipfftHandle, void*) { return 0; }
inline hipfftResult hipfftSetStream(hipfftHandle, void*) { return 0; }
inline hipfftResult hipfftExecD2Z(hipfftHandle, double*, hipfftDoubleComplex*) { return 0; }
inline hipfftResult hipfftExecZ2D(hipfftHandle, hipfftDoubleComplex*, double*) { return 0; }
"""

MAIN = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "fftplan.h"
int cur_dev = 0, live_work = 0, fail_malloc = 0, made = 0, fail_make = 0, live_plans = 0, wrong_dev = 0;
int plan_dev[1000]; bool alive[1000];
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (plans %d, work %d)\n", __LINE__, #x, live_plans, live_work); return 1; } } while (0)
int main() {
  using namespace cg;
  cg_ctx c{{0, 8, 8, 8}, ""};
  fft_pool_enter();
  { FftPlan a, b; CHECK(a.take(&c, HIPFFT_D2Z, 0) == 0 && b.take(&c, HIPFFT_D2Z, 0) == 0); CHECK(made == 2 && live_work == 2); }
  CHECK(live_plans == 2 && live_work == 0);
  { FftPlan a, b; CHECK(a.take(&c, HIPFFT_D2Z, 0) == 0 && b.take(&c, HIPFFT_Z2D, 0) == 0); CHECK(made == 3); }
  for (int n = 10; n < 30; ++n) { c.p.nx = n; FftPlan a; CHECK(a.take(&c, HIPFFT_D2Z, 0) == 0); }
  CHECK(live_plans == 8 && live_work == 0);
  // an error leaves no plan or work area behind
  c.p.nx = 40;
  { FftPlan a; fail_make = 1; CHECK(a.take(&c, HIPFFT_D2Z, 0) == CG_ERR_HIP); fail_make = 0; }
  { FftPlan a; fail_malloc = 1; CHECK(a.take(&c, HIPFFT_D2Z, 0) == CG_ERR_HIP); fail_malloc = 0; }
  CHECK(live_plans == 8 && live_work == 0);
  // a second context on another device; the first to go takes nothing
  cg_ctx d{{1, 8, 8, 8}, ""};
  fft_pool_enter();
  cur_dev = 1;
  { FftPlan a; CHECK(a.take(&d, HIPFFT_D2Z, 0) == 0); }
  cur_dev = 0;
  fft_pool_leave();
  CHECK(live_plans == 8);
  wrong_dev = 0;
  fft_pool_leave();
  CHECK(live_plans == 0 && live_work == 0 && wrong_dev == 0 && cur_dev == 0);
  // ... and it starts again
  fft_pool_enter();
  { FftPlan a; CHECK(a.take(&c, HIPFFT_D2Z, 0) == 0); }
  CHECK(live_plans == 1);
  fft_pool_leave();
  CHECK(live_plans == 0);
  // contexts of several threads
  std::vector<std::thread> t;
  for (int q = 0; q < 6; ++q) t.emplace_back([] { for (int k = 0; k < 2000; ++k) { fft_pool_enter(); fft_pool_leave(); } });
  for (auto& x : t) x.join();
  CHECK(live_plans == 0);
  return 0;
}
"""


def test_pool(tmp_path):
    for sub, name, text in (("", "runtime.h", RUNTIME), ("hip", "hip_runtime.h", "#pragma once\n"), ("hipfft", "hipfft.h", HIPFFT),
                            ("", "main.cc", MAIN)):
        (tmp_path / sub).mkdir(exist_ok=True)
        (tmp_path / sub / name).write_text(text)
    shutil.copy(os.path.join(CSRC, "fftplan.h"), tmp_path)
    shutil.copy(os.path.join(CSRC, "fftplan.hip"), tmp_path / "fftplan.cc")
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(tmp_path), str(tmp_path / "main.cc"),
                    str(tmp_path / "fftplan.cc"), "-pthread", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
