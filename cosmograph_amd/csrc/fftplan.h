// fftplan.h -- hipFFT plans of the 3D real transforms, kept between calls.
//
// Making a plan loads and builds its kernels' modules: 6 to 9 ms per plan at
// every size from 64^3 to 256^3, against 0.2 ms for the 192^3 transform it
// is for.  Plans are therefore taken from a pool and put back.  A plan in use
// belongs to one FftPlan alone (its stream and work area are set on it), so
// any number of threads and streams may hold plans of one size.  The pool
// holds at most kIdlePlans unused plans of the process, the oldest is
// destroyed first, and none of them holds a work area: that is allocated by
// the FftPlan and freed with it.  Contexts are counted: with the last one the
// unused plans go too, so a program that has destroyed its contexts holds
// nothing on the device.
#pragma once
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include "runtime.h"

namespace cg {

void fft_pool_enter();  // a context begins
void fft_pool_leave();  // a context, its FftPlans put back, ends

class FftPlan {
 public:
  FftPlan() = default;
  FftPlan(const FftPlan&) = delete;
  FftPlan& operator=(const FftPlan&) = delete;
  ~FftPlan() { put_back(); }
  // a plan of the context's grid on stream s; CG_OK or an error on c
  int take(cg_ctx* c, hipfftType type, hipStream_t s);
  // back to the pool; the stream's work with it must be done
  void put_back();
  hipfftResult d2z(double* in, void* out) { return hipfftExecD2Z(h_, in, (hipfftDoubleComplex*)out); }
  hipfftResult z2d(void* in, double* out) { return hipfftExecZ2D(h_, (hipfftDoubleComplex*)in, out); }

 private:
  hipfftHandle h_ = 0;
  bool have_ = false;
  int key_[5] = {0, 0, 0, 0, 0};  // device, nx, ny, nz, type
  size_t bytes_ = 0;
  void* work_ = nullptr;
};

#define FFTCHK(ctx, expr)                                                                          \
  do {                                                                                             \
    hipfftResult r_ = (expr);                                                                      \
    if (r_ != HIPFFT_SUCCESS) return fail(ctx, CG_ERR_HIP, std::string(#expr) + ": hipFFT error " + std::to_string((int)r_)); \
  } while (0)

}  // namespace cg
