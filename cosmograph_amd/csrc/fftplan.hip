// fftplan.hip -- the pool behind FftPlan (see fftplan.h).
#include "fftplan.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace cg {
namespace {

constexpr size_t kIdlePlans = 8;
struct Idle {
  int key[5];
  size_t bytes;
  hipfftHandle h;
};
std::mutex g_mu;
int g_contexts = 0;
// never destroyed: at process end the runtime may already be gone
std::vector<Idle>& idle() {
  static std::vector<Idle>* v = new std::vector<Idle>();
  return *v;
}

}  // namespace

void fft_pool_enter() {
  std::lock_guard<std::mutex> lock(g_mu);
  idle().reserve(kIdlePlans + 1);  // put_back, which a destructor calls, does not allocate
  ++g_contexts;
}

void fft_pool_leave() {
  std::vector<Idle> drop;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_contexts > 0) return;
    drop.swap(idle());
  }
  if (drop.empty()) return;
  int dev = 0;
  const bool have_dev = hipGetDevice(&dev) == hipSuccess;
  for (const Idle& e : drop) {
    (void)hipSetDevice(e.key[0]);
    (void)hipfftDestroy(e.h);
  }
  if (have_dev) (void)hipSetDevice(dev);
}

int FftPlan::take(cg_ctx* c, hipfftType type, hipStream_t s) {
  put_back();
  const int key[5] = {c->p.device, c->p.nx, c->p.ny, c->p.nz, (int)type};
  std::copy(key, key + 5, key_);
  {
    std::lock_guard<std::mutex> lock(g_mu);
    auto& v = idle();
    for (size_t q = v.size(); q-- > 0;)
      if (std::equal(key, key + 5, v[q].key)) {
        h_ = v[q].h;
        bytes_ = v[q].bytes;
        have_ = true;
        v.erase(v.begin() + (long)q);
        break;
      }
  }
  if (!have_) {
    FFTCHK(c, hipfftCreate(&h_));
    have_ = true;
    key_[0] = -1;  // destroyed, not kept, unless everything below succeeds
    FFTCHK(c, hipfftSetAutoAllocation(h_, 0));
    FFTCHK(c, hipfftMakePlan3d(h_, c->p.nx, c->p.ny, c->p.nz, type, &bytes_));
    key_[0] = c->p.device;
  }
  if (bytes_) {
    HIPCHK(c, hipMalloc(&work_, bytes_));
    FFTCHK(c, hipfftSetWorkArea(h_, work_));
  }
  FFTCHK(c, hipfftSetStream(h_, s));
  return CG_OK;
}

void FftPlan::put_back() {
  if (work_) (void)hipFree(work_);
  work_ = nullptr;
  if (!have_) return;
  have_ = false;
  hipfftHandle drop = h_;
  bool dropping = true;
  if (key_[0] >= 0) {
    std::lock_guard<std::mutex> lock(g_mu);
    auto& v = idle();
    Idle e;
    std::copy(key_, key_ + 5, e.key);
    e.bytes = bytes_;
    e.h = h_;
    v.push_back(e);
    dropping = v.size() > kIdlePlans;
    if (dropping) {
      drop = v.front().h;
      v.erase(v.begin());
    }
  }
  if (dropping) (void)hipfftDestroy(drop);
}

}  // namespace cg
