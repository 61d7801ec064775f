// afq_ham_and_overlap_dev: the local energies of caller-supplied determinants with no
// device allocation.  afq_ham_and_overlap builds a temporary population (orbitals,
// theta, overlap matrices, force bias, exchange partials, energies) in memory its
// context allocates; here that population lives in `scratch`, a
// file-scope device array of AFQ_NOALLOC_SCRATCH_BYTES that every GPU the library runs
// on holds until the process ends.  The kernels and their order are those of
// afq_ham_and_overlap, so both entry points return the same numbers.
//
// In host code `scratch` names a host-side stand-in, not device memory: its device
// address on a GPU comes from hipGetSymbolAddress, called once per device with that
// device current and kept in g_scratch; only that address reaches the kernels and the
// copies.  Every call on one GPU shares that GPU's array: calls that overlap on one GPU
// (two streams, two contexts, two host threads) race.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "afq_internal.hpp"

static __device__ __align__(256) unsigned char scratch[AFQ_NOALLOC_SCRATCH_BYTES];

namespace {

struct ScratchSlot {
  bool looked_up = false;
  unsigned char* ptr = nullptr;   // device address of `scratch` on this GPU
  std::string err;
};
std::mutex g_mu;
std::vector<ScratchSlot> g_scratch;   // indexed by device ordinal

// This GPU's scratch address (looked up on the first call on the device); nullptr with
// err set when the lookup failed.
unsigned char* scratch_on(int dev, std::string& err) {
  std::lock_guard<std::mutex> lk(g_mu);
  if ((int)g_scratch.size() <= dev) g_scratch.resize(dev + 1);
  ScratchSlot& sl = g_scratch[dev];
  if (!sl.looked_up) {
    // the lookup runs with the context's device current; the caller's current device is
    // restored afterwards
    int prev = 0;
    hipError_t e = hipGetDevice(&prev);
    if (e == hipSuccess) e = hipSetDevice(dev);
    void* p = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    const hipError_t e2 = hipSetDevice(prev);
    if (e == hipSuccess) e = e2;
    sl.looked_up = true;
    if (e != hipSuccess || !p) sl.err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
    else sl.ptr = static_cast<unsigned char*>(p);
  }
  err = sl.err;
  return sl.ptr;
}

int fail_ctx(afq_ctx* c, int code, const std::string& m) {
  c->err = m;
  return code;
}

}  // namespace

extern "C" int afq_ham_and_overlap_dev(afq_ctx* c, const double* dets_dev, int32_t ndet, int32_t nchol_ene,
                                       double* out_dev) {
  if (!c) return AFQ_ERR_ARG;
  if (!dets_dev || !out_dev || ndet <= 0) return fail_ctx(c, AFQ_ERR_ARG, "bad arguments");
  if (nchol_ene < 0 || nchol_ene > c->s.G) return fail_ctx(c, AFQ_ERR_ARG, "nchol_ene out of range");
  std::string err;
  unsigned char* base = scratch_on(c->params.device, err);
  if (!base) return fail_ctx(c, AFQ_ERR_DEVICE, err);
  afq::DevState t = afq::temporary_population(c->s, ndet, nchol_ene);
  afq::Carve size{nullptr};
  afq::carve_population(t, ndet, size);
  if (size.off > (size_t)AFQ_NOALLOC_SCRATCH_BYTES) {
    afq::Carve one{nullptr};
    afq::DevState t1 = t;
    afq::carve_population(t1, 1, one);
    return fail_ctx(c, AFQ_ERR_ARG,
                    "afq_ham_and_overlap_dev: " + std::to_string(ndet) + " determinants need " +
                        std::to_string(size.off) + " bytes of scratch; the allocation-free entry point has " +
                        std::to_string((size_t)AFQ_NOALLOC_SCRATCH_BYTES) + " (about " +
                        std::to_string((size_t)AFQ_NOALLOC_SCRATCH_BYTES / (one.off + 1024)) +
                        " determinants of this shape)");
  }
  afq::Carve cv{base};
  afq::carve_population(t, ndet, cv);
  const hipStream_t st = c->stream;
  hipError_t e = hipMemcpyAsync(t.psi, dets_dev, 2 * sizeof(double) * (size_t)ndet * t.ms, hipMemcpyDeviceToDevice, st);
  if (e != hipSuccess) return fail_ctx(c, AFQ_ERR_DEVICE, std::string("hipMemcpyAsync: ") + hipGetErrorString(e));
  afq::launch_temporary(t, st);
  e = hipGetLastError();
  if (e != hipSuccess) return fail_ctx(c, AFQ_ERR_DEVICE, std::string("ham_and_overlap_dev: ") + hipGetErrorString(e));
  e = hipMemcpyAsync(out_dev, t.ho, 4 * sizeof(double) * (size_t)ndet, hipMemcpyDeviceToDevice, st);
  if (e != hipSuccess) return fail_ctx(c, AFQ_ERR_DEVICE, std::string("hipMemcpyAsync: ") + hipGetErrorString(e));
  return AFQ_OK;
}
