// gd_noalloc.hip -- gd_energy_eval_noalloc: the energy of arbitrary poses with
// no allocation at all, for callers that cannot allocate device memory
// (code under HIP graph capture, tight serving loops, harnesses that forbid
// it).  The kernels' scratch -- the evaluation's copy of the job struct, its
// poses, transformed ligands and partial sums -- lives in one file-scope device
// array of GD_NOALLOC_SCRATCH_BYTES, held by every GPU the library runs on until
// the process ends.
//
// Same kernels and the same tiling as gd_energy_eval, so the results are the
// same bits.  Poses run in passes of whole 64-lane blocks that fit the scratch
// and the device's host buffer for inputs and results, which was made with its
// first job (without it they are copied).  Every call on a GPU shares both: calls
// that overlap on one GPU race (the scratch keeps the last call's contents).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/geauxdock_amd.h"
#include "gd_device.h"
#include "gd_internal.h"

#define GD_NOALLOC_MAX_DEVICES 64

static __device__ __align__(256) unsigned char scratch[GD_NOALLOC_SCRATCH_BYTES];

namespace {

// The device address of `scratch` on each device, from hipGetSymbolAddress
// with that device current (each GPU holds its own copy of the array).
void *g_scratch[GD_NOALLOC_MAX_DEVICES];
std::mutex g_scratch_mu;

gd_status scratch_ptr(void **out) {
  const int dev = gdr::device();
  if (dev < 0 || dev >= GD_NOALLOC_MAX_DEVICES) return GD_ERR_STATE;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return gdr::hip_fail(e, "hipGetSymbolAddress(scratch)");
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return GD_OK;
}

// The scratch a one-block evaluation is held to: its buffers, and room for its
// work items, inputs and results.
size_t one_block_bytes(const GdJob &g) {
  const auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  return gdr::eval_carve(g, 1, nullptr, nullptr) + up((size_t)g.nL * g.nG * sizeof(GdItem)) + up(64 * 2 * 4) +
         up(64 * 6 * 4) + up(64 * 10 * 4) + up(64 * 9 * 4);
}

}  // namespace

extern "C" gd_status gd_energy_eval_noalloc(gd_job *j, int n, const int *conf, const float *pose,
                                            float *terms, float *raw) {
  if (!j || n < 0 || (n > 0 && (!conf || !pose || !terms))) return GD_ERR_ARG;
  if (n == 0) return GD_OK;
  gd_status st = gdr::ensure_device();
  if (st != GD_OK) return st;
  const GdJob &g = j->h;
  for (int i = 0; i < n; ++i)
    if (conf[2 * i] < 0 || conf[2 * i] >= g.n_lig || conf[2 * i + 1] < 0 || conf[2 * i + 1] >= g.n_prt)
      return GD_ERR_ARG;
  void *base = nullptr;
  if ((st = scratch_ptr(&base)) != GD_OK) return st;
  float *host = gdr::noalloc_host();
  if (one_block_bytes(g) > (size_t)GD_NOALLOC_SCRATCH_BYTES) {
    char buf[200];
    std::snprintf(buf, sizeof buf,
                  "gd_energy_eval_noalloc: one 64-pose block of this job needs %zu bytes of scratch, "
                  "more than the %d-byte static workspace",
                  one_block_bytes(g), (int)GD_NOALLOC_SCRATCH_BYTES);
    gdr::set_error(buf);
    return GD_ERR_SIZE;
  }
  // blocks of a pass: as many as fit the scratch and the host buffer
  int nb = (int)(gdr::kNoallocHostBytes / (64 * gdr::kEvalHostWords * sizeof(float)));
  if (nb > (n - 1) / 64 + 1) nb = (n - 1) / 64 + 1;
  // without a host buffer (there was no memory for it) inputs and results are copied
  // through the scratch
  const auto pass_bytes = [&](int k) {
    return gdr::eval_carve(g, k, nullptr, nullptr) + (host ? 0 : (size_t)k * 64 * gdr::kEvalHostWords * sizeof(float));
  };
  while (pass_bytes(nb) > (size_t)GD_NOALLOC_SCRATCH_BYTES) --nb;  // one block fits
  float *dev = host ? nullptr : (float *)((char *)base + gdr::eval_carve(g, nb, nullptr, nullptr));
  gdr::EvalBufs b;
  gdr::eval_carve(g, nb, (char *)base, &b);
  for (int at = 0; at < n && st == GD_OK; at += nb * 64) {
    const int cnt = n - at < nb * 64 ? n - at : nb * 64;
    st = gdr::eval_pass(j, b, cnt, conf + 2 * (size_t)at, pose + 6 * (size_t)at, terms + 10 * (size_t)at,
                        raw ? raw + 9 * (size_t)at : nullptr, host, dev);
  }
  return st;
}
