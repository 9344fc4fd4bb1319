// Schwarz integrals without any device allocation: liberi_c_schwarz_noalloc.
//
// liberi_c_schwarz allocates a device buffer (pair list, shells, primitive-pair
// records, results) and a stream per call, and frees them again; hipFree
// synchronises the whole device, which stalls every other build in flight, and
// neither call is allowed under HIP graph capture.  This variant stages the same
// data in one library-owned device array, `scratch`, and runs on the caller's
// stream.
//
// The array lives as long as the process, once per GPU the library runs on.
// Host code never passes its name to the runtime or to a kernel: its device
// address on each GPU comes from hipGetSymbolAddress, called once per device
// with that device current, and only that address is used.  Calls that
// overlap on one GPU share the array and race; callers serialise them.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "../../include/liberi_hip.h"
#include "liberi_internal.hpp"

using namespace liberi;

// The staged form takes less than the records the limit counts (16 bytes a
// pair and 32 a shell against 68 a pair) but for the exponents and
// coefficients, 16 bytes a primitive; K primitives make at least K^2/2
// primitive pairs of 64 bytes, so at the limit of 64 MiB they take at most 16
// sqrt(2^26/32) = 23 KB.
constexpr size_t kScratchBytes = (size_t)LIBERI_SCHWARZ_SCRATCH_BYTES + (32 << 10);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` per device (nullptr: not looked up yet)

// address of this device's copy of `scratch` (looked up on first use)
int scratch_address(const char *who, void **ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_last_error(LIBERI_EDEVICE, std::string(who) + ": no usable current device");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_last_error(LIBERI_EDEVICE, std::string(who) + ": hipGetSymbolAddress(scratch): " +
                                                hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return LIBERI_OK;
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

}  // namespace

extern "C" int liberi_c_schwarz_noalloc(int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                                        const int32_t *ang_mom, const int32_t *contr_num, const int32_t *sh_loc,
                                        const int32_t *atom_num, const int32_t *atom_loc, const double *exponents,
                                        const double *cs, const double *cp, const double *cd, const double *cf,
                                        const double *coords, double *schwrz_int, void *stream) {
  const char *who = "liberi_c_schwarz_noalloc";
  if (!schwrz_int) return set_last_error(LIBERI_EARG, std::string(who) + ": NULL output");
  SchwarzStage s;
  if (int rc = schwarz_stage(who, nsh, natoms, num_bas, mxgtot, ang_mom, contr_num, sh_loc, atom_num, atom_loc,
                             exponents, cs, cp, cd, cf, coords, s))
    return rc;
  // the accepted bases are those whose whole records fit: 64 bytes per shell
  // pair and per primitive pair, 12 for its index and result
  const size_t np = s.pairs.size();
  const size_t need = align256(np * sizeof(PairRec)) + align256((size_t)s.nprims * sizeof(PrimRec)) +
                      align256(np * sizeof(int32_t)) + np * sizeof(double);
  if (need > (size_t)LIBERI_SCHWARZ_SCRATCH_BYTES)
    return set_last_error(LIBERI_ESIZE, std::string(who) + ": the basis needs " + std::to_string(need) +
                                            " bytes of staging (" + std::to_string(s.pairs.size()) +
                                            " shell pairs, " + std::to_string(s.nprims) +
                                            " primitive pairs), above the fixed " +
                                            std::to_string((long long)LIBERI_SCHWARZ_SCRATCH_BYTES) +
                                            " bytes; use liberi_c_schwarz");
  if (int rc = schwarz_check_device(who)) return rc;
  void *base = nullptr;
  if (int rc = scratch_address(who, &base)) return rc;
  unsigned char *b = (unsigned char *)base;
  if (s.bytes > kScratchBytes)
    return set_last_error(LIBERI_ESIZE, std::string(who) + ": staging area");  // (cannot happen, see kScratchBytes)
  hipStream_t st = (hipStream_t)stream;
  std::vector<unsigned char> host;
  std::vector<double> out(np);
  hipError_t e = (hipError_t)schwarz_enqueue(s, b, host, st);
  if (e == hipSuccess) e = hipMemcpyAsync(out.data(), b + s.o_out, np * sizeof(double), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return set_last_error(LIBERI_EDEVICE, std::string(who) + ": " + hipGetErrorString(e));
  schwarz_scatter(s, out.data(), schwrz_int);
  return LIBERI_OK;
}
