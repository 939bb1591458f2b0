// ctx_probe.cpp -- state of a context that the C ABI does not show, for the
// tests (libfsph_probe.so, built beside libfsph.so from the same header).
#include "fsph_internal.h"

using fsph::Ctx;

extern "C" {

// Candidate capacity and stack tier of the gather tiles.
int64_t fsph_probe_gather(const fsph_ctx *ctx, int64_t out[2]) {
  const Ctx *c = reinterpret_cast<const Ctx *>(ctx);
  out[0] = c->gccap;
  out[1] = c->stack_tier[1];
  return 0;
}

// Whether a scan's stall is on record; set: records one first.
int64_t fsph_probe_scan_stall(const fsph_ctx *ctx, int set) {
  const Ctx *c = reinterpret_cast<const Ctx *>(ctx);
  int *word = c->flags.as<int>() + fsph::kScanWord, v = fsph::kFlagScanStall;
  if (set && hipMemcpy(word, &v, sizeof(v), hipMemcpyHostToDevice)) return -1;
  if (hipMemcpy(&v, word, sizeof(v), hipMemcpyDeviceToHost)) return -1;
  return v == fsph::kFlagScanStall;
}

// Bytes of the scratch buffer that the reductions share.
int64_t fsph_probe_scratch_bytes(const fsph_ctx *ctx) {
  return (int64_t) reinterpret_cast<const Ctx *>(ctx)->red_tmp.bytes;
}

// Whether the sort takes all key bits.
int64_t fsph_probe_sort_full(const fsph_ctx *ctx) {
  return reinterpret_cast<const Ctx *>(ctx)->sort_full;
}

}  // extern "C"
