// The repairs of a kernels.speculate prediction with inline fallback in one
// launch (the drop-in repair, repair_fused, repair_signed, repair_signed_fused).
#pragma once

#include "common.hpp"

namespace stk {

struct SRepairArgs {
  KV kv;                                   // q, k, v, hq, hkv, n, b, d
  const void* a; int atype; int sa;        // selected [hq, sa]
  const void* p; int ptype; int sp;        // predicted [hq, sp]
  int hybrid;                              // 1: hybrid or compact prediction, 0: saved
  int sc;                                  // state rows per head (sp unless compact)
  const void* rids;                        // compact: retained IDs [hq, sc] (ptype), else null
  int split;                               // kernels.repair's guards (merged frame)
  const float* pm; const float* pl; const float* pu;   // prediction states [hq, sc(, d)]
  const uint8_t* high;                     // [hq, sp] (hybrid, compact)
  const float* lm; const float* ll;        // low group [hq] (hybrid, compact)
  const float* lu; const float* labs;      // [hq, d] (hybrid, compact)
  const float* mass_m; const float* mass_l;   // [hq, sp] (eps > 0)
  float min_remain, cancel, eps;
  void* queue; int qtype; int cap;         // [hq, cap] job queue out (null: no queue, counts)
  int32_t* pos; int32_t* total;            // [hq] job counts out
  float* out; uint8_t* bad; float* remain; // [hq, d], [hq], [hq]
  uint8_t* approx; float* extra;           // [hq] when eps > 0
};

// Whether the one-launch kernel covers the shape: bf16 / fp16, D in
// {64, 128, 256}, B a multiple of 16, SA, SP and SC <= 256, SC * D <= 32768,
// 16-byte aligned q / k / v / state rows.  It is the faster form over all of
// it, the compact instances with B = 32 at D = 256 included, whose tiles and two
// sums spill 400 to 470 bytes per lane: speculation and repair of 16 heads x 60
// slots, four layers, 1306 us in the separate launches and 393 here (30 and 120
// slots: 462 and 214, 2428 and 706; D = 128: 591 and 132; hybrid at D = 256: 299
// and 137).
bool srepair_covers(int dtype, int b, int d, int sa, int sp, int sc, uintptr_t align);

int launch_srepair(int dtype, const SRepairArgs& a, hipStream_t st);
int launch_srepair_compact(int dtype, const SRepairArgs& a, hipStream_t st);

}  // namespace stk
