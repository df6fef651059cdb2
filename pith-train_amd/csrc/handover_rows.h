// Query rows worth handing dS over for at 128 features, whose dQ kernel takes 512 of them per workgroup (measurements: ds_handover_pays in
// host/torch_ops.cpp). Asked there, where a call is decided on, and by the head split, which is another one where a call hands over.
#pragma once
#include <cstdint>

namespace pith {

inline bool handover_fills_device(int64_t b, int64_t sq, int64_t hq, int64_t cus) { return (sq + 511) / 512 * hq * b >= cus; }

inline bool handover_rows_pay(int64_t b, int64_t sq, int64_t hq, bool causal, int64_t cus) {
  if (sq <= 256 || (!causal && sq > 512 && sq < 640)) return false;  // few rows to a workgroup
  return handover_fills_device(b, sq, hq, cus) || (sq <= 16384 && 100 * sq * hq * b >= 69 * 512 * cus);
}

}  // namespace pith
