// tanh of a bf16 argument by table: gelu_approx's tanh always sees a value
// rounded to bf16 (src/ming_fused.zig:232-235 rounds c1 * inner before the
// tanh), so f32 tanh(u) for every bf16 u in [0, 16] -- 0x4181 bit patterns,
// 67 KB -- covers it, with tanh(-u) = -tanh(u), and tanh(u) rounding to 1 in
// f32 from u = 9.0625 on.  The entries are (float)tanh((double)u), computed on
// the host in double precision and rounded once: the CPU restatement
// evaluates that expression itself, so kernel and restatement agree bit for
// bit, for one table load instead of a double-precision tanh per element.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ming {

constexpr int kTanhTabN = 0x4181;  // bf16 bits 0x0000 .. 0x4180: +0 .. 16

// tanh(u) for a bf16-valued f32 u; NaN stays NaN, +-inf and |u| > 16 give +-1.
__device__ __forceinline__ float tanh_bf16(const float* __restrict__ tab, float u) {
    const uint32_t b = __float_as_uint(u) >> 16;  // exact: u is a bf16 value
    const uint32_t m = b & 0x7fffu;
    const float t = m < (uint32_t)kTanhTabN ? tab[m] : (m > 0x7f80u ? u : 1.0f);
    return (b & 0x8000u) ? -t : t;
}

// The same from an entry loaded beforehand: e = tab[min(m, kTanhTabN - 1)].
__device__ __forceinline__ float tanh_bf16_of(float e, float u) {
    const uint32_t b = __float_as_uint(u) >> 16, m = b & 0x7fffu;
    const float t = m < (uint32_t)kTanhTabN ? e : (m > 0x7f80u ? u : 1.0f);
    return (b & 0x8000u) ? -t : t;
}

// The table on the host (computed once).
const float* tanh_table_host();

// Per kernel file: upload into that file's device array (current device).
hipError_t tanh_upload_dit(const float* host);
hipError_t tanh_upload_dit_batch(const float* host);
hipError_t tanh_upload_cfmp(const float* host);

}  // namespace ming
