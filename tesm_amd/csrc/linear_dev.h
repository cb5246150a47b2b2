// Device helpers shared by the BitLinear product kernels (bitlinear.hip, mfma32.hip).
#pragma once

#include <algorithm>

#include "tesm_hip_internal.h"

namespace tesm {

typedef int v16i __attribute__((ext_vector_type(16)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t unpack_u(uint32_t w, int s) { return (w >> (2 * s)) & 0x03030303u; }

__device__ __forceinline__ v4i unpack_frag(uint32_t w) {
  return v4i{static_cast<int>(unpack_u(w, 0)), static_cast<int>(unpack_u(w, 1)), static_cast<int>(unpack_u(w, 2)),
             static_cast<int>(unpack_u(w, 3))};
}

// Tile order for a 1-D grid: workgroups are handed to the 8 XCDs round-robin by id, so id is
// mapped to a tile such that each XCD gets a contiguous run of tiles (row-major over
// (M tile, N tile)); consecutive tiles of one XCD share A rows in that XCD's L2.
template <int GM>
__device__ __forceinline__ void xcd_tile_of(int64_t pid, int64_t ntm, int64_t ntn, int64_t& tm, int64_t& tn) {
  constexpr int64_t kXcd = 8;
  const int64_t total = ntm * ntn;
  const int64_t x = pid % kXcd, i = pid / kXcd;
  const int64_t q = total / kXcd, r = total % kXcd;
  const int64_t tile = x * q + (x < r ? x : r) + i;
  // groups of GM M-tile rows with M fastest: the tiles an XCD runs at once cover a few M rows
  // and N columns, so both operands' K slabs are shared through its L2
  constexpr int64_t kGroupM = GM;
  const int64_t g = tile / (kGroupM * ntn);
  const int64_t first_m = g * kGroupM;
  const int64_t gsz = ntm - first_m < kGroupM ? ntm - first_m : kGroupM;
  const int64_t local = tile - g * kGroupM * ntn;
  tm = first_m + local % gsz;
  tn = local / gsz;
}

// With the weights as the A operand, element r of lane L's accumulator is output row L%16 and
// output column 4*(L/16) + r of the 16 x 16 tile.
template <int OUT_DT>
__device__ __forceinline__ void store4(void* out, int64_t idx, const float (&v)[4], bool vec) {
  if (vec) {
    if constexpr (OUT_DT == kBF16) {
      const uint32_t lo = pack_bf16x2(v[0], v[1]);
      const uint32_t hi = pack_bf16x2(v[2], v[3]);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + idx) = make_uint2(lo, hi);
    } else {
      *reinterpret_cast<float4*>(static_cast<float*>(out) + idx) = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) st<OUT_DT>(out, idx + r, v[r]);
  }
}

// 4-element vector access at element (m * ld + n) is aligned for every m and every n % 4 == 0.
template <int DT>
__device__ __forceinline__ bool vec4_ok(const void* p, int64_t ld) {
  constexpr int64_t bytes = DT == kBF16 ? 8 : 16;
  return (reinterpret_cast<uintptr_t>(p) % bytes) == 0 && (ld * (DT == kBF16 ? 2 : 4)) % bytes == 0;
}

// Two-product epilogues on the rounded products p0 = rnd(v0), p1 = rnd(v1):
//   output gate  y = rnd(rnd(local + rnd(sigmoid(gate) * p0)) + p1)      (tesm.py:1256-1261)
//   SwiGLU       h = rnd(rnd(silu(p0)) * p1), silu(x) = x * sigmoid(x)  (mixer_seq_simple.py:63-64)
template <int EPI, int OUT_DT>
__device__ __forceinline__ float dual_epi(float p0, float p1, float local, float gate) {
  if constexpr (EPI == kEpiOutputGate) {
    const float g = rnd<OUT_DT>(sigmoidf_(gate));
    return rnd<OUT_DT>(rnd<OUT_DT>(local + rnd<OUT_DT>(g * p0)) + p1);
  } else {
    return rnd<OUT_DT>(rnd<OUT_DT>(p0 * sigmoidf_(p0)) * p1);
  }
}

// kEpiGates: the region of the 32-column tile that starts at column n (0: stored as is, 1: tanh,
// 2: biased sigmoid, 3: sigmoid).  act_n0 and act_w are multiples of 32, so a tile lies in one region
// and the region is uniform over the wave.
__device__ __forceinline__ int gate_region(const LinearArgs& a, int64_t n) {
  const int64_t r = n - a.act_n0;
  return r < 0 ? 0 : r < a.act_w ? 1 : r < 2 * a.act_w ? 2 : r < 3 * a.act_w ? 3 : 0;
}

// The MIMO gates on four consecutive columns n .. n + 3 of one region (tesm_mimo.py:958-961), each
// on the product rounded to the output dtype: the float ops a scan would apply to the stored
// products, so the values it reads are the ones it would have computed.
template <int DT>
__device__ __forceinline__ void gate_act4(const LinearArgs& a, int kind, int64_t n, float (&v)[4]) {
  if (kind == 1) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = rnd<DT>(tanhf_(rnd<DT>(v[r])));
  } else if (kind == 2) {
    const int64_t c = n - a.act_n0 - a.act_w;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = rnd<DT>(sigmoidf_(rnd<DT>(rnd<DT>(v[r]) + ld<DT>(a.act_bias, c + r))));
  } else if (kind == 3) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = rnd<DT>(sigmoidf_(rnd<DT>(v[r])));
  }
}

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding: vmcnt bits [3:0] and
// [15:14], expcnt [6:4] and lgkmcnt [11:8] left at their maxima)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Compute units and LDS bytes per workgroup of the current device (queried once per device).
struct DeviceLimits {
  int cus = 0;
  int64_t lds = 0;
};
DeviceLimits device_limits();

// Products of more than 32 rows, and wide ones of up to 32, on v_mfma_i32_32x32x32_i8 (mfma32.hip);
// operands and epilogue are checked by launch_linear.
int launch_mfma32(const LinearArgs& a, hipStream_t st);

}  // namespace tesm
