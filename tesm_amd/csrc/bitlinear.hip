// INT2 x INT8 BitLinear products for gfx950.
//
// Reference semantics (tesm_ssm/modules/tesm.py:238-290, torch branch):
//   y = F.linear(q_x / s_x, q_w / s_w) with q_x int8 per-token codes and q_w ternary codes.
// Here the contraction is done exactly in int32 on the codes and scaled once:
//   acc = sum_k q_x[m,k] * q_w[n,k];   y = acc / s_x[m] * c_w     (c_w = 1 / s_w rounded)
// Weights arrive packed (code + 1 in {0,1,2}, four per byte), so the kernels form
//   acc = sum_k q_x * u_w - sum_k q_x      (u = code + 1)
// and the per-row sum of activation codes (from the quantization kernel) removes the offset.
//
// Kernels:
//   * gemv_kernel  (M <= 4): bandwidth-bound decode path.  Each lane streams 16-byte packed
//     chunks (64 codes) with one 128-bit load, unpacks in registers with shift/and and
//     multiplies with v_dot4_i32_i8 against activation codes held in registers.
//   * skinny_kernel / skinny_fq_kernel (M <= 32): 16x16x64 int8 MFMA with the K loop split over a workgroup's
//     waves, operands straight from memory.
//   * the 32x32x32 kernels of mfma32.hip (M > 32).
//   * the output gate's row kernels (gate32_kernel, gate_rowq_lds_kernel, gate_rowq_kernel).
#include <cstdlib>

#include "linear_dev.h"

namespace tesm {

namespace {

// ---------------------------------------------------------------------------
// GEMV
// ---------------------------------------------------------------------------
// RPG: output rows per lane group (independent loads in flight per lane).
template <int LPR, int MR, int NCH, int OUT_DT, int RPG = 4>
__global__ __launch_bounds__(256) void gemv_kernel(LinearArgs a) {
  constexpr int GPW = 64 / LPR;   // lane groups per wave
  const LinearOperand& o = a.op[0];
  const int lane = threadIdx.x & 63;
  const int g = lane & (LPR - 1);
  const int64_t group = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * GPW + lane / LPR;
  const int64_t n0 = group * RPG;
  if (n0 >= a.N) return;
  const int64_t nch = a.Kp / 64;

  // the epilogue's operands first, from clamped indices (raw bits, converted where used): requested
  // after the products they would each cost one more memory round trip at the end of the kernel
  float sxv[MR];
  int32_t rsv[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    const int64_t mc = m < a.M ? m : a.M - 1;
    sxv[m] = o.s_x[mc];
    rsv[m] = o.rowsum[mc];
  }
  float cwv[RPG];
  uint32_t bias_bits[RPG];
  const void* bias_src = a.bias ? a.bias : static_cast<const void*>(o.c_w);  // a valid address either way
#pragma unroll
  for (int r = 0; r < RPG; ++r) {
    const int64_t nc = n0 + r < a.N ? n0 + r : a.N - 1;
    cwv[r] = o.c_w[o.c_w_per_row ? nc : 0];
    bias_bits[r] = ld_bits<OUT_DT>(bias_src, a.bias ? nc : 0);
  }

  // unconditional loads from clamped rows / chunks (masked afterwards): all in flight at once
  uint4 W[RPG][NCH];
#pragma unroll
  for (int r = 0; r < RPG; ++r) {
    const int64_t n = n0 + r;
    const int64_t nc = n < a.N ? n : a.N - 1;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int64_t c = g + LPR * i;
      const int64_t cc = c < nch ? c : nch - 1;
      // rows past N only feed outputs that are never stored; chunks past the row are masked at use
      W[r][i] = *reinterpret_cast<const uint4*>(o.w + nc * o.ldw + 16 * cc);
    }
  }
  uint32_t X[MR][NCH][16];
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    const int64_t mc = m < a.M ? m : a.M - 1;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int64_t c = g + LPR * i;
      const int64_t cc = c < nch ? c : nch - 1;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint4 v = *reinterpret_cast<const uint4*>(o.q + mc * o.ldq + 64 * cc + 16 * d);
        X[m][i][4 * d + 0] = v.x;
        X[m][i][4 * d + 1] = v.y;
        X[m][i][4 * d + 2] = v.z;
        X[m][i][4 * d + 3] = v.w;
      }
    }
  }
  // the row scales and sums are wave-uniform (scalar loads): pinned here, while the vector loads above
  // are in flight, so the compiler does not sink them past the products into the storing lanes' branch
#pragma unroll
  for (int m = 0; m < MR; ++m) asm volatile("" : "+s"(sxv[m]), "+s"(rsv[m]));
  int acc[RPG][MR];
#pragma unroll
  for (int r = 0; r < RPG; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[r][m] = 0;

#pragma unroll
  for (int r = 0; r < RPG; ++r) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      // a lane's chunk past the end of the row contributes nothing (code 0 everywhere)
      const bool live = g + LPR * i < nch;
      const uint32_t wd[4] = {live ? W[r][i].x : 0u, live ? W[r][i].y : 0u, live ? W[r][i].z : 0u,
                              live ? W[r][i].w : 0u};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int u = static_cast<int>(unpack_u(wd[d], s));
#pragma unroll
          for (int m = 0; m < MR; ++m)
            acc[r][m] = __builtin_amdgcn_sdot4(u, static_cast<int>(X[m][i][4 * d + s]), acc[r][m], false);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RPG; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      acc[r][m] = wave_sum_i<LPR>(acc[r][m]);  // DPP / swizzle steps (integer sums: any order is exact)
    }
  // every lane forms the outputs (so the epilogue's loads are waited for here, not after the branch)
  float outv[RPG][MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    const float inv = 1.0f / sxv[m];
#pragma unroll
    for (int r = 0; r < RPG; ++r) {
      acc[r][m] -= rsv[m];
      float v = (static_cast<float>(acc[r][m]) * inv) * cwv[r];
      if (a.bias) v = v + from_bits<OUT_DT>(bias_bits[r]);
      outv[r][m] = v;
    }
  }
  if (g != 0) return;
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    if (m >= a.M) break;
#pragma unroll
    for (int r = 0; r < RPG; ++r) {
      const int64_t n = n0 + r;
      if (n >= a.N) break;
      if (a.acc_dump) a.acc_dump[m * a.N + n] = acc[r][m];
      st<OUT_DT>(a.out, m * a.ldo + n, outv[r][m]);
    }
  }
}

// General epilogue of the 16 x 16 tiles of one wave (tile rows wm*TM.., columns wn*TN..): scale the
// exact accumulators, optional bias / accumulator dump, or the output gate
// y = local + sigmoid(gate) * state_proj + ent_proj in the module dtype's op order.
// Operands of one 16·TM × 16·TN epilogue tile (activation scales and code sums, weight scales, bias,
// output-gate inputs) for the split-K kernels, read in straight-line code with rows and columns clamped into range (values
// at clamped positions are never stored), so they are all in flight together and can be issued
// before the K loop.
template <int TM, int TN, int EPI, int OUT_DT>
struct Epi16In {
  float sx0[TM], sx1[TM];  // activation scales and code sums of the lane's rows
  int32_t rs0[TM], rs1[TM];
  float cw0[TN][4], cw1[TN][4];
  uint32_t bias[TN][4];
  uint32_t lo[TM][TN][4], gt[TM][TN][4];
};

template <int TM, int TN, int EPI, int OUT_DT>
__device__ __forceinline__ void epi16_load(const LinearArgs& a, Epi16In<TM, TN, EPI, OUT_DT>& e, int64_t m0,
                                           int64_t n0, int lane) {
  const LinearOperand& o0 = a.op[0];
  const LinearOperand& o1 = a.op[1];
  const void* bias = a.bias ? a.bias : static_cast<const void*>(o0.c_w);  // no bias: a valid dummy address
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t nb = n0 + j * 16 + 4 * (lane >> 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t n = nb + r < a.N ? nb + r : a.N - 1;
      e.cw0[j][r] = o0.c_w[o0.c_w_per_row ? n : 0];
      if constexpr (epi_dual(EPI)) e.cw1[j][r] = o1.c_w[o1.c_w_per_row ? n : 0];
      if constexpr (EPI == kEpiStore) e.bias[j][r] = ld_bits<OUT_DT>(bias, a.bias ? n : 0);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + i * 16 + (lane & 15), mc = m < a.M ? m : a.M - 1;
    e.sx0[i] = o0.s_x[mc];
    e.rs0[i] = o0.rowsum[mc];
    if constexpr (epi_dual(EPI)) {
      e.sx1[i] = o1.s_x[mc];
      e.rs1[i] = o1.rowsum[mc];
    }
  }
  if constexpr (EPI == kEpiOutputGate) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t m = m0 + i * 16 + (lane & 15), mc = m < a.M ? m : a.M - 1;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t nb = n0 + j * 16 + 4 * (lane >> 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t n = nb + r < a.N ? nb + r : a.N - 1;
          e.lo[i][j][r] = ld_bits<OUT_DT>(a.local, mc * a.ld_local + n);
          e.gt[i][j][r] = ld_bits<OUT_DT>(a.gate, mc * a.ld_gate + n);
        }
      }
    }
  }
}

// The split-K kernels' epilogue (one wave owns the whole tile) on operands read by epi16_load.
template <int TM, int TN, int EPI, int OUT_DT>
__device__ __forceinline__ void epilogue16_pre(const LinearArgs& a, const v4i (&acc0)[TM][TN],
                                               const v4i (&acc1)[TM][TN], const Epi16In<TM, TN, EPI, OUT_DT>& e,
                                               int64_t m0, int64_t n0, int lane) {
  const bool vout = vec4_ok<OUT_DT>(a.out, a.ldo);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + i * 16 + (lane & 15);
    if (m >= a.M) continue;
    const float inv0 = 1.0f / e.sx0[i];
    const int32_t rs0 = e.rs0[i];
    float inv1 = 0.0f;
    int32_t rs1 = 0;
    if constexpr (epi_dual(EPI)) {
      inv1 = 1.0f / e.sx1[i];
      rs1 = e.rs1[i];
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t nb = n0 + j * 16 + 4 * (lane >> 4);
      if (nb >= a.N) continue;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t n = nb + r;
        const int32_t a0 = acc0[i][j][r] - rs0;
        if (a.acc_dump && n < a.N) a.acc_dump[m * a.N + n] = a0;
        const float v0 = (static_cast<float>(a0) * inv0) * e.cw0[j][r];
        if constexpr (EPI == kEpiStore) {
          v[r] = a.bias ? v0 + from_bits<OUT_DT>(e.bias[j][r]) : v0;
        } else {
          const float v1 = rnd<OUT_DT>((static_cast<float>(acc1[i][j][r] - rs1) * inv1) * e.cw1[j][r]);
          if constexpr (EPI == kEpiOutputGate)
            v[r] = dual_epi<EPI, OUT_DT>(rnd<OUT_DT>(v0), v1, from_bits<OUT_DT>(e.lo[i][j][r]),
                                         from_bits<OUT_DT>(e.gt[i][j][r]));
          else
            v[r] = dual_epi<EPI, OUT_DT>(rnd<OUT_DT>(v0), v1, 0.0f, 0.0f);
        }
      }
      if (nb + 3 < a.N) {
        store4<OUT_DT>(a.out, m * a.ldo + nb, v, vout);
      } else {
        for (int r = 0; r < 4 && nb + r < a.N; ++r) st<OUT_DT>(a.out, m * a.ldo + nb + r, v[r]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Small-M products (decode batches, M <= 16*TM): one workgroup per 16*TM x 16*TN output tile, the K
// loop split over its NW waves.  Wave w takes the 256-code blocks w, w + NW, ...; per block, lane L
// (weight column / activation row L%16, group g = L/16) reads one b128 of packed weights per column
// tile (codes 64g .. 64g+63 of the block) and four b128 of activation codes per row tile (the same
// 64 codes of its row).  In k-step s the lane feeds codes 64g + 16s .. +15 to both MFMA operands, so
// every code of the block meets its weight exactly once.  Operands come straight from global
// memory with the next block's loads issued before the current block's MFMAs; the waves' int32
// partial sums are added through LDS (exact, order-free) and wave 0 runs the epilogue.  This gives
// N/(16*TN) workgroups of NW waves instead of the LDS-staged kernel's N/64 single-stream tiles.
template <int TM, int TN>
struct SkinnyRegs {
  uint4 w[TN];      // packed weights of the block: dword s feeds k-step s
  v4i x[TM][4];     // activation codes: x[i][s] feeds k-step s of row tile i
};

template <int TM, int TN>
__device__ __forceinline__ void skinny_load(SkinnyRegs<TM, TN>& r, const uint8_t* const (&pw)[TN],
                                            const int8_t* const (&pa)[TM], int64_t kb, bool live) {
  if (live) {
#pragma unroll
    for (int j = 0; j < TN; ++j) r.w[j] = *reinterpret_cast<const uint4*>(pw[j] + 64 * kb);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) r.x[i][s] = *reinterpret_cast<const v4i*>(pa[i] + 256 * kb + 16 * s);
  } else {  // codes past Kp: zero activations contribute nothing whatever the weights
#pragma unroll
    for (int j = 0; j < TN; ++j) r.w[j] = make_uint4(0x55555555u, 0x55555555u, 0x55555555u, 0x55555555u);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) r.x[i][s] = v4i{0, 0, 0, 0};
  }
}

template <int TM, int TN>
__device__ __forceinline__ void skinny_mma(const SkinnyRegs<TM, TN>& r, v4i (&acc)[TM][TN]) {
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const uint32_t wd = s == 0 ? r.w[j].x : s == 1 ? r.w[j].y : s == 2 ? r.w[j].z : r.w[j].w;
      const v4i bf = unpack_frag(wd);
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf, r.x[i][s], acc[i][j], 0, 0, 0);
    }
}

// K loop of one wave over the blocks w, w + NW, ... of Kp (a trailing 128-code half block is read by
// groups 0 and 1 only).
template <int NW, int TM, int TN>
__device__ __forceinline__ void skinny_loop(const LinearOperand& o, int64_t M, int64_t N, int64_t m0, int64_t n0,
                                            int64_t Kp, int w, int lane, v4i (&acc)[TM][TN]) {
  const int g = lane >> 4, l16 = lane & 15;
  const uint8_t* pw[TN];
  const int8_t* pa[TM];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t n = n0 + 16 * j + l16;
    pw[j] = o.w + (n < N ? n : N - 1) * o.ldw + 16 * g;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + 16 * i + l16;
    pa[i] = o.q + (m < M ? m : M - 1) * o.ldq + 64 * g;
  }
  const int64_t nblk = (Kp + 255) / 256;
  const bool half_tail = (Kp & 255) != 0;  // last block holds 128 codes: groups 0 and 1
  auto live = [&](int64_t kb) { return kb < nblk && (!half_tail || kb + 1 < nblk || g < 2); };
  SkinnyRegs<TM, TN> r0, r1;
  int64_t kb = w;
  skinny_load<TM, TN>(r0, pw, pa, kb, live(kb));
  for (; kb < nblk; kb += 2 * NW) {
    skinny_load<TM, TN>(r1, pw, pa, kb + NW, live(kb + NW));
    skinny_mma<TM, TN>(r0, acc);
    if (kb + NW >= nblk) break;
    skinny_load<TM, TN>(r0, pw, pa, kb + 2 * NW, live(kb + 2 * NW));
    skinny_mma<TM, TN>(r1, acc);
  }
}

template <int NW, int TM, int TN, int EPI, int OUT_DT>
__device__ __forceinline__ void skinny_body(const LinearArgs& a, int64_t m0, int64_t n0) {
  constexpr int NOP = epi_dual(EPI) ? 2 : 1;
  __shared__ v4i red[(NW - 1) * NOP * TM * TN * 64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Epi16In<TM, TN, EPI, OUT_DT> ein;  // wave 0's epilogue operands, in flight during the K loop
  if (w == 0) epi16_load<TM, TN, EPI, OUT_DT>(a, ein, m0, n0, lane);
  v4i acc0[TM][TN], acc1[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc0[i][j] = v4i{0, 0, 0, 0};
      acc1[i][j] = v4i{0, 0, 0, 0};
    }
  skinny_loop<NW, TM, TN>(a.op[0], a.M, a.N, m0, n0, a.Kp, w, lane, acc0);
  if constexpr (epi_dual(EPI)) skinny_loop<NW, TM, TN>(a.op[1], a.M, a.N, m0, n0, a.Kp, w, lane, acc1);
  const int nblk = static_cast<int>((a.Kp + 255) / 256), nact = nblk < NW ? nblk : NW;  // waves with blocks
  if (w > 0 && w < nact) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        red[((((w - 1) * NOP) * TM + i) * TN + j) * 64 + lane] = acc0[i][j];
        if constexpr (NOP == 2) red[((((w - 1) * NOP + 1) * TM + i) * TN + j) * 64 + lane] = acc1[i][j];
      }
  }
  __syncthreads();
  if (w != 0) return;
  for (int src = 0; src < nact - 1; ++src)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc0[i][j] += red[(((src * NOP) * TM + i) * TN + j) * 64 + lane];
        if constexpr (NOP == 2) acc1[i][j] += red[(((src * NOP + 1) * TM + i) * TN + j) * 64 + lane];
      }
  epilogue16_pre<TM, TN, EPI, OUT_DT>(a, acc0, acc1, ein, m0, n0, lane);
}

template <int NW, int TM, int TN, int EPI, int OUT_DT>
__global__ __launch_bounds__(NW * 64) void skinny_kernel(LinearArgs a) {
  const int64_t ntn = (a.N + 16 * TN - 1) / (16 * TN);
  const int64_t tm = blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
  skinny_body<NW, TM, TN, EPI, OUT_DT>(a, tm * 16 * TM, tn * 16 * TN);
}

// The same product with the activation quantization fused (decode-size batches): the workgroup
// quantizes its 16 TM rows of x into LDS exactly as quant_act_kernel does (absmax scale per row,
// int8 codes in layout 1, code sums), then runs the split-K body on them.  Every workgroup of a row
// tile repeats the quantization (a few KB of L2 reads each) in exchange for one launch fewer.  LDS
// rows are Kp + 16 bytes apart, so the 16 rows a K-step reads fall on distinct banks.
// G > 0: a lane's at most G groups stay in registers between the amax and the code pass (one read
// of the row, all loads issued before the first use; needs VEC rows with K % 16 == 0); G == 0: the
// row is read twice.
template <int NW, int TM, int TN, int OUT_DT, int DT, bool VEC, int G>
__global__ __launch_bounds__(NW * 64) void skinny_fq_kernel(LinearArgs a, FusedQuantIn f) {
  extern __shared__ __attribute__((aligned(16))) char lds_fq[];
  constexpr int R = 16 * TM, LPR = NW * 64 / R;  // rows of the tile, lanes per row
  const int64_t ntn = (a.N + 16 * TN - 1) / (16 * TN);
  const int64_t tm = blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
  const int64_t m0 = tm * 16 * TM, n0 = tn * 16 * TN;
  const int64_t lstride = a.Kp + 16;
  int8_t* codes = reinterpret_cast<int8_t*>(lds_fq);
  float* sc_l = reinterpret_cast<float*>(lds_fq + R * lstride);
  int32_t* rs_l = reinterpret_cast<int32_t*>(sc_l + R);
  {
    const int r = threadIdx.x / LPR, g0 = threadIdx.x % LPR;  // LPR consecutive lanes per row
    const int64_t m = m0 + r, ngroups = a.Kp / 16;
    int8_t* crow = codes + r * lstride;
    if (G > 0) {
      // Straight-line code: the lane's G groups are loaded (16-byte loads, all issued before the first
      // use) from row min(m, M - 1), groups past K re-reading the row's last group; both are zeroed
      // or discarded below.  Needs 16-byte aligned rows and K % 16 == 0.
      const int64_t mc = m < a.M ? m : a.M - 1;
      float v[G > 0 ? G : 1][16];
      load_groups<DT, (G > 0 ? G : 1), LPR>(f.x, mc * f.ldx, f.K, g0, v);
      float amax = 0.0f;
#pragma unroll
      for (int gi = 0; gi < G; ++gi)
#pragma unroll
        for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[gi][i]));
      amax = wave_max<LPR>(amax);
      const bool live = m < a.M;  // rows past M: zero codes, scale 1, sum 0
      const float sc = act_scale<DT>(amax, f.eps);
      int32_t rs = 0;
#pragma unroll
      for (int gi = 0; gi < G; ++gi) {
        const int64_t g = g0 + LPR * gi;
        const uint4 c = group_codes<DT>(v[gi], sc, 1, rs);
        if (g < ngroups) *reinterpret_cast<uint4*>(crow + 16 * g) = live ? c : make_uint4(0, 0, 0, 0);
      }
      rs = wave_sum_i<LPR>(rs);
      if (g0 == 0) {
        sc_l[r] = live ? sc : 1.0f;
        rs_l[r] = live ? rs : 0;
      }
    } else if (m < a.M) {
      const int64_t base = m * f.ldx;
      float amax = 0.0f;
      for (int64_t g = g0; g < ngroups; g += LPR) {
        float v[16];
        load_group<DT, VEC>(f.x, base, f.K, g, v);
#pragma unroll
        for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
      }
      amax = wave_max<LPR>(amax);
      const float sc = act_scale<DT>(amax, f.eps);
      int32_t rs = 0;
      for (int64_t g = g0; g < ngroups; g += LPR) {
        float v[16];
        load_group<DT, VEC>(f.x, base, f.K, g, v);
        *reinterpret_cast<uint4*>(crow + 16 * g) = group_codes<DT>(v, sc, 1, rs);
      }
      rs = wave_sum_i<LPR>(rs);
      if (g0 == 0) {
        sc_l[r] = sc;
        rs_l[r] = rs;
      }
    } else {  // rows past M: zero codes (never stored)
      for (int64_t g = g0; g < ngroups; g += LPR) *reinterpret_cast<uint4*>(crow + 16 * g) = make_uint4(0, 0, 0, 0);
      if (g0 == 0) {
        sc_l[r] = 1.0f;
        rs_l[r] = 0;
      }
    }
  }
  __syncthreads();
  LinearArgs b = a;  // operand 0 now reads the LDS copy, indexed by global row as before
  b.op[0].q = codes - m0 * lstride;
  b.op[0].ldq = lstride;
  b.op[0].s_x = sc_l - m0;
  b.op[0].rowsum = rs_l - m0;
  skinny_body<NW, TM, TN, kEpiStore, OUT_DT>(b, m0, n0);
}

// ---------------------------------------------------------------------------
// Output gate over whole rows: a workgroup owns 16 rows and all N = d_model columns (NW waves side
// by side, NCT 16-column tiles each), so after y = local + sigmoid(gate)*state_proj + ent_proj it
// can quantize y per token for out_proj without writing y.  Every global operand of the epilogue
// (local, gate, s_x, rowsum) is requested before the K loop and kept as raw bits, so the whole
// workgroup's memory traffic is in flight at once; the K loop runs two k-steps per iteration on
// ping-pong registers so each MFMA group waits only for its own operands.
// ---------------------------------------------------------------------------

// Raw 32-bit words holding four consecutive epilogue values of one row: two bf16 pairs when the
// row can be read with one 8-byte load, else one word per value.
template <int DT, bool VEC>
struct EpRaw {
  static constexpr int W = (DT == kBF16 && VEC) ? 2 : 4;
};

// Columns past N read the last valid ones (their results are never stored).
template <int DT, bool VEC>
__device__ __forceinline__ void ep_load(const void* base, int64_t ld, int64_t m, int64_t nb, int64_t N,
                                        uint32_t (&raw)[EpRaw<DT, VEC>::W]) {
  if constexpr (VEC) {
    const int64_t c = nb < N ? nb : N - 4;  // N % 4 == 0
    if constexpr (DT == kBF16) {
      const v2u x = *reinterpret_cast<const v2u*>(static_cast<const uint16_t*>(base) + m * ld + c);
      raw[0] = x.x;
      raw[1] = x.y;
    } else {
      const v4i x = *reinterpret_cast<const v4i*>(static_cast<const float*>(base) + m * ld + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) raw[r] = static_cast<uint32_t>(x[r]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t c = nb + r < N ? nb + r : N - 1;
      if constexpr (DT == kBF16)
        raw[r] = static_cast<const uint16_t*>(base)[m * ld + c];
      else
        raw[r] = static_cast<const uint32_t*>(base)[m * ld + c];
    }
  }
}

template <int DT, bool VEC>
__device__ __forceinline__ float ep_get(const uint32_t (&raw)[EpRaw<DT, VEC>::W], int r) {
  if constexpr (DT == kF32) {
    return __uint_as_float(raw[r]);
  } else if constexpr (VEC) {
    return __uint_as_float((r & 1) ? (raw[r >> 1] & 0xffff0000u) : (raw[r >> 1] << 16));
  } else {
    return __uint_as_float(raw[r] << 16);
  }
}

// One k-step of both operands for the lanes' row (A: 16 code bytes) and tiles (B: a packed dword).
template <int NCT>
__device__ __forceinline__ void rowq_load(const LinearArgs& a, int64_t mc, int64_t col0, int lane, int64_t ks,
                                          v4i& x0, v4i& x1, uint32_t (&w0)[NCT], uint32_t (&w1)[NCT]) {
  const LinearOperand& o0 = a.op[0];
  const LinearOperand& o1 = a.op[1];
  const int64_t ko = 64 * ks + 16 * (lane >> 4);
  x0 = *reinterpret_cast<const v4i*>(o0.q + mc * o0.ldq + ko);
  x1 = *reinterpret_cast<const v4i*>(o1.q + mc * o1.ldq + ko);
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    const int64_t n = col0 + 16 * j + (lane & 15);
    const int64_t nc = n < a.N ? n : a.N - 1;
    w0[j] = *reinterpret_cast<const uint32_t*>(o0.w + nc * o0.ldw + ko / 4);
    w1[j] = *reinterpret_cast<const uint32_t*>(o1.w + nc * o1.ldw + ko / 4);
  }
}

template <int NCT>
__device__ __forceinline__ void rowq_mma(v4i (&acc0)[NCT], v4i (&acc1)[NCT], const v4i& x0, const v4i& x1,
                                         const uint32_t (&w0)[NCT], const uint32_t (&w1)[NCT]) {
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    acc0[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack_frag(w0[j]), x0, acc0[j], 0, 0, 0);
    acc1[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack_frag(w1[j]), x1, acc1[j], 0, 0, 0);
  }
}

// y = local + sigmoid(gate) * state_proj + ent_proj in the reference's op order (tesm.py:1256-1260),
// every op rounded to the layer dtype; entries outside the matrix are 0.  PER_ROW: c_w0 / c_w1
// index per output column, else they point at one scalar each.
template <int NCT, int DT, bool VEC, bool PER_ROW>
__device__ __forceinline__ void rowq_gate(const LinearArgs& a, const uint32_t (&lraw)[NCT][EpRaw<DT, VEC>::W],
                                          const uint32_t (&graw)[NCT][EpRaw<DT, VEC>::W], const v4i (&acc0)[NCT],
                                          const v4i (&acc1)[NCT], int32_t rs0, int32_t rs1, float inv0, float inv1,
                                          const float* c_w0, const float* c_w1, bool mok, int64_t col0, int lane,
                                          float (&y)[NCT][4]) {
  const float cws0 = c_w0[0], cws1 = c_w1[0];
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t n = col0 + 16 * j + 4 * (lane >> 4) + r;
      const int64_t nc = n < a.N ? n : a.N - 1;
      const float cw0 = PER_ROW ? c_w0[nc] : cws0;
      const float cw1 = PER_ROW ? c_w1[nc] : cws1;
      const float sp = rnd<DT>((static_cast<float>(acc0[j][r] - rs0) * inv0) * cw0);
      const float ep = rnd<DT>((static_cast<float>(acc1[j][r] - rs1) * inv1) * cw1);
      const float g = rnd<DT>(sigmoidf_(ep_get<DT, VEC>(graw[j], r)));
      const float v = rnd<DT>(rnd<DT>(ep_get<DT, VEC>(lraw[j], r) + rnd<DT>(g * sp)) + ep);
      y[j][r] = (mok && n < a.N) ? v : 0.0f;
    }
  }
}

template <int NW, int NCT, int DT, bool VEC, int NKS>
__global__ __launch_bounds__(NW * 64) void gate_rowq_kernel(LinearArgs a, RowQuant o) {
  constexpr int RW = EpRaw<DT, VEC>::W;
  extern __shared__ __attribute__((aligned(16))) char lds_rowq[];
  int8_t* codes = reinterpret_cast<int8_t*>(lds_rowq);                          // [16][ldq]
  float* red = reinterpret_cast<float*>(lds_rowq + 16 * o.ldq);                 // [16 rows][NW waves]
  int32_t* redi = reinterpret_cast<int32_t*>(red + 16 * NW);                   // [16 rows][NW waves]
  float* cwl = reinterpret_cast<float*>(redi + 16 * NW);                       // [2][N] per-row scales
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * 16;
  const int64_t col0 = static_cast<int64_t>(w) * NCT * 16;
  const LinearOperand& o0 = a.op[0];
  const LinearOperand& o1 = a.op[1];
  const int row = lane & 15;  // the activation row this lane feeds and the output row it holds
  const int64_t m = m0 + row;
  const bool mok = m < a.M;
  const int64_t mc = mok ? m : a.M - 1;
  const int64_t nks = a.Kp / 64;  // even: Kp is a multiple of 128
  const bool per_row = o0.c_w_per_row || o1.c_w_per_row;

  if (per_row) {
    for (int64_t i = tid; i < a.N; i += NW * 64) {
      cwl[i] = o0.c_w_per_row ? o0.c_w[i] : o0.c_w[0];
      cwl[a.N + i] = o1.c_w_per_row ? o1.c_w[i] : o1.c_w[0];
    }
  }
  // epilogue operands first, as raw bits: nothing waits on them before the K loop is done
  uint32_t lraw[NCT][RW], graw[NCT][RW];
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    const int64_t nb = col0 + 16 * j + 4 * (lane >> 4);
    ep_load<DT, VEC>(a.local, a.ld_local, mc, nb, a.N, lraw[j]);
    ep_load<DT, VEC>(a.gate, a.ld_gate, mc, nb, a.N, graw[j]);
  }
  const float sx0 = o0.s_x[mc], sx1 = o1.s_x[mc];
  const int32_t rs0 = o0.rowsum[mc], rs1 = o1.rowsum[mc];
  const float cws0 = o0.c_w[0], cws1 = o1.c_w[0];
  for (int64_t i = tid; i < 16 * o.ldq / 16; i += NW * 64) reinterpret_cast<uint4*>(codes)[i] = make_uint4(0, 0, 0, 0);

  v4i acc0[NCT], acc1[NCT];
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    acc0[j] = v4i{0, 0, 0, 0};
    acc1[j] = v4i{0, 0, 0, 0};
  }
  if constexpr (NKS > 0) {
    // the whole K extent at once (NKS == Kp / 64): one round trip for all of the wave's operands
    v4i x0[NKS], x1[NKS];
    uint32_t w0[NKS][NCT], w1[NKS][NCT];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) rowq_load<NCT>(a, mc, col0, lane, ks, x0[ks], x1[ks], w0[ks], w1[ks]);
    __builtin_amdgcn_sched_barrier(0);  // keep every load ahead of the first MFMA
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) rowq_mma<NCT>(acc0, acc1, x0[ks], x1[ks], w0[ks], w1[ks]);
  } else {
    v4i xa0, xa1, xb0, xb1;
    uint32_t wa0[NCT], wa1[NCT], wb0[NCT], wb1[NCT];
    rowq_load<NCT>(a, mc, col0, lane, 0, xa0, xa1, wa0, wa1);
    for (int64_t ks = 0; ks < nks; ks += 2) {
      rowq_load<NCT>(a, mc, col0, lane, ks + 1, xb0, xb1, wb0, wb1);
      rowq_mma<NCT>(acc0, acc1, xa0, xa1, wa0, wa1);
      // the last iteration re-reads k-step ks + 1 instead of branching (the values are unused)
      rowq_load<NCT>(a, mc, col0, lane, ks + 2 < nks ? ks + 2 : ks + 1, xa0, xa1, wa0, wa1);
      rowq_mma<NCT>(acc0, acc1, xb0, xb1, wb0, wb1);
    }
  }
  if (per_row) __syncthreads();

  // epilogue: lane holds row m, columns col0 + 16j + 4*(lane/16) + r
  const float inv0 = 1.0f / sx0, inv1 = 1.0f / sx1;
  float y[NCT][4];
  if (per_row)
    rowq_gate<NCT, DT, VEC, true>(a, lraw, graw, acc0, acc1, rs0, rs1, inv0, inv1, cwl, cwl + a.N, mok, col0, lane, y);
  else
    rowq_gate<NCT, DT, VEC, false>(a, lraw, graw, acc0, acc1, rs0, rs1, inv0, inv1, &cws0, &cws1, mok, col0, lane, y);
  float mx = 0.0f;
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, fabsf(y[j][r]));
  }
  if (o.y && mok) {
    const bool vout = vec4_ok<DT>(o.y, o.ldy);
#pragma unroll
    for (int j = 0; j < NCT; ++j) {
      const int64_t nb = col0 + 16 * j + 4 * (lane >> 4);
      if (vout && nb + 3 < a.N) {
        store4<DT>(o.y, m * o.ldy + nb, y[j], true);
      } else {
        for (int r = 0; r < 4 && nb + r < a.N; ++r) st<DT>(o.y, m * o.ldy + nb + r, y[j][r]);
      }
    }
  }
  // row max over the 4 lanes sharing the row, then over the NW waves
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (lane < 16) red[row * NW + w] = mx;
  __syncthreads();
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) amax = fmaxf(amax, red[row * NW + i]);
  const float sc = act_scale<DT>(amax, o.eps);
  int sum = 0;
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t n = col0 + 16 * j + 4 * (lane >> 4) + r;
      if (!mok || n >= a.N) continue;
      const int q = act_code<DT>(y[j][r], sc);
      // layout 1: element e = n % 16 = 4 * (lane / 16) + r sits at byte 4 * r + lane / 16 of its group
      codes[row * o.ldq + (n & ~static_cast<int64_t>(15)) + 4 * r + (lane >> 4)] = static_cast<int8_t>(q);
      sum += q;
    }
  }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  if (lane < 16) redi[row * NW + w] = sum;
  __syncthreads();
  if (tid < 16 && m0 + tid < a.M) {
    float am = 0.0f;
    int32_t rsum = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      am = fmaxf(am, red[tid * NW + i]);
      rsum += redi[tid * NW + i];
    }
    o.s[m0 + tid] = act_scale<DT>(am, o.eps);
    o.rs[m0 + tid] = rsum;
  }
  const int64_t chunks = o.ldq / 16;
  for (int r = w; r < 16; r += NW) {
    if (m0 + r >= a.M) continue;
    for (int64_t ck = lane; ck < chunks; ck += 64)
      reinterpret_cast<uint4*>(o.q + (m0 + r) * o.ldq)[ck] = reinterpret_cast<const uint4*>(codes + r * o.ldq)[ck];
  }
}

// ---------------------------------------------------------------------------
// Persistent output gate with both packed weight matrices resident in LDS (gfx950: 160 KB per
// workgroup).  Each workgroup stages state_proj and ent_proj once with coalesced 16-byte loads and
// then walks 16-row tiles blockIdx.x, blockIdx.x + gridDim.x, ...; the next tile's activation codes
// (one 16-byte piece per thread, staged through LDS) and local/gate operands are requested before
// the current tile is computed.
//
// Staged weight row n of operand p sits at (p * N + n) * RS bytes, RS = 16 * NKS + 16; dword
// q * NKS + ks of a row holds codes 64 ks + 16 q .. + 15, so one lane reads all its k-steps with
// wide LDS loads and a 16-lane row group covers all 64 banks once.  Activation rows are staged at
// a pitch of Kp + 16 bytes for the same reason.
// ---------------------------------------------------------------------------
template <int NKS>
struct RowqLds {
  static constexpr int RS = 16 * NKS + 16;           // staged weight row pitch
  static constexpr int ARS = 64 * NKS + 16;          // staged activation row pitch
  static constexpr int ABUF = 2 * 16 * ARS;          // one tile of both operands
};

inline int64_t rowq_lds_bytes(int64_t N, int64_t nks, int64_t ldq, int nw) {
  const int64_t stage = nks <= 4 ? 0 : 2 * N * (16 * nks + 16);  // register-resident weights for K <= 256
  return stage + 2 * 2 * 16 * (64 * nks + 16) + 16 * (ldq + 16) + 2 * 2 * 16 * nw * 4 + 2 * N * 4;
}

template <int NCT, int AC, int RW>
struct RowqIn {
  v4i ac[AC];                          // this thread's share of the tile's activation codes
  uint32_t lr[NCT][RW], gr[NCT][RW];   // raw local / gate values of the lane's row
  float sx0, sx1;
  int32_t rs0, rs1;
};

// Requests for tile t; rows past M read the last row (never stored).
template <int NW, int NCT, int NKS, int DT, int AC>
__device__ __forceinline__ void rowq_in_load(const LinearArgs& a, int64_t t, int64_t col0, int tid,
                                             RowqIn<NCT, AC, EpRaw<DT, true>::W>& in) {
  const int lane = tid & 63;
  const int64_t m0 = t * 16;
  const int64_t m = m0 + (lane & 15);
  const int64_t mc = m < a.M ? m : a.M - 1;
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    int g = tid + i * NW * 64;
    g = g < 128 * NKS ? g : 128 * NKS - 1;
    const int p = g / (64 * NKS), rem = g - p * 64 * NKS;
    const int r = rem / (4 * NKS), c = rem - r * 4 * NKS;
    const int64_t mr = m0 + r < a.M ? m0 + r : a.M - 1;
    const LinearOperand& op = a.op[0];
    const int8_t* src = p == 0 ? op.q + mr * op.ldq : a.op[1].q + mr * a.op[1].ldq;
    in.ac[i] = *reinterpret_cast<const v4i*>(src + 16 * c);
  }
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    const int64_t nb = col0 + 16 * j + 4 * (lane >> 4);
    ep_load<DT, true>(a.local, a.ld_local, mc, nb, a.N, in.lr[j]);
    ep_load<DT, true>(a.gate, a.ld_gate, mc, nb, a.N, in.gr[j]);
  }
  in.sx0 = a.op[0].s_x[mc];
  in.sx1 = a.op[1].s_x[mc];
  in.rs0 = a.op[0].rowsum[mc];
  in.rs1 = a.op[1].rowsum[mc];
}

// NKS consecutive dwords of staged LDS (16-byte aligned when NKS % 4 == 0, else 8-byte aligned).
template <int NKS>
__device__ __forceinline__ void lds_frag(const char* p, uint32_t (&f)[NKS]) {
  if constexpr (NKS % 4 == 0) {
#pragma unroll
    for (int i = 0; i < NKS / 4; ++i) {
      const v4i v = reinterpret_cast<const v4i*>(p)[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) f[4 * i + r] = static_cast<uint32_t>(v[r]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < NKS / 2; ++i) {
      const v2u v = reinterpret_cast<const v2u*>(p)[i];
      f[2 * i] = v.x;
      f[2 * i + 1] = v.y;
    }
  }
}

struct RowqShared {
  const char* wl;     // staged weights
  char* abuf;         // staged activation tile (this tile's buffer)
  int8_t* codes;      // [16][ldq]
  float* red;         // [16][NW] (this tile's buffer)
  int32_t* redi;      // [16][NW] (this tile's buffer)
  const float* cwl;   // [2][N] output scale of every column (c_w, or its one scalar repeated)
};

// Packed-weight fragments of the lane's columns for the register-resident variant (NKS <= 4).  The
// lanes of group q take the 16-code groups q NKS .. q NKS + NKS - 1 of their column (k-step ks: group
// q NKS + ks, for weights and activation codes alike), so each lane's fragments are one contiguous
// load and a column's four lanes read its packed row whole.
template <int NCT, int NKS>
struct RowqW {
  uint32_t w0[NCT][NKS], w1[NCT][NKS];
};

template <int NW, int NCT, int DT, int NKS, int AC, bool RW = false>
__device__ __forceinline__ void rowq_tile(const LinearArgs& a, const RowQuant& o, int64_t t,
                                          const RowqIn<NCT, AC, EpRaw<DT, true>::W>& in, const RowqShared& sh,
                                          int tid, const RowqW<NCT, NKS>* rw = nullptr) {
  using L = RowqLds<NKS>;
  // all in-tile indices fit 32 bits: N <= 1024 and the LDS is 160 KB
  const int N = static_cast<int>(a.N);
  const int cp = static_cast<int>(o.ldq) + 16;  // staged code row pitch (16 rows spread over all banks)
  const int lane = tid & 63, w = tid >> 6, q = lane >> 4;
  const int col0 = w * NCT * 16;
  const int row = lane & 15;
  const int64_t m0 = t * 16;

  // activation tile into LDS, then each lane's row fragments for every k-step
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    const int g = tid + i * NW * 64;
    if (g >= 128 * NKS) continue;
    const int p = g / (64 * NKS), rem = g - p * 64 * NKS;
    const int r = rem / (4 * NKS), c = rem - r * 4 * NKS;
    *reinterpret_cast<v4i*>(sh.abuf + (p * 16 + r) * L::ARS + 16 * c) = in.ac[i];
  }
  __syncthreads();
  v4i x0[NKS], x1[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int kb = RW ? 16 * (q * NKS + ks) : 64 * ks + 16 * q;  // the k-step's code group of lane group q
    x0[ks] = *reinterpret_cast<const v4i*>(sh.abuf + row * L::ARS + kb);
    x1[ks] = *reinterpret_cast<const v4i*>(sh.abuf + (16 + row) * L::ARS + kb);
  }

  // per 16-column tile: both products, then y = local + sigmoid(gate) * state_proj + ent_proj in the
  // reference's op order (tesm.py:1256-1260), every op rounded to the layer dtype.  Rows past M
  // compute finite values from clamped operands and are never stored.
  const float inv0 = 1.0f / in.sx0, inv1 = 1.0f / in.sx1;
  float y[NCT][4];
  float mx = 0.0f;
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    const int n = col0 + 16 * j + row;
    const int nc = n < N ? n : N - 1;
    uint32_t f0[NKS], f1[NKS];
    if constexpr (RW) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        f0[ks] = rw->w0[j][ks];
        f1[ks] = rw->w1[j][ks];
        // opaque copies: the unpacking below stays per tile instead of being hoisted out of the tile
        // loop as 4x as many live registers
        asm volatile("" : "+v"(f0[ks]));
        asm volatile("" : "+v"(f1[ks]));
      }
    } else {
      lds_frag<NKS>(sh.wl + nc * L::RS + q * NKS * 4, f0);
      lds_frag<NKS>(sh.wl + (N + nc) * L::RS + q * NKS * 4, f1);
    }
    v4i acc0 = v4i{0, 0, 0, 0}, acc1 = v4i{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      acc0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack_frag(f0[ks]), x0[ks], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack_frag(f1[ks]), x1[ks], acc1, 0, 0, 0);
    }
    const int nb = col0 + 16 * j + 4 * q;
    const int nbc = nb < N ? nb : N - 4;  // N % 4 == 0
    const float4 cw0 = *reinterpret_cast<const float4*>(sh.cwl + nbc);
    const float4 cw1 = *reinterpret_cast<const float4*>(sh.cwl + N + nbc);
    const float c0[4] = {cw0.x, cw0.y, cw0.z, cw0.w}, c1[4] = {cw1.x, cw1.y, cw1.z, cw1.w};
    const bool nok = nb < N;  // N % 4 == 0: the lane's 4 columns are all in range or all out
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float sp = rnd<DT>((static_cast<float>(acc0[r] - in.rs0) * inv0) * c0[r]);
      const float ep = rnd<DT>((static_cast<float>(acc1[r] - in.rs1) * inv1) * c1[r]);
      const float g = rnd<DT>(sigmoidf_(ep_get<DT, true>(in.gr[j], r)));
      const float v = rnd<DT>(rnd<DT>(ep_get<DT, true>(in.lr[j], r) + rnd<DT>(g * sp)) + ep);
      y[j][r] = nok ? v : 0.0f;
      mx = fmaxf(mx, fabsf(y[j][r]));
    }
  }
  const int64_t m = m0 + row;
  if (o.y && m < a.M) {
    const bool vout = vec4_ok<DT>(o.y, o.ldy);
#pragma unroll
    for (int j = 0; j < NCT; ++j) {
      const int nb = col0 + 16 * j + 4 * q;
      if (vout && nb < N) {
        store4<DT>(o.y, m * o.ldy + nb, y[j], true);
      } else {
        for (int r = 0; r < 4 && nb + r < N; ++r) st<DT>(o.y, m * o.ldy + nb + r, y[j][r]);
      }
    }
  }
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (lane < 16) sh.red[row * NW + w] = mx;
  __syncthreads();
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) amax = fmaxf(amax, sh.red[row * NW + i]);
  const float sc = act_scale<DT>(amax, o.eps);
  // layout 1: column n = 16 g + 4 q + r sits at byte 16 g + 4 r + q of its row
  int sum = 0;
  int8_t* crow = sh.codes + row * cp + col0 + q;
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    if (col0 + 16 * j + 4 * q >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int qv = act_code<DT>(y[j][r], sc);
      crow[16 * j + 4 * r] = static_cast<int8_t>(qv);
      sum += qv;
    }
  }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  if (lane < 16) sh.redi[row * NW + w] = sum;
  __syncthreads();
  if (tid < 16 && m0 + tid < a.M) {
    float am = 0.0f;
    int32_t rsum = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      am = fmaxf(am, sh.red[tid * NW + i]);
      rsum += sh.redi[tid * NW + i];
    }
    o.s[m0 + tid] = act_scale<DT>(am, o.eps);
    o.rs[m0 + tid] = rsum;
  }
  const int chunks = static_cast<int>(o.ldq / 16);
  for (int r = w; r < 16; r += NW) {
    if (m0 + r >= a.M) continue;
    uint4* dst = reinterpret_cast<uint4*>(o.q + (m0 + r) * o.ldq);
    const uint4* src = reinterpret_cast<const uint4*>(sh.codes + r * cp);
    for (int ck = lane; ck < chunks; ck += 64) dst[ck] = src[ck];
  }
}

// NKS <= 4 (K <= 256): each wave's packed-weight fragments (its NCT column tiles of both products, 2 NCT
// NKS dwords per lane) stay in registers for the whole kernel, read straight from global memory;
// otherwise both weight matrices are staged once per workgroup in LDS.
template <int NKS>
constexpr bool rowq_reg_weights() {
  return NKS <= 4;
}

template <int NW, int NCT, int DT, int NKS>
__global__ __launch_bounds__(NW * 64) void gate_rowq_lds_kernel(LinearArgs a, RowQuant o, int64_t ntiles) {
  using L = RowqLds<NKS>;
  constexpr bool RW = rowq_reg_weights<NKS>();
  constexpr int NT = NW * 64;
  constexpr int SB = RW ? 1 : (2 * NW * NCT * 16 * NKS + NT - 1) / NT;  // staged weight chunks per thread
  constexpr int AC = (128 * NKS + NT - 1) / NT;                          // activation chunks per thread per tile
  using In = RowqIn<NCT, AC, EpRaw<DT, true>::W>;
  extern __shared__ __attribute__((aligned(16))) char lds_rowq[];
  char* wl = lds_rowq;                                                    // [2][N][RS] (LDS weights only)
  char* abuf = wl + (RW ? 0 : 2 * a.N * L::RS);                           // [2 tiles][2][16][ARS]
  int8_t* codes = reinterpret_cast<int8_t*>(abuf + 2 * L::ABUF);          // [16][ldq + 16]
  float* red = reinterpret_cast<float*>(codes + 16 * (o.ldq + 16));       // [2 tiles][16][NW]
  int32_t* redi = reinterpret_cast<int32_t*>(red + 2 * 16 * NW);         // [2 tiles][16][NW]
  float* cwl = reinterpret_cast<float*>(redi + 2 * 16 * NW);             // [2][N]
  const int tid = threadIdx.x;
  const int64_t col0 = static_cast<int64_t>(tid >> 6) * NCT * 16;

  // weights: every load first (registers, or the LDS stage), then this workgroup's first tile, then
  // the LDS writes
  RowqW<NCT, NKS> rw;
  v4i sb[SB];
  const int64_t total = 2 * a.N * NKS;
  if constexpr (RW) {
    // lane (q, row) of column tile j: column col0 + 16 j + row, dwords q NKS .. q NKS + NKS - 1 of its row
    const int lane = tid & 63, q = lane >> 4, row = lane & 15;
#pragma unroll
    for (int j = 0; j < NCT; ++j) {
      const int64_t n = col0 + 16 * j + row, nc = n < a.N ? n : a.N - 1;
      const uint32_t* p0 = reinterpret_cast<const uint32_t*>(a.op[0].w + nc * a.op[0].ldw) + q * NKS;
      const uint32_t* p1 = reinterpret_cast<const uint32_t*>(a.op[1].w + nc * a.op[1].ldw) + q * NKS;
      if constexpr (NKS == 4) {
        const uint4 v0 = *reinterpret_cast<const uint4*>(p0), v1 = *reinterpret_cast<const uint4*>(p1);
        rw.w0[j][0] = v0.x, rw.w0[j][1] = v0.y, rw.w0[j][2] = v0.z, rw.w0[j][3] = v0.w;
        rw.w1[j][0] = v1.x, rw.w1[j][1] = v1.y, rw.w1[j][2] = v1.z, rw.w1[j][3] = v1.w;
      } else {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          rw.w0[j][ks] = p0[ks];
          rw.w1[j][ks] = p1[ks];
        }
      }
    }
  } else {
#pragma unroll
    for (int b = 0; b < SB; ++b) {
      const int64_t g = tid + static_cast<int64_t>(b) * NT;
      const int64_t gc = g < total ? g : total - 1;
      const int64_t pn = gc / NKS, c = gc - pn * NKS;  // pn = p * N + n
      const uint8_t* wp = pn < a.N ? a.op[0].w + pn * a.op[0].ldw : a.op[1].w + (pn - a.N) * a.op[1].ldw;
      sb[b] = *reinterpret_cast<const v4i*>(wp + 16 * c);
    }
  }
  RowqShared sh0, sh1;
  sh0.wl = sh1.wl = wl;
  sh0.abuf = abuf;
  sh1.abuf = abuf + L::ABUF;
  sh0.codes = sh1.codes = codes;
  sh0.red = red;
  sh1.red = red + 16 * NW;
  sh0.redi = redi;
  sh1.redi = redi + 16 * NW;
  sh0.cwl = sh1.cwl = cwl;
  In ta, tb;
  int64_t t = blockIdx.x;
  rowq_in_load<NW, NCT, NKS, DT, AC>(a, t, col0, tid, ta);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!RW) {
#pragma unroll
    for (int b = 0; b < SB; ++b) {
      const int64_t g = tid + static_cast<int64_t>(b) * NT;
      if (g >= total) continue;
      const int64_t pn = g / NKS, c = g - pn * NKS;
      uint32_t* dst = reinterpret_cast<uint32_t*>(wl + pn * L::RS) + c;
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) dst[qq * NKS] = static_cast<uint32_t>(sb[b][qq]);
    }
  }
  for (int64_t i = tid; i < a.N; i += NT) {
    cwl[i] = a.op[0].c_w_per_row ? a.op[0].c_w[i] : a.op[0].c_w[0];
    cwl[a.N + i] = a.op[1].c_w_per_row ? a.op[1].c_w[i] : a.op[1].c_w[0];
  }
  for (int64_t i = tid; i < (o.ldq + 16); i += NT) reinterpret_cast<uint4*>(codes)[i] = make_uint4(0, 0, 0, 0);
  // (the first tile's barrier after its activation staging also orders these LDS writes)

  // two tiles per iteration on ping-pong registers and LDS buffers; a prefetch past the end
  // re-reads the current tile
  for (;;) {
    const int64_t t1 = t + gridDim.x;
    rowq_in_load<NW, NCT, NKS, DT, AC>(a, t1 < ntiles ? t1 : t, col0, tid, tb);
    rowq_tile<NW, NCT, DT, NKS, AC, RW>(a, o, t, ta, sh0, tid, &rw);
    if (t1 >= ntiles) break;
    const int64_t t2 = t1 + gridDim.x;
    rowq_in_load<NW, NCT, NKS, DT, AC>(a, t2 < ntiles ? t2 : t1, col0, tid, ta);
    rowq_tile<NW, NCT, DT, NKS, AC, RW>(a, o, t1, tb, sh1, tid, &rw);
    if (t2 >= ntiles) break;
    t = t2;
  }
}

// ---------------------------------------------------------------------------
// Output gate on 32-row tiles (v_mfma_i32_32x32x32_i8).  A workgroup of NW waves owns 32 tokens and
// all N = d_model columns (wave w: NCT 32-column tiles from 32 NCT w), so it can quantize y per
// token for out_proj without writing y.  Per 32x32 product each unpacked weight dword serves 32
// tokens (twice the 16-row kernel's reuse), and the epilogue is cut to the operations the reference
// rounds (one conversion per bf16 rounding), codes written to LDS byte by byte in layout 1 (no VALU)
// and their sums formed with v_dot4 while the tile is copied out.
//
// Operands: weights are the MFMA's A operand (D rows = output columns), activation codes the B
// operand (D columns = tokens), so lane (t, h) holds token t and output columns 8 g + 4 h + r of each
// 32-column tile.  Lane half h takes the 16-code groups h NKS .. h NKS + NKS - 1 of a row (K step ks:
// group h NKS + ks, for both operands), so a lane's packed weight fragments are one contiguous read.
// ---------------------------------------------------------------------------
template <int NKS>
struct G32 {
  static constexpr int ARS = 32 * NKS + 16;  // staged activation row pitch: 16 rows span all banks
};

// bf16 local / gate are staged per wave in LDS (G32S: slab row pitch of NCT 32-column tiles)
template <int NCT>
struct G32S {
  // 16 NCT + 2 words: an odd multiple of two words, so the 32 rows of an 8-byte read hit 64 distinct banks
  static constexpr int SP = NCT * 64 + 8;
};

inline int64_t gate32_lds_bytes(int64_t Kp, int64_t ldq, int64_t nct, int nw, bool staged) {
  const int64_t slab = staged ? nw * 2 * 32 * (nct * 64 + 8) : 0;
  const int64_t codes = 32 * (ldq + 16);  // aliases the slabs when they are staged (used after them)
  return 2 * 32 * (Kp + 16) + std::max(slab, codes) + 32 * nw * 4 + 32 * 4;
}

// a and b rounded to the layer dtype
template <int DT>
__device__ __forceinline__ void rnd2(float& a, float& b) {
  a = rnd<DT>(a);
  b = rnd<DT>(b);
}

// The out_proj a 32-row output-gate workgroup runs on its own rows' y codes (gate32_kernel with NKO > 0).
struct G32Out {
  const uint8_t* w = nullptr;  // (N, ldw) packed weights, K = N
  int64_t ldw = 0;
  const float* c_w = nullptr;  // per-tensor +1 value
  void* out = nullptr;         // (M, ldo) in the output dtype
  int64_t ldo = 0;
};

// NKO > 0: out_proj (NKO K steps of 32 over y's codes, K = N) follows the gate in the same workgroup.
template <int NW, int NCT, int DT, int NKS, int NKO>
__global__ __launch_bounds__(NW * 64) void gate32_kernel(LinearArgs a, RowQuant o, G32Out op) {
  constexpr int NT = NW * 64;
  constexpr int ARS = G32<NKS>::ARS;
  constexpr int ACH = 2 * 32 * 2 * NKS;        // 16-byte chunks of both operands' activation tiles
  constexpr int AC = (ACH + NT - 1) / NT;
  constexpr int RW = EpRaw<DT, true>::W;
  static_assert(NKS % 4 == 0, "K steps come in 16-byte fragment loads");
  // bf16: each wave stages its own columns of local and gate (32 rows x NCT 32-column tiles) in LDS
  // through row-contiguous 16-byte loads, instead of one 8-byte load per lane and token row
  constexpr bool STG = DT == kBF16;
  constexpr int SP = G32S<NCT>::SP;
  constexpr int SPL = 2 * 32 * NCT * 4 / 64;   // 16-byte slab chunks per lane: 4 per column tile
  extern __shared__ __attribute__((aligned(16))) char lds_g32[];
  char* abuf = lds_g32;                                                  // [2][32][ARS]
  // in-tile indices fit 32 bits: N <= 1024
  const int cp = static_cast<int>(o.ldq) + 16;                           // staged code row pitch
  char* slabs = lds_g32 + 2 * 32 * ARS;                                  // [NW][2][32][SP] (bf16)
  int8_t* codes = reinterpret_cast<int8_t*>(slabs);                      // [32][cp], after the slabs are read
  const int region = STG ? NW * 2 * 32 * SP : 0;
  float* red = reinterpret_cast<float*>(slabs + (region > 32 * cp ? region : 32 * cp));  // [NW][32]
  int32_t* rsl = reinterpret_cast<int32_t*>(red + NW * 32);                            // [32] y code sums
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  __builtin_assume(tid < NT);
  const int h = lane >> 5, row = lane & 31;
  const int N = static_cast<int>(a.N);
  const int col0 = w * NCT * 32;
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * 32;
  const int64_t m = m0 + row, mc = m < a.M ? m : a.M - 1;  // rows past M compute from row M - 1, never stored

  // 1. every global load first, in straight-line code: packed weight fragments (lane (t, h) of column
  //    tile c: column col0 + 32 c + t, dwords h NKS .. h NKS + NKS - 1), the activation tiles, the row
  //    scales and sums, and the lane's local / gate values
  uint32_t w0[NCT][NKS], w1[NCT][NKS];
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int n = col0 + 32 * c + row, nc = n < N ? n : N - 1;
    const uint4* p0 = reinterpret_cast<const uint4*>(a.op[0].w + nc * a.op[0].ldw + h * NKS * 4);
    const uint4* p1 = reinterpret_cast<const uint4*>(a.op[1].w + nc * a.op[1].ldw + h * NKS * 4);
#pragma unroll
    for (int i = 0; i < NKS / 4; ++i) {
      const uint4 v0 = p0[i], v1 = p1[i];
      w0[c][4 * i] = v0.x, w0[c][4 * i + 1] = v0.y, w0[c][4 * i + 2] = v0.z, w0[c][4 * i + 3] = v0.w;
      w1[c][4 * i] = v1.x, w1[c][4 * i + 1] = v1.y, w1[c][4 * i + 2] = v1.z, w1[c][4 * i + 3] = v1.w;
    }
  }
  v4i ac[AC];
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    int g = tid + i * NT;
    g = g < ACH ? g : ACH - 1;
    const int p = g / (64 * NKS), rem = g - p * 64 * NKS;
    const int r = rem / (2 * NKS), c = rem - r * 2 * NKS;
    const int64_t mr = m0 + r < a.M ? m0 + r : a.M - 1;
    // operand fields selected by value (a lane-dependent choice of the struct itself would be read
    // from the kernel arguments with a vector load and a full wait)
    const int8_t* q = p == 0 ? a.op[0].q : a.op[1].q;
    const int64_t ldq = p == 0 ? a.op[0].ldq : a.op[1].ldq;
    ac[i] = *reinterpret_cast<const v4i*>(q + mr * ldq + 16 * c);
  }
  // the loads above land first: the products wait for them only, the epilogue's below stay in flight
  __builtin_amdgcn_sched_barrier(0);
  const float sx0 = a.op[0].s_x[mc], sx1 = a.op[1].s_x[mc];
  const int32_t rs0 = a.op[0].rowsum[mc], rs1 = a.op[1].rowsum[mc];
  const float cw0 = a.op[0].c_w[0], cw1 = a.op[1].c_w[0];
  uint32_t lr[NCT][4][RW], gr[NCT][4][RW];
  uint4 sg[STG ? SPL : 1];
  if constexpr (STG) {
    // column tile by column tile (the epilogue of tile c needs only its own chunks): chunk i = 4 c + q
    // of a lane is operand q / 2 (local, gate), row (lane + 64 (q % 2)) / 4, 16-byte chunk lane % 4
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
      const int c = i / 4, q = i % 4;
      const int r = (lane >> 2) + 16 * (q & 1);
      const int64_t mr = m0 + r < a.M ? m0 + r : a.M - 1;
      const int cb = col0 + 32 * c + 8 * (lane & 3);
      const int col = cb < N ? cb : N - 8;  // columns past N: never stored
      if (q < 2)
        sg[i] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.local) + mr * a.ld_local + col);
      else
        sg[i] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.gate) + mr * a.ld_gate + col);
    }
  } else {
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int64_t nb = col0 + 32 * c + 8 * g + 4 * h;
        ep_load<DT, true>(a.local, a.ld_local, mc, nb, a.N, lr[c][g]);
        ep_load<DT, true>(a.gate, a.ld_gate, mc, nb, a.N, gr[c][g]);
      }
  }
  __builtin_amdgcn_sched_barrier(0);

  // 2. activation tiles into LDS; the code tile's padding columns [N, ldq) are zero
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    const int g = tid + i * NT;
    if (ACH % NT != 0 && g >= ACH) continue;
    const int p = g / (64 * NKS), rem = g - p * 64 * NKS;
    const int r = rem / (2 * NKS), c = rem - r * 2 * NKS;
    *reinterpret_cast<v4i*>(abuf + (p * 32 + r) * ARS + 16 * c) = ac[i];
  }
  // LDS-only barriers throughout: the local / gate loads stay in flight under the products
  lds_barrier();

  // 3. both products: per K step, one B fragment per operand from LDS and NCT weight fragments each
  v16i acc0[NCT], acc1[NCT];
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    acc0[c] = v16i{};
    acc1[c] = v16i{};
  }
  const char* xr0 = abuf + row * ARS + 16 * h * NKS;
  const char* xr1 = abuf + (32 + row) * ARS + 16 * h * NKS;
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const v4i x0 = *reinterpret_cast<const v4i*>(xr0 + 16 * ks);
    const v4i x1 = *reinterpret_cast<const v4i*>(xr1 + 16 * ks);
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      acc0[c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(unpack_frag(w0[c][ks]), x0, acc0[c], 0, 0, 0);
      acc1[c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(unpack_frag(w1[c][ks]), x1, acc1[c], 0, 0, 0);
    }
  }

  // out_proj's weight fragments (same lane assignment as the gate's: column col0 + 32 c + t, dwords
  // h NKO .. h NKO + NKO - 1): requested now, they land under the gate's epilogue arithmetic
  uint32_t w2[NKO > 0 ? NCT : 1][NKO > 0 ? NKO : 1];
  if constexpr (NKO > 0) {
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      const int n = col0 + 32 * c + row, nc = n < N ? n : N - 1;
      const uint4* p2 = reinterpret_cast<const uint4*>(op.w + nc * op.ldw + h * NKO * 4);
#pragma unroll
      for (int i = 0; i < NKO / 4; ++i) {
        const uint4 v = p2[i];
        w2[c][4 * i] = v.x, w2[c][4 * i + 1] = v.y, w2[c][4 * i + 2] = v.z, w2[c][4 * i + 3] = v.w;
      }
    }
  }

  // the wave's local / gate slab into its own LDS region (read back by the same wave only: LDS
  // operations of one wave complete in order, the wave barrier keeps the compiler from moving them)
  char* slab = slabs + w * 2 * 32 * SP;

  // 4. y = local + sigmoid(gate) * state_proj + ent_proj in the reference's op order (tesm.py:1256-1260),
  //    every op rounded to the layer dtype; columns past N are 0
  const float inv0 = 1.0f / sx0, inv1 = 1.0f / sx1;
  float y[NCT][16];
  float mx = 0.0f;
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    if (col0 + 32 * c >= N) continue;  // N % 32 == 0: a column tile is all in range or all out (uniform)
    if constexpr (STG) {
      // this tile's local / gate chunks into the wave's own LDS slab, read back by the same wave only
      // (LDS operations of one wave complete in order; the wave barriers keep the compiler from moving them)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = (lane >> 2) + 16 * (q & 1);
        uint2* d = reinterpret_cast<uint2*>(slab + ((q >> 1) * 32 + r) * SP + 64 * c + 16 * (lane & 3));
        d[0] = make_uint2(sg[4 * c + q].x, sg[4 * c + q].y);
        d[1] = make_uint2(sg[4 * c + q].z, sg[4 * c + q].w);
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if constexpr (STG) {
        const int off = (32 * c + 8 * g + 4 * h) * 2;
        const uint2 l2 = *reinterpret_cast<const uint2*>(slab + row * SP + off);
        const uint2 g2 = *reinterpret_cast<const uint2*>(slab + (32 + row) * SP + off);
        lr[c][g][0] = l2.x, lr[c][g][1] = l2.y, gr[c][g][0] = g2.x, gr[c][g][1] = g2.y;
      }
      float sp[4], ep[4], gv[4], v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // (acc / s_x) * c_w as the tiled kernels form it, so that every output-gate kernel agrees bit for bit
        sp[r] = (static_cast<float>(acc0[c][4 * g + r] - rs0) * inv0) * cw0;
        ep[r] = (static_cast<float>(acc1[c][4 * g + r] - rs1) * inv1) * cw1;
        gv[r] = sigmoidf_(ep_get<DT, true>(gr[c][g], r));
      }
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        rnd2<DT>(sp[r], sp[r + 1]);
        rnd2<DT>(ep[r], ep[r + 1]);
        rnd2<DT>(gv[r], gv[r + 1]);
        v[r] = gv[r] * sp[r];
        v[r + 1] = gv[r + 1] * sp[r + 1];
        rnd2<DT>(v[r], v[r + 1]);
        v[r] = ep_get<DT, true>(lr[c][g], r) + v[r];
        v[r + 1] = ep_get<DT, true>(lr[c][g], r + 1) + v[r + 1];
        rnd2<DT>(v[r], v[r + 1]);
        v[r] = v[r] + ep[r];
        v[r + 1] = v[r + 1] + ep[r + 1];
        rnd2<DT>(v[r], v[r + 1]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y[c][4 * g + r] = v[r];
        mx = fmaxf(mx, fabsf(v[r]));
      }
    }
  }
  if (o.y && m < a.M) {  // the optional y itself (decision taps)
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int nb = col0 + 32 * c + 8 * g + 4 * h;
        if (nb < N) {
          const float yy[4] = {y[c][4 * g], y[c][4 * g + 1], y[c][4 * g + 2], y[c][4 * g + 3]};
          store4<DT>(o.y, m * o.ldy + nb, yy, vec4_ok<DT>(o.y, o.ldy));
        }
      }
  }

  // 5. per-token absmax over the workgroup's columns, then int8 codes into LDS in layout 1: column
  //    n = 16 G + e sits at byte 16 G + 4 (e & 3) + (e >> 2); here e = 8 (g & 1) + 4 h + r
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (h == 0) red[w * 32 + row] = mx;
  lds_barrier();  // every wave is past its slab reads: the code tile may overwrite them
  const int padw = (static_cast<int>(o.ldq) - N) / 4;  // N % 32 == 0, ldq % 16 == 0
  if (padw > 0)
    for (int i = tid; i < 32 * padw; i += NT)
      reinterpret_cast<uint32_t*>(codes + (i / padw) * cp + N)[i % padw] = 0u;
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) amax = fmaxf(amax, red[i * 32 + row]);
  const float sc = act_scale<DT>(amax, o.eps);
  int8_t* crow = codes + row * cp + col0 + h;
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    if (col0 + 32 * c >= N) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float t[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] = y[c][4 * g + r] * sc;
      rnd2<DT>(t[0], t[1]);
      rnd2<DT>(t[2], t[3]);
#pragma unroll
      for (int r = 0; r < 4; ++r)  // clamp, then + 1.5 * 2^23 rounds to the code, left in the low byte (group_codes)
        reinterpret_cast<uint8_t*>(crow)[32 * c + 16 * (g >> 1) + 4 * r + 2 * (g & 1)] =
            static_cast<uint8_t>(__float_as_uint(fminf(fmaxf(t[r], -128.0f), 127.0f) + 12582912.0f));
    }
  }
  lds_barrier();

  // 6. the code tile out, row by row in 16-byte chunks; each row's code sum by v_dot4 over its chunks
  constexpr int TPR = NT / 32;  // threads per row
  const int r = tid / TPR, tr = tid % TPR;
  const int chunks = static_cast<int>(o.ldq / 16);
  const int64_t mr = m0 + r;
  int sum = 0;
  for (int ck = tr; ck < chunks; ck += TPR) {
    const uint4 v = *reinterpret_cast<const uint4*>(codes + r * cp + 16 * ck);
    sum = __builtin_amdgcn_sdot4(static_cast<int>(v.x), 0x01010101, sum, false);
    sum = __builtin_amdgcn_sdot4(static_cast<int>(v.y), 0x01010101, sum, false);
    sum = __builtin_amdgcn_sdot4(static_cast<int>(v.z), 0x01010101, sum, false);
    sum = __builtin_amdgcn_sdot4(static_cast<int>(v.w), 0x01010101, sum, false);
    if (o.q && mr < a.M) reinterpret_cast<uint4*>(o.q + mr * o.ldq)[ck] = v;
  }
  sum = wave_sum_i<TPR>(sum);  // the row's TPR consecutive lanes; DPP steps, an integer sum in any order
  if (tr == 0 && o.q && mr < a.M) {
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < NW; ++i) am = fmaxf(am, red[i * 32 + r]);
    o.s[mr] = act_scale<DT>(am, o.eps);
    o.rs[mr] = sum;
  }
  if constexpr (NKO > 0) {
    if (tr == 0) rsl[r] = sum;
    lds_barrier();
    // 7. out_proj on the workgroup's y codes (the B operand from the code tile, K split between the lane
    //    halves as the gate's products split it), then its plain epilogue (acc - rowsum) / s_x * c_w, the
    //    tiled kernels' op order, so the result equals a separate out_proj bit for bit
    v16i acc2[NCT];
#pragma unroll
    for (int c = 0; c < NCT; ++c) acc2[c] = v16i{};
    const char* xr = reinterpret_cast<const char*>(codes) + row * cp + 16 * h * NKO;
#pragma unroll
    for (int ks = 0; ks < NKO; ++ks) {
      const v4i x = *reinterpret_cast<const v4i*>(xr + 16 * ks);
#pragma unroll
      for (int c = 0; c < NCT; ++c)
        acc2[c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(unpack_frag(w2[c][ks]), x, acc2[c], 0, 0, 0);
    }
    const int32_t rsy = rsl[row];
    const float invy = 1.0f / sc, cwo = op.c_w[0];
    if (DT == kBF16 && reinterpret_cast<uintptr_t>(op.out) % 16 == 0 && op.ldo % 8 == 0) {
      // staged through the wave's own 32 x 80-byte LDS slab, one column tile at a time, so that a store
      // instruction covers 16 rows x 64 contiguous bytes instead of 32 rows x 8
      char* os = reinterpret_cast<char*>(rsl + 32) + w * 32 * 80;
#pragma unroll
      for (int c = 0; c < NCT; ++c) {
        if (col0 + 32 * c >= N) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float v[4];
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) v[rr] = (static_cast<float>(acc2[c][4 * g + rr] - rsy) * invy) * cwo;
          *reinterpret_cast<uint2*>(os + row * 80 + (8 * g + 4 * h) * 2) =
              make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          const int idx = 64 * it + lane, rr = idx >> 2, ch = idx & 3;
          const uint4 d = *reinterpret_cast<const uint4*>(os + rr * 80 + 16 * ch);
          if (m0 + rr < a.M)
            *reinterpret_cast<uint4*>(static_cast<uint16_t*>(op.out) + (m0 + rr) * op.ldo + col0 + 32 * c + 8 * ch) = d;
        }
        __builtin_amdgcn_wave_barrier();
      }
      return;
    }
    if (m >= a.M) return;
    const bool vo = vec4_ok<DT>(op.out, op.ldo);
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int nb = col0 + 32 * c + 8 * g + 4 * h;
        if (nb >= N) continue;
        float v[4];
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) v[rr] = (static_cast<float>(acc2[c][4 * g + rr] - rsy) * invy) * cwo;
        store4<DT>(op.out, m * op.ldo + nb, v, vo);
      }
  }
}

// Compute units and LDS bytes per workgroup of the current device (queried once per device).
}  // namespace

DeviceLimits device_limits() {
  static DeviceLimits cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return DeviceLimits{};
  DeviceLimits& d = cache[dev];
  if (d.cus == 0) {
    int cus = 0, lds = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
      return DeviceLimits{};
    d.lds = lds;
    d.cus = cus;
  }
  return d;
}

namespace {

template <int NW, int TM, int TN, int EPI>
int run_skinny(const LinearArgs& a, hipStream_t st) {
  const int64_t tiles = ((a.M + 16 * TM - 1) / (16 * TM)) * ((a.N + 16 * TN - 1) / (16 * TN));
  TESM_REQUIRE(tiles <= 0x7fffffff, kErrUnsupported, "bitlinear: too many tiles");
  if (a.out_dt == kBF16)
    skinny_kernel<NW, TM, TN, EPI, kBF16><<<static_cast<unsigned>(tiles), NW * 64, 0, TESM_LOGGED(st, skinny_kernel<NW, TM, TN, EPI, kBF16>)>>>(a);
  else
    skinny_kernel<NW, TM, TN, EPI, kF32><<<static_cast<unsigned>(tiles), NW * 64, 0, TESM_LOGGED(st, skinny_kernel<NW, TM, TN, EPI, kF32>)>>>(a);
  return check_launch("bitlinear skinny");
}

inline bool host_vec4_ok(const void* p, int64_t ld, int dt) {
  const int64_t bytes = dt == kBF16 ? 8 : 16;
  return (reinterpret_cast<uintptr_t>(p) % bytes) == 0 && (ld * (dt == kBF16 ? 2 : 4)) % bytes == 0;
}

template <int NW, int NCT, int NKS>
void launch_rowq_lds(const LinearArgs& a, const RowQuant& o, int64_t ntiles, int64_t lds, int cus, hipStream_t st) {
  // register-resident weights: one workgroup per CU (VGPR-bound), its tiles prefetched one ahead
  const int64_t per_cu = rowq_reg_weights<NKS>() ? 1 : std::max<int64_t>(1, std::min<int64_t>(4, (160 * 1024) / lds));
  const unsigned grid = static_cast<unsigned>(std::min<int64_t>(ntiles, cus * per_cu));
  if (a.out_dt == kBF16)
    gate_rowq_lds_kernel<NW, NCT, kBF16, NKS><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_lds_kernel<NW, NCT, kBF16, NKS>)>>>(a, o, ntiles);
  else
    gate_rowq_lds_kernel<NW, NCT, kF32, NKS><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_lds_kernel<NW, NCT, kF32, NKS>)>>>(a, o, ntiles);
}

template <int NW, int NCT>
int run_rowq(const LinearArgs& a, const RowQuant& o, hipStream_t st) {
  const bool per_row = a.op[0].c_w_per_row || a.op[1].c_w_per_row;
  const int64_t ntiles = (a.M + 15) / 16;
  const bool vec = a.N % 4 == 0 && host_vec4_ok(a.local, a.ld_local, a.out_dt) &&
                   host_vec4_ok(a.gate, a.ld_gate, a.out_dt);
  const int64_t nks = a.Kp / 64;
  if (vec && (nks == 2 || nks == 4 || nks == 8)) {
    const DeviceLimits dl = device_limits();
    const int64_t lds = rowq_lds_bytes(a.N, nks, o.ldq, NW);
    if (dl.cus > 0 && lds <= dl.lds) {
      if (nks == 2)
        launch_rowq_lds<NW, NCT, 2>(a, o, ntiles, lds, dl.cus, st);
      else if (nks == 4)
        launch_rowq_lds<NW, NCT, 4>(a, o, ntiles, lds, dl.cus, st);
      else
        launch_rowq_lds<NW, NCT, 8>(a, o, ntiles, lds, dl.cus, st);
      return check_launch("output gate rowq (LDS weights)");
    }
  }
  const size_t lds = static_cast<size_t>(16 * o.ldq + 2 * 16 * NW * 4 + (per_row ? 2 * a.N * 4 : 0));
  const unsigned grid = static_cast<unsigned>(ntiles);
  if (a.out_dt == kBF16) {
    if (vec)
      gate_rowq_kernel<NW, NCT, kBF16, true, 0><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_kernel<NW, NCT, kBF16, true, 0>)>>>(a, o);
    else
      gate_rowq_kernel<NW, NCT, kBF16, false, 0><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_kernel<NW, NCT, kBF16, false, 0>)>>>(a, o);
  } else {
    if (vec)
      gate_rowq_kernel<NW, NCT, kF32, true, 0><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_kernel<NW, NCT, kF32, true, 0>)>>>(a, o);
    else
      gate_rowq_kernel<NW, NCT, kF32, false, 0><<<grid, NW * 64, lds, TESM_LOGGED(st, gate_rowq_kernel<NW, NCT, kF32, false, 0>)>>>(a, o);
  }
  return check_launch("output gate rowq");
}

template <int NW, int NCT, int NKS, int NKO = 0>
void launch_gate32(const LinearArgs& a, const RowQuant& o, int64_t lds, hipStream_t st, const G32Out& op = G32Out{}) {
  const unsigned grid = static_cast<unsigned>((a.M + 31) / 32);
  if (a.out_dt == kBF16)
    gate32_kernel<NW, NCT, kBF16, NKS, NKO><<<grid, NW * 64, lds, TESM_LOGGED(st, gate32_kernel<NW, NCT, kBF16, NKS, NKO>)>>>(a, o, op);
  else if constexpr (NKO == 0)  // the fused out_proj is bf16 only (in float32 its registers would spill)
    gate32_kernel<NW, NCT, kF32, NKS, NKO><<<grid, NW * 64, lds, TESM_LOGGED(st, gate32_kernel<NW, NCT, kF32, NKS, NKO>)>>>(a, o, op);
}

template <int NCT>
void launch_gate32_k(const LinearArgs& a, const RowQuant& o, int64_t nks, int64_t lds, hipStream_t st) {
  if (nks == 4)
    launch_gate32<8, NCT, 4>(a, o, lds, st);
  else if (nks == 8)
    launch_gate32<8, NCT, 8>(a, o, lds, st);
  else
    launch_gate32<8, NCT, 12>(a, o, lds, st);
}

// The 32-row kernel when it applies: per-tensor weight scales, N a multiple of 32 up to 1024, K up to
// 384 (register-resident weights), vector-aligned local / gate rows and an LDS budget that fits.
int try_gate32(const LinearArgs& a, const RowQuant& o, hipStream_t st) {
  // TESM_HIP_NO_GATE32=1 keeps the 16-row kernel (a diagnostic switch for side-by-side timing)
  static const bool off = [] {
    const char* e = std::getenv("TESM_HIP_NO_GATE32");
    return e != nullptr && e[0] == '1';
  }();
  const int64_t nks = a.Kp / 32;
  if (off) return -1;
  // bf16 slabs are read in 16-byte chunks: rows and bases 16-byte aligned
  const bool a16 = a.out_dt != kBF16 || (reinterpret_cast<uintptr_t>(a.local) % 16 == 0 && a.ld_local % 8 == 0 &&
                                        reinterpret_cast<uintptr_t>(a.gate) % 16 == 0 && a.ld_gate % 8 == 0);
  if (a.op[0].c_w_per_row || a.op[1].c_w_per_row || a.N % 32 != 0 || a.N > 1024 ||
      !(nks == 4 || nks == 8 || nks == 12) || !host_vec4_ok(a.local, a.ld_local, a.out_dt) ||
      !host_vec4_ok(a.gate, a.ld_gate, a.out_dt) || !a16 || (o.y && !host_vec4_ok(o.y, o.ldy, a.out_dt)))
    return -1;
  const DeviceLimits dl = device_limits();
  const int64_t nct = (a.N / 32 + 7) / 8;
  const int64_t lds = gate32_lds_bytes(a.Kp, o.ldq, nct, 8, a.out_dt == kBF16);
  if (dl.cus <= 0 || lds > dl.lds) return -1;
  if (nct == 1)
    launch_gate32_k<1>(a, o, nks, lds, st);
  else if (nct == 2)
    launch_gate32_k<2>(a, o, nks, lds, st);
  else if (nct == 3)
    launch_gate32_k<3>(a, o, nks, lds, st);
  else
    launch_gate32_k<4>(a, o, nks, lds, st);
  return check_launch("output gate (32-row tiles)");
}

template <int LPR, int MR, int NCH, int RPG = 4>
int run_gemv(const LinearArgs& a, hipStream_t st) {
  constexpr int GPW = 64 / LPR;
  const int64_t groups = (a.N + RPG - 1) / RPG;
  const int64_t waves = (groups + GPW - 1) / GPW;
  const unsigned blocks = static_cast<unsigned>((waves + 3) / 4);
  if (a.out_dt == kBF16)
    gemv_kernel<LPR, MR, NCH, kBF16, RPG><<<blocks, 256, 0, TESM_LOGGED(st, gemv_kernel<LPR, MR, NCH, kBF16, RPG>)>>>(a);
  else
    gemv_kernel<LPR, MR, NCH, kF32, RPG><<<blocks, 256, 0, TESM_LOGGED(st, gemv_kernel<LPR, MR, NCH, kF32, RPG>)>>>(a);
  return check_launch("bitlinear gemv");
}

template <int MR>
int dispatch_gemv(const LinearArgs& a, int64_t nch, hipStream_t st) {
  if (nch <= 4) return run_gemv<4, MR, 1>(a, st);
  if (nch <= 8) return run_gemv<8, MR, 1>(a, st);
  if (nch <= 16) return run_gemv<16, MR, 1>(a, st);
  if (nch <= 32) return run_gemv<32, MR, 1>(a, st);
  // two rows per lane group: twice the waves of four, 3-7 % faster at K = 4096 (N 4096 / 11008)
  if (nch <= 64) return run_gemv<64, MR, 1, 2>(a, st);
  if (nch <= 128) return run_gemv<64, MR, 2, 2>(a, st);
  return run_gemv<64, MR, 4, 2>(a, st);
}

int check_operand(const LinearOperand& o, int64_t Kp, const char* which) {
  std::string p = std::string("bitlinear ") + which + ": ";
  TESM_REQUIRE(o.q && o.s_x && o.rowsum && o.w && o.c_w, kErrInvalidArg, p + "null pointer");
  TESM_REQUIRE(o.ldq >= Kp && o.ldq % 16 == 0, kErrInvalidArg, p + "ldq must be >= Kp and a multiple of 16");
  TESM_REQUIRE(o.ldw >= Kp / 4 && o.ldw % 16 == 0, kErrInvalidArg, p + "ldw must be >= Kp/4 and a multiple of 16");
  TESM_REQUIRE(aligned(o.q, 16) && aligned(o.w, 16), kErrAlignment, p + "codes and packed weights must be 16-byte aligned");
  return kOk;
}

}  // namespace

// Waves of a fused-quantization workgroup (16 waves, four per SIMD, were measured no faster at the
// decode shapes: the quantization phase is bound by its dependent load / reduction / LDS steps).
constexpr int kFqNW = 4;

// LDS of one fused-quantization workgroup: 16 TM code rows of Kp + 16 bytes with their scales and sums
// (dynamic), and skinny_body's static split-K reduction buffer (kFqNW - 1 waves' TM partial tiles, 16
// bytes per lane each).
static int64_t linear_fq_lds_bytes(int64_t M, int64_t Kp) {
  const int64_t TM = M <= 16 ? 1 : 2;
  return 16 * TM * (Kp + 16) + 16 * TM * 8 + (kFqNW - 1) * TM * 64 * 16;
}

// Kp <= 1920 keeps a workgroup at most 68 KB of LDS; the device's per-workgroup limit is checked too (a
// build for a target with less LDS takes the two-launch path).
bool linear_fq_ok(const LinearArgs& a) {
  if (!(a.epilogue == kEpiStore && a.M > 4 && a.M <= 32 && a.N >= 1 && a.N < 16384 && a.Kp >= kKTile &&
        a.Kp % kKTile == 0 && a.Kp <= 1920))
    return false;
  const DeviceLimits dl = device_limits();
  return dl.lds > 0 && linear_fq_lds_bytes(a.M, a.Kp) <= dl.lds;
}

namespace {
template <int TM, int DT, bool VEC, int G>
void run_skinny_fq(const LinearArgs& a, const FusedQuantIn& f, hipStream_t st) {
  const int64_t tiles = ((a.M + 16 * TM - 1) / (16 * TM)) * ((a.N + 15) / 16);
  const size_t lds = static_cast<size_t>(16 * TM * (a.Kp + 16) + 16 * TM * 8);
  if (a.out_dt == kBF16)
    skinny_fq_kernel<kFqNW, TM, 1, kBF16, DT, VEC, G><<<static_cast<unsigned>(tiles), kFqNW * 64, lds, TESM_LOGGED(st, skinny_fq_kernel<kFqNW, TM, 1, kBF16, DT, VEC, G>)>>>(a, f);
  else
    skinny_fq_kernel<kFqNW, TM, 1, kF32, DT, VEC, G><<<static_cast<unsigned>(tiles), kFqNW * 64, lds, TESM_LOGGED(st, skinny_fq_kernel<kFqNW, TM, 1, kF32, DT, VEC, G>)>>>(a, f);
}
template <int TM>
void dispatch_skinny_fq(const LinearArgs& a, const FusedQuantIn& f, bool vec, hipStream_t st) {
  // groups per lane: Kp / 16 over kFqNW * 64 / (16 TM) lanes per row; the register-held variants (one read
  // of the row, straight-line loads) need 16-byte aligned rows of whole 16-element groups
  const int64_t lpr = kFqNW * 64 / (16 * TM), gpl = (a.Kp / 16 + lpr - 1) / lpr;
  const bool held = vec && f.K % 16 == 0;
  if (f.dt == kBF16) {
    if (held) {
      if (gpl <= 2) return run_skinny_fq<TM, kBF16, true, 2>(a, f, st);
      if (gpl <= 4) return run_skinny_fq<TM, kBF16, true, 4>(a, f, st);
      if (gpl <= 6) return run_skinny_fq<TM, kBF16, true, 6>(a, f, st);
      if (gpl <= 8) return run_skinny_fq<TM, kBF16, true, 8>(a, f, st);
    }
    if (vec) return run_skinny_fq<TM, kBF16, true, 0>(a, f, st);
    return run_skinny_fq<TM, kBF16, false, 0>(a, f, st);
  }
  if (held) {
    if (gpl <= 2) return run_skinny_fq<TM, kF32, true, 2>(a, f, st);
    if (gpl <= 4) return run_skinny_fq<TM, kF32, true, 4>(a, f, st);
  }
  if (vec) return run_skinny_fq<TM, kF32, true, 0>(a, f, st);
  return run_skinny_fq<TM, kF32, false, 0>(a, f, st);
}
}  // namespace

int launch_linear_fq(const LinearArgs& a, const FusedQuantIn& f, hipStream_t st) {
  TESM_REQUIRE(linear_fq_ok(a), kErrUnsupported, "bitlinear fused quant: needs 4 < M <= 32, N < 16384, Kp <= 1920");
  TESM_REQUIRE(f.dt == kF32 || f.dt == kBF16, kErrInvalidArg, "bitlinear fused quant: x dtype must be 0 or 1");
  TESM_REQUIRE(f.x && f.K >= 1 && f.K <= a.Kp && f.ldx >= f.K, kErrInvalidArg, "bitlinear fused quant: bad x");
  TESM_REQUIRE(a.out_dt == kF32 || a.out_dt == kBF16, kErrInvalidArg, "bitlinear: out dtype must be 0 or 1");
  TESM_REQUIRE(a.out && a.ldo >= a.N, kErrInvalidArg, "bitlinear: need out and ldo >= N");
  const LinearOperand& o = a.op[0];
  TESM_REQUIRE(o.w && o.c_w && o.ldw >= a.Kp / 4 && o.ldw % 16 == 0 && aligned(o.w, 16), kErrInvalidArg,
               "bitlinear fused quant: bad packed weights");
  const int esz = f.dt == kBF16 ? 2 : 4;
  const bool vec = aligned(f.x, 16) && (f.ldx * esz) % 16 == 0;
  if (a.M <= 16)
    dispatch_skinny_fq<1>(a, f, vec, st);
  else
    dispatch_skinny_fq<2>(a, f, vec, st);
  return check_launch("bitlinear skinny (fused quant)");
}

// The 32x32x32 kernels address a tile's rows (up to 128 of codes, 256 of weights) with 32-bit offsets; longer rows
// take the split-K kernel, which walks any number of 32-row tiles.
static bool tiles32_ok(const LinearArgs& a) {
  const int np = epi_dual(a.epilogue) ? 2 : 1;
  for (int p = 0; p < np; ++p)
    if (a.op[p].ldq >= (int64_t(1) << 24) || a.op[p].ldw >= (int64_t(1) << 23)) return false;
  return true;
}

int launch_linear(const LinearArgs& a, hipStream_t st) {
  TESM_REQUIRE(a.M >= 0 && a.N >= 0, kErrInvalidArg, "bitlinear: negative size");
  TESM_REQUIRE(a.Kp >= kKTile && a.Kp % kKTile == 0, kErrInvalidArg, "bitlinear: Kp must be a positive multiple of 128");
  TESM_REQUIRE(a.out_dt == kF32 || a.out_dt == kBF16, kErrInvalidArg, "bitlinear: out dtype must be 0 or 1");
  TESM_REQUIRE(a.epilogue == kEpiStore || a.epilogue == kEpiOutputGate || a.epilogue == kEpiSwiGLU ||
                   a.epilogue == kEpiGates,
               kErrInvalidArg, "bitlinear: bad epilogue");
  if (a.M == 0 || a.N == 0) return kOk;
  TESM_REQUIRE(a.out && a.ldo >= a.N, kErrInvalidArg, "bitlinear: need out and ldo >= N");
  if (int rc = check_operand(a.op[0], a.Kp, "op0")) return rc;
  if (a.epilogue == kEpiGates) {
    TESM_REQUIRE(a.M > 32 && !a.bias && !a.acc_dump && !a.op[0].c_w_per_row && a.act_bias && a.act_w > 0 &&
                     a.act_n0 >= 0 && a.act_n0 % 32 == 0 && a.act_w % 32 == 0 && a.act_n0 + 3 * a.act_w <= a.N,
                 kErrUnsupported, "bitlinear gates epilogue: needs M > 32, 32-aligned regions inside N, no bias");
    TESM_REQUIRE(tiles32_ok(a), kErrUnsupported, "bitlinear gates epilogue: code rows too long");
    return launch_mfma32(a, st);
  }
  if (a.epilogue != kEpiStore) {
    if (int rc = check_operand(a.op[1], a.Kp, "op1")) return rc;
    TESM_REQUIRE(a.bias == nullptr, kErrInvalidArg, "bitlinear two-product epilogue: bias unsupported");
  }
  if (a.epilogue == kEpiOutputGate)
    TESM_REQUIRE(a.local && a.gate && a.ld_local >= a.N && a.ld_gate >= a.N, kErrInvalidArg,
                 "bitlinear output gate: need local and gate operands");
  const int64_t nch = a.Kp / 64;
  if (a.epilogue == kEpiStore && a.M <= 4 && nch <= 256) {
    if (a.M == 1) return dispatch_gemv<1>(a, nch, st);
    if (a.M == 2) return dispatch_gemv<2>(a, nch, st);
    return dispatch_gemv<4>(a, nch, st);
  }
  if (a.epilogue == kEpiStore) {
    // decode-size batches: the split-K kernel while the LDS-staged one would have too few 64-column
    // tiles to fill the chip (measured at M = 32: N = 768 .. 4096 faster split, N = 34816 staged)
    if (a.M <= 16 && a.N < 16384) return run_skinny<4, 1, 1, kEpiStore>(a, st);
    if ((a.M <= 32 && a.N < 16384) || !tiles32_ok(a)) return run_skinny<4, 2, 1, kEpiStore>(a, st);
    return launch_mfma32(a, st);
  }
  // two-product epilogues: split-K for decode-size batches, else the 32x32 kernels
  if (a.M <= 16) return a.epilogue == kEpiOutputGate ? run_skinny<4, 1, 1, kEpiOutputGate>(a, st) : run_skinny<4, 1, 1, kEpiSwiGLU>(a, st);
  if (a.M <= 32 || !tiles32_ok(a)) return a.epilogue == kEpiOutputGate ? run_skinny<4, 2, 1, kEpiOutputGate>(a, st) : run_skinny<4, 2, 1, kEpiSwiGLU>(a, st);
  return launch_mfma32(a, st);
}

int launch_gate_out(const LinearArgs& a, const RowQuant& o, const LinearOperand& out_proj, void* out, int64_t ldout,
                    hipStream_t st) {
  static const bool off = [] {
    const char* e = std::getenv("TESM_HIP_NO_GATE32");
    return e != nullptr && e[0] == '1';
  }();
  if (off || a.epilogue != kEpiOutputGate || a.M <= 0 || a.N != 768 || a.out_dt != kBF16) return -1;
  const int64_t nks = a.Kp / 32;
  // out_proj over y's codes: K = N = 768 (24 K steps), per-tensor scale, rows of the code pitch
  if (!out_proj.w || !out_proj.c_w || out_proj.c_w_per_row || o.ldq != kpad(a.N) || out_proj.ldw * 4 != o.ldq ||
      !aligned(out_proj.w, 16) || !out || ldout < a.N)
    return -1;
  if (o.q && !(o.s && o.rs && o.ldq % 16 == 0 && aligned(o.q, 16))) return -1;
  const bool a16 = a.out_dt != kBF16 || (reinterpret_cast<uintptr_t>(a.local) % 16 == 0 && a.ld_local % 8 == 0 &&
                                        reinterpret_cast<uintptr_t>(a.gate) % 16 == 0 && a.ld_gate % 8 == 0);
  if (a.op[0].c_w_per_row || a.op[1].c_w_per_row || !(nks == 4 || nks == 8 || nks == 12) ||
      !host_vec4_ok(a.local, a.ld_local, a.out_dt) || !host_vec4_ok(a.gate, a.ld_gate, a.out_dt) || !a16 ||
      (o.y && !host_vec4_ok(o.y, o.ldy, a.out_dt)))
    return -1;
  if (int rc = check_operand(a.op[0], a.Kp, "op0")) return rc;
  if (int rc = check_operand(a.op[1], a.Kp, "op1")) return rc;
  const DeviceLimits dl = device_limits();
  // plus the out_proj output's staging slabs: 8 waves x 32 rows x 80 bytes
  const int64_t lds = gate32_lds_bytes(a.Kp, o.ldq, 3, 8, a.out_dt == kBF16) + 8 * 32 * 80;
  if (dl.cus <= 0 || lds > dl.lds) return -1;
  G32Out op;
  op.w = out_proj.w;
  op.ldw = out_proj.ldw;
  op.c_w = out_proj.c_w;
  op.out = out;
  op.ldo = ldout;
  if (nks == 4)
    launch_gate32<8, 3, 4, 24>(a, o, lds, st, op);
  else if (nks == 8)
    launch_gate32<8, 3, 8, 24>(a, o, lds, st, op);
  else
    launch_gate32<8, 3, 12, 24>(a, o, lds, st, op);
  return check_launch("output gate + out_proj (32-row tiles)");
}

int launch_gate_rowq(const LinearArgs& a, const RowQuant& o, hipStream_t st) {
  TESM_REQUIRE(a.epilogue == kEpiOutputGate, kErrInvalidArg, "gate_rowq: needs the output-gate operands");
  TESM_REQUIRE(a.M >= 0 && a.N >= 1 && a.N <= 1024, kErrUnsupported, "gate_rowq: needs 1 <= d_model <= 1024");
  TESM_REQUIRE(a.Kp >= kKTile && a.Kp % kKTile == 0, kErrInvalidArg, "gate_rowq: Kp must be a multiple of 128");
  TESM_REQUIRE(a.out_dt == kF32 || a.out_dt == kBF16, kErrInvalidArg, "gate_rowq: dtype must be 0 or 1");
  if (a.M == 0) return kOk;
  if (int rc = check_operand(a.op[0], a.Kp, "op0")) return rc;
  if (int rc = check_operand(a.op[1], a.Kp, "op1")) return rc;
  TESM_REQUIRE(a.local && a.gate && a.ld_local >= a.N && a.ld_gate >= a.N, kErrInvalidArg,
               "gate_rowq: need local and gate operands");
  TESM_REQUIRE(o.q && o.s && o.rs && o.ldq >= a.N && o.ldq % 16 == 0 && aligned(o.q, 16), kErrInvalidArg,
               "gate_rowq: bad code outputs");
  TESM_REQUIRE(!o.y || o.ldy >= a.N, kErrInvalidArg, "gate_rowq: bad y output");
  if (const int rc = try_gate32(a, o, st); rc >= 0) return rc;
  const int64_t tiles = (a.N + 15) / 16;
  if (tiles <= 4) return run_rowq<4, 1>(a, o, st);
  if (tiles <= 8) return run_rowq<4, 2>(a, o, st);
  if (tiles <= 12) return run_rowq<4, 3>(a, o, st);
  if (tiles <= 16) return run_rowq<4, 4>(a, o, st);
  if (tiles <= 24) return run_rowq<8, 3>(a, o, st);
  if (tiles <= 32) return run_rowq<8, 4>(a, o, st);
  if (tiles <= 48) return run_rowq<8, 6>(a, o, st);
  return run_rowq<8, 8>(a, o, st);
}

}  // namespace tesm
