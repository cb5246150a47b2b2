// Local-window ternary entanglement of wide bf16 layers (d_state above 512) on the matrix cores, with the
// per-token int8 codes of tanh(E) and C formed in place (the arithmetic is in entangle.hip's header).
//
// Both halves are banded contractions: the scores q . k over the window's keys and the window sums
// weights x states.  One workgroup of 16 waves owns 16 positions and all D channels:
//   1. RoPE'd q rows (16) and k rows (16 + W - 1) are staged in LDS as bf16, the products' exact operands;
//      one wave per 16-key tile forms its scores with v_mfma_f32_16x16x32_bf16 (keys are the A operand, so a
//      lane holds four consecutive keys of one position) and the ternary decisions stay in its registers
//      until the workgroup has counted them; the weights go to LDS as a 16 x keys bf16 matrix.
//   2. the states of 256 channels at a time (16 + W - 1 rows, the next 256 prefetched into registers) are
//      staged in LDS in their natural order and read with ds_read_b64_tr_b16, which hands each lane four
//      consecutive keys of one channel: the A operand of the window sums without a transposed copy.  A wave
//      owns 16 channels of each block; a lane ends with four consecutive channels of one position, forms
//      E, tanh(E) and C, and keeps both as packed bf16 in registers (4 per block).
//   3. row maxima over the workgroup give the two scales; codes are formed from the registers, gathered in
//      LDS (over the staging buffers) and stored as whole 16-code groups.
// So the window weights and the float tanh(E) / C never reach memory, and 16 positions x 2048 channels keep
// 16 waves per CU busy.
//
// 4096 positions, D 2048, rank 256, window 64: 37 us in the layer (33 at best), where the scores kernel (114), the mix
// kernel (309) and the quantization launch (10) took 433; by this alone the whole layer (d_model 4096) went from 927 to
// 526 us.
// Bound by the staging of the states (each CU reads (16 + W - 1) / 16 of its share of them: 5x at window 64,
// from its XCD's L2) and by the barriers between the blocks; the contractions are a few microseconds.
#include "entangle.h"
#include "tesm_hip_internal.h"

namespace tesm {

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMmTP = 16;               // positions per workgroup
constexpr int kMmNW = 16;               // waves per workgroup
constexpr int kMmSC = 16 * kMmNW;       // channels staged at a time, 16 per wave
constexpr int kMmSP = kMmSC + 16;       // state row pitch (elements): 32 bytes past a multiple of 256
constexpr int kMmNT = 64 * kMmNW;

struct MmLds {
  int kp = 0;     // q / k row pitch (elements)
  int s_off = 0;  // staged states
  int t_off = 0;  // weights [16][16 NKT + 8]
  int m_off = 0;  // counts, maxima and code sums of the 16 positions
  int total = 0;
};

MmLds mm_lds(int64_t R, int64_t D, int nkt) {
  MmLds f;
  f.kp = static_cast<int>(round_up(R, 32)) + 8;
  f.s_off = (16 * nkt + kMmTP) * f.kp * 2;
  const int e1 = f.s_off + 16 * nkt * kMmSP * 2;
  const int e2 = 2 * kMmTP * (static_cast<int>(D) + 16);  // the codes, once the stages are consumed
  f.t_off = static_cast<int>(round_up(std::max(e1, e2), 16));
  f.m_off = f.t_off + kMmTP * (16 * nkt + 8) * 2;
  f.total = f.m_off + kMmTP * 5 * 4;
  return f;
}

__device__ __forceinline__ uint2 lds_tr16(const char* p) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
  return __builtin_bit_cast(uint2, v);
}

// Four rotated pairs of one row: x[i .. i + 3] and x[i + half ..], the cross-layer addend, rounded as rope_pair.
__device__ __forceinline__ void mm_rope4(uint2 xa, uint2 xb, const float2 (&cs)[4], bool add, uint2 aa, uint2 ab,
                                         uint2& o1, uint2& o2) {
  const uint32_t wa[2] = {xa.x, xa.y}, wb[2] = {xb.x, xb.y}, va[2] = {aa.x, aa.y}, vb[2] = {ab.x, ab.y};
  float r1[4], r2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = __uint_as_float(j & 1 ? wa[j >> 1] & 0xffff0000u : wa[j >> 1] << 16);
    const float b = __uint_as_float(j & 1 ? wb[j >> 1] & 0xffff0000u : wb[j >> 1] << 16);
    rope_pair<kBF16>(a, b, cs[j], r1[j], r2[j]);
    if (add) {
      r1[j] = rnd<kBF16>(r1[j] + __uint_as_float(j & 1 ? va[j >> 1] & 0xffff0000u : va[j >> 1] << 16));
      r2[j] = rnd<kBF16>(r2[j] + __uint_as_float(j & 1 ? vb[j >> 1] & 0xffff0000u : vb[j >> 1] << 16));
    }
  }
  o1 = make_uint2(pack_bf16x2(r1[0], r1[1]), pack_bf16x2(r1[2], r1[3]));
  o2 = make_uint2(pack_bf16x2(r2[0], r2[1]), pack_bf16x2(r2[2], r2[3]));
}

// NKT: 16-key tiles of the 16 + weff - 1 keys (2, 3 or 5: windows up to 17, 33 and 64); PASSES: blocks of kMmSC
// channels; VEC: q, k, q_add and S rows can be read in 8- and 16-byte vectors.
template <int NKT, int PASSES, bool VEC>
__global__ __launch_bounds__(kMmNT) void ent_mfma_kernel(EntArgs e, int weff, MmLds f) {
  extern __shared__ __attribute__((aligned(16))) char lds_mm[];
  constexpr int ROWS = 16 * NKT;  // staged key / state rows (those past 16 + weff - 1 are zero)
  constexpr int TP = 16 * NKT + 8;
  uint16_t* qk = reinterpret_cast<uint16_t*>(lds_mm);  // [ROWS] keys, then [16] queries
  char* sst = lds_mm + f.s_off;
  uint16_t* tw = reinterpret_cast<uint16_t*>(lds_mm + f.t_off);
  int* cnt = reinterpret_cast<int*>(lds_mm + f.m_off);  // [16] nonzero decisions
  int* amx = cnt + kMmTP;                               // [2][16] row maxima (bits of non-negative floats)
  int* rsum = amx + 2 * kMmTP;                          // [2][16] code sums
  const int tid = threadIdx.x;
  __builtin_assume(tid < kMmNT);
  const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane & 15, q4 = lane >> 4;
  const int64_t b = blockIdx.y, L = e.L;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kMmTP, tk0 = t0 - (weff - 1);
  const int rows = kMmTP + weff - 1;
  const int half = static_cast<int>(e.R / 2), D = static_cast<int>(e.D);

  // states of block `pass`: 16-byte vectors, rows outside [0, L) or past the window and channels past D are zero
  constexpr int NV = ROWS * (kMmSC / 8), SI = (NV + kMmNT - 1) / kMmNT;
  uint4 pre[SI];
  const uint16_t* Sb = static_cast<const uint16_t*>(e.S) + b * L * e.ld_s;
  auto fetch = [&](int pass) {
#pragma unroll
    for (int k = 0; k < SI; ++k) {
      const int i = tid + k * kMmNT, r = i / (kMmSC / 8), c = pass * kMmSC + 8 * (i % (kMmSC / 8));
      const int64_t t = tk0 + r;
      const bool in = r < rows && t >= 0 && t < L && c < D;
      const uint16_t* src = Sb + (t < 0 ? 0 : (t < L ? t : L - 1)) * e.ld_s + (c < D ? c : 0);
      uint4 v;
      if constexpr (VEC) {
        v = *reinterpret_cast<const uint4*>(src);
      } else {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = src[2 * j] | (static_cast<uint32_t>(src[2 * j + 1]) << 16);
        v = make_uint4(w[0], w[1], w[2], w[3]);
      }
      pre[k] = in ? v : make_uint4(0, 0, 0, 0);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int k = 0; k < SI; ++k) {
      const int i = tid + k * kMmNT, r = i / (kMmSC / 8);
      if (NV % kMmNT == 0 || i < NV) *reinterpret_cast<uint4*>(sst + (r * kMmSP + 8 * (i % (kMmSC / 8))) * 2) = pre[k];
    }
  };

  // 1. RoPE'd keys and queries into LDS
  if (tid < 5 * kMmTP) cnt[tid] = 0;
  const int qrow0 = ROWS;
  if constexpr (VEC) {
    const int h4 = half / 4, n = (rows + kMmTP) * h4;
    constexpr int KB = 3;
    for (int base = 0; base < n; base += kMmNT * KB) {
      uint2 xa[KB], xb[KB], aa[KB], ab[KB];
      float2 cs[KB][4];
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        int i = base + tid + k * kMmNT;
        i = i < n ? i : n - 1;
        const int r = i / h4, c = 4 * (i - r * h4);
        const bool isq = r >= rows;
        int64_t t = isq ? t0 + (r - rows) : tk0 + r;
        t = t < 0 ? 0 : (t < L ? t : L - 1);
        const uint16_t* src = static_cast<const uint16_t*>(isq ? e.q : e.k) + (b * L + t) * (isq ? e.ld_q : e.ld_k) + c;
        xa[k] = *reinterpret_cast<const uint2*>(src);
        xb[k] = *reinterpret_cast<const uint2*>(src + half);
        const float4* ct = reinterpret_cast<const float4*>(e.rope + t * half + c);
        const float4 c0 = ct[0], c1 = ct[1];
        cs[k][0] = make_float2(c0.x, c0.y);
        cs[k][1] = make_float2(c0.z, c0.w);
        cs[k][2] = make_float2(c1.x, c1.y);
        cs[k][3] = make_float2(c1.z, c1.w);
        aa[k] = ab[k] = make_uint2(0, 0);
        if (e.q_add) {
          const uint16_t* ad = static_cast<const uint16_t*>(e.q_add) + (b * L + t) * e.ld_qadd + c;
          aa[k] = *reinterpret_cast<const uint2*>(ad);
          ab[k] = *reinterpret_cast<const uint2*>(ad + half);
        }
      }
      if (base == 0) fetch(0);  // behind the q / k loads, ahead of their use
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        const int i = base + tid + k * kMmNT;
        if (i >= n) break;
        const int r = i / h4, c = 4 * (i - r * h4);
        const bool isq = r >= rows;
        const int64_t t = isq ? t0 + (r - rows) : tk0 + r;
        uint2 o1, o2;
        mm_rope4(xa[k], xb[k], cs[k], isq && e.q_add != nullptr, aa[k], ab[k], o1, o2);
        if (t < 0 || t >= L) o1 = o2 = make_uint2(0, 0);
        uint16_t* dst = qk + (isq ? qrow0 + (r - rows) : r) * f.kp + c;
        *reinterpret_cast<uint2*>(dst) = o1;
        *reinterpret_cast<uint2*>(dst + half) = o2;
      }
    }
  } else {
    fetch(0);
    for (int i = tid; i < (rows + kMmTP) * half; i += kMmNT) {
      const int r = i / half, c = i - r * half;
      const bool isq = r >= rows;
      const int64_t t = isq ? t0 + (r - rows) : tk0 + r;
      float o1 = 0.0f, o2 = 0.0f;
      if (t >= 0 && t < L) {
        const int64_t o = (b * L + t) * (isq ? e.ld_q : e.ld_k) + c;
        const void* src = isq ? e.q : e.k;
        rope_pair<kBF16>(ld<kBF16>(src, o), ld<kBF16>(src, o + half), e.rope[t * half + c], o1, o2);
        if (isq && e.q_add) {
          const int64_t ao = (b * L + t) * e.ld_qadd + c;
          o1 = rnd<kBF16>(o1 + ld<kBF16>(e.q_add, ao));
          o2 = rnd<kBF16>(o2 + ld<kBF16>(e.q_add, ao + half));
        }
      }
      uint16_t* dst = qk + (isq ? qrow0 + (r - rows) : r) * f.kp + c;
      dst[0] = f32_to_bf16(o1);
      dst[half] = f32_to_bf16(o2);
    }
  }
  // columns R .. round_up(R, 32) - 1 are zero; key rows past the window feed only masked scores
  const int R = 2 * half, padc = f.kp - 8 - R;
  for (int i = tid; i < (ROWS + kMmTP) * padc; i += kMmNT) qk[(i / padc) * f.kp + R + i % padc] = 0;
  stage();
  if (PASSES > 1) fetch(1);
  // window bias of the lane's four keys (decisions outside the window are masked)
  const int jr0 = 16 * wv + 4 * q4;  // first key row of the lane in its wave's tile
  float wb[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    int w = jr0 + r - p;
    w = w < 0 ? 0 : (w < weff ? w : weff - 1);
    wb[r] = e.bias[e.W - weff + w];
  }
  __syncthreads();

  // scores of 16 keys x 16 positions per wave: ternary decisions, counted per position
  float tern[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const int64_t t = t0 + p;
  if (wv < NKT) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* pa = qk + (16 * wv + p) * f.kp + 8 * q4;
    const uint16_t* pb = qk + (qrow0 + p) * f.kp + 8 * q4;
    for (int s = 0; s < f.kp - 8; s += 32)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const b16x8*>(pa + s),
                                                   *reinterpret_cast<const b16x8*>(pb + s), acc, 0, 0, 0);
    const float sq = static_cast<float>(sqrt(static_cast<double>(e.R)));
    int n = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int w = jr0 + r - p;
      const bool in = w >= 0 && w < weff && t < L;
      float sc = rnd<kBF16>(rnd<kBF16>(acc[r]) / sq);
      sc = rnd<kBF16>(sc + wb[r]);
      const float v = sc > e.thr ? 1.0f : (sc < -e.thr ? -1.0f : 0.0f);
      tern[r] = in && tk0 + jr0 + r >= 0 ? v : 0.0f;
      if (e.tern && in) e.tern[(b * L + t) * weff + w] = static_cast<int8_t>(tern[r]);
      n += tern[r] != 0.0f;
    }
    if (n) atomicAdd(&cnt[p], n);
  }
  __syncthreads();
  if (wv < NKT) {
    const float n = fmaxf(static_cast<float>(cnt[p]), 1.0f);
    *reinterpret_cast<uint2*>(tw + p * TP + jr0) =
        make_uint2(pack_bf16x2(tern[0] / n, tern[1] / n), pack_bf16x2(tern[2] / n, tern[3] / n));
  }
  __syncthreads();

  // 2. window sums, E, tanh(E), C; both kept as packed bf16
  // 32 keys per product; with an odd number of key tiles the last product's upper 16 (lanes 32-63) are zeros in
  // both operands.  (A closing 16x16x16 product is not used: right behind a 16x16x32 one, whose result it adds
  // to, it read that result too early.)
  constexpr int N32 = (NKT + 1) / 2;
  const bool upper = q4 >= 2;
  uint4 wf[N32];
#pragma unroll
  for (int s = 0; s < N32; ++s) {
    const bool odd = 2 * s + 1 >= NKT;
    const uint4 v = *reinterpret_cast<const uint4*>(tw + p * TP + 32 * s + 8 * (odd ? q4 & 1 : q4));
    wf[s] = odd && upper ? make_uint4(0, 0, 0, 0) : v;
  }
  uint2 te[PASSES], cc[PASSES];
  float mte = 0.0f, mcc = 0.0f;
  const char* lrow = sst + ((8 * q4 + (p >> 2)) * kMmSP + 16 * wv + 4 * (p & 3)) * 2;
  const char* lodd = sst + ((8 * (q4 & 1) + (p >> 2)) * kMmSP + 16 * wv + 4 * (p & 3)) * 2;
  const char* lown = sst + ((p + weff - 1) * kMmSP + 16 * wv + 4 * q4) * 2;
#pragma unroll
  for (int ps = 0; ps < PASSES; ++ps) {
    te[ps] = cc[ps] = make_uint2(0, 0);
    if (ps * kMmSC + 16 * wv < D) {  // (wave-uniform)
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < N32; ++s) {
        const bool odd = 2 * s + 1 >= NKT;
        const char* lr = (odd ? lodd : lrow) + 32 * s * kMmSP * 2;
        const uint2 a0 = lds_tr16(lr), a1 = lds_tr16(lr + 4 * kMmSP * 2);
        const bool z = odd && upper;
        const uint4 av = make_uint4(z ? 0u : a0.x, z ? 0u : a0.y, z ? 0u : a1.x, z ? 0u : a1.y);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b16x8, av), __builtin_bit_cast(b16x8, wf[s]),
                                                     acc, 0, 0, 0);
      }
      // a weight 0 times an infinite or NaN state outside the position's own window must not reach its sum:
      // such a tile (its sums are then not finite) takes the window's slots alone, in order
      if (__any(!(fabsf(acc[0]) + fabsf(acc[1]) + fabsf(acc[2]) + fabsf(acc[3]) < __builtin_inff()))) {
        acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int w = 0; w < weff; ++w) {
          const float wt = bf16_to_f32(tw[p * TP + p + w]);
          const uint16_t* srow = reinterpret_cast<const uint16_t*>(sst) + (p + w) * kMmSP + 16 * wv + 4 * q4;
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(wt, bf16_to_f32(srow[r]), acc[r]);
        }
      }
      const uint2 own = *reinterpret_cast<const uint2*>(lown);
      const uint32_t ow[2] = {own.x, own.y};
      float tv[4], cv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float s0 = __uint_as_float(r & 1 ? ow[r >> 1] & 0xffff0000u : ow[r >> 1] << 16);
        const float avg = rnd<kBF16>(acc[r]);
        const float ev = rnd<kBF16>(s0 + rnd<kBF16>(e.ent_scale * rnd<kBF16>(avg - s0)));
        cv[r] = rnd<kBF16>(ev - s0);
        tv[r] = rnd<kBF16>(tanhf_(ev));
        mte = fmaxf(mte, fabsf(tv[r]));
        mcc = fmaxf(mcc, fabsf(cv[r]));
      }
      te[ps] = make_uint2(pack_bf16x2(tv[0], tv[1]), pack_bf16x2(tv[2], tv[3]));
      cc[ps] = make_uint2(pack_bf16x2(cv[0], cv[1]), pack_bf16x2(cv[2], cv[3]));
      if (t < L && (e.e_tanh || e.c_out)) {
        const int64_t o = (b * L + t) * e.ld_out + ps * kMmSC + 16 * wv + 4 * q4;
        if (e.e_tanh)
#pragma unroll
          for (int r = 0; r < 4; ++r) st<kBF16>(e.e_tanh, o + r, tv[r]);
        if (e.c_out)
#pragma unroll
          for (int r = 0; r < 4; ++r) st<kBF16>(e.c_out, o + r, cv[r]);
      }
    }
    if (ps + 1 < PASSES) {
      lds_barrier();  // every wave is done with this block's states
      stage();
      if (ps + 2 < PASSES) fetch(ps + 2);
      lds_barrier();
    }
  }

  // 3. per-token codes: maxima of the row, then a lane's four codes per block as one dword in LDS
  atomicMax(&amx[p], __float_as_int(mte));
  atomicMax(&amx[kMmTP + p], __float_as_int(mcc));
  __syncthreads();
  uint32_t* code = reinterpret_cast<uint32_t*>(lds_mm);  // [2][16][(D + 16) / 4], natural order
  const int cp = (D + 16) / 4;
  float sc2[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    sc2[q] = act_scale<kBF16>(__int_as_float(amx[q * kMmTP + p]), e.eps);
    int32_t rs = 0;
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      if (ps * kMmSC + 16 * wv >= D) continue;
      const uint2 v2 = q == 0 ? te[ps] : cc[ps];
      const uint32_t vw[2] = {v2.x, v2.y};
      uint32_t c[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {  // group_codes' clamp and rounding
        const float v = __uint_as_float(r & 1 ? vw[r >> 1] & 0xffff0000u : vw[r >> 1] << 16);
        c[r] = __float_as_uint(fminf(fmaxf(rnd<kBF16>(v * sc2[q]), -128.0f), 127.0f) + 12582912.0f);
      }
      const uint32_t w = pack_low_bytes(c[0], c[1], c[2], c[3]);
      rs = __builtin_amdgcn_sdot4(static_cast<int>(w), 0x01010101, rs, false);
      code[(q * kMmTP + p) * cp + (ps * kMmSC + 16 * wv) / 4 + q4] = w;
    }
    atomicAdd(&rsum[q * kMmTP + p], rs);
  }
  __syncthreads();
  const int groups = D / 16, ngq = static_cast<int>(e.ldq / 16);
  for (int i = tid; i < 2 * kMmTP * ngq; i += kMmNT) {
    const int g = i % ngq, row = i / ngq, pp = row & (kMmTP - 1), q = row >> 4;
    if (t0 + pp >= L) continue;
    const uint4 o = g < groups ? natural_to_layout1(*reinterpret_cast<const uint4*>(code + row * cp + 4 * g))
                               : make_uint4(0, 0, 0, 0);
    reinterpret_cast<uint4*>((q == 0 ? e.q_te : e.q_c) + (b * L + t0 + pp) * e.ldq)[g] = o;
  }
  if (wv == 0 && q4 < 2 && t < L) {  // lanes 0-15: tanh(E)'s scale and code sum, lanes 16-31: C's
    (q4 == 0 ? e.s_te : e.s_c)[b * L + t] = q4 == 0 ? sc2[0] : sc2[1];
    (q4 == 0 ? e.rs_te : e.rs_c)[b * L + t] = rsum[q4 * kMmTP + p];
  }
}

template <int NKT, int PASSES>
void launch_mm(const EntArgs& a, int weff, const MmLds& f, bool vec, hipStream_t st) {
  dim3 grid(static_cast<unsigned>((a.L + kMmTP - 1) / kMmTP), static_cast<unsigned>(a.B));
  if (vec)
    ent_mfma_kernel<NKT, PASSES, true><<<grid, kMmNT, f.total, TESM_LOGGED(st, ent_mfma_kernel<NKT, PASSES, true>)>>>(a, weff, f);
  else
    ent_mfma_kernel<NKT, PASSES, false><<<grid, kMmNT, f.total, TESM_LOGGED(st, ent_mfma_kernel<NKT, PASSES, false>)>>>(a, weff, f);
}

template <int NKT>
void launch_mm_p(const EntArgs& a, int weff, const MmLds& f, bool vec, hipStream_t st) {
  const int64_t passes = (a.D + kMmSC - 1) / kMmSC;
  if (passes <= 4)
    launch_mm<NKT, 4>(a, weff, f, vec, st);
  else if (passes <= 8)
    launch_mm<NKT, 8>(a, weff, f, vec, st);
  else
    launch_mm<NKT, 16>(a, weff, f, vec, st);
}

int mm_key_tiles(int64_t weff) { return weff <= 17 ? 2 : (weff <= 33 ? 3 : 5); }

}  // namespace

// bf16 rows wider than the other fused kernels take (they hold D <= 512), in whole 16-channel tiles, and an LDS
// budget of one workgroup per CU (ranks up to about 550 at window 64).  Shapes only: the workspace plan asks too.
bool ent_mfma_ok(const EntArgs& a, int64_t weff) {
  if (a.mimo || a.H != 1 || a.dt != kBF16 || a.D <= 512 || a.D > 16 * kMmSC || a.D % 16 != 0 || weff > 64) return false;
  return mm_lds(a.R, a.D, mm_key_tiles(weff)).total <= 160 * 1024;
}

int launch_ent_mfma(const EntArgs& a, int64_t weff, hipStream_t st) {
  TESM_REQUIRE(ent_mfma_ok(a, weff), kErrUnsupported, "local_ent: shape outside the matrix-core kernel's range");
  const int nkt = mm_key_tiles(weff);
  const MmLds f = mm_lds(a.R, a.D, nkt);
  const bool vec = a.R % 8 == 0 && aligned(a.q, 8) && aligned(a.k, 8) && a.ld_q % 4 == 0 && a.ld_k % 4 == 0 &&
                   aligned(a.rope, 16) && (!a.q_add || (aligned(a.q_add, 8) && a.ld_qadd % 4 == 0)) &&
                   aligned(a.S, 16) && a.ld_s % 8 == 0;
  if (nkt == 2)
    launch_mm_p<2>(a, static_cast<int>(weff), f, vec, st);
  else if (nkt == 3)
    launch_mm_p<3>(a, static_cast<int>(weff), f, vec, st);
  else
    launch_mm_p<5>(a, static_cast<int>(weff), f, vec, st);
  return check_launch("entanglement fused (matrix cores)");
}

}  // namespace tesm
