// Global causal ternary entanglement of bf16 single-head layers in one pass over the keys (the arithmetic is in
// global.h and global.hip).
//
// A workgroup of 8 waves owns 16 queries and 256 channels and walks the keys in blocks of 128:
//   scores   each wave forms one 16-key x 16-query tile (v_mfma_f32_16x16x32_bf16, queries in registers for the whole
//            kernel, key rows straight from the RoPE'd copy, requested a block ahead), rounds it to decisions and
//            writes them as bf16 into a 16 x 128 LDS matrix: each decision is formed once and never leaves the CU;
//   mix      each wave adds decisions x states for its 32 channels.  States are loaded to LDS in their natural
//            (key, channel) order, two buffers of 64 keys so the next block's loads run under this block's scores
//            and the other half's products, and read with ds_read_b64_tr_b16 as the operand of 8 consecutive keys
//            per channel; 32-byte units are XORed with three of the key's bits, so the reads hit all banks.
// The normalisation by the decision count is applied once at the end, where the layer's E, tanh(E) and C are formed
// and, when the workgroup holds whole rows (D <= 256), quantized in place.
//
// Two workgroups fit a CU, so one's decisions (vector arithmetic, about 25 operations per score) run under the other's
// products (LDS reads).  The causal triangle makes the last queries' workgroups twice the mean: where all workgroups
// are resident at once the second half of the grid runs in ascending order, so a CU pairs a long with a short one.
// Bound by the chain of one workgroup's key blocks (about 1.9 us per 128 keys with its three barriers) and, with the
// chip full, by LDS bandwidth (128 bytes per state and block written and read).  4 x 2048 tokens, rank 64, 256
// channels: 31 us and 5 us for the bias table and RoPE, against scores 33, transposed copy 5, mix 35, table 5, RoPE 4
// and quantization 5 us with 17 MB of decisions written and read four times (32 queries per workgroup and one
// workgroup per CU: 54 us).
#include <type_traits>

#include "global.h"
#include "linear_dev.h"

namespace tesm {

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kGQ = 16;                  // queries per workgroup
constexpr int kGK = 128;                 // keys per block, 16 per wave
constexpr int kGC = 256;                 // channels per workgroup, 32 per wave
constexpr int kGNW = 8, kGNT = 64 * kGNW;
constexpr int kGRow = kGC * 2;           // bytes of a staged state row
constexpr int kGHalf = kGK / 2 * kGRow;  // bytes of one state buffer
constexpr int kGLoads = kGK / 2 / 2 / kGNW;  // load instructions of a wave per state buffer, two rows each
constexpr int kGTP = kGK + 8;            // decision row pitch (bf16)
constexpr int kGTab = kGNT;              // staged bias entries
constexpr int64_t kGMaxL = 32768;        // positions for which they hold a block's
constexpr int kGLds = 2 * kGHalf + kGQ * kGTP * 2 + kGTab * 4 + kGQ * 5 * 4;
static_assert(2 * kGLds <= 160 * 1024, "two workgroups' LDS");

// Loads to LDS through a buffer resource (see mfma32.hip: global_load_lds would make every LDS read wait for all)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffffu, 0x00027000);
}
typedef __attribute__((address_space(3))) const char* lds_cptr;

// The transposed operands of two 32-key steps for a wave's two 16-channel tiles: v[step][tile] holds 8 keys of a
// channel.  One block that waits for its own reads: before the builtin the compiler would wait for every load to LDS
// in flight.  x0, x1: the tiles' places in the first step's rows; 2048 and 16384 bytes are 4 and 32 rows on.
__device__ __forceinline__ void tr_step2(lds_cptr x0, lds_cptr x1, uint2 (&v)[2][2][2]) {
  static_assert(kGRow == 512, "row offsets below");
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:2048\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:2048\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:16384\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:18432\n\t"
      "ds_read_b64_tr_b16 %6, %9 offset:16384\n\t"
      "ds_read_b64_tr_b16 %7, %9 offset:18432\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[0][1][0]), "=&v"(v[0][1][1]), "=&v"(v[1][0][0]),
        "=&v"(v[1][0][1]), "=&v"(v[1][1][0]), "=&v"(v[1][1][1])
      : "v"(x0), "v"(x1)
      : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wg_barrier() {  // LDS accesses done, no wait for loads in flight
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// LDS stores past loads to LDS in flight (the compiler would wait for those); wg_barrier waits for them
__device__ __forceinline__ void lds_put8(lds_cptr p, uint32_t x, uint32_t y) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(p), "v"(make_uint2(x, y)) : "memory");
}
__device__ __forceinline__ void lds_put4(lds_cptr p, float x) {
  asm volatile("ds_write_b32 %0, %1" ::"v"(p), "v"(x) : "memory");
}

// x / d rounded to nearest as the division is: one correction of x * inv by the exact residual (inv = 1 / d rounded;
// Markstein's theorem), the plain product where it is not finite
__device__ __forceinline__ float div_by(float x, float d, float inv) {
  const float q = x * inv;
  const float r = __builtin_fmaf(-q, d, x);
  return fabsf(q) < __builtin_inff() ? __builtin_fmaf(r, inv, q) : q;
}

// RoPE'd bf16 rows of pitch rp (zeros past R), and the bias table, in one launch: workgroups below nrope rotate.
__global__ __launch_bounds__(256) void global_prep_kernel(GlobalArgs a, uint16_t* qr, uint16_t* kr, int rp,
                                                          unsigned nrope, int64_t ntab, float* table) {
  if (blockIdx.x >= nrope) {  // the bias table: eight lanes per entry, as global_bias_table_kernel
    global_bias_entry<kBF16>(static_cast<int64_t>(blockIdx.x - nrope) * 256 + threadIdx.x, ntab, a.embed, a.P,
                             a.rel_scale, a.rel_bias, table);
    return;
  }
  const int half = static_cast<int>(a.R / 2);
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t bt = e / half;
  if (bt >= a.B * a.L) return;
  const int p = static_cast<int>(e - bt * half);
  const float2 cs = a.rope[(bt % a.L) * half + p];
  const int64_t qo = bt * a.ld_q, ko = bt * a.ld_k, o = bt * rp;
  float q1, q2, k1, k2;
  rope_pair<kBF16>(ld<kBF16>(a.q, qo + p), ld<kBF16>(a.q, qo + half + p), cs, q1, q2);
  rope_pair<kBF16>(ld<kBF16>(a.k, ko + p), ld<kBF16>(a.k, ko + half + p), cs, k1, k2);
  if (a.q_add) {
    const int64_t ao = bt * a.ld_qadd;
    q1 = rnd<kBF16>(q1 + ld<kBF16>(a.q_add, ao + p));
    q2 = rnd<kBF16>(q2 + ld<kBF16>(a.q_add, ao + half + p));
  }
  qr[o + p] = f32_to_bf16(q1);
  qr[o + half + p] = f32_to_bf16(q2);
  kr[o + p] = f32_to_bf16(k1);
  kr[o + half + p] = f32_to_bf16(k2);
  for (int c = 2 * half + p; c < rp; c += half) qr[o + c] = kr[o + c] = 0;
}

// Unit of 32 bytes that holds channels 16 u .. of buffer row r
__device__ __forceinline__ int swz(int u, int r) { return u ^ ((r & 3) | ((r >> 1) & 4)); }

// RS: 32-value steps of a RoPE'd row.  QUANT: whole rows in the workgroup, codes of tanh(E) and C formed here.
template <int RS, bool QUANT>
__global__ __launch_bounds__(kGNT, 4) void global_mfma_kernel(GlobalArgs a, const uint16_t* qr, const uint16_t* kr,
                                                              int64_t nqb, unsigned fold) {
  extern __shared__ __attribute__((aligned(16))) char lds_g[];
  uint16_t* T = reinterpret_cast<uint16_t*>(lds_g + 2 * kGHalf);
  float* tab = reinterpret_cast<float*>(lds_g + 2 * kGHalf + kGQ * kGTP * 2);
  int* cnt = reinterpret_cast<int*>(tab + kGTab);  // [16] decision counts, [2][16] row maxima, [2][16] code sums
  int* amx = cnt + kGQ;
  int* rsum = amx + 2 * kGQ;
  const int tid = threadIdx.x;
  __builtin_assume(tid < kGNT);
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, l16 = lane & 15;
  // heaviest (latest) query blocks first, in ascending order from `fold` on
  const unsigned nb = static_cast<unsigned>(a.B), bx = blockIdx.x;
  const unsigned bo = bx < fold ? bx : static_cast<unsigned>(nqb) * nb - 1 - (bx - fold);
  const int64_t b = bo % nb;
  const int L = static_cast<int>(a.L);  // (at most kGMaxL)
  const int i0 = static_cast<int>(nqb - 1 - bo / nb) * kGQ, kend = L < i0 + kGQ ? L : i0 + kGQ;
  const int cbase = static_cast<int>(blockIdx.y) * kGC, D = static_cast<int>(a.D);
  const int i = i0 + l16, ir = i < L ? i : L - 1;
  constexpr int RP = 32 * RS;
  const uint16_t* kb_ = kr + b * L * RP;

  b16x8 qf[RS], kf[RS];
#pragma unroll
  for (int s = 0; s < RS; ++s) qf[s] = *reinterpret_cast<const b16x8*>(qr + (b * L + ir) * RP + 32 * s + 8 * g);
  auto load_keys = [&](int k0) {
    const int j = k0 + 16 * w + l16, jr = j < L ? j : L - 1;
#pragma unroll
    for (int s = 0; s < RS; ++s)
      kf[s] = *reinterpret_cast<const b16x8*>(kb_ + static_cast<int64_t>(jr) * RP + 32 * s + 8 * g);
  };
  // states of keys k0 + 64 hf ..: two rows per load instruction; rows past the last key re-read it
  const __amdgpu_buffer_rsrc_t sbuf = rows_buffer(static_cast<const uint16_t*>(a.S) + b * L * a.ld_s + cbase);
  auto load_states = [&](int k0, int hf) {
#pragma unroll
    for (int n = 0; n < kGLoads; ++n) {
      const int blk = w + n * kGNW, r = 2 * blk + (lane >> 5);  // row of the buffer
      const int key = k0 + kGK / 2 * hf + r, kc = key < kend ? key : kend - 1;
      int ch = 8 * (2 * swz((lane & 31) >> 1, r) + (lane & 1));
      ch = cbase + ch < D ? ch : 0;  // (channels past D feed only outputs that are never stored)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          sbuf, (__attribute__((address_space(3))) void*)(lds_g + hf * kGHalf + blk * 1024), 16,
          (static_cast<uint32_t>(kc) * static_cast<uint32_t>(a.ld_s) + ch) * 2, 0, 0, 0);
    }
  };
  // first bias entry the block's scores reach: rel is monotone in both positions, and up to kGMaxL the entries of a
  // block span at most 257 (positions round by up to 64 there)
  auto rel_of = [](int x, int y) {
    return static_cast<int>(rnd<kBF16>(rnd<kBF16>(static_cast<float>(x)) - rnd<kBF16>(static_cast<float>(y))));
  };
  auto table_from = [&](int k0) {
    const int r0 = rel_of(i0, k0 + kGK - 1);
    return r0 > 0 ? r0 : 0;
  };
  auto table_entry = [&](int lo) { return a.table[lo + tid < 2 * L ? lo + tid : 2 * L - 1]; };

  int rlo = table_from(0);
  if (tid < 5 * kGQ) cnt[tid] = 0;
  load_keys(0);
  tab[tid] = table_entry(rlo);
  load_states(0, 0);
  load_states(0, 1);
  wg_barrier();

  const float pi = rnd<kBF16>(static_cast<float>(i)), dinv = 1.0f / a.sqrt_div;
  const int ilast = i < L ? i : -1;
  int n = 0;
  f32x4 acc[2] = {};
  // the lane's place in a state row: keys 8 g + l16 / 4 of a 32-key step, four channels
  const int arow = 8 * g + (l16 >> 2);
  const int aoff[2] = {arow * kGRow + swz(2 * w, arow) * 32 + 8 * (l16 & 3),
                       arow * kGRow + swz(2 * w + 1, arow) * 32 + 8 * (l16 & 3)};
  auto block = [&](int k0, auto last_tag) {
    constexpr bool last = decltype(last_tag)::value;
    int nlo = 0;
    float nt = 0.0f;
    // scores of keys k0 + 16 w .. + 15 (rows of the product) for the 16 queries: four keys of one query per lane
    {
      f32x4 sc = {};
#pragma unroll
      for (int s = 0; s < RS; ++s) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s], qf[s], sc, 0, 0, 0);
      if constexpr (!last) {  // (in flight until the block's end)
        nlo = table_from(k0 + kGK);
        load_keys(k0 + kGK);
        nt = table_entry(nlo);
        asm volatile("" ::: "memory");
      }
      const int jt = 16 * w + 4 * g;
      uint32_t t16[4], t8 = 0;
      float tb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = k0 + jt + u;
        const float rel = rnd<kBF16>(pi - rnd<kBF16>(static_cast<float>(j)));
        const int r = static_cast<int>(rel);
        tb[u] = tab[r > rlo ? r - rlo : 0];  // (past the diagonal: any entry, unused)
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float sv = rnd<kBF16>(rnd<kBF16>(div_by(rnd<kBF16>(sc[u]), a.sqrt_div, dinv)) + tb[u]);
        int t = static_cast<int>(sv > a.thr) - static_cast<int>(sv < -a.thr);
        t = k0 + jt + u <= ilast ? t : 0;
        n += t != 0;
        t16[u] = (static_cast<uint32_t>(t) & 0x8000u) | (t != 0 ? 0x3f80u : 0u);
        t8 |= static_cast<uint32_t>(static_cast<uint8_t>(t)) << (8 * u);
      }
      lds_put8((lds_cptr)(reinterpret_cast<const char*>(T + l16 * kGTP + jt)), t16[0] | (t16[1] << 16),
               t16[2] | (t16[3] << 16));
      if (a.tap_tern && i < L && blockIdx.y == 0 && k0 + jt < round_up64(i + 1))
        *reinterpret_cast<uint32_t*>(a.tern + (b * L + i) * round_up64(L) + k0 + jt) = t8;
    }
    if constexpr (last)
      wait_loads<0>();
    else
      wait_loads<kGLoads + RS + 1>();  // the first half's states have landed; what came after may be in flight
    wg_barrier();
    const int steps = (kend - k0 + 31) / 32;  // 32-key steps that hold a key (decisions past kend are 0)
    auto mix = [&](int hf) {
      if (last && steps <= 2 * hf) return;  // (uniform)
      const uint16_t* tr = T + l16 * kGTP + 8 * g + kGK / 2 * hf;
      const b16x8 tv[2] = {*reinterpret_cast<const b16x8*>(tr), *reinterpret_cast<const b16x8*>(tr + 32)};
      uint2 v[2][2][2];
      const char* cur = lds_g + hf * kGHalf;
      tr_step2((lds_cptr)(cur + aoff[0]), (lds_cptr)(cur + aoff[1]), v);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(b16x8, make_uint4(v[s][t][0].x, v[s][t][0].y, v[s][t][1].x, v[s][t][1].y)), tv[s],
              acc[t], 0, 0, 0);
    };
    mix(0);
    if constexpr (!last) wait_loads<RS + 1>();  // the second half's states
    wg_barrier();
    if constexpr (!last) load_states(k0 + kGK, 0);
    mix(1);
    if constexpr (!last) {
      lds_put4((lds_cptr)(reinterpret_cast<const char*>(tab + tid)), nt);  // (every wave is past its scores)
      wg_barrier();
      load_states(k0 + kGK, 1);
      asm volatile("" ::: "memory");  // the waits count on these loads before the next block's keys and bias entries
      rlo = nlo;
    }
  };
  int kl = 0;
  for (; kl + kGK < kend; kl += kGK) block(kl, std::false_type{});
  block(kl, std::true_type{});
  if (n) atomicAdd(&cnt[l16], n);
  __syncthreads();

  // E, tanh(E) and C of the lane's 8 channels of its query (two groups of four)
  const int nn = cnt[l16];
  const float winv = rnd<kBF16>(1.0f / rnd<kBF16>(static_cast<float>(nn > 1 ? nn : 1)));
  uint2 te[2], cc[2], own[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = cbase + 32 * w + 16 * t + 4 * g;
    const uint16_t* src = static_cast<const uint16_t*>(a.S) + (b * L + ir) * a.ld_s + (c < D ? c : 0);
    own[t] = *reinterpret_cast<const uint2*>(src);
  }
  float mte = 0.0f, mcc = 0.0f;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = cbase + 32 * w + 16 * t + 4 * g;
    const uint32_t ow[2] = {own[t].x, own[t].y};
    float t4[4], c4[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float s0 = __uint_as_float(r & 1 ? ow[r >> 1] & 0xffff0000u : ow[r >> 1] << 16);
      const float avg = rnd<kBF16>(acc[t][r] * winv);
      const float ev = rnd<kBF16>(s0 + rnd<kBF16>(a.ent_scale * rnd<kBF16>(avg - s0)));
      c4[r] = rnd<kBF16>(ev - s0);
      t4[r] = rnd<kBF16>(tanhf_(ev));
    }
    te[t] = make_uint2(pack_bf16x2(t4[0], t4[1]), pack_bf16x2(t4[2], t4[3]));
    cc[t] = make_uint2(pack_bf16x2(c4[0], c4[1]), pack_bf16x2(c4[2], c4[3]));
    if (c < D) {  // D is a multiple of 4
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        mte = fmaxf(mte, fabsf(t4[r]));
        mcc = fmaxf(mcc, fabsf(c4[r]));
      }
      if (i < L) {
        const int64_t o = (b * L + i) * a.ld_out + c;
        if (a.e_tanh) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.e_tanh) + o) = te[t];
        if (a.c_out) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.c_out) + o) = cc[t];
      }
    }
  }
  if constexpr (QUANT) {  // per-token codes, as entangle_mfma.hip forms them
    atomicMax(&amx[l16], __float_as_int(mte));
    atomicMax(&amx[kGQ + l16], __float_as_int(mcc));
    __syncthreads();
    uint32_t* code = reinterpret_cast<uint32_t*>(lds_g);  // [2][16][(D + 16) / 4], natural order (the states are done)
    const int cp = (D + 16) / 4;
    float sc2[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      sc2[q] = act_scale<kBF16>(__int_as_float(amx[q * kGQ + l16]), a.eps);
      int32_t rs = 0;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int c = 32 * w + 16 * t + 4 * g;
        const uint2 v2 = q == 0 ? te[t] : cc[t];
        const uint32_t vw[2] = {v2.x, v2.y};
        uint32_t cb[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = __uint_as_float(r & 1 ? vw[r >> 1] & 0xffff0000u : vw[r >> 1] << 16);
          cb[r] = __float_as_uint(fminf(fmaxf(rnd<kBF16>(v * sc2[q]), -128.0f), 127.0f) + 12582912.0f);
        }
        const uint32_t wd = pack_low_bytes(cb[0], cb[1], cb[2], cb[3]);
        if (c < D) {
          rs = __builtin_amdgcn_sdot4(static_cast<int>(wd), 0x01010101, rs, false);
          code[(q * kGQ + l16) * cp + c / 4] = wd;
        }
      }
      atomicAdd(&rsum[q * kGQ + l16], rs);
    }
    __syncthreads();
    const int groups = D / 16, ngq = static_cast<int>(a.ldq / 16);
    for (int x = tid; x < 2 * kGQ * ngq; x += kGNT) {
      const int gr = x % ngq, row = x / ngq, qq = row & (kGQ - 1), q = row / kGQ;
      if (i0 + qq >= L) continue;
      const uint4 o = gr < groups ? natural_to_layout1(*reinterpret_cast<const uint4*>(code + row * cp + 4 * gr))
                                  : make_uint4(0, 0, 0, 0);
      reinterpret_cast<uint4*>((q == 0 ? a.q_te : a.q_c) + (b * L + i0 + qq) * a.ldq)[gr] = o;
    }
    if (w == 0 && g < 2 && i < L) {  // lanes 0-15: tanh(E)'s scale and code sum, lanes 16-31: C's
      (g == 0 ? a.s_te : a.s_c)[b * L + i] = g == 0 ? sc2[0] : sc2[1];
      (g == 0 ? a.rs_te : a.rs_c)[b * L + i] = rsum[g * kGQ + l16];
    }
  }
}

template <int RS>
void launch_rs(const GlobalArgs& a, int64_t nqb, unsigned ncb, bool quant, hipStream_t st) {
  const uint16_t* qr = reinterpret_cast<const uint16_t*>(a.qr);
  const uint16_t* kr = reinterpret_cast<const uint16_t*>(a.kr);
  const unsigned nwg = static_cast<unsigned>(nqb * a.B);
  const unsigned ncu = static_cast<unsigned>(device_limits().cus);
  const unsigned fold = ncb == 1 && nwg <= 2 * ncu ? (nwg < ncu ? nwg : ncu) : nwg;
  const dim3 grid(nwg, ncb);
  if (quant)
    global_mfma_kernel<RS, true><<<grid, kGNT, kGLds, TESM_LOGGED(st, global_mfma_kernel<RS, true>)>>>(a, qr, kr, nqb,
                                                                                                 fold);
  else
    global_mfma_kernel<RS, false><<<grid, kGNT, kGLds, TESM_LOGGED(st, global_mfma_kernel<RS, false>)>>>(a, qr, kr, nqb,
                                                                                                 fold);
}

}  // namespace

// bf16 single-head layers with rows that can be read in 16-byte vectors, ranks from 16 to 128 (queries and the next
// keys are held in registers, and the rows fit the general path's workspace), lengths whose bias entries fit the
// staged slice, and offsets of one batch row's states within 32 bits.  There it is the faster path at every size
// tried, from 5 x 84 tokens (52 against 60 us for the layer) to 4 x 2048 (103 against 150).
bool global_mfma_ok(const GlobalArgs& a) {
  return a.dt == kBF16 && a.L <= kGMaxL && !a.mimo && a.H == 1 && a.R >= 16 && a.R <= 128 &&
         a.D % 16 == 0 && a.ld_s % 8 == 0 &&
         a.L * a.ld_s * 2 < (int64_t(1) << 32) && aligned(a.S, 16) && a.ld_out % 4 == 0 && aligned(a.e_tanh, 8) &&
         aligned(a.c_out, 8);
}
bool global_mfma_quantizes(const GlobalArgs& a) { return global_mfma_ok(a) && a.D <= kGC; }

int launch_global_mfma(const GlobalArgs& a, hipStream_t st) {
  const int rc = check_global(a);
  if (rc || a.B == 0 || a.L == 0) return rc;
  TESM_REQUIRE(global_mfma_ok(a), kErrInvalidArg, "global ent: not a one-pass layer");
  TESM_REQUIRE(a.embed && a.rel_scale && a.rel_bias && a.P >= 1, kErrInvalidArg, "global ent: null bias parameters");
  const bool quant = global_mfma_quantizes(a) && a.q_te != nullptr;
  TESM_REQUIRE(quant || (a.e_tanh && a.c_out), kErrInvalidArg, "global ent: null outputs");
  // 32-value steps of a row: 32 rs <= 2 R values, so bf16 rows fit the workspace of R floats each
  const int rs = a.R <= 32 ? 1 : a.R <= 64 ? 2 : 4, rp = 32 * rs;
  const int64_t half = a.R / 2, nr = (a.B * a.L * half + 255) / 256, nt = (8 * 2 * a.L + 255) / 256;
  const int64_t nqb = (a.L + kGQ - 1) / kGQ, ncb = (a.D + kGC - 1) / kGC;
  TESM_REQUIRE(nr + nt <= 0x7fffffff && nqb * a.B <= 0x7fffffff && ncb <= 65535, kErrUnsupported,
               "global ent: too large");
  global_prep_kernel<<<static_cast<unsigned>(nr + nt), 256, 0, TESM_LOGGED(st, global_prep_kernel)>>>(
      a, reinterpret_cast<uint16_t*>(a.qr), reinterpret_cast<uint16_t*>(a.kr), rp, static_cast<unsigned>(nr), 2 * a.L,
      const_cast<float*>(a.table));
  const unsigned nc = static_cast<unsigned>(ncb);
  switch (rs) {
    case 1: launch_rs<1>(a, nqb, nc, quant, st); break;
    case 2: launch_rs<2>(a, nqb, nc, quant, st); break;
    default: launch_rs<4>(a, nqb, nc, quant, st); break;
  }
  return check_launch("global ent (one pass)");
}

}  // namespace tesm
