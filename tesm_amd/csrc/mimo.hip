// TESMMIMO_Optimized (tesm_ssm/modules/tesm_mimo.py:914-1062) around the shared kernels.
//
// The reference expands every head's update into mimo_rank copies, scans each copy and runs the
// window entanglement on each, then merges with mimo_o.  Decay and window weights are shared by the
// ranks and the scan and the window mix are linear in the update, so
//   states_r = S * mimo_x[:, r]^2,  sum_r entangled_r * mimo_o[:, r] = E * c,  c = sum_r mimo_x_r^2 mimo_o_r,
// with S the scan of write * tanh(sv) and E its entangled state.  Here the one scan and the one mix
// run on S and the merge is a per-channel factor (float32 throughout, as the reference's rank tensors).
#include "linear_dev.h"
#include "mimo.h"

namespace tesm {

namespace {

template <int DT>
__global__ __launch_bounds__(256) void mimo_coef_kernel(const void* x, const void* o, int64_t H, int64_t Rm, int64_t D,
                                                        float* coef, float* x0sq) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= H * D) return;
  const int64_t h = i / D, d = i - h * D;
  float c = 0.0f;
  for (int64_t r = 0; r < Rm; ++r) {
    const int64_t k = (h * Rm + r) * D + d;
    const float xv = ld<DT>(x, k);
    c += (xv * xv) * ld<DT>(o, k);
  }
  const float x0 = ld<DT>(x, h * Rm * D + d);
  coef[i] = c;
  x0sq[i] = x0 * x0;
}

constexpr int kMixTP = 64;           // positions per workgroup
constexpr int kMixDS = 32;           // channels per block
constexpr int kMixSP = kMixDS + 8;   // state row pitch (floats): rows r and r + 4 fall in opposite bank halves
constexpr int kMixWP = kMixTP + 4;   // weight row pitch (floats)
constexpr int kMixCB = 16;           // channel blocks per workgroup
constexpr int kMixLD = 4;            // float4 state loads per thread per block: (kMixTP + 63) * 8 <= 4 * 256

// Window mix for one (batch row, head) pair, kMixTP positions x kMixCB blocks of kMixDS channels.
// Key position of window slot w is t - W + 1 + w (tesm_mimo.py:536-586); slots the reference drops
// carry weight 0.  The weights (transposed, [w][position]) are staged in LDS once; the states of one
// channel block plus its W - 1 row halo are staged per block, and the next block's states are loaded
// into registers while the current one is mixed and stored.  Each thread owns 2 positions x 4 channels
// and walks the window keeping the 2 state rows it needs in registers, so every 8 multiply-adds cost
// one state and one weight read.  Sums run over w in increasing order.  WT: 64 for mix64, else 0.
//
// W = 64 with whole 16-byte rows (the largest window, and the large preset's) takes mix64 below: here a thread reads
// 24 bytes of LDS per 8 multiply-adds, three bytes each where two keep up with the vector units.  Its loop would serve
// any window that is a multiple of 8; for smaller ones it is neither instantiated nor measured.
constexpr int kM64C = 128;                           // channels per block
constexpr int kM64Rows = kMixTP + 64;                // state rows per block (the last one is not used)
constexpr int kM64CB = 4;                            // channel blocks per workgroup
constexpr size_t kM64Lds = (kM64Rows * kM64C + 64 * kMixTP) * sizeof(float);
static_assert(2 * kM64Lds <= 160 * 1024, "two workgroups per CU");

// The general form's plan at W = 64 with 8 positions x 4 channels per thread: the 8 state rows a slot needs stay in
// registers and move up by one, so a slot's 32 multiply-adds cost one state and two weight reads of 16 bytes (half the
// general form's LDS traffic), and the last slot's rows are the positions' own states.  States go straight to LDS; two
// workgroups per CU overlap one's loads with the other's sums.  Each sum runs over the window in increasing order, as
// in the general form (same bits).  32768 positions x 8192 channels: 886 us (925 in the layer on another box), before
// 1017, with the next block's states held in registers instead 951; the vector units alone need 440 us for these 17 G
// multiply-adds, and weights as scalar operands (16 positions x 1 channel per lane) took 1560, the scalar cache being
// too small for 20 waves' weights.
template <int DT>
__device__ __forceinline__ void mix64(const MimoMixArgs& a, float* lds) {
  float* srow = lds;                         // [kM64Rows][kM64C]
  float* wtT = lds + kM64Rows * kM64C;       // [64][kMixTP]
  const int64_t b = blockIdx.z / a.H, h = blockIdx.z - b * a.H;
  const int64_t t0 = static_cast<int64_t>(blockIdx.y) * kMixTP;
  const int D = static_cast<int>(a.D), nblk = (D + kM64C - 1) / kM64C;
  const int cb0 = static_cast<int>(blockIdx.x) * kM64CB, cb1 = cb0 + kM64CB < nblk ? cb0 + kM64CB : nblk;
  const int tid = threadIdx.x;
  const int64_t C = a.H * a.D, tlo = t0 - 63;
  const int nvalid = static_cast<int>(a.L - t0 < kMixTP ? a.L - t0 : kMixTP);
  const float* Sh = a.S + b * a.L * C + h * a.D;
  // Straight to LDS, two rows per instruction.  Rows before the sequence re-read row 0 (their weights are 0, and row 0
  // is in those positions' windows), rows past it and channels past D feed only outputs that are dropped.
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  auto stage = [&](int cb) {
    const int dc = cb * kM64C + 4 * (lane & 31);
    const float* src = Sh + (dc < D ? dc : 0);
#pragma unroll
    for (int k = 0; k < kM64Rows / 8; ++k) {
      const int r = 2 * (wv + 4 * k);
      const int64_t t = tlo + r + (lane >> 5), tc = t < 0 ? 0 : (t < a.L ? t : a.L - 1);
      __builtin_amdgcn_global_load_lds(src + tc * C, (__attribute__((address_space(3))) void*)(srow + r * kM64C), 16, 0,
                                       0);
    }
  };
  stage(cb0);
  const float* wb = a.wts + ((b * a.L + t0) * a.H + h) * 64;
  const int64_t wrow = a.H * 64;
  for (int i = tid; i < kMixTP * 64; i += 256) {
    const int p = i & (kMixTP - 1), w = i / kMixTP;  // (reads by position: the stores go to consecutive words)
    wtT[w * kMixTP + p] = p < nvalid ? wb[p * wrow + w] : 0.0f;
  }
  __syncthreads();
  const int p0 = 8 * (tid >> 5), c0 = 4 * (tid & 31);
  const float* sp = srow + p0 * kM64C + c0;
  for (int cb = cb0; cb < cb1; ++cb) {
    float acc[8][4];
    float4 s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
      s[i] = *reinterpret_cast<const float4*>(sp + i * kM64C);
    }
#pragma unroll 1
    for (int w0 = 0; w0 < 64; w0 += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {  // slot w0 + u: position i's row is s[(i + u) % 8]
        const float4 wa = *reinterpret_cast<const float4*>(wtT + (w0 + u) * kMixTP + p0);
        const float4 wc = *reinterpret_cast<const float4*>(wtT + (w0 + u) * kMixTP + p0 + 4);
        const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wc.x, wc.y, wc.z, wc.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float4 x = s[(i + u) & 7];
          acc[i][0] = __builtin_fmaf(wv[i], x.x, acc[i][0]);
          acc[i][1] = __builtin_fmaf(wv[i], x.y, acc[i][1]);
          acc[i][2] = __builtin_fmaf(wv[i], x.z, acc[i][2]);
          acc[i][3] = __builtin_fmaf(wv[i], x.w, acc[i][3]);
        }
        // the row the window's move brings in; after the last slot position 0's own row stays in s[7]
        if (u < 7 || w0 < 56) s[u] = *reinterpret_cast<const float4*>(sp + (w0 + u + 8) * kM64C);
      }
    }
    const int d = cb * kM64C + c0;
    if (d < D) {
      float cf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) cf[j] = a.coef[h * a.D + d + j];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (p0 + i >= nvalid) break;
        const float4 own = s[(i + 7) & 7];  // slot 63
        const float sv[4] = {own.x, own.y, own.z, own.w};
        float te[4], cc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = sv[j] + a.ent_scale * (acc[i][j] - sv[j]);
          te[j] = tanhf_(e * cf[j]);
          cc[j] = (e - sv[j]) * cf[j];
        }
        const int64_t o = (b * a.L + t0 + p0 + i) * C + h * a.D + d;
        st4<DT>(a.te, o, te);
        st4<DT>(a.cc, o, cc);
      }
    }
    __syncthreads();  // every thread is done with this block's states
    if (cb + 1 < cb1) {
      stage(cb + 1);
      __syncthreads();
    }
  }
}

template <int DT, bool VEC, int WT>
__global__ __launch_bounds__(256, WT == 64 ? 2 : 1) void mimo_mix_kernel(MimoMixArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds_mimo[];
  if constexpr (WT == 64) {
    mix64<DT>(a, lds_mimo);
    return;
  }
  const int W = static_cast<int>(a.W);
  const int rows = kMixTP + W - 1;
  float* srow = lds_mimo;                  // [rows][kMixSP]
  float* wtT = lds_mimo + rows * kMixSP;   // [W][kMixWP]
  const int64_t bh = blockIdx.z;
  const int64_t b = bh / a.H, h = bh - b * a.H;
  const int64_t t0 = static_cast<int64_t>(blockIdx.y) * kMixTP;
  const int64_t nblk = (a.D + kMixDS - 1) / kMixDS;
  const int64_t cb0 = static_cast<int64_t>(blockIdx.x) * kMixCB;
  const int64_t cb1 = cb0 + kMixCB < nblk ? cb0 + kMixCB : nblk;
  const int tid = threadIdx.x;
  const int64_t C = a.H * a.D;
  const int64_t tlo = t0 - (W - 1);  // position of LDS row 0
  const int nvalid = static_cast<int>(a.L - t0 < kMixTP ? a.L - t0 : kMixTP);
  const float* Sh = a.S + (b * a.L) * C + h * a.D;

  // state prefetch of channel block cb into registers (rows outside [0, L) and channels past D are 0)
  float4 pre[kMixLD];
  auto prefetch = [&](int64_t cb) {
#pragma unroll
    for (int k = 0; k < kMixLD; ++k) {
      const int i = tid + k * 256;
      const int r = i >> 3, c4 = 4 * (i & 7);
      const int64_t t = tlo + r;
      const int64_t dc = cb * kMixDS + c4;
      float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (r < rows && t >= 0 && t < a.L) {
        const float* src = Sh + t * C + dc;
        if (VEC && dc + 3 < a.D) {
          v = *reinterpret_cast<const float4*>(src);
        } else {
          if (dc + 0 < a.D) v.x = src[0];
          if (dc + 1 < a.D) v.y = src[1];
          if (dc + 2 < a.D) v.z = src[2];
          if (dc + 3 < a.D) v.w = src[3];
        }
      }
      pre[k] = v;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int k = 0; k < kMixLD; ++k) {
      const int i = tid + k * 256;
      const int r = i >> 3, c4 = 4 * (i & 7);
      if (r < rows) *reinterpret_cast<float4*>(srow + r * kMixSP + c4) = pre[k];
    }
  };
  prefetch(cb0);
  const float* wb = a.wts + ((b * a.L + t0) * a.H + h) * W;
  const int64_t wrow = a.H * W;  // floats between the weights of consecutive positions
  for (int i = tid; i < kMixTP * W; i += 256) {
    const int p = i / W, w = i - p * W;
    wtT[w * kMixWP + p] = p < nvalid ? wb[p * wrow + w] : 0.0f;
  }
  stage();
  __syncthreads();
  const int p0 = 2 * (tid >> 3), c0 = 4 * (tid & 7);
  const float* sp = srow + p0 * kMixSP + c0;
  for (int64_t cb = cb0; cb < cb1; ++cb) {
    prefetch(cb + 1 < cb1 ? cb + 1 : cb);  // the last block re-reads itself (never staged)
    float acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
    float4 s0 = *reinterpret_cast<const float4*>(sp);
#pragma unroll 4
    for (int w = 0; w < W; ++w) {
      const float4 s1 = *reinterpret_cast<const float4*>(sp + (w + 1) * kMixSP);
      const float2 wv = *reinterpret_cast<const float2*>(wtT + w * kMixWP + p0);
      acc[0][0] = __builtin_fmaf(wv.x, s0.x, acc[0][0]);
      acc[0][1] = __builtin_fmaf(wv.x, s0.y, acc[0][1]);
      acc[0][2] = __builtin_fmaf(wv.x, s0.z, acc[0][2]);
      acc[0][3] = __builtin_fmaf(wv.x, s0.w, acc[0][3]);
      acc[1][0] = __builtin_fmaf(wv.y, s1.x, acc[1][0]);
      acc[1][1] = __builtin_fmaf(wv.y, s1.y, acc[1][1]);
      acc[1][2] = __builtin_fmaf(wv.y, s1.z, acc[1][2]);
      acc[1][3] = __builtin_fmaf(wv.y, s1.w, acc[1][3]);
      s0 = s1;
    }
    const int64_t d = cb * kMixDS + c0;
    float cf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) cf[j] = d + j < a.D ? a.coef[h * a.D + d + j] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (p0 + i >= nvalid) break;
      const int64_t t = t0 + p0 + i;
      const float* srq = srow + (p0 + i + W - 1) * kMixSP + c0;  // the query position's own state
      float te[4], cc[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float sv = srq[j];
        const float e = sv + a.ent_scale * (acc[i][j] - sv);
        te[j] = tanhf_(e * cf[j]);
        cc[j] = (e - sv) * cf[j];
      }
      const int64_t o = (b * a.L + t) * C + h * a.D + d;
      if (VEC && d + 3 < a.D) {
        st4<DT>(a.te, o, te);
        st4<DT>(a.cc, o, cc);
      } else {
        for (int j = 0; j < 4 && d + j < a.D; ++j) {
          st<DT>(a.te, o + j, te[j]);
          st<DT>(a.cc, o + j, cc[j]);
        }
      }
    }
    __syncthreads();  // every thread is done with this block's states
    if (cb + 1 < cb1) {
      stage();
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(256) void mimo_final_kernel(const float* S, const float* x0sq, int64_t B, int64_t L,
                                                         int64_t C, double* h_final, float* last) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= B * C) return;
  const int64_t b = i / C, c = i - b * C;
  const float v = S[(b * L + L - 1) * C + c] * x0sq[c];
  if (h_final) h_final[i] = static_cast<double>(v);
  if (last) last[i] = v;
}

// One workgroup of 16 waves per batch row.  The RoPE'd q and k rows of the sampled positions are staged in LDS once
// per group of hb heads (as many as fill the threads and fit), then a thread forms one score: its products in natural
// (h, r) order, each rounded, from two rows.  Rows longer than a slice of sl values are staged slice by slice, and the
// global branch's scores run over all heads.  VEC: rows of whole 16-byte groups; the pitch (R + 4 or R + 1) spreads
// the lanes' key rows over all banks. Bound by the staging's loads and the chain of additions.  us for 1 x 64
// positions (before: one thread per score over its own rows of q and k, bf16 and f32; in brackets a wave's lanes
// forming a score's products side by side): 4 heads of rank 256, window 64 37 and 33 (97, 39 [49, 45]); rank 64,
// window 32 30 and 26 (398, 150 [239, 219]); 2 heads of rank 16, window 8 5 (17, 10 [55, 50]); global, 4 heads of rank
// 32 10 and 11 (190, 71 [76, 68]).  A rank whose rows do not fit whole rotates each pair twice: window 1, rank 400,
// the layer 142, 131 in the bracketed form.
constexpr int kStNT = 1024;
constexpr int kStNW = kStNT / 64;
constexpr int kStLds = 144 * 1024;

template <int DT, bool VEC>
__global__ __launch_bounds__(kStNT) void mimo_stats_kernel(MimoStatsArgs a, int hb, int sl, int pitch) {
  extern __shared__ __attribute__((aligned(16))) float lds_st[];
  __shared__ int32_t cnt[2][kStNW];
  const int64_t b = blockIdx.x;
  const int R = static_cast<int>(a.R), half = R / 2, S = static_cast<int>(a.S), H = static_cast<int>(a.H);
  const int W = static_cast<int>(a.W), tid = threadIdx.x;
  // window branch: (v, h, w) over S - W + 1 complete windows; global branch: (s, t) over S x S, all heads
  const int q0 = a.global ? 0 : W - 1, nq = S - q0, rows = nq + S;
  const int per = a.global ? S * S : nq * W;  // scores of a head (global: of all)
  const bool whole = sl >= R;
  // elements r0 .. r0 + m - 1 of the rows of heads h0 .. h0 + nh - 1 (more than one only where rows are whole)
  auto stage = [&](int h0, int nh, int r0, int m) {
    const int width = whole ? half : m, n = nh * rows * width;
#pragma unroll 4
    for (int x = tid; x < n; x += kStNT) {
      const int row = x / width, c = x - row * width, hl = row / rows, rr = row - hl * rows;
      const int r = whole ? c : r0 + c, i = r < half ? r : r - half;
      const bool isq = rr < nq;
      const int64_t t = isq ? q0 + rr : rr - nq;
      const int64_t o = (b * a.L + t) * (isq ? a.ld_q : a.ld_k) + static_cast<int64_t>(h0 + hl) * R + i;
      const void* src = isq ? a.q : a.k;
      float x1, x2;
      rope_pair<DT>(ld<DT>(src, o), ld<DT>(src, o + half), a.rope[t * half + i], x1, x2);
      float* dst = lds_st + row * pitch;
      if (whole) {
        dst[i] = x1;
        dst[i + half] = x2;
      } else {
        dst[c] = r < half ? x1 : x2;
      }
    }
  };
  int32_t pos = 0, neg = 0;
  for (int h0 = 0; h0 < (a.global ? 1 : H); h0 += hb) {  // (uniform, as are the loops in it)
    const int nh = H - h0 < hb ? H - h0 : hb, n = per * nh;
    for (int e0 = 0; e0 < n; e0 += kStNT) {
      const int e = e0 + tid, hl = e / per, es = e - hl * per;
      const int qr = es / (a.global ? S : W), w = es - qr * (a.global ? S : W), kr = a.global ? w : qr + w;
      float acc = 0.0f;
      for (int h = h0; h < (a.global ? H : h0 + 1); ++h)
        for (int r0 = 0; r0 < R; r0 += sl) {
          const int m = R - r0 < sl ? R - r0 : sl;
          if (!whole || a.global || e0 == 0) {
            __syncthreads();  // every thread is done with the rows before
            stage(h, a.global ? 1 : nh, r0, m);
            __syncthreads();
          }
          if (e >= n) continue;
          const float* pq = lds_st + (hl * rows + qr) * pitch;
          const float* pk = lds_st + (hl * rows + nq + kr) * pitch;
          if constexpr (VEC) {
#pragma unroll 4
            for (int r = 0; r < m; r += 4) {
              const float4 x = *reinterpret_cast<const float4*>(pq + r), y = *reinterpret_cast<const float4*>(pk + r);
              acc += rnd<DT>(x.x * y.x);
              acc += rnd<DT>(x.y * y.y);
              acc += rnd<DT>(x.z * y.z);
              acc += rnd<DT>(x.w * y.w);
            }
          } else {
#pragma unroll 8
            for (int r = 0; r < m; ++r) acc += rnd<DT>(pq[r] * pk[r]);
          }
        }
      if (e < n) {
        const float sc = rnd<DT>(rnd<DT>(acc) / a.sqrt_r);
        const float t = sc > a.thr ? 1.0f : (sc < -a.thr ? -1.0f : 0.0f);
        pos += t > 0.0f;
        neg += t < 0.0f;
        st<DT>(a.ternary, a.global ? b * per + e : ((b * nq + qr) * a.H + h0 + hl) * a.W + w, t);
      }
    }
  }
  // wave sums, then the workgroup's
  for (int o = 32; o > 0; o >>= 1) {
    pos += __shfl_xor(pos, o);
    neg += __shfl_xor(neg, o);
  }
  if ((tid & 63) == 0) {
    cnt[0][tid >> 6] = pos;
    cnt[1][tid >> 6] = neg;
  }
  __syncthreads();
  if (tid == 0) {
    int32_t p = 0, q = 0;
    for (int k = 0; k < kStNW; ++k) {
      p += cnt[0][k];
      q += cnt[1][k];
    }
    a.counts[b * 3 + 0] = p;
    a.counts[b * 3 + 1] = q;
    a.counts[b * 3 + 2] = static_cast<int32_t>(per * (a.global ? 1 : a.H)) - p - q;
  }
}

}  // namespace

int launch_mimo_stats(const MimoStatsArgs& a, hipStream_t st) {
  TESM_REQUIRE(a.dt == kF32 || a.dt == kBF16, kErrInvalidArg, "mimo stats: dtype must be 0 or 1");
  if (a.B == 0) return kOk;
  TESM_REQUIRE(a.q && a.k && a.rope && a.ternary && a.counts, kErrInvalidArg, "mimo stats: null pointer");
  TESM_REQUIRE(a.global ? (a.S >= 1 && a.S <= a.L) : (a.W >= 1 && a.S >= a.W && a.S <= a.L), kErrInvalidArg,
               "mimo stats: need 1 <= W <= S <= L");
  TESM_REQUIRE(a.R >= 2 && a.R % 2 == 0 && a.H >= 1, kErrInvalidArg, "mimo stats: need an even R");
  TESM_REQUIRE((a.S - a.W + 1) * a.H * a.W <= 0x7fffffff, kErrUnsupported, "mimo stats: too many scores");
  TESM_REQUIRE(!a.global || a.S <= 0x7fff, kErrUnsupported, "mimo stats: too many scores");
  // whole rows where they fit, in slices of a multiple of 4 values where not; heads side by side as long as they fit
  // and the threads are not filled
  const int64_t rows = (a.global ? a.S : a.S - a.W + 1) + a.S, per = a.global ? a.S * a.S : (a.S - a.W + 1) * a.W;
  const int64_t room = kStLds / 4 / rows;  // floats of a row
  TESM_REQUIRE(room >= 16, kErrUnsupported, "mimo stats: too many sampled positions");
  const bool vec = a.R % 4 == 0;
  const int64_t whole = a.R + (a.R % 8 == 0 ? 4 : vec ? 8 : 1);
  const int64_t sl = whole <= room ? a.R : (room - 8) / 8 * 8, pitch = whole <= room ? whole : sl + 4;
  const int64_t hb = a.global || sl < a.R ? 1 : std::min({a.H, room / pitch, (kStNT + per - 1) / per});
  const size_t lds = static_cast<size_t>(hb * rows * pitch) * sizeof(float);
  if (a.dt == kBF16) {
    if (vec) mimo_stats_kernel<kBF16, true><<<static_cast<unsigned>(a.B), kStNT, lds, TESM_LOGGED(st, mimo_stats_kernel<kBF16, true>)>>>(a, static_cast<int>(hb), static_cast<int>(sl), static_cast<int>(pitch));
    else mimo_stats_kernel<kBF16, false><<<static_cast<unsigned>(a.B), kStNT, lds, TESM_LOGGED(st, mimo_stats_kernel<kBF16, false>)>>>(a, static_cast<int>(hb), static_cast<int>(sl), static_cast<int>(pitch));
  } else {
    if (vec) mimo_stats_kernel<kF32, true><<<static_cast<unsigned>(a.B), kStNT, lds, TESM_LOGGED(st, mimo_stats_kernel<kF32, true>)>>>(a, static_cast<int>(hb), static_cast<int>(sl), static_cast<int>(pitch));
    else mimo_stats_kernel<kF32, false><<<static_cast<unsigned>(a.B), kStNT, lds, TESM_LOGGED(st, mimo_stats_kernel<kF32, false>)>>>(a, static_cast<int>(hb), static_cast<int>(sl), static_cast<int>(pitch));
  }
  return check_launch("mimo stats");
}

int launch_mimo_coef(const void* mimo_x, const void* mimo_o, int dt, int64_t H, int64_t Rm, int64_t D, float* coef,
                     float* x0sq, hipStream_t st) {
  TESM_REQUIRE(dt == kF32 || dt == kBF16, kErrInvalidArg, "mimo coef: dtype must be 0 or 1");
  TESM_REQUIRE(H >= 1 && Rm >= 1 && D >= 1, kErrInvalidArg, "mimo coef: bad sizes");
  TESM_REQUIRE(mimo_x && mimo_o && coef && x0sq, kErrInvalidArg, "mimo coef: null pointer");
  const unsigned nb = static_cast<unsigned>((H * D + 255) / 256);
  if (dt == kBF16)
    mimo_coef_kernel<kBF16><<<nb, 256, 0, TESM_LOGGED(st, mimo_coef_kernel<kBF16>)>>>(mimo_x, mimo_o, H, Rm, D, coef, x0sq);
  else
    mimo_coef_kernel<kF32><<<nb, 256, 0, TESM_LOGGED(st, mimo_coef_kernel<kF32>)>>>(mimo_x, mimo_o, H, Rm, D, coef, x0sq);
  return check_launch("mimo coef");
}

int launch_mimo_mix(const MimoMixArgs& a, hipStream_t st) {
  TESM_REQUIRE(a.dt == kF32 || a.dt == kBF16, kErrInvalidArg, "mimo mix: dtype must be 0 or 1");
  TESM_REQUIRE(a.W >= 1 && a.W <= 64 && a.H >= 1 && a.D >= 1, kErrInvalidArg, "mimo mix: bad sizes");
  TESM_REQUIRE(a.S && a.wts && a.coef && a.te && a.cc, kErrInvalidArg, "mimo mix: null pointer");
  if (a.B == 0 || a.L == 0) return kOk;
  TESM_REQUIRE(a.B * a.H <= 65535 && (a.L + kMixTP - 1) / kMixTP <= 65535, kErrUnsupported, "mimo mix: grid too large");
  static_assert((kMixTP + 63) * (kMixDS / 4) <= kMixLD * 256, "state prefetch must cover the block and its halo");
  const int64_t nblk = (a.D + kMixDS - 1) / kMixDS;
  const dim3 grid(static_cast<unsigned>((nblk + kMixCB - 1) / kMixCB), static_cast<unsigned>((a.L + kMixTP - 1) / kMixTP),
                  static_cast<unsigned>(a.B * a.H));
  const size_t lds = static_cast<size_t>(((kMixTP + a.W - 1) * kMixSP + a.W * kMixWP) * sizeof(float));
  // float4 state loads and 4-wide stores need every channel group 4-aligned in memory
  const bool vec = a.D % 4 == 0 && (a.H * a.D) % 4 == 0 && reinterpret_cast<uintptr_t>(a.S) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(a.te) % (a.dt == kBF16 ? 8 : 16) == 0 &&
                   reinterpret_cast<uintptr_t>(a.cc) % (a.dt == kBF16 ? 8 : 16) == 0;
  // mix64's blocks are 128 channels, the general form's 32, so a last block that is mostly padding costs more there than
  // the form gains.  The layer in us, mix64 and (general): 8 x 800 positions, 8 heads, f32 D 64 140 (133), 96 169 (164),
  // 112 178 (181), 192 246 (239), 256 279 (282); 1 x 4000, 4 heads, whose workgroups are all resident at once, D 32 81.5
  // (80.0), 64 84.8 (85.9), 132 109 (107), 160 107 (108), 192 112 (115).
  const int64_t nb64 = (a.D + kM64C - 1) / kM64C, last = a.D - (nb64 - 1) * kM64C;
  const dim3 g64(static_cast<unsigned>((nb64 + kM64CB - 1) / kM64CB), grid.y, grid.z);
  const bool resident = static_cast<int64_t>(g64.x) * g64.y * g64.z <= 2 * std::max(device_limits().cus, 1);
  const bool full = 6 * (kM64C - last) <= nb64 * kM64C || (resident && last >= (nb64 == 1 ? kM64C / 2 : kM64C / 4));
  const bool m64 = vec && a.W == 64 && a.D < (int64_t(1) << 30) && full;
  if (a.dt == kBF16) {
    if (m64) mimo_mix_kernel<kBF16, true, 64><<<g64, 256, kM64Lds, TESM_LOGGED(st, mimo_mix_kernel<kBF16, true, 64>)>>>(a);
    else if (vec) mimo_mix_kernel<kBF16, true, 0><<<grid, 256, lds, TESM_LOGGED(st, mimo_mix_kernel<kBF16, true, 0>)>>>(a);
    else mimo_mix_kernel<kBF16, false, 0><<<grid, 256, lds, TESM_LOGGED(st, mimo_mix_kernel<kBF16, false, 0>)>>>(a);
  } else {
    if (m64) mimo_mix_kernel<kF32, true, 64><<<g64, 256, kM64Lds, TESM_LOGGED(st, mimo_mix_kernel<kF32, true, 64>)>>>(a);
    else if (vec) mimo_mix_kernel<kF32, true, 0><<<grid, 256, lds, TESM_LOGGED(st, mimo_mix_kernel<kF32, true, 0>)>>>(a);
    else mimo_mix_kernel<kF32, false, 0><<<grid, 256, lds, TESM_LOGGED(st, mimo_mix_kernel<kF32, false, 0>)>>>(a);
  }
  return check_launch("mimo mix");
}

int launch_mimo_final(const float* S, const float* x0sq, int64_t B, int64_t L, int64_t C, double* h_final,
                      float* last, hipStream_t st) {
  if (B == 0 || L == 0 || (!h_final && !last)) return kOk;
  TESM_REQUIRE(S && x0sq, kErrInvalidArg, "mimo final: null pointer");
  const unsigned nb = static_cast<unsigned>((B * C + 255) / 256);
  mimo_final_kernel<<<nb, 256, 0, TESM_LOGGED(st, mimo_final_kernel)>>>(S, x0sq, B, L, C, h_final, last);
  return check_launch("mimo final");
}

}  // namespace tesm
