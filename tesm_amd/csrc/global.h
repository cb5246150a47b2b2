// Global (causal, full-history) ternary entanglement: TESM_SISO with entanglement_window = 0
// (tesm_ssm/modules/tesm.py:963-1063, torch branch 1040-1052) and TESMMIMO_Optimized's global branch
// (tesm_mimo.py:590-687, torch branch 655-687).
#pragma once

#include "entangle.h"

namespace tesm {

// Relative-position bias (tesm.py:970-982).  Positions are arange(L) in the layer dtype and the bias
// of a (query, key) pair is a function of rel = dt(pos_q - pos_k) alone, an integer-valued number in
// [0, 2L) for causal pairs; table[r] = that function at rel = r, a float holding a dt value:
//   ang_p = dt(r * freq_p), freq_p = dt(dt(p * pi) / 1000), p = 1 .. P
//   b = dt(dt(sum_p dt(dt(sin ang_p) * e_p)) + dt(sum_p dt(dt(cos ang_p) * e_p)))
//   table[r] = dt(dt(b * scale) + bias)
// embed (P), scale and bias are float32 arrays holding the parameters rounded to dt.
int launch_global_bias_table(int dt, int64_t n, const float* embed, int64_t P, const float* scale, const float* bias,
                             float* table, hipStream_t st);

struct GlobalArgs {
  int dt = 0;
  int mimo = 0;                  // 0: SISO (E = S + scale (A - S)); 1: MIMO (E = A, outputs scaled by coef)
  int64_t B = 0, L = 0, H = 1, R = 0, D = 0;  // q / k: H heads of R (RoPE per head); states: H*D channels
  const void* q = nullptr;       // (b, t, h, r) raw at q[(b*L + t)*ld_q + h*R + r]
  int64_t ld_q = 0;
  const void* k = nullptr;
  int64_t ld_k = 0;
  const float2* rope = nullptr;  // (L, R/2), positions 0..L-1
  const void* q_add = nullptr;   // optional SISO cross-layer query bias, added after RoPE
  int64_t ld_qadd = 0;
  const float* table = nullptr;  // bias table over rel in [0, 2L)
  float thr = 0.0f;              // rounded to dt
  float sqrt_div = 1.0f;         // float(sqrt(H*R))
  float ent_scale = 0.0f;
  const void* S = nullptr;       // states (b, t, c) at S[(b*L + t)*ld_s + c], c < H*D; dt (SISO) or f32 (MIMO)
  int64_t ld_s = 0;
  const float* coef = nullptr;   // MIMO: (H*D) rank merge factors
  void* e_tanh = nullptr;        // (b, t, c) at [(b*L + t)*ld_out + c], dt: tanh(E) (MIMO: tanh(E * coef))
  void* c_out = nullptr;         // E - S (MIMO: (E - S) * coef)
  int64_t ld_out = 0;
  int8_t* tern = nullptr;        // workspace (B, L, ldt) ternary decisions, ldt = round_up(L, 64); a row's
                                 // columns past its 64-key diagonal tile are left unwritten
  int32_t* count = nullptr;      // workspace (B, L) nonzero decisions per query
  uint16_t* states_t = nullptr;  // workspace (B, H*D, ldt) bf16 states transposed (bf16 SISO layers only)
  float* qr = nullptr;           // workspace (B, L, H*R) RoPE'd queries (+ cross-layer bias)
  float* kr = nullptr;           // workspace (B, L, H*R) RoPE'd keys
  // the one-pass kernel (global_mfma.hip): the bias parameters (it fills the table itself), whether to leave the
  // decisions in tern, and the int8 codes of tanh(E) and C (layout 1), formed in place where q_te is set and
  // global_mfma_quantizes; e_tanh and c_out may then be null
  const float* embed = nullptr;
  int64_t P = 0;
  const float* rel_scale = nullptr;
  const float* rel_bias = nullptr;
  bool tap_tern = false;
  int8_t* q_te = nullptr;
  float* s_te = nullptr;
  int32_t* rs_te = nullptr;
  int8_t* q_c = nullptr;
  float* s_c = nullptr;
  int32_t* rs_c = nullptr;
  int64_t ldq = 0;
  float eps = 1e-5f;
};

__device__ __forceinline__ int64_t round_up64(int64_t v) { return (v + 63) & ~int64_t(63); }

// One entry of the bias table per eight lanes (lane `e & 7` of entry `e >> 3`, each over every eighth frequency; the
// partial sums meet by shuffles).
template <int DT>
__device__ __forceinline__ void global_bias_entry(int64_t e, int64_t n, const float* embed, int64_t P,
                                                  const float* scale, const float* bias, float* table) {
  const int64_t r = e >> 3;
  const int part = static_cast<int>(e & 7);
  const float rel = rnd<DT>(static_cast<float>(r < n ? r : 0));
  constexpr float kPi = 3.14159265358979323846f;
  float ssum = 0.0f, csum = 0.0f;
  for (int64_t p = part; p < P; p += 8) {
    const float fr = rnd<DT>(rnd<DT>(static_cast<float>(p + 1) * kPi) / 1000.0f);
    const float ang = rnd<DT>(rel * fr);
    const float em = embed[p];
    ssum += rnd<DT>(rnd<DT>(sinf(ang)) * em);
    csum += rnd<DT>(rnd<DT>(cosf(ang)) * em);
  }
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) {
    ssum += __shfl_xor(ssum, o);
    csum += __shfl_xor(csum, o);
  }
  if (r >= n || part != 0) return;
  const float b = rnd<DT>(rnd<DT>(ssum) + rnd<DT>(csum));
  table[r] = rnd<DT>(rnd<DT>(b * scale[0]) + bias[0]);
}

int64_t global_tern_pitch(int64_t L);
// bytes of the transposed-states workspace (zero where the states are float32)
int64_t global_states_t_bytes(int dt, int mimo, int64_t B, int64_t L, int64_t C);
int check_global(const GlobalArgs& a);  // sizes and inputs, as both paths need them
int launch_global_ent(const GlobalArgs& a, hipStream_t st);

// Scores, decisions and mix in one pass over the keys: the layers it takes, whether it also quantizes, its launch.
bool global_mfma_ok(const GlobalArgs& a);
bool global_mfma_quantizes(const GlobalArgs& a);
int launch_global_mfma(const GlobalArgs& a, hipStream_t st);

}  // namespace tesm
