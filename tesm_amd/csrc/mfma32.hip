// INT2 x INT8 products of more than 32 rows (and wide ones of fewer) on v_mfma_i32_32x32x32_i8, which on
// gfx950 delivers about twice the int8 rate of the 16x16x64 form.
//
// A workgroup owns BM x BN outputs: WM x WN waves, each TM x TN tiles of 32 x 32.  Weights are the MFMA's A
// operand: in k-step s (of the 4 of a 128-code K tile) lane L feeds weight column L%32 with chunk 4*(L/32) + s
// (one packed dword, unpacked in registers) and activation row L%32 with the same 16-code chunk; any pairing
// of chunks to k-steps gives the same sums as long as both operands use it, and this one makes a lane's four
// weight dwords of a K tile one 16-byte read.  Accumulator element r of lane L is weight column
// 8*(r/4) + 4*(L/32) + r%4 and activation row L%32.
//
// Pipeline.  K tiles go straight from memory to LDS (16-byte buffer loads with the LDS destination, no staging
// registers) into NS stages.  A fragment's LDS reads are issued one k-step ahead of its MFMAs, across the K tile
// boundary too: the one barrier of a K tile stands in its middle, where a wave (a) knows its loads of the next tile
// landed (vmcnt), (b) meets the others, so the next tile may be read from the last k-step on and the previous tile's
// stage may be refilled.  With the wait at a tile's start instead, and two stages, every tile paid an LDS round
// trip and the slowest wave's load (2048 x 4096 x 4096 37.7 us, now 36.8; 4095 x 3744 x 1024 27.5, now 23.8).
//
// What bounds it: products of many rounds of tiles run at 2.1-2.3 POP/s, where the chip's power limit lies for these
// operands (the library int8 product reaches 2.25 on random codes; the same kernel on all-zero codes is 1.4 times
// faster, 167 against 233 us at 4096 x 14848 x 4096; tiles from 128x128 to 256x256, 64x64 to 128x64 per wave and 2 to
// 4 stages all end within 10 % of each other): 8192 x 34816 x 4096 1025 us, 4096 x 14848 x 4096 233 (the two-stage
// loop 1099 and 265).  A round or two lose part of that to the first K tiles' latency, the stores and the rounds' ends
// (2048 x 4096 x 4096 1.87 POP/s, 4095 x 1024 x 2816 1.36, 8192 x 2432 x 768 1.22), the output gate to its one
// workgroup per CU (4096 x 4096 x 2 x 2048 1.64).  Small ones are bound by the latency of the first tiles and by idle
// CUs, hence the K groups: KS groups of waves in one workgroup take K tiles g, g + KS, ... into stages of their own,
// and their exact int32 sums are added in LDS, so a 32 x 64 tile with a quarter of the K loop per group replaces
// 64 x 128 tiles on a fifth of the CUs (512 x 768 x 3072 11.8 -> 6.0 us; 512 x 768 x 768 5.5 -> 4.3).
//
// Two-product epilogues: SwiGLU's products share the activations, so one K loop reads them once against both
// weight tiles (it ran one K loop after the other: 4095 x 2816 x 1024 53.8 us); the output gate's products follow
// each other in one pipeline.
//
// LDS images (bank model measured on the device: 16-byte reads are served 16 lanes per pass over 256 bytes): one
// load instruction moves 64 lanes x 16 bytes into 1 KB in lane order, so the layouts are chosen through the lanes'
// global addresses: activation rows in blocks of 8 rows x 8 chunks (chunk q of row r in slot
// r*8 + (q ^ ((r/2) % 8))), weights in blocks of 32 columns x 2 halves (half h of column n in slot
// 2n + (h ^ ((n/8) % 2))); both make the fragment reads hit 16 distinct 16-byte slots of 256 bytes.
#include "linear_dev.h"

namespace tesm {

namespace {

// Loads to LDS through a buffer resource rather than global_load_lds: the compiler counts that instruction as one
// that may also touch LDS out of order, and waits for every outstanding LDS read (lgkmcnt(0)) wherever one is
// needed while such a load is in flight, which undoes the fragment prefetch (4096 x 14848 x 4096: 242 us, 231 with
// buffer loads; 8192 x 34816 x 4096, then walked by fours: 1108, 1056).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffffu, 0x00027000);
}
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t buf, char* dst, uint32_t off, int koff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (__attribute__((address_space(3))) void*)(dst), 16, off, koff, 0, 0);
}

__device__ __forceinline__ int a32_off(int row, int q) { return 16 * (row * 8 + (q ^ ((row >> 1) & 7))); }
__device__ __forceinline__ int b32_off(int col, int h) { return 16 * (col * 2 + (h ^ ((col >> 3) & 1))); }

template <int WM, int WN, int TM, int TN, int KS, int NS, int EPI, int OUT_DT>
struct Tile32 {
  static constexpr bool DUAL = epi_dual(EPI);
  static constexpr bool SHARE = EPI == kEpiSwiGLU;  // both products read one set of activations
  static constexpr int NACC = DUAL ? 2 : 1;
  static constexpr int NWT = SHARE ? 2 : 1;  // weight tiles per K tile
  static constexpr int NG = WM * WN, NW = NG * KS, NT = NW * 64;
  static constexpr int BM = WM * TM * 32, BN = WN * TN * 32, BK = 128;
  static constexpr int A_BYTES = BM * BK, W_BYTES = BN * BK / 4;
  static constexpr int SUB = A_BYTES + NWT * W_BYTES;  // one group's K tile
  static constexpr int STAGE = SUB * KS;
  static constexpr int NA = BM / 8, NB = BN / 32, PER = NA + NWT * NB;  // 1 KB blocks
  static constexpr int D = (PER * KS + NW - 1) / NW;  // loads per wave and stage (the last block is loaded twice
                                                      // where they do not divide: the same bytes to the same place)
  static constexpr int ES = OUT_DT == kBF16 ? 2 : 4;
  static constexpr int RED = (KS - 1) * NG * NACC * TM * TN * 4096;  // partial sums of the other K groups
  static constexpr int SLAB = 32 * (TN * 32 * ES + 16);              // a wave's 32 rows x TN column tiles
  static constexpr int SMEM = std::max(NS * STAGE, RED + NG * SLAB);
  static_assert(NS >= 3 && (NS - 2) * D < 64, "loads in flight");
};

// acc[p][i][j]: product p, row tile i, column tile j of the wave's group (with KS > 1 a partial sum).
template <class T, int WN, int TM, int TN, int KS, int NS>
__device__ __forceinline__ void mfma32_loop(const LinearArgs& a, int64_t m0, int64_t n0, v16i (&acc)[T::NACC][TM][TN],
                                            char* smem) {
  const int t = threadIdx.x;
  __builtin_assume(t < T::NT);
  const int lane = t & 63, wall = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kg = wall / T::NG, w = wall % T::NG;
  const int wm = w / WN, wn = w % WN;
  constexpr int SEQ = T::DUAL && !T::SHARE ? 2 : 1;  // products one after the other
  // Each of the wave's D blocks: its buffer (the tile's rows of an operand, so offsets fit 32 bits), the lane's
  // offset in it (rows past M and columns past N re-read the last one and feed only outputs that are never stored),
  // and its K group.  The K position is the scalar offset, so a load costs no address arithmetic.
  __amdgpu_buffer_rsrc_t buf[SEQ][T::D];
  uint32_t off[SEQ][T::D];
  int dst[T::D], adv[T::D], grp[T::D];
#pragma unroll
  for (int i = 0; i < T::D; ++i) {
    const int b0 = wall + i * T::NW, blk = b0 < T::PER * KS ? b0 : T::PER * KS - 1;
    const int g = blk / T::PER, bb = blk % T::PER;
    const bool is_q = bb < T::NA;
    const int wt = T::SHARE && bb >= T::NA + T::NB ? 1 : 0, cb = (bb - T::NA) % T::NB;
    const int row = is_q ? bb * 8 + (lane >> 3) : cb * 32 + (lane >> 1);  // row of the tile, or column
    const int chunk = is_q ? (lane & 7) ^ ((row >> 1) & 7) : (lane & 1) ^ ((row >> 3) & 1);
    const int64_t last = is_q ? a.M - 1 - m0 : a.N - 1 - n0;
#pragma unroll
    for (int p = 0; p < SEQ; ++p) {
      const LinearOperand& o = a.op[p];
      const LinearOperand& ow = a.op[T::SHARE ? wt : p];
      const char* base = is_q ? reinterpret_cast<const char*>(o.q) + m0 * o.ldq
                              : reinterpret_cast<const char*>(ow.w) + n0 * ow.ldw;
      buf[p][i] = tile_buffer(base);
      off[p][i] = static_cast<uint32_t>((row < last ? row : last) * (is_q ? o.ldq : ow.ldw)) + 16 * chunk;
    }
    grp[i] = g;
    adv[i] = is_q ? T::BK : T::BK / 4;
    dst[i] = g * T::SUB + bb * 1024;  // (A_BYTES and W_BYTES are whole blocks)
  }
  const int nk = static_cast<int>(a.Kp / T::BK);
  const int ns = (nk + KS - 1) / KS;  // steps of one product: a K tile per group
  const int steps = SEQ * ns;
  auto issue_p = [&](int kt, char* stage, const __amdgpu_buffer_rsrc_t (&bf)[T::D], const uint32_t (&of)[T::D]) {
#pragma unroll
    for (int i = 0; i < T::D; ++i) {
      int k = kt * KS + grp[i];
      k = k < nk ? k : nk - 1;  // (past the last tile: re-reads it, so every wave's count stays the same)
      lds_dma16(bf[i], stage + dst[i], of[i], k * adv[i]);
    }
  };
  auto issue = [&](int kt, int st) {
    char* stage = smem + st * T::STAGE;
    if (SEQ == 2 && kt >= ns)
      issue_p(kt - ns, stage, buf[SEQ - 1], off[SEQ - 1]);
    else
      issue_p(kt, stage, buf[0], off[0]);
  };
  const int hq = 4 * (lane >> 5);
  int ar[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) ar[s] = kg * T::SUB + a32_off(wm * TM * 32 + (lane & 31), hq + s);
  const int br = kg * T::SUB + T::A_BYTES + b32_off(wn * TN * 32 + (lane & 31), lane >> 5);
  constexpr int NB = T::NWT * TN;
  v4i bw[2][NB], af[2][TM];
  auto read_a = [&](const char* cur, int s, v4i (&f)[TM]) {
#pragma unroll
    for (int i = 0; i < TM; ++i) f[i] = *reinterpret_cast<const v4i*>(cur + ar[s] + i * 4096);
  };
  auto read_b = [&](const char* cur, v4i (&f)[NB]) {
#pragma unroll
    for (int p = 0; p < T::NWT; ++p)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        f[p * TN + j] = *reinterpret_cast<const v4i*>(cur + br + p * T::W_BYTES + j * 1024);
  };
  auto mma = [&](int prod, const v4i (&b)[NB], const v4i (&f)[TM], int s) {
#pragma unroll
    for (int p = 0; p < T::NWT; ++p)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const v4i bf = unpack_frag(static_cast<uint32_t>(b[p * TN + j][s]));
        v16i(&c)[TM][TN] = acc[T::SHARE ? p : prod];
#pragma unroll
        for (int i = 0; i < TM; ++i) c[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf, f[i], c[i][j], 0, 0, 0);
      }
  };
  // scheduling barriers keep the compiler from sinking the next fragments' reads behind the MFMAs
  int st = 0;
  auto tile = [&](int kt, int prod, v4i (&b)[NB], v4i (&bn)[NB]) {
    const char* cur = smem + st * T::STAGE;
    const int nx = st + 1 == NS ? 0 : st + 1, pv = st == 0 ? NS - 1 : st - 1;
    const char* nxt = smem + nx * T::STAGE;
    const bool live = KS == 1 || (kt - prod * ns) * KS + kg < nk;  // (wave-uniform)
    read_a(cur, 1, af[1]);
    __builtin_amdgcn_sched_barrier(0);
    if (live) mma(prod, b, af[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(cur, 2, af[0]);
    __builtin_amdgcn_sched_barrier(0);
    if (live) mma(prod, b, af[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    read_a(cur, 3, af[1]);
    wait_vmcnt<(NS - 3) * T::D>();  // this wave's loads of tile kt + 1 have landed
    __builtin_amdgcn_s_barrier();   // ... every wave's, and every wave is done with tile kt - 1
    asm volatile("" ::: "memory");  // (orders the compiler only: an acquire fence would wait for the reads above)
    issue(kt + NS - 1, pv);         // into the stage tile kt - 1 used
    __builtin_amdgcn_sched_barrier(0);
    if (live) mma(prod, b, af[0], 2);
    __builtin_amdgcn_sched_barrier(0);
    read_b(nxt, bn);
    read_a(nxt, 0, af[0]);
    __builtin_amdgcn_sched_barrier(0);
    if (live) mma(prod, b, af[1], 3);
    __builtin_amdgcn_sched_barrier(0);
    st = nx;
  };
#pragma unroll
  for (int g = 0; g < NS - 1; ++g) issue(g, g);
  wait_vmcnt<(NS - 2) * T::D>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  read_b(smem, bw[0]);
  read_a(smem, 0, af[0]);
  if constexpr (SEQ == 2) {
    int kt = 0;
    for (; kt + 2 <= ns; kt += 2) {
      tile(kt, 0, bw[0], bw[1]);
      tile(kt + 1, 0, bw[1], bw[0]);
    }
    if (kt < ns) {  // an odd number of steps: the second product starts on the other weight registers
      tile(kt, 0, bw[0], bw[1]);
      ++kt;
      for (; kt + 2 <= steps; kt += 2) {
        tile(kt, 1, bw[1], bw[0]);
        tile(kt + 1, 1, bw[0], bw[1]);
      }
      if (kt < steps) tile(kt, 1, bw[1], bw[0]);
    } else {
      for (; kt + 2 <= steps; kt += 2) {
        tile(kt, 1, bw[0], bw[1]);
        tile(kt + 1, 1, bw[1], bw[0]);
      }
    }
  } else {
    int kt = 0;
    for (; kt + 2 <= steps; kt += 2) {
      tile(kt, 0, bw[0], bw[1]);
      tile(kt + 1, 0, bw[1], bw[0]);
    }
    if (kt < steps) tile(kt, 0, bw[0], bw[1]);
  }
  wait_vmcnt<0>();  // the re-reads past the last tile: the stages are reused by the epilogue
  __syncthreads();
}

// Orders a wave's own LDS accesses (its slab is private: no other wave waits for it).
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); }

// A wave's 32 rows x TN column tiles to its LDS slab, four consecutive columns per lane and group.  v(j, g, out)
// gives the four values of tile j's group g (columns 8g + 4*(lane/32) ..).
template <int OUT_DT, int TN, class F>
__device__ __forceinline__ void fill_slab32(char* slab, F v) {
  constexpr int ES = OUT_DT == kBF16 ? 2 : 4, PITCH = TN * 32 * ES + 16;
  const int lane = threadIdx.x & 63;
  wave_lds_fence();  // the slab's previous contents are consumed
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float x[4];
      v(j, g, x);
      char* p = slab + (lane & 31) * PITCH + (32 * j + 8 * g + 4 * (lane >> 5)) * ES;
      if constexpr (OUT_DT == kBF16)
        *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
      else
        *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
    }
  wave_lds_fence();
}

// The slab's rows as 16-byte chunks, so a store instruction covers whole row segments (128 bytes for two bf16 tiles).
template <int OUT_DT, int TN>
__device__ __forceinline__ void store_tiles32(const LinearArgs& a, const char* slab, int64_t mb, int64_t nb) {
  constexpr int ES = OUT_DT == kBF16 ? 2 : 4, RB = TN * 32 * ES, PITCH = RB + 16, CPR = RB / 16, VPC = 16 / ES;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int it = 0; it < 32 * CPR / 64; ++it) {
    const int idx = it * 64 + lane, row = idx / CPR, ch = idx % CPR;
    const int64_t m = mb + row, n = nb + ch * VPC;
    if (m >= a.M || n >= a.N) continue;
    const uint4 d = *reinterpret_cast<const uint4*>(slab + row * PITCH + ch * 16);
    char* dst = static_cast<char*>(a.out) + (m * a.ldo + n) * ES;
    if (n + VPC <= a.N) {
      *reinterpret_cast<uint4*>(dst) = d;
    } else {
      const uint32_t wd[4] = {d.x, d.y, d.z, d.w};
      for (int e = 0; e < a.N - n; ++e) {
        if constexpr (OUT_DT == kBF16)
          reinterpret_cast<uint16_t*>(dst)[e] = static_cast<uint16_t>(wd[e >> 1] >> (16 * (e & 1)));
        else
          reinterpret_cast<uint32_t*>(dst)[e] = wd[e];
      }
    }
  }
}

// The slab's rows to outputs that are not in whole 16-byte rows: U (an element, a bf16 pair where rows start on four
// bytes, or 8 bytes where all rows are in whole ones) per lane, a store instruction covering whole rows again.  From the accumulators, four columns of 32 rows
// per instruction, the stores touched a memory line per lane and cost as much as the product (us, M x N x K: 4093 x 4093
// x 512 31.6 -> 20.3, f32 4093 x 3965 x 512 57.0 -> 19.3; 964 x 7932 x 1100 20.7 -> 16.6, f32 964 x 7835 x 4096 54.4 ->
// 35.9; geometric mean of 120 sizes 1.48).
template <class U, int ES, int RB>
__device__ __forceinline__ void store_rows32(const LinearArgs& a, const char* slab, int64_t mb, int64_t nb) {
  constexpr int S = sizeof(U), UPR = RB / S, RPI = 64 / UPR, PITCH = RB + 16;  // units per row, rows per instruction
  static_assert(UPR <= 64 && 64 % UPR == 0);
  const int lane = threadIdx.x & 63, u = lane % UPR;
  const int64_t n = nb + u * (S / ES), rows = a.M - mb;
  if (n >= a.N) return;
  const bool whole = n + S / ES <= a.N;  // (else the first element of a pair)
  const char* src = slab + (lane / UPR) * PITCH + u * S;
  char* dst = static_cast<char*>(a.out) + ((mb + lane / UPR) * a.ldo + n) * ES;
#pragma unroll 8
  for (int row = lane / UPR; row < 32; row += RPI) {
    if (row >= rows) break;
    const U d = *reinterpret_cast<const U*>(src);
    if (whole)
      *reinterpret_cast<U*>(dst) = d;
    else
      *reinterpret_cast<uint16_t*>(dst) = static_cast<uint16_t>(d);
    src += RPI * PITCH;
    dst += RPI * a.ldo * ES;
  }
}

// A wave's 32 rows x TN column tiles of an input, in 16-byte chunks along the rows (past M and N the last row and the
// row's last whole chunk again), ...
using Chunk16 = uint32_t __attribute__((ext_vector_type(4)));
template <int OUT_DT, int TN>
__device__ __forceinline__ void load_rows32(const LinearArgs& a, const void* p, int64_t ld, int64_t mb, int64_t nb,
                                            Chunk16 (&d)[TN * (OUT_DT == kBF16 ? 2 : 4)]) {
  constexpr int ES = OUT_DT == kBF16 ? 2 : 4, CPR = TN * 2 * ES, VPC = 16 / ES;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int it = 0; it < TN * ES; ++it) {
    const int64_t m = mb + (it * 64 + lane) / CPR, n = nb + lane % CPR * VPC;
    const int64_t e = (m < a.M ? m : a.M - 1) * ld + (n < a.N ? n : a.N - VPC);
    d[it] = *reinterpret_cast<const Chunk16*>(static_cast<const char*>(p) + e * ES);
  }
}

// ... to the slab, ...
template <int OUT_DT, int TN>
__device__ __forceinline__ void slab_chunks32(char* slab, const Chunk16 (&d)[TN * (OUT_DT == kBF16 ? 2 : 4)]) {
  constexpr int ES = OUT_DT == kBF16 ? 2 : 4, PITCH = TN * 32 * ES + 16, CPR = TN * 2 * ES;
  const int lane = threadIdx.x & 63;
  wave_lds_fence();  // the slab's previous contents are consumed
#pragma unroll
  for (int it = 0; it < TN * ES; ++it)
    *reinterpret_cast<Chunk16*>(slab + (it * 64 + lane) / CPR * PITCH + lane % CPR * 16) = d[it];
  wave_lds_fence();
}

// (both for rows that are not in whole 16-byte chunks: an element per lane, or a bf16 pair or 8 bytes where all rows
// are in whole ones)
template <class U, int ES, int RB>
__device__ __forceinline__ void slab_units32(const LinearArgs& a, char* slab, const void* p, int64_t ld, int64_t mb,
                                             int64_t nb) {
  constexpr int S = sizeof(U), UPR = RB / S, RPI = 64 / UPR, PITCH = RB + 16;  // units per row, rows per instruction
  static_assert(UPR <= 64 && 64 % UPR == 0);
  const int lane = threadIdx.x & 63, u = lane % UPR, r0 = lane / UPR;
  const int64_t n = nb + u * (S / ES);
  const char* src = static_cast<const char*>(p) + (n < a.N ? n : a.N - S / ES) * ES;
  wave_lds_fence();  // the slab's previous contents are consumed
#pragma unroll 4
  for (int r = 0; r < 32; r += RPI) {
    const int64_t m = mb + r + r0;
    *reinterpret_cast<U*>(slab + (r + r0) * PITCH + u * S) = *reinterpret_cast<const U*>(src + (m < a.M ? m : a.M - 1) * ld * ES);
  }
  wave_lds_fence();
}

// ... and into the accumulators' order: f[j][g] holds the lane's four columns of tile j's group g, float32 bits or two
// bf16 pairs.
template <int OUT_DT>
using Group4 = uint32_t __attribute__((ext_vector_type(OUT_DT == kBF16 ? 2 : 4)));
template <int OUT_DT, int TN>
__device__ __forceinline__ void slab_groups32(const char* slab, Group4<OUT_DT> (&f)[TN][4]) {
  constexpr int ES = OUT_DT == kBF16 ? 2 : 4, PITCH = TN * 32 * ES + 16;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      f[j][g] = *reinterpret_cast<const Group4<OUT_DT>*>(slab + (lane & 31) * PITCH + (32 * j + 8 * g + 4 * (lane >> 5)) * ES);
}
template <int OUT_DT>
__device__ __forceinline__ float group_at(Group4<OUT_DT> f, int r) {
  if constexpr (OUT_DT == kF32) return __uint_as_float(f[r]);
  else return __uint_as_float(r & 1 ? f[r >> 1] & 0xffff0000u : f[r >> 1] << 16);
}

// The outputs of one wave (tile rows wm*TM .., columns wn*TN ..).  slab: SLAB bytes of the wave's own.
template <int TM, int TN, int EPI, int OUT_DT>
__device__ __forceinline__ void epilogue32(const LinearArgs& a, const v16i (&acc)[epi_dual(EPI) ? 2 : 1][TM][TN],
                                           int64_t m0, int64_t n0, int wm, int wn, char* slab) {
  constexpr bool DUAL = epi_dual(EPI);
  constexpr int es = OUT_DT == kBF16 ? 2 : 4;
  const int lane = threadIdx.x & 63;
  const LinearOperand& o0 = a.op[0];
  const LinearOperand& o1 = a.op[1];
  float inv0[TM], inv1[TM];
  int32_t rs0[TM], rs1[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + (wm * TM + i) * 32 + (lane & 31);
    const int64_t mc = m < a.M ? m : a.M - 1;
    inv0[i] = o0.s_x[mc];
    rs0[i] = o0.rowsum[mc];
    inv1[i] = DUAL ? o1.s_x[mc] : 1.0f;
    rs1[i] = DUAL ? o1.rowsum[mc] : 0;
  }
  const float cws = o0.c_w[0], cws1 = DUAL ? o1.c_w[0] : 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    inv0[i] = 1.0f / inv0[i];
    inv1[i] = 1.0f / inv1[i];
  }
  const bool a16 = reinterpret_cast<uintptr_t>(a.out) % 16 == 0 && (a.ldo * es) % 16 == 0;
  const bool tensor = !o0.c_w_per_row && !(DUAL && o1.c_w_per_row) && !a.acc_dump;
  if (a16 && tensor && EPI != kEpiOutputGate && !a.bias) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t nb = n0 + wn * TN * 32;
      int kind[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) kind[j] = EPI == kEpiGates ? gate_region(a, nb + 32 * j) : 0;
      fill_slab32<OUT_DT, TN>(slab, [&](int j, int g, float (&v)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (static_cast<float>(acc[0][i][j][4 * g + r] - rs0[i]) * inv0[i]) * cws;
        if constexpr (EPI == kEpiGates) gate_act4<OUT_DT>(a, kind[j], nb + 32 * j + 8 * g + 4 * (lane >> 5), v);
        if constexpr (DUAL) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v1 = (static_cast<float>(acc[DUAL ? 1 : 0][i][j][4 * g + r] - rs1[i]) * inv1[i]) * cws1;
            v[r] = dual_epi<EPI, OUT_DT>(rnd<OUT_DT>(v[r]), rnd<OUT_DT>(v1), 0.0f, 0.0f);
          }
        }
      });
      store_tiles32<OUT_DT, TN>(a, slab, m0 + (wm * TM + i) * 32, nb);
    }
    return;
  }
  if (EPI == kEpiStore && tensor && !a.bias) {  // unaligned: apart, so that the aligned stores stay as short
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t mb = m0 + (wm * TM + i) * 32, nb = n0 + wn * TN * 32;
      fill_slab32<OUT_DT, TN>(slab, [&](int j, int g, float (&v)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (static_cast<float>(acc[0][i][j][4 * g + r] - rs0[i]) * inv0[i]) * cws;
      });
      if constexpr (OUT_DT == kBF16)
        if ((reinterpret_cast<uintptr_t>(a.out) | static_cast<uintptr_t>(a.ldo * es)) % 4 != 0) {
          store_rows32<uint16_t, es, TN * 32 * es>(a, slab, mb, nb);
          continue;
        }
      store_rows32<uint32_t, es, TN * 32 * es>(a, slab, mb, nb);
    }
    return;
  }
  if constexpr (EPI == kEpiOutputGate) {
    // The gate's inputs go the outputs' way back, so that loads and stores cover row segments: with short K they are
    // most of the time, and in the accumulators' order each touches a memory line per lane (4095 x 5056 x 2 x 64 55.0 us ->
    // 37.9, f32 121.6 -> 44.2; 4096 x 4096 x 2 x 2048 103.5 -> 83.7, 147.7 -> 91.5; 512 x 768 x 2 x 384 7.9 -> 5.9; over
    // 330 sizes 1.38 times faster).
    // Other rows go by smaller units (3000 x 2050 x 2 x 300 38.4 us -> 25.7, f32 4095 x 2050 55.0
    // -> 36.5), in code of their own: inside one loop with these they cost the whole chunks 2 %.
    constexpr int RB = TN * 32 * es;
    auto bits = [](const void* p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) | static_cast<uintptr_t>(ld * es); };
    const uintptr_t in = bits(a.local, a.ld_local) | bits(a.gate, a.ld_gate) | static_cast<uintptr_t>(a.N * es);
    auto rows = [&](auto chunks) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int64_t mb = m0 + (wm * TM + i) * 32, nb = n0 + wn * TN * 32;
        Group4<OUT_DT> lo[TN][4], gt[TN][4];
        if constexpr (decltype(chunks)::value) {
          Chunk16 dl[TN * es], dg[TN * es];
          load_rows32<OUT_DT, TN>(a, a.local, a.ld_local, mb, nb, dl);
          load_rows32<OUT_DT, TN>(a, a.gate, a.ld_gate, mb, nb, dg);
          slab_chunks32<OUT_DT, TN>(slab, dl);
          slab_groups32<OUT_DT, TN>(slab, lo);
          slab_chunks32<OUT_DT, TN>(slab, dg);
          slab_groups32<OUT_DT, TN>(slab, gt);
        } else {
          auto units = [&](const void* p, int64_t ld) {
            if (in % 8 == 0) return slab_units32<uint64_t, es, RB>(a, slab, p, ld, mb, nb);
            if constexpr (OUT_DT == kBF16)
              if (in % 4 != 0) return slab_units32<uint16_t, es, RB>(a, slab, p, ld, mb, nb);
            slab_units32<uint32_t, es, RB>(a, slab, p, ld, mb, nb);
          };
          units(a.local, a.ld_local);
          slab_groups32<OUT_DT, TN>(slab, lo);
          units(a.gate, a.ld_gate);
          slab_groups32<OUT_DT, TN>(slab, gt);
        }
        fill_slab32<OUT_DT, TN>(slab, [&](int j, int g, float (&v)[4]) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v0 = (static_cast<float>(acc[0][i][j][4 * g + r] - rs0[i]) * inv0[i]) * cws;
            const float v1 = (static_cast<float>(acc[1][i][j][4 * g + r] - rs1[i]) * inv1[i]) * cws1;
            v[r] = dual_epi<EPI, OUT_DT>(rnd<OUT_DT>(v0), rnd<OUT_DT>(v1), group_at<OUT_DT>(lo[j][g], r),
                                         group_at<OUT_DT>(gt[j][g], r));
          }
        });
        if constexpr (decltype(chunks)::value) {
          store_tiles32<OUT_DT, TN>(a, slab, mb, nb);
        } else {
          if ((bits(a.out, a.ldo) | static_cast<uintptr_t>(a.N * es)) % 8 == 0) {
            store_rows32<uint64_t, es, RB>(a, slab, mb, nb);
            continue;
          }
          if constexpr (OUT_DT == kBF16)
            if (bits(a.out, a.ldo) % 4 != 0) {
              store_rows32<uint16_t, es, RB>(a, slab, mb, nb);
              continue;
            }
          store_rows32<uint32_t, es, RB>(a, slab, mb, nb);
        }
      }
    };
    if (a16 && tensor && in % 16 == 0) return rows(std::true_type{});
    if (tensor) return rows(std::false_type{});
  }
  // General form: per-row weight scales, bias, accumulator dump, and what is not in whole 16-byte rows of SwiGLU and the
  // gates.  The output gate's inputs of one 32 x 32 tile (four groups of four columns per lane) are requested together in
  // straight-line code (indices clamped into range, raw bits) before any is used, so the tile waits for memory once
  // instead of once per group.
  const bool vout = vec4_ok<OUT_DT>(a.out, a.ldo);
  const bool vin = EPI == kEpiOutputGate && vec4_ok<OUT_DT>(a.local, a.ld_local) &&
                   vec4_ok<OUT_DT>(a.gate, a.ld_gate) && a.N % 4 == 0;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + (wm * TM + i) * 32 + (lane & 31), mc = m < a.M ? m : a.M - 1;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      uint32_t lo[4][4], gt[4][4];
      if constexpr (EPI == kEpiOutputGate) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int64_t nb = n0 + (wn * TN + j) * 32 + 8 * g + 4 * (lane >> 5);
          if (vin) {  // whole groups of four: a group past N re-reads the last one
            const int64_t nv = nb < a.N ? nb : a.N - 4;
            const char* pl = static_cast<const char*>(a.local) + (mc * a.ld_local + nv) * es;
            const char* pg = static_cast<const char*>(a.gate) + (mc * a.ld_gate + nv) * es;
#pragma unroll
            for (int q = 0; q < es / 2; ++q) {  // bf16: one 8-byte load, f32: two
              const uint2 wl = reinterpret_cast<const uint2*>(pl)[q], wg = reinterpret_cast<const uint2*>(pg)[q];
              lo[g][2 * q] = wl.x;
              lo[g][2 * q + 1] = wl.y;
              gt[g][2 * q] = wg.x;
              gt[g][2 * q + 1] = wg.y;
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int64_t n = nb + r < a.N ? nb + r : a.N - 1;
              lo[g][r] = ld_bits<OUT_DT>(a.local, mc * a.ld_local + n);
              gt[g][r] = ld_bits<OUT_DT>(a.gate, mc * a.ld_gate + n);
            }
          }
        }
      }
      if (m >= a.M) continue;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int64_t nb = n0 + (wn * TN + j) * 32 + 8 * g + 4 * (lane >> 5);
        if (nb >= a.N) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t n = nb + r, nc = n < a.N ? n : a.N - 1;
          const float cw0 = o0.c_w_per_row ? o0.c_w[nc] : cws;
          const int32_t a0 = acc[0][i][j][4 * g + r] - rs0[i];
          if (a.acc_dump && n < a.N) a.acc_dump[m * a.N + n] = a0;
          const float v0 = (static_cast<float>(a0) * inv0[i]) * cw0;
          if constexpr (!DUAL) {
            v[r] = a.bias ? v0 + ld<OUT_DT>(a.bias, nc) : v0;
          } else {
            const float cw1 = o1.c_w_per_row ? o1.c_w[nc] : cws1;
            const float v1 = rnd<OUT_DT>((static_cast<float>(acc[1][i][j][4 * g + r] - rs1[i]) * inv1[i]) * cw1);
            float lv = 0.0f, gv = 0.0f;
            if constexpr (EPI == kEpiOutputGate) {
              if (vin && OUT_DT == kBF16) {
                const uint32_t wl = lo[g][r >> 1], wg = gt[g][r >> 1];
                lv = __uint_as_float(r & 1 ? wl & 0xffff0000u : wl << 16);
                gv = __uint_as_float(r & 1 ? wg & 0xffff0000u : wg << 16);
              } else {
                lv = from_bits<OUT_DT>(lo[g][r]);
                gv = from_bits<OUT_DT>(gt[g][r]);
              }
            }
            v[r] = dual_epi<EPI, OUT_DT>(rnd<OUT_DT>(v0), v1, lv, gv);
          }
        }
        if constexpr (EPI == kEpiGates) gate_act4<OUT_DT>(a, gate_region(a, n0 + (wn * TN + j) * 32), nb, v);
        if (nb + 3 < a.N) {
          store4<OUT_DT>(a.out, m * a.ldo + nb, v, vout);
        } else {
          for (int r = 0; r < 4 && nb + r < a.N; ++r) st<OUT_DT>(a.out, m * a.ldo + nb + r, v[r]);
        }
      }
    }
  }
}

// One output tile at (m0, n0); smem holds at least the tile's SMEM bytes.
template <int WM, int WN, int TM, int TN, int KS, int NS, int EPI, int OUT_DT>
__device__ __forceinline__ void mfma32_tile(const LinearArgs& a, int64_t m0, int64_t n0, char* smem) {
  using T = Tile32<WM, WN, TM, TN, KS, NS, EPI, OUT_DT>;
  v16i acc[T::NACC][TM][TN];
#pragma unroll
  for (int p = 0; p < T::NACC; ++p)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[p][i][j] = v16i{};
  mfma32_loop<T, WN, TM, TN, KS, NS>(a, m0, n0, acc, smem);
  const int lane = threadIdx.x & 63, wall = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int kg = wall / T::NG, w = wall % T::NG;
  if constexpr (KS > 1) {  // the other groups' partial sums, added by group 0 (integers: any order is exact)
    constexpr int TQ = T::NACC * TM * TN * 4;
    v4i* red = reinterpret_cast<v4i*>(smem);
    if (kg > 0) {
#pragma unroll
      for (int q = 0; q < TQ; ++q) {
        const v16i& c = acc[q / (4 * TM * TN)][q / (4 * TN) % TM][q / 4 % TN];
        red[(((kg - 1) * T::NG + w) * TQ + q) * 64 + lane] =
            v4i{c[4 * (q % 4)], c[4 * (q % 4) + 1], c[4 * (q % 4) + 2], c[4 * (q % 4) + 3]};
      }
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int h = 0; h < KS - 1; ++h)
#pragma unroll
      for (int q = 0; q < TQ; ++q) {
        v16i& c = acc[q / (4 * TM * TN)][q / (4 * TN) % TM][q / 4 % TN];
        const v4i v = red[((h * T::NG + w) * TQ + q) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) c[4 * (q % 4) + r] += v[r];
      }
  }
  epilogue32<TM, TN, EPI, OUT_DT>(a, acc, m0, n0, w / WN, w % WN, smem + T::RED + w * T::SLAB);
}

// One group of WM x WN waves per tile.  ORD: the tile order, 4 (ORD 0) or 8 (ORD 2) M tiles per group of the
// XCD-aware walk: the fewer for grids of about one round, whose XCDs then share weights across fewer rows
// (2048 x 4096 x 4096: 34.7 us with 4, 38.1 with 8), the more for grids of many rounds (8192 x 34816 x 4096:
// 1016 us with 8, 1054 with 4).
template <int WM, int WN, int TM, int TN, int EPI, int OUT_DT, int ORD>
__global__ __launch_bounds__(WM* WN * 64, WM * WN >= 8 && EPI != kEpiOutputGate ? 4 : 1) void mfma32_kernel(LinearArgs a) {
  using T = Tile32<WM, WN, TM, TN, 1, 3, EPI, OUT_DT>;
  __shared__ __attribute__((aligned(16))) char smem[T::SMEM];
  int64_t tm, tn;
  xcd_tile_of<ORD == 0 ? 4 : 8>(blockIdx.x, (a.M + T::BM - 1) / T::BM, (a.N + T::BN - 1) / T::BN, tm, tn);
  mfma32_tile<WM, WN, TM, TN, 1, 3, EPI, OUT_DT>(a, tm * T::BM, tn * T::BN, smem);
}

// KS groups of WM x WN waves per tile, each with K tiles of its own.  (The output gate's eight groups keep 64 of their
// registers in scratch memory, 244-264 bytes a lane: two products' loads in flight beside two accumulator sets.)
template <int WM, int WN, int TM, int TN, int KS, int NS, int EPI, int OUT_DT>
__global__ __launch_bounds__(WM* WN* KS * 64) void mfma32k_kernel(LinearArgs a) {
  using T = Tile32<WM, WN, TM, TN, KS, NS, EPI, OUT_DT>;
  __shared__ __attribute__((aligned(16))) char smem[T::SMEM];
  int64_t tm, tn;
  xcd_tile_of<4>(blockIdx.x, (a.M + T::BM - 1) / T::BM, (a.N + T::BN - 1) / T::BN, tm, tn);
  mfma32_tile<WM, WN, TM, TN, KS, NS, EPI, OUT_DT>(a, tm * T::BM, tn * T::BN, smem);
}

// Plain product whose 128x256 tiles would run in more rounds than the CUs hold (the SISO in_proj, 640
// tiles): columns [0, nA) in 128x256 tiles, two per CU, and the remaining N - nA columns in 128x128
// tiles launched after them, so the last round runs half-size tiles on more CUs.
template <int OUT_DT, int TMB, int EPI>
__global__ __launch_bounds__(512, 4) void mfma32_split_kernel(LinearArgs a, int64_t nA) {
  using A = Tile32<2, 4, 2, 2, 1, 3, EPI, OUT_DT>;
  using B = Tile32<2, 4, TMB, 1, 1, 3, EPI, OUT_DT>;
  __shared__ __attribute__((aligned(16))) char smem[A::SMEM > B::SMEM ? A::SMEM : B::SMEM];
  const int64_t ntm = (a.M + A::BM - 1) / A::BM, ntnA = nA / A::BN, tilesA = ntm * ntnA;
  int64_t tm, tn;
  if (static_cast<int64_t>(blockIdx.x) < tilesA) {
    xcd_tile_of<8>(blockIdx.x, ntm, ntnA, tm, tn);
    mfma32_tile<2, 4, 2, 2, 1, 3, EPI, OUT_DT>(a, tm * A::BM, tn * A::BN, smem);
  } else {
    xcd_tile_of<8>(blockIdx.x - tilesA, (a.M + B::BM - 1) / B::BM, (a.N - nA + B::BN - 1) / B::BN, tm, tn);
    mfma32_tile<2, 4, TMB, 1, 1, 3, EPI, OUT_DT>(a, tm * B::BM, nA + tn * B::BN, smem);
  }
}

template <int WM, int WN, int TM, int TN, int EPI, int ORD>
int run_mfma32(const LinearArgs& a, hipStream_t st) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, NT = WM * WN * 64;
  const int64_t tiles = ((a.N + BN - 1) / BN) * ((a.M + BM - 1) / BM);
  TESM_REQUIRE(tiles <= 0x7fffffff, kErrUnsupported, "bitlinear: too many tiles");
  const unsigned grid = static_cast<unsigned>(tiles);
  if (a.out_dt == kBF16)
    mfma32_kernel<WM, WN, TM, TN, EPI, kBF16, ORD><<<grid, NT, 0, TESM_LOGGED(st, mfma32_kernel<WM, WN, TM, TN, EPI, kBF16, ORD>)>>>(a);
  else
    mfma32_kernel<WM, WN, TM, TN, EPI, kF32, ORD><<<grid, NT, 0, TESM_LOGGED(st, mfma32_kernel<WM, WN, TM, TN, EPI, kF32, ORD>)>>>(a);
  return check_launch("bitlinear mfma32");
}

template <int WM, int WN, int TM, int TN, int KS, int NS, int EPI>
int run_mfma32k(const LinearArgs& a, hipStream_t st) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, NT = WM * WN * KS * 64;
  const int64_t tiles = ((a.N + BN - 1) / BN) * ((a.M + BM - 1) / BM);
  TESM_REQUIRE(tiles <= 0x7fffffff, kErrUnsupported, "bitlinear: too many tiles");
  const unsigned grid = static_cast<unsigned>(tiles);
  if (a.out_dt == kBF16)
    mfma32k_kernel<WM, WN, TM, TN, KS, NS, EPI, kBF16><<<grid, NT, 0, TESM_LOGGED(st, mfma32k_kernel<WM, WN, TM, TN, KS, NS, EPI, kBF16>)>>>(a);
  else
    mfma32k_kernel<WM, WN, TM, TN, KS, NS, EPI, kF32><<<grid, NT, 0, TESM_LOGGED(st, mfma32k_kernel<WM, WN, TM, TN, KS, NS, EPI, kF32>)>>>(a);
  return check_launch("bitlinear mfma32 (K groups)");
}

// Tile sizes by grid.  Times in us on one box, bf16 outputs unless noted; "before" is the two-stage, one-group form.
//   * 128x256 tiles (8 waves of 64x64, two workgroups per CU) when they give every CU one: 2048 x 4096 x 4096 36.2
//     (64x256 tiles 40), 4095 x 3744 x 1024 21.2 (64x128: 26.3); past short K already when they give three CUs in four
//     one: 1500 x 4096 x 11008 72.4 (64x128: 79.2), 520 x 11008 x 4096 30.5 (35.2), and 400 x 11008 x 4096, below
//     that, 26.9 against 26.0; above K 4096 from five CUs in eight (with the quantization: 1400 x 4096 x 11008 78.2,
//     64x128 84.3; 1200 77.5, 78.6; 1100 no difference).  Grids past two rounds walk 8 M tiles per group, past short K
//     those past one (3000 x 4096 x 4096 54.5, by fours 59.2), at K above 4096 all (1500 x 4096 x 11008 f32 77.0, by
//     fours 85.9), and those of five M tiles, where four and one leave one by itself (513 x 12992 x 4096 32.6, by fours
//     33.5, f32 34.2, 35.8; the less of the fifth tile is filled the more: over 27 sizes of K 1536-4096 from 4.5 %
//     faster to 0.7 slower, 1.3 in the mean, none at 640 rows).  Other counts gain nothing to speak of: six or seven
//     3 % faster to 3 slower, 0.4 in the mean; one to four and 8 to 21 within 1.6 %, with 9, 13, 17 and 21 among them.
//     Up to K 2048 only when 64x128 tiles would go past three per CU: below that the rows or columns they need not fill
//     up count for more (402 x 12544 x 1100 13.2, 64x128 12.4, f32 14.6, 13.7; x 2048 17.9, 17.0, f32 19.7, 18.0; past
//     the line 700 x 8960 x 1100 13.5, 14.8).
//   * with short K and a narrow remainder past two tiles per CU (the SISO in_proj, 8192 x 2432 x 768), the split
//     kernel: 23.5 against 26.1 for 128x256 tiles throughout.
//   * 64x128 tiles (4 waves of 64x32) when they give two workgroups per CU, past short K one: 8192 x 768 x 768 10.6
//     (128x256: 10.9), 4095 x 1024 x 2816 15.4 (before 21.5), 1000 x 4096 x 4096 21.2 (before 28.3), 666 x 4096 x 11008
//     41.0 (two K groups on 32x64: 50.6), 200 x 11008 x 4096 16.7 (20.7).
//   * a K loop of at most three tiles, where the first loads and the stores are most of the time: 128x256 tiles when
//     they give every CU two (32768 x 4096 x 64 63.1, 64x128 82.6; f32 97.9, 101.8) or, in bf16, one (4096 x 2048 x 256
//     8.6, 9.1; f32 11.1, 32x128 10.4); then 32x128, in bf16 as long as 64x128 ones would not give every CU two (800 x
//     768 x 384 3.8, 64x128 4.9; 4096 x 768 x 384 5.8, 6.3; 8192 x 768 x 384 8.8, 8.5), and for up to 64 rows (32 x
//     151936 x 384 7.5, 64x128 10.2, 128x256 14.3; 64 rows 11.3, 11.6, 15.7).  One column tile of up to 512 rows
//     stays on 64x128: its call is bound by the launch (512 x 96 x 384 4.7, 32x128 3.8).
//   * 32x128 tiles when those do, at short K and up to three 64x128 tiles per two CUs (two per CU where those would be
//     half empty): 512 x 2944 x 768 4.9 (64x128: 5.8), 666 x 2944 x 768 f32 6.1 (7.1); with the quantization
//     1300 x 2432 x 768 f32 12.4 (11.8), 1600 13.2 (12.8), 4095 x 768 x 768 12.1 (11.6).  Around the line it also
//     depends on the remainders: 3500 x 1000 x 768 16.5 (17.0), 1100 x 2816 x 1024 11.7 (12.1).
//   * else K groups: two on 32x128 tiles past short K when those give three workgroups per two CUs (400 x 4096 x 11008
//     30.1, on 32x64 tiles 35.4; 300 rows 28.8 against 25.0), or on 32x64 tiles two (512 x 768 x 768 4.2, before 5.3;
//     32 x 34816 x 4096 12.3, before 14.0), or
//     four when K is long and two would leave CUs idle (512 x 768 x 3072 5.7, before 11.8; 200 x 4096 x 11008 18.2,
//     two groups 21.1).
template <int EPI>
int dispatch_store32(const LinearArgs& a, hipStream_t st) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
  const int64_t cus = std::max(device_limits().cus, 1);
  const int64_t big = tiles(128, 256);
  if (big >= 2 * cus && a.Kp <= 1024) {
    const int64_t ntm = (a.M + 127) / 128, ntnA = std::min<int64_t>(a.N / 256, (2 * cus) / ntm), nA = ntnA * 256;
    if (ntnA >= 1 && a.N > nA && a.N - nA <= 512) {
      const int64_t grid = ntm * ntnA + ntm * ((a.N - nA + 127) / 128);
      TESM_REQUIRE(grid <= 0x7fffffff, kErrUnsupported, "bitlinear: too many tiles");
      if (a.out_dt == kBF16)
        mfma32_split_kernel<kBF16, 2, EPI><<<static_cast<unsigned>(grid), 512, 0, TESM_LOGGED(st, mfma32_split_kernel<kBF16, 2, EPI>)>>>(a, nA);
      else
        mfma32_split_kernel<kF32, 2, EPI><<<static_cast<unsigned>(grid), 512, 0, TESM_LOGGED(st, mfma32_split_kernel<kF32, 2, EPI>)>>>(a, nA);
      return check_launch("bitlinear mfma32 split");
    }
  }
  if (a.Kp > 3 * kKTile) {
    const bool most = a.Kp > 4096 ? 8 * big >= 5 * cus : 4 * big >= 3 * cus;
    const int64_t mid = tiles(64, 128);
    const bool wide = big >= cus || (most && a.Kp > 1024 && a.M > 64 && (a.Kp > 2048 || mid >= 3 * cus));
    const bool five = a.M > 512 && a.M <= 640;  // M tiles: by fours the fifth shares no weights in its XCD
    if (big >= 2 * cus || (wide && (a.Kp > 4096 || ((big > cus || five) && a.Kp > 1024)))) return run_mfma32<2, 4, 2, 2, EPI, 2>(a, st);
    if (wide) return run_mfma32<2, 4, 2, 2, EPI, 0>(a, st);
    if (2 * mid < (a.M <= 32 ? 4 : 3) * cus && a.Kp <= 1024 && tiles(32, 128) >= cus) return run_mfma32<1, 4, 1, 1, EPI, 0>(a, st);
    if (mid < cus || a.M <= 32) {
      if (a.Kp >= 2048 && tiles(32, 64) < 2 * cus) return run_mfma32k<1, 2, 1, 1, 4, 3, EPI>(a, st);
      if (a.Kp > 1024 && 2 * tiles(32, 128) >= 3 * cus) return run_mfma32k<1, 4, 1, 1, 2, 3, EPI>(a, st);
      return run_mfma32k<1, 2, 1, 1, 2, 3, EPI>(a, st);
    }
  } else if constexpr (EPI == kEpiStore) {
    const bool full = a.M > 64 && a.N > 128;  // (not most of a 128x256 tile for padding)
    if (full && big >= 2 * cus) return run_mfma32<2, 4, 2, 2, EPI, 2>(a, st);
    if (full && big >= cus && a.out_dt == kBF16) return run_mfma32<2, 4, 2, 2, EPI, 0>(a, st);
    if ((a.N > 128 || a.M > 512) && (a.out_dt == kF32 || a.M <= 64 || tiles(64, 128) < 2 * cus))
      return run_mfma32<1, 4, 1, 1, EPI, 0>(a, st);
  }
  return run_mfma32<1, 4, 2, 1, EPI, 2>(a, st);
}

// The output gate.  us, bf16 / f32 (M x N x 2 x K):
//   * 128x256 tiles: two accumulator sets, so one workgroup per CU and whole rounds of the CUs; taken where the rounds
//     are nearly full, the fuller the shorter the K loop: 4096 x 4096 x 2 x 2048 83.3 / 91.4 (eight-wave 64x128 102 / 107),
//     7000 x 1024 x 2 x 4096 64.7 / 67.2 (86.1 / 88.7), 4095 x 2048 x 2 x 1024 29.4 / 32.2 (34.6 / 37.6); not 7000 x 2432
//     x 2 x 1280 (2.15 rounds) 83.7 / 88.1 (79.9 / 87.0), 3000 x 4096 x 2 x 2048 (1.5) 74.0 / 79.5 (75.8 / 79.6).  These
//     lines were drawn when bf16 inputs and outputs went in the accumulators' order, which favoured small tiles: bf16 at
//     one round and K up to 1024 would now gain from the large ones, as above.  At two K tiles they stand from two rounds
//     on, though 64x128 ones would be a little faster (4095 x 4096 x 2 x 256 38.1 / 47.5, 36.1 / 45.6; 4100 x 4104 x 2 x
//     200 47.5 / 52.7, 38.9 / 47.8).
//   * 64x128 tiles when they give every CU one: eight waves in bf16 (4095 x 1024 x 2 x 512 13.2, one-group form 27.8); in
//     f32 32x64 tiles just past two per CU (3000 x 1536 x 2 x 768 23.2, 25.9 with 64x128; 2048 x 2432 x 2 x 1280 32.4,
//     32.9) and four waves beyond (7000 x 2432 x 2 x 1280 82.7, eight 87.0; 8300 x 2048 x 2 x 1024 72.6, 77.3); at long K
//     32x64 up to three per two CUs (2048 x 1024 x 2 x 4096 32.2 / 32.8, 38.4 / 39.0).
//   * else 32x64 tiles of two waves: 512 x 768 x 2 x 384 5.9 (one-group form 12.3); at long K with CUs left over, eight K
//     groups on 32x32 tiles or four on 32x64: 64 x 4096 x 2 x 8192 21.9 (51.8), 100 rows 31.5.
int dispatch_gate32(const LinearArgs& a, hipStream_t st) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
  const int64_t cus = std::max(device_limits().cus, 1), big = tiles(128, 256), mid = tiles(64, 128);
  const int64_t rounds = (big + cus - 1) / cus, fill = 100 * big / (rounds * cus);  // percent of the rounds' CUs
  const bool f32 = a.out_dt == kF32;
  const bool wide = a.Kp < 512      ? a.Kp == 256 && big >= 2 * cus
                    : a.Kp <= 1024  ? fill >= 95 && (f32 || rounds > 1)
                    : a.Kp < 2048   ? fill >= (a.Kp < 1536 ? 90 : 85)
                    : a.Kp < 4096   ? fill >= (f32 ? 85 : 75) + (rounds > 1 ? 5 : 0)
                                    : fill >= 75;
  if (wide && big >= 8 * cus) return run_mfma32<2, 4, 2, 2, kEpiOutputGate, 2>(a, st);
  if (wide) return run_mfma32<2, 4, 2, 2, kEpiOutputGate, 0>(a, st);
  if (mid >= cus && !(a.Kp >= 4096 && 2 * mid <= 3 * cus)) {
    if (f32 && mid > 2 * cus) {
      if (4 * mid <= 11 * cus) return run_mfma32<1, 2, 1, 1, kEpiOutputGate, 0>(a, st);
      if (a.Kp > 256) return run_mfma32<1, 4, 2, 1, kEpiOutputGate, 0>(a, st);
    }
    return run_mfma32<2, 4, 1, 1, kEpiOutputGate, 0>(a, st);
  }
  if (a.Kp >= 4096 && tiles(32, 64) < cus) return run_mfma32k<1, 1, 1, 1, 8, 3, kEpiOutputGate>(a, st);
  if (a.Kp >= 4096 && tiles(32, 64) < 2 * cus) return run_mfma32k<1, 2, 1, 1, 4, 3, kEpiOutputGate>(a, st);
  return run_mfma32<1, 2, 1, 1, kEpiOutputGate, 0>(a, st);
}

// SwiGLU over 128 + 128 columns when those tiles give two workgroups per CU (4095 x 2 x 2816 x 1024 35.2, before 53.8;
// one per CU is enough at long K: 200 x 2 x 16384 x 4096 34.5, before 58), else over 64 + 64 (512 x 2 x 3072 x 768
// 7.6, before 12.5).
int dispatch_swiglu32(const LinearArgs& a, hipStream_t st) {
  const int64_t cus = std::max(device_limits().cus, 1), big = ((a.M + 127) / 128) * ((a.N + 127) / 128);
  if (big >= 2 * cus || (big >= cus && a.Kp >= 2048)) return run_mfma32<2, 4, 2, 1, kEpiSwiGLU, 2>(a, st);
  return run_mfma32<2, 2, 1, 1, kEpiSwiGLU, 0>(a, st);
}

}  // namespace

int launch_mfma32(const LinearArgs& a, hipStream_t st) {
  if (a.epilogue == kEpiGates) return dispatch_store32<kEpiGates>(a, st);
  if (a.epilogue == kEpiStore) return dispatch_store32<kEpiStore>(a, st);
  if (a.epilogue == kEpiOutputGate) return dispatch_gate32(a, st);
  return dispatch_swiglu32(a, st);
}

}  // namespace tesm
