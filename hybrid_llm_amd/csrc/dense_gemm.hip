// Tiled bf16 MFMA GEMM on gfx950: the dense projections of a sequence
// prefill (llmy_linear_bf16 with many rows), out[M, N] = x[M, K] . w[N, K]^T
// with the linear epilogues, and an N tail (rows past N re-read row N-1,
// their columns are not stored).  The MoE prefill GEMMs are the grouped
// kernel of moe_grouped.hip.
//
// Tiling: a workgroup of 4 wavefronts (one per SIMD) computes a BM x BN tile of
// the x rows times the weight rows; wavefront (wm, wn) of the 2 x 2 grid owns a
// (BM/2) x (BN/2) sub-tile as FA x FB blocks of v_mfma_f32_32x32x16_bf16, so
// LDS traffic is FA + FB fragment reads per FA FB MFMAs.  128 x 128 tiles run
// two workgroups per CU, the larger ones one.  The MFMA takes the weight
// fragment as its first operand.
//
// Work order: work items (n-tile, m-tile) are grouped 4 m-tiles x all
// n-tiles, m fastest inside a group, and each XCD (block id mod 8) takes a
// contiguous range of them, so the tiles an XCD runs together share few x
// and weight tiles in its L2.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "abi_util.hpp"

namespace llmy {

// Dense epilogues (values of the linear entry's epilogue argument).
enum DenseEpi : int { kDenseBf16 = 0, kDenseF32 = 1, kDenseResid = 2, kDenseGated = 3 };

struct TileArgs {
  const uint16_t* x;  // [M, K]
  const uint16_t* w;  // weights, row-major [N, K] or packed
  void* out;          // [M, ldo] (bf16 or fp32 by epilogue)
  const float* aux;   // gated residual: out += acc * aux[m * ldo + n]
  int K, ldo, M;
  int N;        // output columns (last n-tile may be partial)
  int n_tiles;  // output column tiles
  int m_tiles;  // row tiles
  int group_m;  // m-tiles per work group (0: m fastest over all rows)
  int packed;
};

namespace {

constexpr int kThreads = 256;  // 4 wavefronts: one per SIMD
constexpr int kNumXcd = 8;

// Packed operand order of llmy_pack_weights_bf16 (see linear.hip): the 8
// elements W[n][k .. k+7] (k % 8 == 0) are contiguous at this index.
__device__ __forceinline__ long long packed_at(int n, int k, int K) {
  const int nb = n >> 4, r = n & 15;
  const int kb = k >> 8, kk = k & 255;
  const int j = kk >> 5, g = (kk >> 3) & 3;
  const int lane = g * 16 + r;
  return (((static_cast<long long>(nb) * (K >> 8) + kb) * 8 + j) * 64 + lane) << 3;
}

typedef __attribute__((address_space(3))) void lds_void;
// A __shared__ address in the LDS address space (the destination operand of
// global_load_lds).
__device__ __forceinline__ lds_void* as_lds(void* p) { return (lds_void*)p; }

// One global_load_lds_dwordx4: 16 bytes per lane from src into LDS at dst
// (+16 bytes per lane).  Kept in a device function: the builtin inside a
// kernel template body stops the host pass from emitting the launch stub.
__device__ __forceinline__ void dma16(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(src, as_lds(dst), 16, 0, 0);
}

// 16-byte LDS read at byte address addr + OFF, as inline asm: the compiler's
// LDS-DMA tracking cannot separate the stage being read from the stage being
// filled and would make every read wait for all loads in flight.  The result
// is valid only after a settle below.
template <int OFF>
__device__ __forceinline__ u32x4 lds_frag(uint32_t addr) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(OFF) : "memory");
  return v;
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_void*)p));
}

__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// vmcnt <= n, expcnt and lgkmcnt left open.
constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

}  // namespace

// ---- epilogue of a wavefront's FA x FB blocks: block i's rows from m0 +
// row_of(i), block j's columns from n0 + col + 32 j.  acc[i][j] = (weight block
// j) . (row block i)^T, so in the 32 x 32 D layout lane l holds row 32 i + (l &
// 31) and, in registers 4 g .. 4 g + 3, the columns 32 j + 8 g + 4 (l >> 5) ..
// +3.  Stored as they lie, an instruction would write 32 rows of 16 or 32
// bytes; so each 32-row block goes through this wave's LDS (lds, 32 rows of
// FB * 32 values + 16 bytes; the ring is no longer in use) and leaves, and its
// residual and gate arrive, as whole row segments of 16 bytes a lane.
template <int EPI, int FA, int FB, typename Row>
__device__ __forceinline__ void tile_store(const TileArgs& a, const f32x16 (&acc)[FA][FB], int m0,
                                           int n0, Row row_of, int col, int lane,
                                           unsigned char* lds) {
  constexpr int ES = EPI == kDenseBf16 ? 2 : 4;         // bytes of a value
  constexpr int PITCH = FB * 32 * ES + 16;
  constexpr int CPW = FB * 32 * ES / 16;                // 16-byte chunks of a row
  constexpr int IT = 32 * CPW / 64, VPC = 16 / ES;
  static_assert(IT * 64 == 32 * CPW, "whole instructions");
  unsigned char* const wr = lds + (lane & 31) * PITCH + (lane >> 5) * 4 * ES;
#pragma unroll
  for (int i = 0; i < FA; ++i) {
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float v0 = acc[i][j][4 * g], v1 = acc[i][j][4 * g + 1];
        const float v2 = acc[i][j][4 * g + 2], v3 = acc[i][j][4 * g + 3];
        unsigned char* const w = wr + (32 * j + 8 * g) * ES;
        if (EPI == kDenseBf16)
          *reinterpret_cast<uint2*>(w) = make_uint2(pack_bf2(v0, v1), pack_bf2(v2, v3));
        else
          *reinterpret_cast<float4*>(w) = make_float4(v0, v1, v2, v3);
      }
    wave_lds_order();  // the block is written: other lanes' values are read below
    const int mb = m0 + row_of(i);
#pragma unroll
    for (int t0 = 0; t0 < IT; t0 += 8) {
      // Eight chunks at a time: their residual (and gate) loads go out before the
      // first store, which they could not be moved across, and are waited for once:
      // after the branches below the compiler no longer knows what is in flight, and
      // would wait before each chunk's sum for the store before it too (256 x 16 x
      // 256, gated residual: 7.4 -> 6.0 us, 2048 x 1024 x 1024 15.2 -> 13.0; with four
      // chunks at a time 6.2 and 13.4).
      constexpr int G = IT < 8 ? IT : 8;
      float4 res[G], gat[G];
      bool on[G];
      long long at[G];
      const unsigned char* src[G];
#pragma unroll
      for (int t = 0; t < G; ++t) {
        const int e = (t0 + t) * 64 + lane, r = e / CPW, c = e % CPW;
        const int m = mb + r, n = n0 + col + VPC * c;
        on[t] = t0 + t < IT && m < a.M && n < a.N;  // N % 16 == 0: a chunk is all in or out
        at[t] = static_cast<long long>(m) * a.ldo + n;
        src[t] = lds + r * PITCH + 16 * c;
        res[t] = make_float4(0.f, 0.f, 0.f, 0.f);
        gat[t] = make_float4(1.f, 1.f, 1.f, 1.f);
        if (on[t] && (EPI == kDenseResid || EPI == kDenseGated))
          res[t] = *reinterpret_cast<const float4*>(static_cast<const float*>(a.out) + at[t]);
        if (on[t] && EPI == kDenseGated) gat[t] = *reinterpret_cast<const float4*>(a.aux + at[t]);
      }
      if (EPI == kDenseResid || EPI == kDenseGated) __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
#pragma unroll
      for (int t = 0; t < G; ++t) {
        if (!on[t]) continue;
        if (EPI == kDenseBf16) {
          *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + at[t]) =
              *reinterpret_cast<const uint4*>(src[t]);
          continue;
        }
        const float4 v = *reinterpret_cast<const float4*>(src[t]);
        const float4 r = res[t], g = gat[t];
        float* const o = static_cast<float*>(a.out) + at[t];
        if (EPI == kDenseF32)
          *reinterpret_cast<float4*>(o) = v;
        else if (EPI == kDenseResid)
          *reinterpret_cast<float4*>(o) = make_float4(r.x + v.x, r.y + v.y, r.z + v.z, r.w + v.w);
        else
          *reinterpret_cast<float4*>(o) = make_float4(r.x + v.x * g.x, r.y + v.y * g.y,
                                                      r.z + v.z * g.z, r.w + v.w * g.w);
      }
    }
    wave_lds_order();  // the block is read: the next one takes its place
  }
}

// ---------------------------------------------------------------------------
// 32 k per step through a ring of NS stages.  A stage holds the BM rows of x
// (64 bytes each, 16-byte chunks XOR-swizzled by row: the 16 lanes that a
// ds_read_b128 serves at once take 16 rows at one chunk index and meet all bank
// groups) and the BN weight rows: packed ones as BN / 16 fragments of 16 rows x 32 k
// (1 KiB, lane l: row l % 16 at k 8 (l / 16) .. +7), row-major ones like those of x
// (in fragments an instruction would gather 64 pieces of 16 bytes, four rows' worth
// of lanes apart: 96 x 1024 x 4096 39.9 -> 28.7 us, 4096 x 1024 x 1024 15.2 -> 13.0).
// All by global_load_lds_dwordx4 from scalar bases plus 32-bit lane offsets; every
// wave issues the same copies each step (past the last step they re-read it),
// so its waits count fixed numbers.
//
// With one wave per SIMD nothing covers a stall of the issuing wave, so the
// step's LDS reads and copies are issued one at a time between its MFMAs: half
// 0: the MFMAs of k half 0 with the reads of half 1 and the weight copies of
// step kk + NS - 1; then the wait for step kk + 1's copies and the barrier (stage
// kk is free); half 1: the MFMAs of half 1 with the reads of step kk + 1's half 0
// and the x copies of step kk + NS into the freed stage.
//
// Measured (us, K = 1024, packed weights, bf16 out, three operand sets in turn;
// before: reads and copies in bursts, every output stored as its lane holds it):
// 4096 x 3072: 44.2 -> 27.7 (930 TFLOP/s; 256 x 192 tiles, where 128 x 128 ones
// ran 1.5 rounds), 4096 x 4096: 44.1 -> 33.7, 2048 x 3072: 26.4 -> 15.3, 4096 x
// 1024: 16.0 -> 11.2, gated residual 23.1 -> 17.3.  A further 1024 of K take a 256 x
// 192 tile 12.3 us on an idle chip (its MFMAs alone 10.2 at 2.4 GHz) and 19 on a full
// one: 1.36 PFLOP/s, where power holds the clock (loops of MFMAs alone on random
// operands reach 1.44 to 1.53).  The rest of a call is its first loads, the epilogue
// and the launch, about 8 us.
template <int N>
__device__ __forceinline__ void settle_frags(u32x4 (&f)[N]) {
  static_assert(N >= 4 && N <= 8, "fragments");
  if constexpr (N == 8)
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]),
                   "+v"(f[6]), "+v"(f[7])::"memory");
  else if constexpr (N == 7)
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]),
                   "+v"(f[6])::"memory");
  else if constexpr (N == 6)
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5])::"memory");
  else if constexpr (N == 5)
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4])::"memory");
  else
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3])::"memory");
}

// BLK: the sums restart every 256 k (kSumSteps) and the block sums are added in
// order, the sums of the weight-streaming kernel: bit for bit at K <= 2048, where
// it has a wave per 256 k, so a row's outputs do not change where this kernel takes
// over.  One chain over all of K is 2 to 3 times further from 64 bits (relative
// error at K = 512 / 1024 / 2048 / 4096, fp32 out: 1.25e-7 / 1.84e-7 / 2.71e-7 /
// 3.95e-7 in one chain, 0.90e-7 / 0.95e-7 / 1.03e-7 / 1.15e-7 in blocks), and the
// blocks cost nothing: 96 x 1024 x 1024 takes 8.8 us, in one chain 9.6 (only where
// the chip is full do they: 255 x 32000 x 1024 22.1, 21.1).
constexpr int kSumSteps = 8;

template <int BM, int BN, int NS, int OCC, int EPI, bool BLK>
__global__ __launch_bounds__(kThreads, OCC) void tile_gemm_kernel(TileArgs a) {
  constexpr int FA = BM / 64, FB = BN / 64, NF = FA + FB, NM = FA * FB;
  constexpr int A_STAGE = BM * 64, STAGE = (BM + BN) * 64;
  constexpr int LA = BM / 64, LB = BN / 64, L = LA + LB;  // copies per wave and step
  static_assert(NM >= 2 * LA && NM >= 2 * LB - 1 && NM >= NF, "interleave");
  static_assert((NS - 1) * L <= 63, "vmcnt range");
  __shared__ __align__(1024) unsigned char smem[NS * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 31, lh = lane >> 5;
  const int K = a.K, nk = K >> 5;

  // ---- which tile: work item w = (n-tile, m-tile), m fastest inside a group
  const int per_xcd = (gridDim.x + kNumXcd - 1) / kNumXcd;
  const int w_item = (blockIdx.x % kNumXcd) * per_xcd + blockIdx.x / kNumXcd;
  if (w_item >= a.m_tiles * a.n_tiles) return;
  const int per_group = a.group_m * a.n_tiles;
  const int grp = w_item / per_group, in = w_item % per_group;
  const int gm = min(a.group_m, a.m_tiles - grp * a.group_m);
  const int m0 = (grp * a.group_m + in % gm) * BM, n0 = in / gm * BN;

  // ---- copies: x instruction q of this wave fills stage rows 16 (4 wave + q)
  // .. +15, lane l row l / 4, slot l % 4, holding the row's chunk (l % 4) ^ (l /
  // 16); weight fragments LB wave + q (rows past M or N repeat the last)
  const bool packed = a.packed != 0;
  uint32_t ao[LA], bo[LB];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = 16 * (LA * wave + q) + (lane >> 2);
    ao[q] = static_cast<uint32_t>(
        (static_cast<long long>(min(m0 + r, a.M - 1)) * K + 8 * ((lane & 3) ^ (lane >> 4))) * 2);
  }
#pragma unroll
  for (int q = 0; q < LB; ++q) {
    const int nb = n0 + 16 * (LB * wave + q);
    const long long at =
        packed ? packed_at(min(nb + (lane & 15), a.N - 1), 8 * (lane >> 4), K)
               : static_cast<long long>(min(nb + (lane >> 2), a.N - 1)) * K +
                     8 * ((lane & 3) ^ (lane >> 4));
    bo[q] = static_cast<uint32_t>(at * 2);
  }
  const char* const a_base = reinterpret_cast<const char*>(a.x);
  const char* const b_base = reinterpret_cast<const char*>(a.w);
  const int b_step = packed ? 1024 : 64;
  unsigned char* const a_dst = smem + 1024 * LA * wave;
  unsigned char* const b_dst = smem + A_STAGE + 1024 * LB * wave;

  const uint32_t base = lds_addr(smem);
  const uint32_t xa0 = base + wm * (BM * 32) + lr * 64 + ((lh ^ ((lr >> 2) & 3)) << 4);
  const uint32_t xa1 = base + wm * (BM * 32) + lr * 64 + (((2 + lh) ^ ((lr >> 2) & 3)) << 4);
  const uint32_t xb = base + A_STAGE + wn * (BN * 32);
  const uint32_t xb0 = xb + (packed ? (lr >> 4) * 1024 + lh * 256 + (lane & 15) * 16
                                    : lr * 64 + ((lh ^ ((lr >> 2) & 3)) << 4));
  const uint32_t xb1 = packed ? xb0 + 512 : xb + lr * 64 + (((2 + lh) ^ ((lr >> 2) & 3)) << 4);
  // fragment n of k half H of the stage at byte offset o: n < FA: rows BM / 2 wm
  // + 32 n of x, else the wave's 32-column weight block n - FA
#define TILE_READ(F, n, o, H)                                           \
  do {                                                                 \
    const uint32_t a_ = ((H) ? xa1 : xa0) + (o), b_ = ((H) ? xb1 : xb0) + (o); \
    if ((n) < FA) {                                                    \
      if ((n) == 0) F[0] = lds_frag<0>(a_);                            \
      if ((n) == 1) F[1] = lds_frag<2048>(a_);                         \
      if ((n) == 2) F[2] = lds_frag<4096>(a_);                         \
      if ((n) == 3) F[3] = lds_frag<6144>(a_);                         \
    } else {                                                           \
      if ((n) == FA) F[FA] = lds_frag<0>(b_);                          \
      if ((n) == FA + 1) F[FA + 1] = lds_frag<2048>(b_);               \
      if ((n) == FA + 2) F[NF > FA + 2 ? FA + 2 : 0] = lds_frag<4096>(b_); \
      if ((n) == FA + 3) F[NF > FA + 3 ? FA + 3 : 0] = lds_frag<6144>(b_); \
    }                                                                  \
  } while (0)
#define TILE_FENCE() __builtin_amdgcn_sched_barrier(0)

  f32x16 acc[FA][FB], sum[FA][FB];  // sum: BLK only
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.f;
        if constexpr (BLK) sum[i][j][r] = 0.f;
      }

  // steps 0 .. NS - 2 and step NS - 1's x copies in flight
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int q = 0; q < LA; ++q)
      dma16(a_base + 64 * min(s, nk - 1) + ao[q], a_dst + s * STAGE + 1024 * q);
    if (s < NS - 1)
#pragma unroll
      for (int q = 0; q < LB; ++q)
        dma16(b_base + b_step * min(s, nk - 1) + bo[q], b_dst + s * STAGE + 1024 * q);
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((NS - 2) * L + LA));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  u32x4 h0[NF], h1[NF];
  uint32_t off = 0, last = (NS - 1) * STAGE;  // stages of steps kk and kk + NS - 1
#pragma unroll
  for (int n = 0; n < NF; ++n) TILE_READ(h0, n, 0u, 0);
  settle_frags(h0);
  // one step; FIRST and LAST: of a block of k (BLK), whose products start from zero
  // and join the sums behind the last step's MFMAs
  auto step = [&](int kk, auto FIRST, auto LAST) {
    const int kb = min(kk + NS - 1, nk - 1), ka = min(kk + NS, nk - 1);
    const char* const bb = b_base + static_cast<long long>(b_step) * kb;
    const char* const ab = a_base + 64 * ka;
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      f32x16& c = acc[n / FB][n % FB];
      TILE_FENCE();
      c = mfma32(h0[FA + n % FB], h0[n / FB], FIRST.value ? f32x16{0.f} : c);
      TILE_FENCE();
      if (n < NF) TILE_READ(h1, n, off, 1);
      if (n % 2 == 1 && n / 2 < LB) dma16(bb + bo[n / 2], b_dst + last + 1024 * (n / 2));
    }
    TILE_FENCE();
    settle_frags(h1);
    // step kk + 1 has landed: the NS - 2 steps after it may be in flight
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((NS - 2) * L));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    last = off;
    off = off + STAGE == NS * STAGE ? 0 : off + STAGE;
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      TILE_FENCE();
      acc[n / FB][n % FB] = mfma32(h1[FA + n % FB], h1[n / FB], acc[n / FB][n % FB]);
      TILE_FENCE();
      if (n < NF) TILE_READ(h0, n, off, 0);
      if (n % 2 == 1 && n / 2 < LA) dma16(ab + ao[n / 2], a_dst + last + 1024 * (n / 2));
      if constexpr (LAST.value) {
        if (n > 0) sum[(n - 1) / FB][(n - 1) % FB] += acc[(n - 1) / FB][(n - 1) % FB];
      }
    }
    TILE_FENCE();
    if constexpr (LAST.value) sum[FA - 1][FB - 1] += acc[FA - 1][FB - 1];
    // no read of the loop is in flight across its edge: the compiler knows
    // nothing of them and may move a register that one is still to fill
    settle_frags(h0);
  };
  constexpr std::true_type yes;
  constexpr std::false_type no;
  if constexpr (BLK) {
    for (int kk = 0; kk < nk; kk += kSumSteps) {  // K % 256 == 0: whole blocks
      step(kk, yes, no);
      for (int i = 1; i < kSumSteps - 1; ++i) step(kk + i, no, no);
      step(kk + kSumSteps - 1, no, yes);
    }
  } else {
    for (int kk = 0; kk < nk; ++kk) step(kk, no, no);
  }
#undef TILE_FENCE
#undef TILE_READ
  // every wave's copies have landed and its reads are done: the ring is free
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_assert(4 * 32 * (FB * 128 + 16) <= NS * STAGE, "epilogue rows");
  tile_store<EPI, FA, FB>(a, BLK ? sum : acc, m0, n0, [&](int i) { return 32 * (FA * wm + i); },
                          32 * FB * wn, lane, smem + wave * 32 * (FB * 128 + 16));
}

template <int BM, int BN, int NS, int OCC, int EPI, bool BLK>
int32_t launch_tiles(const TileArgs& g, long long items, hipStream_t s) {
  const unsigned grid = static_cast<unsigned>((items + kNumXcd - 1) / kNumXcd * kNumXcd);
  hipLaunchKernelGGL((tile_gemm_kernel<BM, BN, NS, OCC, EPI, BLK>), dim3(grid), dim3(kThreads), 0, s,
                     g);
  return launch_status();
}

int32_t dense_narrow_ws(const uint16_t* x, const uint16_t* w, void* out, const float* aux, int M,
                        int N, int K, int ldo, int epi, bool packed, hipStream_t s);

// Tile shapes and the time of one round of them (us, packed weights, bf16 out; K 256
// to 4096): on an idle chip (at most 64 tiles) and on a full one (230 to 256), each
// a fixed part and one per k.
struct TileShape {
  int bm, bn;
  float idle, idle_k, full, full_k;
};
constexpr TileShape kTileShapes[] = {{128, 128, 3.6f, 0.0060f, 4.0f, 0.0082f},
                                     {128, 192, 4.5f, 0.0074f, 5.5f, 0.0105f},
                                     {128, 256, 5.0f, 0.0088f, 6.2f, 0.0131f},
                                     {256, 192, 6.1f, 0.0120f, 7.0f, 0.0190f},
                                     {256, 256, 7.1f, 0.0151f, 8.4f, 0.0243f}};

// Modelled time (us) of out[M, N] with a shape: full rounds of workgroups and a last
// one between the idle and the full chip's time by the square of its share of the
// CUs.  A 128 x 128 tile starts beside another on its CU, which hides 2.5 us of each
// further round.  Over 184 calls of 256 to 8192 rows, 16 to 6400 columns and K 256 to
// 4096 the shape (and tail) chosen takes 0.14% more than the best one on average and
// 7% at most (whole rounds at K = 1024's proportions: 0.65% and 24%).
float tile_cost(int shape, int M, int N, int K) {
  const TileShape& t = kTileShapes[shape];
  const long long tiles = static_cast<long long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
  const int cus = compute_units();
  const long long rounds = (tiles + cus - 1) / cus;
  const float idle = t.idle + t.idle_k * K, full = t.full + t.full_k * K;
  const float part = static_cast<float>(tiles - (rounds - 1) * cus) / cus;
  return static_cast<float>(rounds - 1) * (full - (shape == 0 ? 2.5f : 0.f)) + idle +
         (full - idle) * part * part;
}

// Modelled time (us) of the narrow launch that takes a column tail: its own, and
// reading x again.
float tail_cost(int M, int K) { return 3.5f + 3.2e-7f * static_cast<float>(M) * K; }

// Rows below which outputs are summed in 256-wide blocks of k (tiles of 128 rows
// only: the second set of sums takes registers that the larger ones do not have).
constexpr int kBlockSumRows = 256;

// The cheapest shape.  Every shape that a row count allows sums each output over k
// in the same order, so the results do not depend on it (those of a column tail
// depend on whether it is split off, below).
int tile_shape(int M, int N, int K) {
  int best = 0;
  for (int i = 1; i < (M < kBlockSumRows ? 3 : 5); ++i)
    if (tile_cost(i, M, N, K) < tile_cost(best, M, N, K)) best = i;
  return best;
}

// Dense out[M, N] (epilogue epi) = x[M, K] . w[N, K]^T.  Validated by the
// caller: M >= 1, N >= 1, K % 256 == 0, 16-byte aligned x and w, aux given
// for the gated epilogue.
int32_t dense_gemm_mfma(const uint16_t* x, const uint16_t* w, void* out, const float* aux,
                        int M, int N, int K, int epi, bool packed, hipStream_t s) {
  // operand blocks addressed with 32-bit byte offsets
  if (2ll * M * K >= (1ll << 31) || 2ll * N * K >= (1ll << 31))
    return static_cast<int32_t>(hipErrorInvalidValue);
  TileArgs g{};
  g.x = x;
  g.w = w;
  g.out = out;
  g.aux = aux;
  g.K = K;
  g.ldo = N;
  g.M = M;
  g.N = N;
  g.packed = packed;
  g.group_m = 4;
  int shape = tile_shape(M, N, K);
  // A narrow column tail (N = 256 n + 16 .. 64, e.g. a 4096-row projection
  // plus its 16 gate rows) can cost a whole column of tiles, often another
  // round of workgroups: then the whole columns run first and the tail columns
  // follow on the weight-streaming kernel with the rows split 16 per workgroup
  // (the same output rows, column offset and stride N), which sums them in
  // 256-wide blocks of k.  us, split / one launch: 4096 x 4112 x 1024 37.9 / 40.2,
  // 2048 x 4112 x 1024 24.1 / 21.8, 2048 x 4112 x 256 13.8 / 11.2.
  const int tail = N > 256 ? N % 256 : 0;
  if (tail > 0 && tail <= 64) {
    const int whole = tile_shape(M, N - tail, K);
    if (tile_cost(whole, M, N - tail, K) + tail_cost(M, K) < tile_cost(shape, M, N, K)) {
      g.N = N - tail;
      shape = whole;
    }
  }
  g.m_tiles = (M + kTileShapes[shape].bm - 1) / kTileShapes[shape].bm;
  g.n_tiles = (g.N + kTileShapes[shape].bn - 1) / kTileShapes[shape].bn;
  const long long items = static_cast<long long>(g.m_tiles) * g.n_tiles;
  if (items >= (1ll << 31) - kNumXcd) return static_cast<int32_t>(hipErrorInvalidValue);
  int32_t st = 0;
#define LLMY_DENSE(BM_, BN_, NS_, OCC_, BLK_)                                                  \
  switch (epi) {                                                                              \
    case kDenseBf16: st = launch_tiles<BM_, BN_, NS_, OCC_, kDenseBf16, BLK_>(g, items, s); break;   \
    case kDenseF32: st = launch_tiles<BM_, BN_, NS_, OCC_, kDenseF32, BLK_>(g, items, s); break;     \
    case kDenseResid: st = launch_tiles<BM_, BN_, NS_, OCC_, kDenseResid, BLK_>(g, items, s); break; \
    default: st = launch_tiles<BM_, BN_, NS_, OCC_, kDenseGated, BLK_>(g, items, s); break;          \
  }
  if (M < kBlockSumRows) {
    switch (shape) {
      case 0: LLMY_DENSE(128, 128, 5, 2, true) break;
      case 1: LLMY_DENSE(128, 192, 7, 1, true) break;
      default: LLMY_DENSE(128, 256, 6, 1, true) break;
    }
  } else {
    switch (shape) {
      case 0: LLMY_DENSE(128, 128, 5, 2, false) break;
      case 1: LLMY_DENSE(128, 192, 7, 1, false) break;
      case 2: LLMY_DENSE(128, 256, 6, 1, false) break;
      case 3: LLMY_DENSE(256, 192, 5, 1, false) break;
      default: LLMY_DENSE(256, 256, 5, 1, false) break;
    }
  }
#undef LLMY_DENSE
  if (st != 0 || g.N == N) return st;
  // the tail: rows g.N .. N-1 of w (for the packed order too: 16-row groups are
  // contiguous), output columns g.N .. N-1
  return dense_narrow_ws(x, w + static_cast<long long>(g.N) * K,
                         static_cast<char*>(out) +
                             static_cast<long long>(g.N) * (epi == kDenseBf16 ? 2 : 4),
                         aux ? aux + g.N : nullptr, M, N - g.N, K, N, epi, packed, s);
}

}  // namespace llmy
