// Gated delta rule, prefill: the recurrence of model/layers/gated_deltanet.py:140-149
//
//   S_t = g_t S_{t-1} + beta_t k_t (v_t - S_{t-1}^T k_t)^T,   o_t = S_t^T q_t
//
// over T tokens per (batch, head) with an fp32 state S [D, D] (dk = dv = D),
// computed in chunks of C = 64 tokens (the reference is sequential over T
// everywhere: gated_deltanet.py:42-53, runpod/kernels/triton_gdn.py:91-114).
// Within a chunk starting from S0, with Gamma_t = prod_{j<=t} g_j (log-space
// cumulative sums, so every ratio below is <= 1):
//   T  = (I + L)^{-1},  L[t,i] = beta_t (Gamma_{t-1} / Gamma_i) k_t . k_i   (i < t)
//   U  = T Y,  Y = beta o V - (beta Gamma_{t-1}) o (K S0)
//   O  = Gamma o (Q S0) + A U,  A[t,i] = (Gamma_t / Gamma_i) q_t . k_i      (i <= t)
//   S' = Gamma_C S0 + K^T (Gamma_C / Gamma_t o U)
//
// Kernel 1 (gdn_chunk_prep) forms T and the per-token factors of every chunk,
// all chunks in parallel; kernel 2 (gdn_chunk_scan) walks the chunks of one
// (b, h, column slice of the state).  Every product with an fp32 operand uses
// split-bf16 MFMA: x = hi + lo with hi = bf16(x), lo = bf16(x - hi), keeping
// hi*hi + hi*lo + lo*hi (relative error about 2^-16); products of two bf16
// tensors are exact.  The inverse runs on fp32 FMAs and fp32 MFMA.
//
// Resets (gated_deltanet.py:138-142: the state is zeroed before token t's
// update where reset[b, t]): a reset starts a new segment of the chunk.
// Log-decays are cumulated per segment, the couplings L and A vanish between
// tokens of different segments, S0 reaches only the segment before the first
// reset (Gamma masked to 0 after it), and S' takes only the last segment's
// tokens (Gamma_C / Gamma_t masked to 0 before it, Gamma_C to 0 when the
// chunk resets).
//
// Fragments.  v_mfma_f32_16x16x32_bf16: with r = lane % 16, g = lane / 16, the
// A lane holds 8 k-elements of row r, the B lane 8 k-elements of column r, the
// D lane rows 4 g + i (i < 4) of column r.  Both kernels order k inside a
// 32-wide step so that element j of lane group g is k = 4 g + j (j < 4) or
// 16 + 4 g + j - 4: then two stacked 16 x 16 results in D form, rounded and
// packed, ARE the B (or, transposed, the A) operand of the next product, and
// the chain K S -> Y -> T Y -> K^T (dec o U) of a 16-column slice never leaves
// its wave's registers.
#include <mutex>

#include "common.hpp"
#include "abi_util.hpp"

namespace llmy {

constexpr int kC = 64;           // chunk length
constexpr int kTFrag = 6;        // 16 x 32 operand fragments of a causal 64 x 64 matrix
constexpr int kTElems = kTFrag * 2 * 64 * 8;  // bf16 of its (hi, lo) fragments
constexpr int kFac = 6 * kC;     // per-token factors of a chunk

// Fragment (row block m, 32-wide step s) of a lower triangular 64 x 64 matrix:
// row blocks 0 and 1 have one step, 2 and 3 two.
__host__ __device__ constexpr int tri_frag(int m, int s) { return m < 2 ? m : 2 * m - 2 + s; }

// x = hi + lo as 8 packed bf16 each, from two D-form tiles.
__device__ __forceinline__ void split_pair(const f32x4& a, const f32x4& b, uint4& hi, uint4& lo) {
  const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  uint32_t h[4], l[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h[j] = pack_bf2(x[2 * j], x[2 * j + 1]);
    l[j] = pack_bf2(x[2 * j] - __uint_as_float(h[j] << 16),
                    x[2 * j + 1] - __uint_as_float(h[j] & 0xffff0000u));
  }
  hi = uint4{h[0], h[1], h[2], h[3]};
  lo = uint4{l[0], l[1], l[2], l[3]};
}

__device__ __forceinline__ f32x4 mfma16(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// 16 x 16 fp32 product, k ordered as element e of lane group g is k = 4 g + e:
// the operands are D-form tiles (A transposed).
__device__ __forceinline__ f32x4 mfma16_f32(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

// ---------------------------------------------------------------------------
// Kernel 1: one wavefront per chunk; no wave waits for another.  Outputs per
// chunk id cid = (b*H + h) * NC + c: T's six (hi, lo) operand fragments
// [6][2][lane][8] bf16 and the factors [6][64] fp32: Gamma_t, Gamma_C / Gamma_t
// (both masked as above), beta_t, beta_t Gamma_{t-1}, the cumulative log-decay
// and the segment.
//
// K stays in registers (each lane 16 B of 16 rows per 32-wide step, serving
// both operands of K K^T).  The six blocks of N = I + L below the diagonal are
// used in the D form that K K^T leaves them in; the four diagonal blocks go
// through 5 KiB of LDS to be inverted together by forward substitution, lane
// (block, column) owning one column.  Then, in transposed D form,
//   T_ij^T = -T_jj^T (sum_{m=j+1..i} N_mj^T T_im^T)
// is a chain of fp32 MFMAs whose operands are all lane-local, and T_ij^T in D
// form is T in the scan's operand form.  Bound by reading K and writing T and
// the factors (16 + 13.5 KiB per chunk and head of 128): 8 x 4096 tokens, 16
// heads of 128: 46 us, 5.5 TB/s (a four-wave workgroup per chunk with the
// inverse in LDS: 108 us).
template <int D>
__global__ __launch_bounds__(64) void gdn_chunk_prep_kernel(
    const uint16_t* __restrict__ k, const float* __restrict__ beta, const float* __restrict__ g,
    const int32_t* __restrict__ reset, uint16_t* __restrict__ Tg, float* __restrict__ facg, int T,
    int H, int NC) {
  constexpr int NS = D / 32;
  constexpr int PD = 20, BD = 16 * PD + 16;  // row and block pitch of the diagonal blocks
  __shared__ __align__(16) float dg[4 * BD];
  __shared__ __align__(16) float cumS[kC], prvS[kC], betS[kC], segS[kC];

  const int cid = blockIdx.x;
  const int lane = threadIdx.x, r16 = lane & 15, g4 = lane >> 4;
  const int bh = cid / NC, c = cid - bh * NC;
  const int b = bh / H, h = bh - b * H;
  const int t0 = c * kC, Tc = min(kC, T - t0);
  const long long rk = static_cast<long long>(H) * D;
  const uint16_t* kb = k + (static_cast<long long>(b) * T + t0) * rk + static_cast<long long>(h) * D;

  // the per-token scalars first: their chain is the longest
  const long long tok = static_cast<long long>(b) * T + t0 + min(lane, Tc - 1);
  const float gv = g[tok * H + h], bv = beta[tok * H + h];
  const int32_t rv = reset != nullptr ? reset[tok] : 0;
  uint4 kf[4][NS];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int s = 0; s < NS; ++s)
      kf[m][s] = *reinterpret_cast<const uint4*>(kb + min(16 * m + r16, Tc - 1) * rk + 32 * s + 8 * g4);

  // inclusive prefix sum of log g over the chunk (past it: g = 1, beta = 0)
  const float lg = lane < Tc ? logf(gv) : 0.f;
  const float bt = lane < Tc ? bv : 0.f;
  float sc = lg;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float o = __shfl_up(sc, off, kWave);
    if (lane >= off) sc += o;
  }
  // segments: a reset at token r starts a new one; cumulative log-decays
  // restart there (minus the prefix before r)
  const unsigned long long rm = __ballot(lane < Tc && rv != 0);
  const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
  const int sg = __popcll(rm & upto);
  if (rm != 0) {
    const unsigned long long before = rm & upto;
    const int r0 = before ? 63 - __clzll(static_cast<long long>(before)) : lane;
    const float pre = __shfl(sc - lg, r0, kWave);  // cumulative log-decay before token r0
    sc -= before ? pre : 0.f;
  }
  cumS[lane] = sc;
  prvS[lane] = sc - lg;
  betS[lane] = bt;
  segS[lane] = static_cast<float>(sg);
  {
    const float cl = __shfl(sc, kC - 1, kWave);
    const int sl = __shfl(sg, kC - 1, kWave);
    float* f = facg + static_cast<long long>(cid) * kFac + lane;
    f[0] = sg == 0 ? __expf(sc) : 0.f;
    f[kC] = sg == sl ? __expf(cl - sc) : 0.f;
    f[2 * kC] = bt;
    f[3 * kC] = sg == 0 ? bt * __expf(sc - lg) : 0.f;
    f[4 * kC] = sc;
    f[5 * kC] = static_cast<float>(sg);
  }
  wave_lds_order();

  // ---- N = I + L: block (m, j) in D form (rows 4 g4 + i of m, column r16 of j)
  f32x4 nb[4][4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const f32x4 prv = *reinterpret_cast<const f32x4*>(prvS + 16 * m + 4 * g4);
    const f32x4 bet = *reinterpret_cast<const f32x4*>(betS + 16 * m + 4 * g4);
    const f32x4 seg = *reinterpret_cast<const f32x4*>(segS + 16 * m + 4 * g4);
#pragma unroll
    for (int j = 0; j <= m; ++j) {
      const float cj = cumS[16 * j + r16], sj = segS[16 * j + r16];
      f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NS; ++s) a = mfma16(kf[m][s], kf[j][s], a);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * m + 4 * g4 + i;
        const bool on = (16 * j + r16 < t) & (sj == seg[i]) & (t < Tc);
        a[i] = on ? bet[i] * __expf(prv[i] - cj) * a[i] : 0.f;
      }
      nb[m][j] = a;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) dg[m * BD + (4 * g4 + i) * PD + r16] = nb[m][m][i];
  }
  wave_lds_order();

  // ---- the diagonal blocks' inverses: lane (block g4, column r16)
  {
    const float* nd = dg + g4 * BD;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      f32x4 a = f32x4{t == r16 ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i4 = 0; 4 * i4 < t; ++i4) {
        const f32x4 n = *reinterpret_cast<const f32x4*>(nd + t * PD + 4 * i4);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (4 * i4 + i < t) a[i] -= n[i] * x[4 * i4 + i];
      }
      x[t] = t < r16 ? 0.f : (a[0] + a[1]) + (a[2] + a[3]);
    }
    wave_lds_order();
#pragma unroll
    for (int t = 0; t < 16; ++t) dg[g4 * BD + t * PD + r16] = x[t];
  }
  wave_lds_order();

  // ---- T_ij^T in D form; row block i needs only N and its own T_im, m > j
  f32x4 tt[4][4], tj[3];
#pragma unroll
  for (int m = 0; m < 4; ++m)
    tt[m][m] = *reinterpret_cast<const f32x4*>(dg + m * BD + r16 * PD + 4 * g4);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) tj[j][e] = dg[j * BD + (4 * g4 + e) * PD + r16];
#pragma unroll
  for (int d = 1; d < 4; ++d)
#pragma unroll
    for (int i = d; i < 4; ++i) {
      const int j = i - d;
      f32x4 p = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = j + 1; m <= i; ++m) p = mfma16_f32(nb[m][j], tt[i][m], p);
      p = mfma16_f32(tj[j], p, f32x4{0.f, 0.f, 0.f, 0.f});
      tt[i][j] = -p;
    }
  uint16_t* Tw = Tg + static_cast<long long>(cid) * kTElems + lane * 8;
  const f32x4 z = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int s = 0; s <= m / 2; ++s) {
      uint4 hi, lo;
      split_pair(tt[m][2 * s], 2 * s + 1 <= m ? tt[m][2 * s + 1] : z, hi, lo);
      uint16_t* w = Tw + tri_frag(m, s) * 1024;
      *reinterpret_cast<uint4*>(w) = hi;
      *reinterpret_cast<uint4*>(w + 512) = lo;
    }
}

// ---------------------------------------------------------------------------
// Kernel 2: sequential scan over chunks for one (b, h, CW-column state slice),
// CW = 16 NW.  Two kinds of waves share a workgroup:
//   NW state waves own 16 columns of S each, in registers (D form), and carry
//     the recurrence: P1: K S, Y; P2: U = T Y, S = Gamma_C S + K^T (dec o U).
//     S and U are split once and left in LDS as operand fragments;
//   4 helper waves do what the recurrence does not wait for: P1: the previous
//     chunk's + U^T A^T and its output (four columns of a token per lane: 8-byte
//     stores), and the K Q^T tiles of A, already in operand form; P2: A's six
//     fragments, and (Q S)^T of one state wave's columns each.  They also start
//     the next chunk's copies into LDS (buffer loads with the lds bit: no
//     register holds staged data): K, Q, T and the factors, double-buffered, in
//     P1; V, whose last reads are in P1, in P2.
// Two barriers per chunk; the helpers' products hide behind the recurrence.
// Each phase's LDS reads are issued before the phase's first MFMA: the
// compiler would put every read next to its use and wait out some forty LDS
// latencies a chunk.
// The 16-byte chunks of K, Q and V rows are XOR-swizzled by row (on the source
// side of the copies): by the bank map row fragments (16-byte reads of 16 rows)
// meet no conflict, nor do K^T's (ds_read_b64_tr_b16 of 8 rows); the counter still
// shows conflicts in 10% of the cycles, from reads not yet told apart.
// Slices of one (b, h) run on one XCD (block id mod 8) and share its L2.
// 8 x 4096 tokens, 16 heads of 128: 212 us of back-to-back calls (first calls on an
// idle GPU up to 285), about 7.6k cycles a chunk (eight equal waves that passed S, Y
// and U through LDS: 275 us, 9.2k).  No unit is saturated (LDS active 42% of the
// cycles, VALU 37%, matrix cores 30%; 667 MB of HBM traffic, 3.1 TB/s): the
// recurrence's dependent products, the reads in front of them and the two barriers
// set the pace.
template <int D>
__device__ __forceinline__ int kq_swz(int t) {
  return D == 128 ? (4 * (t & 3)) | ((t >> 2) & 3) : (4 * ((t >> 1) & 1)) | ((t >> 2) & 3);
}

template <int NW>
__device__ __forceinline__ int v_swz(int t) {
  return NW == 4 ? 2 * ((t >> 1) & 3) : NW == 2 ? 2 * ((t >> 2) & 1) : 0;
}

// One copy into LDS: 16 (or 4) bytes per lane from rsrc + off to dst + lane *
// 16 (4).  What lanes past the buffer's range leave in LDS is not relied on
// (the kernel clears the rows of a ragged chunk first).  In inline asm so that
// the compiler does not make every later LDS read of the wave wait for it; the
// wave waits (vmcnt) before the barrier that publishes the data.  The compiler
// inserts no wait states for what is inside: s_nop 3 after the move of m0 makes
// the five that a buffer load needs after a VALU write of its descriptor (a
// readfirstlane, or a v_readlane that restores a spilled SGPR).  m0 is reserved
// (nothing is allocated to it, hence the compiler's warning), but the compiler
// itself keeps values there for LDS-DMA builtins and indexed moves: the clobber
// tells it that they are gone.  (The wait states cost 0.4 us of 34.6 at 1 x 1003 tokens,
// 16 heads of 64, and nothing measurable at 128; one wait for several copies in one
// statement was no faster.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_copy16(const u32x4& rsrc, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               ::"s"(dst), "v"(off), "s"(rsrc) : "memory", "m0");
}
__device__ __forceinline__ void lds_copy4(const u32x4& rsrc, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, 0 offen lds"
               ::"s"(dst), "v"(off), "s"(rsrc) : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ u32x4 buffer_of(const void* p, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return u32x4{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a))),
               static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32))),
               static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(bytes)), 0x00020000u};
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}

template <int N>
struct Int {
  static constexpr int value = N;
};

__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// ds_read_b64_tr_b16: in each 16-lane group, lane 4 a + e receives element e of
// the 8 bytes that lanes a, a + 4, a + 8, a + 12 address.
__device__ __forceinline__ uint2 lds_tr(const uint16_t* p) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_s16x4*)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)p);
  return __builtin_bit_cast(uint2, v);
}

template <int D, int NW>
__global__ __launch_bounds__(64 * (NW + 4)) void gdn_chunk_scan_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, const uint16_t* __restrict__ Tg,
    const float* __restrict__ facg, float* __restrict__ state, uint16_t* __restrict__ out, int T,
    int H, int NC, int n_units, int wide) {
  constexpr int NS = D / 32, MT = D / 16, CW = 16 * NW, NSL = D / CW;
  __shared__ __align__(16) uint16_t Ks[2][kC * D], Qs[2][kC * D], Vs[kC * CW];
  __shared__ __align__(16) uint16_t Ts[2][kTElems], As[kTElems];
  __shared__ __align__(16) uint16_t SF[NW * NS * 2 * 512], UF[NW * 4 * 512];
  __shared__ __align__(16) float fc[2][kFac];

  const int per_xcd = (gridDim.x + 7) / 8;
  const int unit = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (unit >= n_units) return;
  const int bh = unit / NSL;
  const int sl = unit - bh * NSL;
  const int b = bh / H, h = bh - b * H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const long long rk = static_cast<long long>(H) * D;

  if (T & (kC - 1)) {
    // a ragged last chunk: rows that no copy fills must not hold NaN patterns
    const uint4 z = uint4{0u, 0u, 0u, 0u};
    for (int i = tid; i < kC * D / 8; i += 64 * (NW + 4)) {
      reinterpret_cast<uint4*>(Ks[0])[i] = z;
      reinterpret_cast<uint4*>(Ks[1])[i] = z;
      reinterpret_cast<uint4*>(Qs[0])[i] = z;
      reinterpret_cast<uint4*>(Qs[1])[i] = z;
      if (i < kC * CW / 8) reinterpret_cast<uint4*>(Vs)[i] = z;
    }
    __syncthreads();
  }

  // fragment (16 rows from 16 m, dims 32 s + 8 g4 .. +7) of a K or Q tile
  auto frag = [&](const uint16_t* base, int m, int s) {
    return *reinterpret_cast<const uint4*>(base + (16 * m + r16) * D +
                                           8 * ((4 * s + g4) ^ kq_swz<D>(r16)));
  };
  // S tiles 2 s and 2 s + 1 in D form hold state rows 32 s + 8 g4 + i and + 4 +
  // i, the latter first for odd g4: they pack (after that swap) to the dims of
  // a fragment, and K^T's fragments read both halves of their 16-byte chunks
  auto srow = [&](int m, int i) {
    return 32 * (m >> 1) + 8 * g4 + 4 * ((m & 1) ^ (g4 & 1)) + i;
  };
  const f32x4 zf = f32x4{0.f, 0.f, 0.f, 0.f};

  if (wave < NW) {
    // ------------------------------------------------------------ state wave
    float* Sg = state + static_cast<long long>(bh) * D * D + CW * sl + 16 * wave + r16;
    f32x4 S[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[m][i] = Sg[srow(m, i) * D];
    uint16_t* const sf = SF + wave * NS * 1024 + lane * 8;
    uint16_t* const uf = UF + wave * 2048 + lane * 8;
    __syncthreads();
    for (int c = 0; c < NC; ++c) {
      const uint16_t* const Kc = Ks[c & 1];
      const float* const f = fc[c & 1];
      // P1: K S with S split once, then Y = beta o V - (beta Gamma_prev) o (K S)
      uint4 a[NS][4];
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int m = 0; m < 4; ++m) a[s][m] = frag(Kc, m, s);
      sched_fence();
      uint4 sh[NS], so[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const bool odd = g4 & 1;
        split_pair(odd ? S[2 * s + 1] : S[2 * s], odd ? S[2 * s] : S[2 * s + 1], sh[s], so[s]);
        *reinterpret_cast<uint4*>(sf + s * 1024) = sh[s];
        *reinterpret_cast<uint4*>(sf + s * 1024 + 512) = so[s];
      }
      uint2 vv[4];  // V[16 m + 4 g4 + i][this lane's column]
      f32x4 bt[4], ws[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int t = 16 * m + 4 * g4 + (r16 >> 2), e = r16 & 3;
        vv[m] = lds_tr(Vs + t * CW + 8 * ((2 * wave + (e >> 1)) ^ v_swz<NW>(t)) + 4 * (e & 1));
        bt[m] = *reinterpret_cast<const f32x4*>(f + 2 * kC + 16 * m + 4 * g4);
        ws[m] = *reinterpret_cast<const f32x4*>(f + 3 * kC + 16 * m + 4 * g4);
      }
      sched_fence();
      f32x4 y[4] = {zf, zf, zf, zf};
#pragma unroll
      for (int s = 0; s < NS; ++s) {
#pragma unroll
        for (int m = 0; m < 4; ++m) y[m] = mfma16(a[s][m], sh[s], y[m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) y[m] = mfma16(a[s][m], so[s], y[m]);
      }
      uint4 th[kTFrag], tl[kTFrag];
#pragma unroll
      for (int i = 0; i < kTFrag; ++i) {
        th[i] = *reinterpret_cast<const uint4*>(Ts[c & 1] + i * 1024 + lane * 8);
        tl[i] = *reinterpret_cast<const uint4*>(Ts[c & 1] + i * 1024 + 512 + lane * 8);
      }
      sched_fence();
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float vf[4] = {__uint_as_float(vv[m].x << 16), __uint_as_float(vv[m].x & 0xffff0000u),
                             __uint_as_float(vv[m].y << 16), __uint_as_float(vv[m].y & 0xffff0000u)};
#pragma unroll
        for (int i = 0; i < 4; ++i) y[m][i] = bt[m][i] * vf[i] - ws[m][i] * y[m][i];
      }
      uint4 yh[2], yl[2];
      split_pair(y[0], y[1], yh[0], yl[0]);
      split_pair(y[2], y[3], yh[1], yl[1]);
      __syncthreads();  // S fragments ready; U fragments, A and V read
      // P2: U = T Y, then S = Gamma_C S + K^T (dec o U)
      uint4 kt[2][MT];
      f32x4 de[4];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int t = 32 * s + 4 * g4 + (r16 >> 2);
          const uint16_t* p =
              Kc + t * D + 8 * ((4 * (m >> 1) + (r16 & 3)) ^ kq_swz<D>(t)) + 4 * ((m ^ r16) & 1);
          const uint2 a0 = lds_tr(p), a1 = lds_tr(p + 16 * D);
          kt[s][m] = uint4{a0.x, a0.y, a1.x, a1.y};
        }
#pragma unroll
      for (int m = 0; m < 4; ++m) de[m] = *reinterpret_cast<const f32x4*>(f + kC + 16 * m + 4 * g4);
      const float gc = f[kC - 1];  // Gamma_C (0 when the chunk resets)
      sched_fence();
      f32x4 u[4] = {zf, zf, zf, zf};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int m = 2 * s; m < 4; ++m) u[m] = mfma16(th[tri_frag(m, s)], yh[s], u[m]);
#pragma unroll
        for (int m = 2 * s; m < 4; ++m) u[m] = mfma16(th[tri_frag(m, s)], yl[s], u[m]);
#pragma unroll
        for (int m = 2 * s; m < 4; ++m) u[m] = mfma16(tl[tri_frag(m, s)], yh[s], u[m]);
      }
      uint4 dh[2], dl[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 uh, ul;
        split_pair(u[2 * s], u[2 * s + 1], uh, ul);
        *reinterpret_cast<uint4*>(uf + s * 1024) = uh;
        *reinterpret_cast<uint4*>(uf + s * 1024 + 512) = ul;
        split_pair(de[2 * s] * u[2 * s], de[2 * s + 1] * u[2 * s + 1], dh[s], dl[s]);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) S[m] *= gc;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int m = 0; m < MT; ++m) S[m] = mfma16(kt[s][m], dh[s], S[m]);
#pragma unroll
        for (int m = 0; m < MT; ++m) S[m] = mfma16(kt[s][m], dl[s], S[m]);
      }
      __syncthreads();  // U fragments and A ready; the next chunk is staged
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) Sg[srow(m, i) * D] = S[m][i];
    return;
  }

  // -------------------------------------------------------------- helper wave
  const int hw = wave - NW;
  // copies: instruction j of an array fills 64 consecutive 16-byte slots; this
  // wave takes j = hw + 4 i.  K and Q slot (row t, p) holds the row's chunk p ^
  // swizzle, V likewise
  constexpr int CK = D / 8, RK = 64 / CK, NK = kC / RK / 4;   // chunks per row, rows, per wave
  constexpr int CV = CW / 8, RV = 64 / CV, IV = kC / RV, NV = (IV + 3) / 4;
  uint32_t ok[NK], ov[NV];
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const int t = (hw + 4 * i) * RK + lane / CK;
    ok[i] = static_cast<uint32_t>(t * rk * 2) + 16 * ((lane % CK) ^ kq_swz<D>(t));
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int t = (hw + 4 * i) * RV + lane / CV;
    ov[i] = static_cast<uint32_t>(t * rk * 2) + 16 * ((lane % CV) ^ v_swz<NW>(t));
  }
  const uint32_t aK = lds_addr(Ks), aQ = lds_addr(Qs), aV = lds_addr(Vs), aT = lds_addr(Ts),
                 aF = lds_addr(fc);
  auto row0 = [&](int c_) {
    return (static_cast<long long>(b) * T + c_ * kC) * rk + static_cast<long long>(h) * D;
  };
  auto copy_next = [&](int c_, int buf) {  // K, Q, T and the factors
    const int Tc = min(kC, T - c_ * kC);
    const uint32_t n = static_cast<uint32_t>(((Tc - 1) * rk + D) * 2);
    const long long cid = static_cast<long long>(bh) * NC + c_;
    const u32x4 rs = buffer_of(k + row0(c_), n), rq = buffer_of(q + row0(c_), n);
    const u32x4 rt = buffer_of(Tg + cid * kTElems, kTElems * 2);
    const u32x4 rf = buffer_of(facg + cid * kFac, kFac * 4);
#pragma unroll
    for (int i = 0; i < NK; ++i) lds_copy16(rs, ok[i], aK + buf * (kC * D * 2) + (hw + 4 * i) * 1024);
    lds_copy4(rf, hw * 256 + lane * 4, aF + buf * (kFac * 4) + hw * 256);
    if (hw < 2) lds_copy4(rf, (4 + hw) * 256 + lane * 4, aF + buf * (kFac * 4) + (4 + hw) * 256);
#pragma unroll
    for (int i = 0; i < NK; ++i) lds_copy16(rq, ok[i], aQ + buf * (kC * D * 2) + (hw + 4 * i) * 1024);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      lds_copy16(rt, (hw + 4 * i) * 1024 + lane * 16, aT + buf * (kTElems * 2) + (hw + 4 * i) * 1024);
  };
  auto copy_v = [&](int c_) {
    const int Tc = min(kC, T - c_ * kC);
    const u32x4 rv = buffer_of(v + row0(c_) + CW * sl, static_cast<uint32_t>(((Tc - 1) * rk + CW) * 2));
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (4 * i + 3 < IV || hw + 4 * i < IV) lds_copy16(rv, ov[i], aV + (hw + 4 * i) * 1024);
  };
  // (Q S)^T of state wave hw's columns, scaled by Gamma: lane holds columns 4
  // g4 + i of token 16 m + r16; finish() adds U^T A^T and stores the chunk
  f32x4 o[4] = {zf, zf, zf, zf};
  auto finish = [&](int c_) {
    const int t0 = c_ * kC, Tc = min(kC, T - t0);
    const uint16_t* const uf = UF + hw * 2048 + lane * 8;
    uint4 uh[2], ul[2], ah[kTFrag], al[kTFrag];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uh[s] = *reinterpret_cast<const uint4*>(uf + s * 1024);
      ul[s] = *reinterpret_cast<const uint4*>(uf + s * 1024 + 512);
    }
#pragma unroll
    for (int i = 0; i < kTFrag; ++i) {
      ah[i] = *reinterpret_cast<const uint4*>(As + i * 1024 + lane * 8);
      al[i] = *reinterpret_cast<const uint4*>(As + i * 1024 + 512 + lane * 8);
    }
    sched_fence();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int m = 2 * s; m < 4; ++m) o[m] = mfma16(uh[s], ah[tri_frag(m, s)], o[m]);
#pragma unroll
      for (int m = 2 * s; m < 4; ++m) o[m] = mfma16(ul[s], ah[tri_frag(m, s)], o[m]);
#pragma unroll
      for (int m = 2 * s; m < 4; ++m) o[m] = mfma16(uh[s], al[tri_frag(m, s)], o[m]);
    }
    // tokens past the chunk lie beyond the buffer's range: dropped
    const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(
        out + row0(c_) + CW * sl, static_cast<short>(0),
        static_cast<int>(((Tc - 1) * rk + CW) * 2), 0x00020000);
    if (wide) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        const int at = static_cast<int>(((16 * m + r16) * rk + 16 * hw + 4 * g4) * 2);
        __builtin_amdgcn_raw_buffer_store_b64(
            u32x2{pack_bf2(o[m][0], o[m][1]), pack_bf2(o[m][2], o[m][3])}, orsrc, at, 0, 0);
      }
    } else {  // out not 8-byte aligned
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          __builtin_amdgcn_raw_buffer_store_b16(
              f2bf(o[m][i]), orsrc,
              static_cast<int>(((16 * m + r16) * rk + 16 * hw + 4 * g4 + i) * 2), 0, 0);
    }
  };
  // A's tiles: each helper forms one fragment of two tiles (token block ti,
  // key blocks tj, tj + 1), two of them also a fragment of one diagonal tile
  const int ti = hw == 0 || hw == 1 ? 3 : hw == 2 ? 2 : 1, tj = hw == 1 ? 2 : 0;
  const int fi = hw == 0 ? 4 : hw == 1 ? 5 : hw == 2 ? 2 : 1;
  const int td = hw == 2 ? 0 : 2, fd = hw == 2 ? 0 : 3;
  copy_next(0, 0);
  copy_v(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int c = 0; c < NC; ++c) {
    const uint16_t* const Kc = Ks[c & 1];
    const uint16_t* const Qc = Qs[c & 1];
    const float* const f = fc[c & 1];
    const int cn = min(c + 1, NC - 1);  // the last chunk copies itself again
    copy_next(cn, (c + 1) & 1);
    // P1: the previous chunk's output, then the K Q^T tiles of A (lane holds
    // token 16 i + r16, keys 16 j + 4 g4 + e)
    if (c > 0 && hw < NW) finish(c - 1);
    f32x4 x = zf, y = zf, z = zf;
    auto tiles = [&](auto TI, auto TJ, auto TD) {
      uint4 ka[NS], kb[NS], kd[NS], qa[NS], qd[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        ka[s] = frag(Kc, TJ.value, s);
        kb[s] = frag(Kc, TJ.value + 1, s);
        qa[s] = frag(Qc, TI.value, s);
        if (TD.value > 0) kd[s] = frag(Kc, TD.value, s);
        if (TD.value >= 0) qd[s] = frag(Qc, TD.value & 3, s);
      }
      sched_fence();
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        x = mfma16(ka[s], qa[s], x);
        y = mfma16(kb[s], qa[s], y);
        if (TD.value >= 0) z = mfma16(TD.value > 0 ? kd[s] : ka[s], qd[s], z);
      }
    };
    if (hw == 0)
      tiles(Int<3>{}, Int<0>{}, Int<-1>{});
    else if (hw == 1)
      tiles(Int<3>{}, Int<2>{}, Int<-1>{});
    else if (hw == 2)
      tiles(Int<2>{}, Int<0>{}, Int<0>{});
    else
      tiles(Int<1>{}, Int<0>{}, Int<2>{});
    __syncthreads();  // S fragments ready; U fragments, A and V read
    // P2: A's fragments and (Q S)^T
    copy_v(cn);
    uint4 sh[NS], so[NS], qf[NS][4];
    float e[4];
    if (hw < NW) {
      const uint16_t* const sf = SF + hw * NS * 1024 + lane * 8;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        sh[s] = *reinterpret_cast<const uint4*>(sf + s * 1024);
        so[s] = *reinterpret_cast<const uint4*>(sf + s * 1024 + 512);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) e[m] = f[16 * m + r16];
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int m = 0; m < 4; ++m) qf[s][m] = frag(Qc, m, s);
    }
    sched_fence();
    auto mask = [&](f32x4 w, int i, int j) {
      const int t = 16 * i + r16, j0 = 16 * j + 4 * g4;
      const float ct = f[4 * kC + t], st = f[5 * kC + t];
      const f32x4 cj = *reinterpret_cast<const f32x4*>(f + 4 * kC + j0);
      const f32x4 sj = *reinterpret_cast<const f32x4*>(f + 5 * kC + j0);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const float d = __expf(ct - cj[n]) * w[n];
        w[n] = ((j0 + n <= t) & (sj[n] == st)) ? d : 0.f;
      }
      return w;
    };
    auto put = [&](int i, const f32x4& w0, const f32x4& w1) {
      uint4 hi, lo;
      split_pair(w0, w1, hi, lo);
      *reinterpret_cast<uint4*>(As + i * 1024 + lane * 8) = hi;
      *reinterpret_cast<uint4*>(As + i * 1024 + 512 + lane * 8) = lo;
    };
    put(fi, mask(x, ti, tj), mask(y, ti, tj + 1));
    if (hw >= 2) put(fd, mask(z, td, td), zf);
    if (hw < NW) {
#pragma unroll
      for (int m = 0; m < 4; ++m) o[m] = zf;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
#pragma unroll
        for (int m = 0; m < 4; ++m) o[m] = mfma16(sh[s], qf[s][m], o[m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) o[m] = mfma16(so[s], qf[s][m], o[m]);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) o[m] *= e[m];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies have landed
    __syncthreads();  // U fragments and A ready; the next chunk is staged
  }
  if (hw < NW) finish(NC - 1);
}

}  // namespace llmy

using namespace llmy;

extern "C" int64_t llmy_gdn_prefill_workspace_bytes(int32_t B, int32_t T, int32_t H, int32_t dk,
                                                    int32_t dv) {
  if (B <= 0 || T <= 0 || H <= 0 || dk <= 0 || dv <= 0) return 0;
  const long long nc = (T + kC - 1) / kC;
  const long long chunks = static_cast<long long>(B) * H * nc;
  return chunks * kC * (static_cast<long long>(dk) + dv + kC + 2) * static_cast<long long>(sizeof(float));
}

namespace {

template <int D, int NW>
void launch_scan(const llmy_bf16* q, const llmy_bf16* k, const llmy_bf16* v, const uint16_t* Tf,
                 const float* fac, float* state, llmy_bf16* out, int B, int T, int H, int NC,
                 hipStream_t s) {
  const int units = B * H * (D / (16 * NW));
  hipLaunchKernelGGL((gdn_chunk_scan_kernel<D, NW>), dim3((units + 7) / 8 * 8), dim3(64 * (NW + 4)),
                     0, s, q, k, v, Tf, fac, state, out, T, H, NC, units,
                     aligned(out, 8) ? 1 : 0);
}

// The prep + scan launches over a caller-sized workspace (validated by the
// entry points below).
template <int D>
int32_t gdn_prefill_run(const llmy_bf16* q, const llmy_bf16* k, const llmy_bf16* v,
                        const float* beta, const float* g, const int32_t* reset, float* state,
                        llmy_bf16* out, void* workspace, int B, int T, int H, hipStream_t s) {
  const int NC = (T + kC - 1) / kC;
  const long long chunks = static_cast<long long>(B) * H * NC;
  // workspace: T's fragments of every chunk, then the per-token factors
  // (kTElems * 2 + kFac * 4 = 13.5 KiB per chunk of the 49 or 82 KiB required)
  uint16_t* Tf = static_cast<uint16_t*>(workspace);
  float* fac = reinterpret_cast<float*>(Tf + chunks * kTElems);
  hipLaunchKernelGGL((gdn_chunk_prep_kernel<D>), dim3(static_cast<unsigned>(chunks)), dim3(64), 0,
                     s, k, beta, g, reset, Tf, fac, T, H, NC);
  const int32_t st = launch_status();
  if (st != 0) return st;
  // Slice width: as narrow as one round of workgroups allows.  A chunk's chain
  // of products does not shrink with the slice, its LDS traffic does (16 heads
  // of 128, us for NW = 1 / 2 / 4: 1 x 4096 tokens, 128 column tiles: 141 / 155
  // / 208; 4 x 1024, 512 tiles: 83 / 54 / 64; 8 x 2048, 1024 tiles: 289 / 175 /
  // 133).
  const long long cols = static_cast<long long>(B) * H * (D / 16), cus = compute_units();
  if (cols <= cus)
    launch_scan<D, 1>(q, k, v, Tf, fac, state, out, B, T, H, NC, s);
  else if (cols <= 2 * cus)
    launch_scan<D, 2>(q, k, v, Tf, fac, state, out, B, T, H, NC, s);
  else
    launch_scan<D, 4>(q, k, v, Tf, fac, state, out, B, T, H, NC, s);
  return launch_status();
}

int32_t gdn_prefill_launch(const llmy_bf16* q, const llmy_bf16* k, const llmy_bf16* v,
                           const float* beta, const float* g, const int32_t* reset, float* state,
                           llmy_bf16* out, void* workspace, int B, int T, int H, int dk,
                           hipStream_t s) {
  return dk == 64 ? gdn_prefill_run<64>(q, k, v, beta, g, reset, state, out, workspace, B, T, H, s)
                  : gdn_prefill_run<128>(q, k, v, beta, g, reset, state, out, workspace, B, T, H, s);
}

// Workspace of the no-allocation entry point: a fixed device array, one copy
// per GPU (each device holds it from module load until the process ends).
// Host code never passes `scratch` itself (in host code the name is a
// stand-in, not a device address): the per-device address comes from
// hipGetSymbolAddress, once per device, with that device current.
constexpr long long kStaticWorkspaceBytes = 64ll << 20;
__device__ __align__(256) unsigned char scratch[kStaticWorkspaceBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's copy of `scratch` (null on failure).
void* static_workspace() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int32_t llmy_gdn_prefill_bf16(const llmy_bf16* q, const llmy_bf16* k,
                                         const llmy_bf16* v, const float* beta, const float* g,
                                         float* state, llmy_bf16* out, void* workspace,
                                         int64_t workspace_bytes, int32_t B, int32_t T,
                                         int32_t H, int32_t dk, int32_t dv, void* stream) {
  LLMY_REQUIRE(B >= 0 && T >= 0 && H > 0);
  LLMY_REQUIRE((dk == 64 && dv == 64) || (dk == 128 && dv == 128));
  if (B == 0 || T == 0) return 0;
  LLMY_REQUIRE(q && k && v && beta && g && state && out && workspace);
  LLMY_REQUIRE(workspace_bytes >= llmy_gdn_prefill_workspace_bytes(B, T, H, dk, dv));
  LLMY_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(state, 16) &&
               aligned(workspace, 16));
  const long long chunks = static_cast<long long>(B) * H * ((T + kC - 1) / kC);
  LLMY_REQUIRE(chunks < (1ll << 31));
  return gdn_prefill_launch(q, k, v, beta, g, nullptr, state, out, workspace, B, T, H, dk,
                            as_stream(stream));
}

extern "C" int32_t llmy_gdn_prefill_reset_bf16(const llmy_bf16* q, const llmy_bf16* k,
                                               const llmy_bf16* v, const float* beta,
                                               const float* g, const int32_t* reset, float* state,
                                               llmy_bf16* out, void* workspace,
                                               int64_t workspace_bytes, int32_t B, int32_t T,
                                               int32_t H, int32_t dk, int32_t dv, void* stream) {
  LLMY_REQUIRE(B >= 0 && T >= 0 && H > 0);
  LLMY_REQUIRE((dk == 64 && dv == 64) || (dk == 128 && dv == 128));
  if (B == 0 || T == 0) return 0;
  LLMY_REQUIRE(q && k && v && beta && g && reset && state && out && workspace);
  LLMY_REQUIRE(workspace_bytes >= llmy_gdn_prefill_workspace_bytes(B, T, H, dk, dv));
  LLMY_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(state, 16) &&
               aligned(workspace, 16));
  const long long chunks = static_cast<long long>(B) * H * ((T + kC - 1) / kC);
  LLMY_REQUIRE(chunks < (1ll << 31));
  return gdn_prefill_launch(q, k, v, beta, g, reset, state, out, workspace, B, T, H, dk,
                            as_stream(stream));
}

extern "C" int32_t llmy_gdn_prefill_bf16_noalloc(const llmy_bf16* q, const llmy_bf16* k,
                                                 const llmy_bf16* v, const float* beta,
                                                 const float* g, float* state, llmy_bf16* out,
                                                 int32_t B, int32_t T, int32_t H, int32_t dk,
                                                 int32_t dv, void* stream) {
  LLMY_REQUIRE(B >= 0 && T >= 0 && H > 0);
  LLMY_REQUIRE((dk == 64 && dv == 64) || (dk == 128 && dv == 128));
  if (B == 0 || T == 0) return 0;
  LLMY_REQUIRE(q && k && v && beta && g && state && out);
  LLMY_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(state, 16));
  // beyond the fixed workspace: a distinct status, before anything runs
  if (llmy_gdn_prefill_workspace_bytes(B, T, H, dk, dv) > kStaticWorkspaceBytes)
    return static_cast<int32_t>(hipErrorOutOfMemory);
  void* ws = static_workspace();
  if (!ws) return static_cast<int32_t>(hipErrorInvalidDevicePointer);
  // every workspace byte the scan reads is written by this call's prep kernel
  // first, so what an earlier call left there does not matter
  return gdn_prefill_launch(q, k, v, beta, g, nullptr, state, out, ws, B, T, H, dk,
                            as_stream(stream));
}
