// gx_mlp.hip -- BF16 MFMA kernels for the learned acceleration surrogate.
//
// The surrogate is an MLP (5 inputs: rotating-frame x, y, z, R, r; four hidden
// layers of 256 with SiLU; 3 outputs) standing in for the expensive part of a
// composite field (a rotating bar plus dozens of co-rotating subhaloes).
// Weights and activations are BF16; every product accumulates in FP32 on the
// matrix cores (v_mfma_f32_16x16x32_bf16).
//
// Forward and backward passes are strided products:
//   C[m, n] = sum_k A(m, k) B(k, n),  A(m,k) = A[m*sam + k*sak],
//                                     B(k,n) = B[k*sbk + n*sbn]   (BF16)
// with a fused epilogue (bias + SiLU storing the pre-activation, bias only,
// SiLU backward, or a plain FP32 store).  k_gemm takes every shape, k_gemm_rows
// and k_gemm_cols the large ones where they are the faster (use_gemm_rows,
// use_gemm_cols).  In k_gemm a 256-thread block computes a 64x64 tile; each wave a 32x32 quarter as 2x2 MFMA tiles; K advances in slabs of
// 32 staged through LDS (16-byte loads when the reduction axis is
// contiguous).
//
// MFMA operand layout (16x16x32 BF16, wave64): lane l supplies
// A[l%16][8(l/16) .. 8(l/16)+7] and B[8(l/16) .. +7][l%16]; it receives
// D[4(l/16) + j][l%16], j = 0..3.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "gx_internal.hpp"
#include "gx_potential.hpp"
#include "gx_tableau.hpp"

namespace gx {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4;

// x, or zero where keep is false, by a bit mask: loads feeding it stay
// unconditional (a select between a loaded value and zero compiled to a
// branch around the load and a wait after it).
__device__ __forceinline__ float keep_or_zero(float x, bool keep) {
  return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) & (keep ? ~0u : 0u));
}

constexpr int BM = 64, BN = 64, BK = 32;
constexpr int LDSK = BK + 8;  // padded row (bf16 elements) against bank conflicts

enum : int {
  EPI_STORE = GX_EPI_STORE,
  EPI_BIAS = GX_EPI_BIAS,
  EPI_BIAS_SILU = GX_EPI_BIAS_SILU,
  EPI_DSILU = GX_EPI_DSILU
};

struct GemmArgs {
  const __bf16* A;
  long long sam, sak;
  const __bf16* B;
  long long sbk, sbn;
  long long M, N, K;
  int epi;
  int accumulate;       // EPI_STORE: add into C (atomically when split over K)
  int ksplit;           // blocks along K (grid z); > 1 only with EPI_STORE
  const float* bias;    // [N]
  float* C;             // fp32 output (EPI_STORE / EPI_BIAS); Z for BIAS_SILU
  long long ldc;
  __bf16* H;            // bf16 output (BIAS_SILU: silu(Z); DSILU: dZ)
  long long ldh;
  const float* Zin;     // DSILU: pre-activation
  long long ldzin;
};

// SiLU and its derivative in FP32 with the hardware reciprocal (1 ulp): the
// results are rounded to BF16 (8 bits), and a correctly rounded division
// took ten instructions per activation.  exp(-z) = +inf for very negative
// z gives 1/inf = 0, so silu -> -0 and dsilu -> 0 there, as in the limit.
__device__ __forceinline__ float sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = sigmoid(z);
  return s * (1.0f + z * (1.0f - s));
}

// Stages a 64 x 32 slab of a strided BF16 operand X(r, k) = X[r*sr + k*sk]
// (rows r0.., reduction index k0..) into LDS as T[r][k], zero-padding out of
// range entries.  Three load shapes: 16-byte loads along k (sk == 1), 16-byte
// loads along r (sr == 1, e.g. the transposed operands of the weight
// gradient), or scalar loads.
template <bool VEC>
__device__ __forceinline__ void stage_tile(__bf16 (*T)[LDSK], const __bf16* X,
                                           long long sr, long long sk,
                                           long long r0, long long R,
                                           long long k0, long long K, int tid) {
  if (VEC && sk == 1) {
    const int r = tid >> 2, kc = (tid & 3) * 8;
    const long long rr = r0 + r, k = k0 + kc;
    const __bf16* src = X + rr * sr + k;
    if (rr < R && k + 8 <= K && ((reinterpret_cast<uintptr_t>(src) & 15) == 0)) {
      *reinterpret_cast<bf16x8*>(&T[r][kc]) = *reinterpret_cast<const bf16x8*>(src);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        T[r][kc + j] = (rr < R && k + j < K) ? X[rr * sr + k + j] : (__bf16)0.0f;
    }
  } else if (VEC && sr == 1) {
    const int kq = tid >> 3, rc = (tid & 7) * 8;
    const long long k = k0 + kq, rr = r0 + rc;
    const __bf16* src = X + k * sk + rr;
    if (k < K && rr + 8 <= R && ((reinterpret_cast<uintptr_t>(src) & 15) == 0)) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(src);
#pragma unroll
      for (int j = 0; j < 8; ++j) T[rc + j][kq] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        T[rc + j][kq] = (k < K && rr + j < R) ? X[k * sk + rr + j] : (__bf16)0.0f;
    }
  } else {
    const int r = tid >> 2, kc = (tid & 3) * 8;
    const long long rr = r0 + r;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const long long k = k0 + kc + j;
      T[r][kc + j] = (rr < R && k < K) ? X[rr * sr + k * sk] : (__bf16)0.0f;
    }
  }
}

template <bool VEC>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs g) {
  __shared__ __bf16 As[BM][LDSK];
  __shared__ __bf16 Bs[BN][LDSK];  // B transposed: [n][k]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  // m tiles on x (up to 2^31 - 1 blocks), n tiles on y
  const long long m0 = (long long)blockIdx.x * BM, n0 = (long long)blockIdx.y * BN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this block's share of the reduction (split-K for the weight gradients,
  // whose reduction runs over the whole batch)
  const long long kper = ((g.K + g.ksplit - 1) / g.ksplit + BK - 1) / BK * BK;
  const long long kbeg = (long long)blockIdx.z * kper;
  const long long kend = kbeg + kper < g.K ? kbeg + kper : g.K;
  for (long long k0 = kbeg; k0 < kend; k0 += BK) {
    // ---- stage A (64 x 32) and B^T (64 x 32) into LDS, [row][k] order
    stage_tile<VEC>(As, g.A, g.sam, g.sak, m0, g.M, k0, kend, tid);
    stage_tile<VEC>(Bs, g.B, g.sbn, g.sbk, n0, g.N, k0, kend, tid);
    __syncthreads();
    // ---- 2x2 MFMA tiles per wave
    const int kk = (lane >> 4) * 8;
    bf16x8 af[2], bfr[2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
      af[a] = *reinterpret_cast<const bf16x8*>(&As[wm + a * 16 + (lane & 15)][kk]);
#pragma unroll
    for (int b = 0; b < 2; ++b)
      bfr[b] = *reinterpret_cast<const bf16x8*>(&Bs[wn + b * 16 + (lane & 15)][kk]);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
    __syncthreads();
  }
  // ---- epilogue
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const long long m = m0 + wm + a * 16 + (lane >> 4) * 4 + j;
        const long long n = n0 + wn + b * 16 + (lane & 15);
        if (m >= g.M || n >= g.N) continue;
        float v = acc[a][b][j];
        switch (g.epi) {
          case EPI_STORE:
            if (g.ksplit > 1) {
              atomicAdd(g.C + m * g.ldc + n, v);
            } else {
              if (g.accumulate) v += g.C[m * g.ldc + n];
              g.C[m * g.ldc + n] = v;
            }
            break;
          case EPI_BIAS:
            g.C[m * g.ldc + n] = v + g.bias[n];
            break;
          case EPI_BIAS_SILU: {
            const float z = v + g.bias[n];
            if (g.C) g.C[m * g.ldc + n] = z;
            g.H[m * g.ldh + n] = (__bf16)silu(z);
            break;
          }
          default: {  // EPI_DSILU
            const float z = g.Zin[m * g.ldzin + n];
            g.H[m * g.ldh + n] = (__bf16)(v * dsilu(z));
            break;
          }
        }
      }
}

// Fragments of an operand whose memory holds columns side by side (rows along
// k): a fragment wants eight k of one column, so a lane reads four columns (8
// bytes) of its eight rows and repacks them in registers into four fragments.
// Which columns make a tile is free: tile t holds columns 4 c + t of 64.
// Columns beyond C read others' values into results that nobody stores; rows
// from kend on count as zero (TAIL).
template <bool TAIL>
__device__ __forceinline__ void load_cols(u32x2 (&v)[8], const __bf16* X, long long sk,
                                          long long k, long long kend) {
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = *reinterpret_cast<const u32x2*>(X + (!TAIL || k + j < kend ? k + j : kend - 1) * sk);
  if (TAIL) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned mask = k + j < kend ? ~0u : 0u;
      v[j] = u32x2{v[j][0] & mask, v[j][1] & mask};
    }
  }
}
// Fragment t (of four): column t of the eight rows.
__device__ __forceinline__ bf16x8 fragment(const u32x2 (&v)[8], int t) {
  u32x4 f;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    f[j] = __builtin_amdgcn_perm(v[2 * j + 1][t >> 1], v[2 * j][t >> 1],
                                 t & 1 ? 0x07060302u : 0x05040100u);
  return __builtin_bit_cast(bf16x8, f);
}

// The large products whose A is read along k (the layers' forward passes and
// the activations' gradients).  Such a product moves 2 (A, H) + 4 (C or Zin)
// bytes an element and is bound by memory: 65,536 x 256 x 256 is 134 MB, 26 us
// at the rate of a copy.  A block takes 128 x 128 of C, a wave 64 x 64 as 4 x
// 4 MFMA tiles.  Fragments come straight from memory, a slab ahead of the
// products: A's from HBM, the weights' from L2, along k (BROWS) or as columns.
// The operands are swapped (D = B^T A^T), so that a lane holds four
// neighbouring columns of a row (or, of a columns' B, the four tiles do), and
// the results pass through LDS to leave in whole rows: 16-byte stores of C,
// 8-byte stores of H, 16-byte loads of Zin.  64 x 64 tiles read A four times
// and stored single elements.  Each
// element's sum runs over k in the order of k_gemm, so the bits are the same.
constexpr int RM = 128, RN = 128;

constexpr int RLD = 64 + 4;  // padded LDS row of a wave's results

// LDS that only one wave uses: its writes are done before its later reads
// (LDS works in order), the compiler keeps them so.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <bool BROWS>
__global__ void __launch_bounds__(256, 2) k_gemm_rows(GemmArgs g, int ntiles) {
  __shared__ float T[4][16][RLD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // Blocks go to the eight XCDs in turn: the n tiles of one m tile are eight
  // blocks apart, so that A's rows are read by one XCD.
  const unsigned group = blockIdx.x / (8 * ntiles), in = blockIdx.x % (8 * ntiles);
  const long long m0 = ((long long)group * 8 + in % 8) * RM, n0 = (long long)(in / 8) * RN;
  if (m0 >= g.M) return;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const int kl = (lane >> 4) * 8;
  f32x4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's rows of A and of B, or B's four columns (in range: rows and
  // columns beyond the end stand for the last)
  const __bf16 *pa[4], *pb[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const long long m = m0 + wm + a * 16 + (lane & 15);
    pa[a] = g.A + (m < g.M ? m : g.M - 1) * g.sam;
    if (BROWS) {
      const long long n = n0 + wn + a * 16 + (lane & 15);
      pb[a] = g.B + (n < g.N ? n : g.N - 1) * g.sbn;
    }
  }
  const long long nc = n0 + wn + (lane & 15) * 4;
  const __bf16* cols = g.B + (nc < g.N ? nc : 0);
  struct Slab {
    u32x4 a[4], b[4];
    u32x2 c[8];
  };
  // k from K on (K is a multiple of eight) counts as zero
  auto load = [&](Slab& s, long long k0) {
    const long long k = k0 + kl;
    const bool keep = k < g.K;
    const long long kk = keep ? k : 0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      s.a[a] = *reinterpret_cast<const u32x4*>(pa[a] + kk);
      if (BROWS) s.b[a] = *reinterpret_cast<const u32x4*>(pb[a] + kk);
    }
    if (!BROWS) load_cols<false>(s.c, cols, g.sbk, kk, 0);
  };
  auto products = [&](const Slab& s, long long k0) {
    const unsigned mask = k0 + kl < g.K ? ~0u : 0u;
    bf16x8 bf[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      bf[b] = BROWS ? __builtin_bit_cast(bf16x8, s.b[b] & mask)
                    : __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fragment(s.c, b)) & mask);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const bf16x8 af = __builtin_bit_cast(bf16x8, s.a[a] & mask);
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[b], af, acc[a][b], 0, 0, 0);
    }
  };
  Slab s0, s1;
  load(s0, 0);
  for (long long k0 = 0; k0 < g.K; k0 += 2 * BK) {
    load(s1, k0 + BK);
    products(s0, k0);
    load(s0, k0 + 2 * BK);
    products(s1, k0 + BK);
  }
  const auto aligned = [](const void* q, int bytes) {
    return (reinterpret_cast<uintptr_t>(q) & (bytes - 1)) == 0;
  };
  // sixteen rows at a time through the wave's own LDS, so that a row's 64
  // columns are loaded and stored together
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float(&t)[16][RLD] = T[wave];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f32x4 c = acc[a][b];
      if (!BROWS) c = f32x4{acc[a][0][b], acc[a][1][b], acc[a][2][b], acc[a][3][b]};
      const int col = BROWS ? b * 16 + (lane >> 4) * 4 : (lane >> 4) * 16 + b * 4;
      *reinterpret_cast<f32x4*>(&t[lane & 15][col]) = c;
    }
    wave_lds_fence();
    f32x4 rows[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      rows[i] = *reinterpret_cast<const f32x4*>(&t[i * 4 + (lane >> 4)][(lane & 15) * 4]);
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long long m = m0 + wm + a * 16 + i * 4 + (lane >> 4);
      const long long n = n0 + wn + (lane & 15) * 4;
      if (m >= g.M || n >= g.N) continue;
      const int cols = g.N - n < 4 ? (int)(g.N - n) : 4;
      float* C = g.C ? g.C + m * g.ldc + n : nullptr;
      __bf16* H = g.H ? g.H + m * g.ldh + n : nullptr;
      f32x4 c = rows[i];
      bf16x4 h = {};
      if (g.epi == EPI_DSILU) {
        const float* Z = g.Zin + m * g.ldzin + n;
        f32x4 z = {};
        if (cols == 4 && aligned(Z, 16)) {
          z = *reinterpret_cast<const f32x4*>(Z);
        } else {
          for (int j = 0; j < cols; ++j) z[j] = Z[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = (__bf16)(c[j] * dsilu(z[j]));
      } else if (g.epi != EPI_STORE) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          c[j] += g.bias[n + (j < cols ? j : 0)];
          h[j] = (__bf16)silu(c[j]);
        }
      } else if (g.accumulate) {
        for (int j = 0; j < cols; ++j) c[j] += C[j];
      }
      if (g.epi != EPI_DSILU && C) {
        if (cols == 4 && aligned(C, 16)) {
          *reinterpret_cast<f32x4*>(C) = c;
        } else {
          for (int j = 0; j < cols; ++j) C[j] = c[j];
        }
      }
      if (g.epi == EPI_BIAS_SILU || g.epi == EPI_DSILU) {
        if (cols == 4 && aligned(H, 8)) {
          *reinterpret_cast<bf16x4*>(H) = h;
        } else {
          for (int j = 0; j < cols; ++j) H[j] = h[j];
        }
      }
    }
  }
}

// The weights' gradients C = sum_k A(m, k) B(k, n) with both operands' rows
// along k (dZ^T H over the batch), fragments straight from memory as columns.
// A block takes 128 x 128 of C over its share of k, four waves 64 x 64 each
// and a second four every other slab; their sums meet in LDS and leave it in
// whole rows.  65,536 x 256 x 256 is 67 MB, 13 us at the rate of a copy, and 17
// MB of atomic sums: 78 -> 37 us.  (Through LDS, transposed by 2-byte writes,
// a slab waited for its own loads.)
constexpr int kColsLd = 128 + 4;

__global__ void __launch_bounds__(512, 2) k_gemm_cols(GemmArgs g) {
  __shared__ float T[128][kColsLd];
  const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3, half = threadIdx.x >> 8;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const long long mb = (long long)blockIdx.x * 128, nb = (long long)blockIdx.y * 128;
  const long long mc = mb + wm + (lane & 15) * 4, nc = nb + wn + (lane & 15) * 4;
  const __bf16* A = g.A + (mc < g.M ? mc : 0);
  const __bf16* B = g.B + (nc < g.N ? nc : 0);
  f32x4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const long long kper = ((g.K + g.ksplit - 1) / g.ksplit + BK - 1) / BK * BK;
  const long long kbeg = (long long)blockIdx.z * kper;
  const long long kend = kbeg + kper < g.K ? kbeg + kper : g.K;
  if (kbeg >= kend) return;
  const int kl = (lane >> 4) * 8;
  auto products = [&](const u32x2 (&va)[8], const u32x2 (&vb)[8]) {
    bf16x8 af[4], bf[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      af[t] = fragment(va, t);
      bf[t] = fragment(vb, t);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bf[b], acc[a][b], 0, 0, 0);
  };
  // whole slabs, two on their way (beyond the last the first is read again)
  const long long whole = kbeg + (kend - kbeg) / BK * BK;
  const long long first = kbeg + half * BK;
  u32x2 va[2][8], vb[2][8];
  auto load = [&](int s, long long k0) {
    const long long k = (k0 < whole ? k0 : kbeg) + kl;
    load_cols<false>(va[s], A, g.sak, k, 0);
    load_cols<false>(vb[s], B, g.sbk, k, 0);
  };
  if (first < whole) {
    load(0, first);
    load(1, first + 2 * BK);
    for (long long k0 = first; k0 < whole; k0 += 4 * BK) {
      products(va[0], vb[0]);
      load(0, k0 + 4 * BK);
      if (k0 + 2 * BK < whole) products(va[1], vb[1]);
      load(1, k0 + 6 * BK);
    }
  }
  if (whole < kend && half == 0) {
    load_cols<true>(va[0], A, g.sak, whole + kl, kend);
    load_cols<true>(vb[0], B, g.sbk, whole + kl, kend);
    products(va[0], vb[0]);
  }
  // tile (a, b), entry j: row 4 (4 (l / 16) + j) + a, column 4 (l % 16) + b
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (half == h) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4* t = reinterpret_cast<f32x4*>(
              &T[wm + 4 * ((lane >> 4) * 4 + j) + a][wn + (lane & 15) * 4]);
          f32x4 v = f32x4{acc[a][0][j], acc[a][1][j], acc[a][2][j], acc[a][3][j]};
          if (h == 1) v += *t;
          *t = v;
        }
    }
    __syncthreads();
  }
  const int c = threadIdx.x & 127;
  if (nb + c >= g.N) return;
  for (int r = threadIdx.x >> 7; r < 128 && mb + r < g.M; r += 4) {
    float* C = g.C + (mb + r) * g.ldc + nb + c;
    const float v = T[r][c];
    if (g.ksplit > 1)
      atomicAdd(C, v);
    else
      *C = g.accumulate ? *C + v : v;
  }
}

// The whole inference pass of an MLP of hidden width 256 in one kernel: a
// block takes 128 points and keeps their activations in LDS, so that they
// never go to HBM; every hidden-to-hidden layer runs on the matrix cores, the
// layer's BF16 weights read from L2.  Each wave owns 64 output columns of a
// layer: 8 x 4 MFMA tiles, weights as the first operand, so that a lane holds four neighbouring columns of a point and packs
// its activations into one 8-byte LDS write.  A layer's results wait in
// registers (as BF16) until all waves have read its inputs, so one buffer of
// 68 KB serves and two blocks share a CU: one's matrix instructions run beside
// the other's exponentials.  The input layer (8 padded inputs) is a short dot
// product in FP32 over the block's inputs staged in LDS; the output layer (at
// most 16 columns, zero-padded) is one MFMA tile column per wave.  Rounding as
// the layer-by-layer path: FP32 accumulation, bias + SiLU in FP32, BF16
// activations.  262,144 points (103 GFLOP): with 64 points a block 242 us,
// bound by the weights' way from L2 (1.6 GB); with 128 (FA = 8) and the next slab's
// weights on their way 168 us back to back (197 to 199 for a launch on its
// own or under the profiler; the products alone take 92 at the rate of a
// large product, the exponentials and reciprocals some 90).
constexpr int FH = 256;      // hidden width
constexpr int FLD = FH + 8;  // padded LDS row (bf16 elements)
constexpr int kMaxFusedLayers = 8;

struct FusedArgs {
  const __bf16* X;  // [n][ldx] inputs (BF16)
  int ldx, nin;     // row stride, inputs used
  long long n;
  int depth;        // hidden layers
  int nout;
  const __bf16* W[kMaxFusedLayers + 1];  // layer l: [out][in] row-major
  const float* b[kMaxFusedLayers + 1];
  float* Y;         // [n][ldy] FP32 outputs
  int ldy;
};

template <int FA>  // MFMA row tiles per block, of 16 points each
__global__ void __launch_bounds__(256, 2) k_mlp_fused(FusedArgs f) {
  constexpr int FM = 16 * FA;
  __shared__ __bf16 act[FM][FLD];
  __shared__ float xin[FM][8];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const long long m0 = (long long)blockIdx.x * FM;
  // ---- the block's inputs, once (zero past n and past nin)
  static_assert(FM * 8 % 256 == 0, "input staging: whole rounds of the block");
#pragma unroll
  for (int j = 0; j < FM * 8 / 256; ++j) {
    const int t = tid + 256 * j;
    const int r = t >> 3, k = t & 7;
    const long long m = m0 + r;
    const bool in = m < f.n && k < f.nin;  // else an in-range stand-in, masked
    xin[r][k] = keep_or_zero((float)f.X[(m < f.n ? m : f.n - 1) * f.ldx + (k < f.nin ? k : 0)], in);
  }
  __syncthreads();
  // ---- input layer: thread tid owns hidden unit tid for all FM points
  {
    const int c = tid;
    float w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      w[k] = keep_or_zero((float)f.W[0][c * f.nin + (k < f.nin ? k : 0)], k < f.nin);
    const float bias = f.b[0][c];
    for (int r = 0; r < FM; ++r) {
      float z = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; ++k) z = fmaf(xin[r][k], w[k], z);
      act[r][c] = (__bf16)silu(z + bias);
    }
  }
  // ---- hidden-to-hidden layers on the matrix cores
  for (int l = 1; l < f.depth; ++l) {
    __syncthreads();
    const __bf16* W = f.W[l];
    const float* bias = f.b[l];
    f32x4 acc[FA][4];
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16* wl = W + (wave * 64 + (lane & 15)) * FH + (lane >> 4) * 8;
    bf16x8 bw[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) bw[b] = *reinterpret_cast<const bf16x8*>(wl + b * 16 * FH);
#pragma unroll 2
    for (int k0 = 0; k0 < FH; k0 += 32) {
      // the next slab's weights on their way during this one's products (the
      // last slab loads its own again)
      const int kn = k0 + 32 < FH ? k0 + 32 : k0;
      bf16x8 next[4];
#pragma unroll
      for (int b = 0; b < 4; ++b)
        next[b] = *reinterpret_cast<const bf16x8*>(wl + b * 16 * FH + kn);
#pragma unroll
      for (int a = 0; a < FA; ++a) {
        const bf16x8 af = *reinterpret_cast<const bf16x8*>(
            &act[a * 16 + (lane & 15)][k0 + (lane >> 4) * 8]);
#pragma unroll
        for (int b = 0; b < 4; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[b], af, acc[a][b], 0, 0, 0);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) bw[b] = next[b];
    }
    bf16x4 out[FA][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float* bn = bias + wave * 64 + b * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j) out[a][b][j] = (__bf16)silu(acc[a][b][j] + bn[j]);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *reinterpret_cast<bf16x4*>(
            &act[a * 16 + (lane & 15)][wave * 64 + b * 16 + (lane >> 4) * 4]) = out[a][b];
  }
  __syncthreads();
  // ---- output layer on the matrix cores: wave w takes the 16-point row
  // tiles w, w + 4, ... against the outputs padded to 16 columns (zero
  // weights past nout)
  {
    const __bf16* Wo = f.W[f.depth];
    const int n = lane & 15;
    // all eight weight fragments in flight at once (row 0 stands in for the
    // padding columns, whose fragments are then masked to zero)
    const int nr = n < f.nout ? n : 0;
    const unsigned mask = n < f.nout ? ~0u : 0u;
    bf16x8 bw[FH / 32];
#pragma unroll
    for (int s = 0; s < FH / 32; ++s) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(Wo + nr * FH + s * 32 + (lane >> 4) * 8);
      bw[s] = __builtin_bit_cast(bf16x8, v & mask);
    }
    // wave w takes row tiles w, w + 4, ...
#pragma unroll
    for (int a = wave; a < FA; a += 4) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < FH / 32; ++s) {
        const int kk = s * 32 + (lane >> 4) * 8;
        const bf16x8 af = *reinterpret_cast<const bf16x8*>(&act[a * 16 + n][kk]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bw[s], acc, 0, 0, 0);
      }
      if (n < f.nout) {
        const float bo = f.b[f.depth][n];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const long long m = m0 + a * 16 + (lane >> 4) * 4 + j;
          if (m < f.n) f.Y[m * f.ldy + n] = acc[j] + bo;
        }
      }
    }
  }
}

// db[n] += sum_m dZ[m, n] (bf16 in, fp32 out) -- partial column sums per
// block of kColsumRows rows, combined with atomics.  A lane keeps four
// independent sums so that four rows' loads are in flight at once; the
// grid has one block row per chunk of rows, enough to fill the device for
// a training batch (65,536 rows: 512 chunks).
constexpr int kColsumRows = 128;
__global__ void k_colsum(const __bf16* __restrict__ dz, long long ld, long long M,
                         long long N, float* __restrict__ out) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const long long rows = (M + gridDim.y - 1) / gridDim.y;
  const long long r0 = (long long)blockIdx.y * rows;
  const long long r1 = r0 + rows < M ? r0 + rows : M;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  long long m = r0;
  for (; m + 3 < r1; m += 4) {
    s0 += (float)dz[m * ld + n];
    s1 += (float)dz[(m + 1) * ld + n];
    s2 += (float)dz[(m + 2) * ld + n];
    s3 += (float)dz[(m + 3) * ld + n];
  }
  for (; m < r1; ++m) s0 += (float)dz[m * ld + n];
  atomicAdd(out + n, (s0 + s1) + (s2 + s3));
}

// The same for rows of 16-byte alignment and whole groups of eight columns
// (the hidden layers): a lane reads eight columns at a time, and a block's
// partial sums meet in LDS before the atomics, which are what bounds it: 512
// blocks of 128 rows took 18 us for 65,536 x 256, 128 blocks of 512 rows 9 (7
// at the rate of a copy; a lane a column: 22).
constexpr int kColsumGroups = 32;    // groups of eight columns a block covers
constexpr int kColsumLanes = 32;     // rows it reads side by side
constexpr int kColsum8Rows = 512;    // rows of a block
__global__ void __launch_bounds__(kColsumGroups * kColsumLanes) k_colsum8(const __bf16* __restrict__ dz, long long ld,
                                                 long long M, long long N,
                                                 float* __restrict__ out) {
  __shared__ float part[kColsumLanes][kColsumGroups][8 + 1];
  const int c = threadIdx.x % kColsumGroups, r = threadIdx.x / kColsumGroups;
  const long long n = ((long long)blockIdx.x * kColsumGroups + c) * 8;
  const long long rows = (M + gridDim.y - 1) / gridDim.y;
  const long long r0 = (long long)blockIdx.y * rows;
  const long long r1 = r0 + rows < M ? r0 + rows : M;
  float s[2][8] = {};
  if (n < N) {
    long long m = r0 + r;
    for (; m + kColsumLanes < r1; m += 2 * kColsumLanes) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(dz + m * ld + n);
      const bf16x8 w = *reinterpret_cast<const bf16x8*>(dz + (m + kColsumLanes) * ld + n);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        s[0][j] += (float)v[j];
        s[1][j] += (float)w[j];
      }
    }
    if (m < r1) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(dz + m * ld + n);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[0][j] += (float)v[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) part[r][c][j] = s[0][j] + s[1][j];
  __syncthreads();
  if (threadIdx.x >= 8 * kColsumGroups) return;
  const int cc = threadIdx.x >> 3, j = threadIdx.x & 7;
  const long long col = ((long long)blockIdx.x * kColsumGroups + cc) * 8 + j;
  if (col >= N) return;
  float t = 0.f;
#pragma unroll
  for (int k = 0; k < kColsumLanes; ++k) t += part[k][cc][j];
  atomicAdd(out + col, t);
}

// Adam on fp32 master parameters (bias-corrected, as Kingma & Ba 2015);
// writes the bf16 copy the GEMMs read.
struct AdamStep {
  float lr, b1, b2, eps, c1, c2;
  __device__ __forceinline__ void at(float* p, const float* g, float* m, float* v, __bf16* pb,
                                     long long i) const {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    p[i] = pi;
    if (pb) pb[i] = (__bf16)pi;
  }
};

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v,
                       __bf16* __restrict__ pb, long long n, AdamStep s) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) s.at(p, g, m, v, pb, i);
}

// Several tensors in one launch (grid y): ten launches of a network's weights
// and biases took 45 us, one takes 5.
constexpr int kAdamTensors = GX_ADAM_TENSORS;
struct AdamTensors {
  float* p[kAdamTensors];
  const float* g[kAdamTensors];
  float *m[kAdamTensors], *v[kAdamTensors];
  __bf16* pb[kAdamTensors];
  long long n[kAdamTensors];
};
__global__ void k_adam_many(AdamTensors a, AdamStep s) {
  const int k = blockIdx.y;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < a.n[k];
       i += (long long)gridDim.x * blockDim.x)
    s.at(a.p[k], a.g[k], a.m[k], a.v[k], a.pb[k], i);
}

// Pseudo-Huber loss on the network's outputs: r = Y - T (first 3 columns),
// loss = delta^2 (sqrt(1 + (r/delta)^2) - 1) summed, gradient
// r / sqrt(1 + (r/delta)^2) times `scale` into dY (bf16, other columns 0).
// The bounded gradient keeps rare large targets (points close to a
// subhalo's core) from dominating training.
__global__ void k_huber(const float* __restrict__ Y, long long ldy,
                        const float* __restrict__ T, long long B, float delta,
                        float scale, __bf16* __restrict__ dY, long long ldd,
                        double* __restrict__ loss) {
  __shared__ double part[256];
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (i < B) {
    const float id = 1.0f / delta;
    for (int c = 0; c < 3; ++c) {
      const float r = Y[i * ldy + c] - T[i * 3 + c];
      const float q = sqrtf(1.0f + (r * id) * (r * id));
      l += (double)(delta * delta * (q - 1.0f));
      dY[i * ldd + c] = (__bf16)(scale * r / q);
    }
    for (long long c = 3; c < ldd; ++c) dY[i * ldd + c] = (__bf16)0.0f;
  }
  part[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, part[0]);
}

// ------------------------------------------------ surrogate field plumbing
// The perturbing part of the field (a bar and subhaloes rotating rigidly at
// omega) is static in the frame rotating with angle th = omega t, so the
// network sees rotating-frame positions and predicts the rotating-frame
// acceleration:  x' = Rz(-th) x,  a = Rz(th) a'.

__device__ __forceinline__ double stage_time(const double* t, int t_stride,
                                             long long i, double dt) {
  return t[t_stride ? i : 0] + dt;
}

// X[i] = (x', y', z, R, r) / L as bf16, zero-padded to width ldx.
__global__ void k_sur_inputs(const double* __restrict__ xyz,
                             const double* __restrict__ t, int t_stride,
                             double dt, long long n, double inv_len, double omega,
                             __bf16* __restrict__ X, long long ldx) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s, c;
  sincos(omega * stage_time(t, t_stride, i, dt), &s, &c);
  const double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
  const double R2 = x * x + y * y;
  __bf16* row = X + i * ldx;
  row[0] = (__bf16)(float)((c * x + s * y) * inv_len);
  row[1] = (__bf16)(float)((c * y - s * x) * inv_len);
  row[2] = (__bf16)(float)(z * inv_len);
  row[3] = (__bf16)(float)(sqrt(R2) * inv_len);
  row[4] = (__bf16)(float)(sqrt(R2 + z * z) * inv_len);
  for (long long k = 5; k < ldx; ++k) row[k] = (__bf16)0.0f;
}

// Training targets: T[i] = Rz(-th) (a_full - a_base)(x_i, t_i) / scale.
__global__ void k_sur_targets(const double* __restrict__ t, int t_stride,
                              long long n, const double* __restrict__ a_full,
                              const double* __restrict__ a_base, double omega,
                              double inv_scale, float* __restrict__ T) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s, c;
  sincos(omega * t[t_stride ? i : 0], &s, &c);
  const double dx = a_full[3 * i] - a_base[3 * i];
  const double dy = a_full[3 * i + 1] - a_base[3 * i + 1];
  const double dz = a_full[3 * i + 2] - a_base[3 * i + 2];
  T[3 * i] = (float)((c * dx + s * dy) * inv_scale);
  T[3 * i + 1] = (float)((c * dy - s * dx) * inv_scale);
  T[3 * i + 2] = (float)(dz * inv_scale);
}

// The surrogate field: a = a_base(x) (exact FP64) + scale Rz(th) Y[i], or the
// exact full field where the gate says so (outside the trained ball
// |x| > r_max, or an orbit flagged by the periodic check).  EB and EF
// evaluate the base and full fields: the compile-time evaluators when the
// tables have their signatures (the Milky Way model; it plus a rotating
// group), else the table loop.
template <class EB, class EF>
__global__ void k_sur_combine(DPot base, DPot full, const double* __restrict__ xyz,
                              const double* __restrict__ t, int t_stride, double dt,
                              long long n, const float* __restrict__ Y,
                              long long ldy, double scale, double omega,
                              double r_max, const int* __restrict__ flag,
                              double* __restrict__ acc) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
  const double ti = stage_time(t, t_stride, i, dt);
  const bool exact = (x * x + y * y + z * z > r_max * r_max) || (flag && flag[i]);
  double ax, ay, az;
  if (exact) {
    EF::acc(full, x, y, z, ti, ax, ay, az);
  } else {
    EB::acc(base, x, y, z, ti, ax, ay, az);
    double s, c;
    sincos(omega * ti, &s, &c);
    const double px = scale * (double)Y[i * ldy], py = scale * (double)Y[i * ldy + 1];
    ax += c * px - s * py;
    ay += s * px + c * py;
    az += scale * (double)Y[i * ldy + 2];
  }
  acc[3 * i] = ax;
  acc[3 * i + 1] = ay;
  acc[3 * i + 2] = az;
}

// The periodic gate check: the surrogate field at the current positions
// against the exact field; an orbit whose relative error exceeds `tol` is
// flagged (sticky) and integrated with the exact field from then on.
template <class EF>
__global__ void k_sur_check(DPot full, const double* __restrict__ xyz,
                            const double* __restrict__ t, int t_stride, long long n,
                            const double* __restrict__ a_sur, double tol,
                            int* __restrict__ flag, float* __restrict__ err) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double ax, ay, az;
  EF::acc(full, xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], t[t_stride ? i : 0], ax, ay, az);
  const double ex = a_sur[3 * i] - ax, ey = a_sur[3 * i + 1] - ay, ez = a_sur[3 * i + 2] - az;
  const double e = sqrt((ex * ex + ey * ey + ez * ez) / (ax * ax + ay * ay + az * az));
  if (err) err[i] = (float)e;
  if (!(e <= tol)) flag[i] = 1;
}

// Lock-step fixed-step Dopri8 (Runge-Kutta-Nystrom form, as the persistent
// integrator) over n orbits sharing one time t[0]; the stage accelerations
// live in HBM, G = [13][n][3], so any batched field (the surrogate) can
// produce them.  Stage positions Q_i = q + h (rs_i p + h sum_l (A^2)_il g_l):
__global__ void k_stage_point(int stage, const double* __restrict__ q,
                              const double* __restrict__ p,
                              const double* __restrict__ G, long long n, double h,
                              double* __restrict__ Q) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  constexpr auto& K = Dopri8::k;
  double s[3] = {0.0, 0.0, 0.0};
  for (int l = 0; l < stage; ++l) {
    const double a = K.aa[stage][l];
    if (a == 0.0) continue;
    for (int m = 0; m < 3; ++m) s[m] = fma(a, G[((long long)l * n + i) * 3 + m], s[m]);
  }
  const double rs = K.rs[stage];
  for (int m = 0; m < 3; ++m)
    Q[3 * i + m] = fma(h, fma(rs, p[3 * i + m], h * s[m]), q[3 * i + m]);
}

// Step update q += h (sb p + h sum bA_l g_l), p += h sum b_l g_l; thread 0
// also advances the shared time t[0] += h.
__global__ void k_step_update(double* __restrict__ q, double* __restrict__ p,
                              const double* __restrict__ G, long long n, double h,
                              double* __restrict__ t) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) t[0] += h;
  if (i >= n) return;
  constexpr auto& K = Dopri8::k;
  double b[3] = {0.0, 0.0, 0.0}, c[3] = {0.0, 0.0, 0.0};
  for (int l = 0; l < 13; ++l) {
    for (int m = 0; m < 3; ++m) {
      const double gl = G[((long long)l * n + i) * 3 + m];
      if (K.b[l] != 0.0) b[m] = fma(K.b[l], gl, b[m]);
      if (K.ba[l] != 0.0) c[m] = fma(K.ba[l], gl, c[m]);
    }
  }
  for (int m = 0; m < 3; ++m) {
    const double pm = p[3 * i + m];
    q[3 * i + m] = fma(h, fma(K.sb, pm, h * c[m]), q[3 * i + m]);
    p[3 * i + m] = fma(h, b[m], pm);
  }
}

long long blocks_for(long long n, int bs) { return (n + bs - 1) / bs; }

bool grid_ok(long long n) { return blocks_for(n, 256) <= 0x7fffffffLL; }

bool aligned(const void* p, int bytes) {
  return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
}

// k_gemm_cols for both operands' rows along k.  Per block it reads more
// slabs than k_gemm and sums fewer results atomically, which needs a reduction
// of some length: it is the faster one wherever a block has 512 or more of k
// (256 x 256 x 65,536 in 64 parts: 78 us with k_gemm, 37 with this; in one
// part 2,240 / 930).  With less, its larger tiles' start and end show, and
// their padding (us with 256 of k a block: 192 x 192 x 131,072 95 / 113, 64 x
// 512 x 262,144 157 / 202, 128 x 128 x 4,096 17.6 / 18.1), except while every
// block has a CU to itself and there is some work (256 x 256 x 8,192 24 / 21,
// 128 x 128 x 65,536 40 / 33).  Rows whose lengths k_gemm cannot read 16 bytes
// at a time (68 x 68 x 65,536: 61 / 31) are always faster here.  N = 8, a
// network's first layer, takes 27 us with k_gemm and 31 with this.
bool use_gemm_cols(const GemmArgs& g) {
  if (g.epi != EPI_STORE || g.sam != 1 || g.sbn != 1 || g.M < 64 || g.N < 64 || g.M % 4 != 0 ||
      g.N % 4 != 0 || g.sak % 4 != 0 || g.sbk % 4 != 0 || g.K < 3072 || !aligned(g.A, 8) ||
      !aligned(g.B, 8))
    return false;
  const long long mt = (g.M + 127) / 128, nt = (g.N + 127) / 128;
  if (mt > 0x7fffffffLL || nt > 65535) return false;
  if (g.sak % 8 != 0 || g.sbk % 8 != 0 || !aligned(g.A, 16) || !aligned(g.B, 16)) return true;
  if (g.K >= 512LL * g.ksplit) return true;
  return mt * nt * g.ksplit <= 256 && g.M * g.N * g.K >= 1LL << 28;
}

// k_gemm_rows for A along k.  Two blocks are resident on each of the 256 CUs,
// and a block's start and end are hidden only by others.
// B's columns along n (the activations' gradients): k_gemm transposes B
// through LDS for every block, and this is faster from three quarters of a
// round of blocks on (us, k_gemm / this: DSILU x 256 x 256 at 24,576 rows
// 41 / 35, 65,536 75 / 47, 262,144 299 / 200; 512 x 512 at 65,536 211 / 131;
// other results from 5/4 rounds: 256 x 256 at 40,960 42 / 34), unless the last
// column tile and the last round are mostly empty (x 64 x 64 at 65,536 18.6 /
// 22.1; 192 x 192 at 70,001 56 / 58; without DSILU's arithmetic 192 x 192 at
// 262,144 121 / 131).
// B along k, or SiLU: k_gemm reads B as well, and what is left to gain is the
// 16-byte results.  Even numbers of rounds gain (x 256 x 256 with SiLU at
// 65,536 rows, two rounds, 62 / 57, at 81,920 72 / 77, at 98,304 86 / 90, at
// 131,072 108 / 103), and from eight rounds on, where the results leave the
// last-level cache, all do (262,144 250 / 203; x 512 x 512 at 196,608 552 /
// 469); with fewer, longer rows of K (x 256 x 512 at 131,072 167 / 172) or
// results in BF16 alone (the first layers' inference, 65,536 56 / 55, 81,920
// 66 / 75) have less to gain than the blocks' tails cost.
bool use_gemm_rows(const GemmArgs& g, bool brows) {
  if (g.sak != 1 || g.sam % 8 != 0 || !aligned(g.A, 16) || g.K % 8 != 0 || g.K < 1 ||
      g.ksplit != 1 || g.N <= 64)
    return false;
  if (brows ? g.sbn % 8 != 0 || !aligned(g.B, 16)
            : g.sbn != 1 || g.sbk % 4 != 0 || !aligned(g.B, 8) || g.N % 4 != 0)
    return false;
  constexpr long long kSlots = 512;
  const long long blocks = ((g.M + RM - 1) / RM) * ((g.N + RN - 1) / RN);
  const bool dsilu = g.epi == EPI_DSILU;
  const long long full = g.M * g.N / (RM * RN);  // the results in whole tiles
  if (full < kSlots * 3 / 4 || blocks < kSlots * (dsilu ? 3 : 5) / 4 || blocks >= 0x7fffff00LL)
    return false;
  const bool half = (g.N + 63) / 64 % 2 != 0;  // half of the last tile's waves idle
  if (!brows && dsilu) {
    const long long rounds = (blocks + kSlots - 1) / kSlots;
    return rounds <= 2 || 5 * full >= 3 * rounds * kSlots;
  }
  if (half) return false;
  if (dsilu) return g.K <= 256;
  if (!brows && g.epi != EPI_BIAS_SILU) return g.K >= 64;
  if (blocks >= 8 * kSlots && g.epi == EPI_BIAS_SILU && g.C) return g.K <= 512;
  return g.K <= (g.C ? 256 : 32) && (blocks >= 8 * kSlots || blocks % (2 * kSlots) == 0);
}

AdamStep adam_step(float lr, float b1, float b2, float eps, int64_t step) {
  return {lr, b1, b2, eps, 1.0f / (1.0f - powf(b1, (float)step)),
          1.0f / (1.0f - powf(b2, (float)step))};
}

}  // namespace
}  // namespace gx

using namespace gx;

extern "C" {

int gx_mlp_gemm(const void* A, int64_t sam, int64_t sak, const void* B,
                int64_t sbk, int64_t sbn, int64_t M, int64_t N, int64_t K,
                int32_t epi, int32_t accumulate, int32_t ksplit, const float* bias,
                float* C, int64_t ldc, void* H, int64_t ldh, const float* Zin,
                int64_t ldzin, void* stream) {
  if (M < 0 || N < 0 || K < 0 || !A || !B) return GX_EINVAL;
  if (M == 0 || N == 0) return GX_OK;
  if (epi < EPI_STORE || epi > EPI_DSILU) return GX_EINVAL;
  if ((epi == EPI_STORE || epi == EPI_BIAS) && !C) return GX_EINVAL;
  if ((epi == EPI_BIAS || epi == EPI_BIAS_SILU) && !bias) return GX_EINVAL;
  if ((epi == EPI_BIAS_SILU || epi == EPI_DSILU) && !H) return GX_EINVAL;
  if (epi == EPI_DSILU && !Zin) return GX_EINVAL;
  if (ksplit < 1 || ksplit > 65535 || (ksplit > 1 && epi != EPI_STORE)) return GX_EINVAL;
  GemmArgs g{};
  g.A = static_cast<const __bf16*>(A);
  g.sam = sam;
  g.sak = sak;
  g.B = static_cast<const __bf16*>(B);
  g.sbk = sbk;
  g.sbn = sbn;
  g.M = M;
  g.N = N;
  g.K = K;
  g.epi = epi;
  g.accumulate = accumulate;
  g.ksplit = ksplit;
  g.bias = bias;
  g.C = C;
  g.ldc = ldc;
  g.H = static_cast<__bf16*>(H);
  g.ldh = ldh;
  g.Zin = Zin;
  g.ldzin = ldzin;
  const long long rt = (M + RM - 1) / RM, ct = (N + RN - 1) / RN;
  if (use_gemm_cols(g)) {
    hipLaunchKernelGGL(k_gemm_cols, dim3((unsigned)rt, (unsigned)ct, (unsigned)ksplit), dim3(512), 0,
                       (hipStream_t)stream, g);
    return check(hipGetLastError());
  }
  const bool brows = sbk == 1;
  if (use_gemm_rows(g, brows)) {
    const long long groups = (rt + 7) / 8;
    const auto kern = brows ? k_gemm_rows<true> : k_gemm_rows<false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)(groups * 8 * ct)), dim3(256), 0, (hipStream_t)stream,
                       g, (int)ct);
    return check(hipGetLastError());
  }
  const long long mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN;
  if (mt > 0x7fffffffLL || nt > 65535) return GX_EINVAL;
  dim3 grid((unsigned)mt, (unsigned)nt, (unsigned)ksplit);
  hipLaunchKernelGGL(k_gemm<true>, grid, dim3(256), 0, (hipStream_t)stream, g);
  return check(hipGetLastError());
}

int gx_mlp_forward_fused(const void* X, int32_t ldx, int32_t nin, int64_t n,
                         int32_t depth, const void* const* W,
                         const float* const* b, int32_t nout, float* Y,
                         int32_t ldy, void* stream) {
  if (n < 0 || depth < 1 || depth > kMaxFusedLayers || nin < 1 || nin > 8 ||
      ldx < nin || nout < 1 || nout > 16 || ldy < nout)
    return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!X || !W || !b || !Y) return GX_EINVAL;
  FusedArgs f{};
  f.X = static_cast<const __bf16*>(X);
  f.ldx = ldx;
  f.nin = nin;
  f.n = n;
  f.depth = depth;
  f.nout = nout;
  f.Y = Y;
  f.ldy = ldy;
  for (int l = 0; l <= depth; ++l) {
    if (!W[l] || !b[l]) return GX_EINVAL;
    // 16-byte fragment loads of the hidden and output layers' rows
    if (l > 0 && (reinterpret_cast<uintptr_t>(W[l]) & 15)) return GX_EINVAL;
    f.W[l] = static_cast<const __bf16*>(W[l]);
    f.b[l] = b[l];
  }
  // 64 points a block while each still has a CU of its own, where a block's
  // latency is all, and in shallow networks, whose weights are little beside
  // the points, for some rounds more (us with 64 / 128 points; depth 4: 100
  // points 30 / 39, 16,384 32 / 40, 20,000 42 / 41, 65,536 67 / 52, 262,144
  // 216 / 168; depth 3: 32,768 33.7 / 33.6, 49,152 42 / 40; depth 2: 49,152
  // 29 / 31, 57,344 34 / 31; depth 1: 131,072 28 / 34)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return GX_ELAUNCH;
  const bool small = depth == 1 || n <= 64LL * num_cus(dev) * (depth < 4 ? 5 - depth : 1);
  const long long blocks = (n + (small ? 63 : 127)) / (small ? 64 : 128);
  if (blocks > 0x7fffffffLL) return GX_EINVAL;
  hipLaunchKernelGGL(small ? k_mlp_fused<4> : k_mlp_fused<8>, dim3((unsigned)blocks), dim3(256), 0,
                     (hipStream_t)stream, f);
  return check(hipGetLastError());
}

int gx_mlp_colsum(const void* dz, int64_t ld, int64_t M, int64_t N, float* out,
                  void* stream) {
  if (!dz || !out || M < 0 || N < 0 || ld < N) return GX_EINVAL;
  if (M == 0 || N == 0) return GX_OK;
  long long ychunks = (M + kColsumRows - 1) / kColsumRows;
  if (ychunks > 65535) ychunks = 65535;  // grid y limit; chunks then grow
  if (N % 8 == 0 && ld % 8 == 0 && (reinterpret_cast<uintptr_t>(dz) & 15) == 0) {
    ychunks = (M + kColsum8Rows - 1) / kColsum8Rows;
    if (ychunks > 65535) ychunks = 65535;
    hipLaunchKernelGGL(k_colsum8, dim3((unsigned)blocks_for(N, 8 * kColsumGroups), (unsigned)ychunks),
                       dim3(kColsumGroups * kColsumLanes), 0, (hipStream_t)stream, static_cast<const __bf16*>(dz),
                       (long long)ld, (long long)M, (long long)N, out);
    return check(hipGetLastError());
  }
  dim3 grid((unsigned)blocks_for(N, 256), (unsigned)ychunks);
  hipLaunchKernelGGL(k_colsum, grid, dim3(256), 0, (hipStream_t)stream,
                     static_cast<const __bf16*>(dz), (long long)ld, (long long)M,
                     (long long)N, out);
  return check(hipGetLastError());
}

int gx_mlp_adam(float* p, const float* g, float* m, float* v, void* pb,
                int64_t n, float lr, float b1, float b2, float eps, int64_t step,
                void* stream) {
  if (!p || !g || !m || !v || n < 0 || step < 1) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  hipLaunchKernelGGL(k_adam, dim3((unsigned)blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, p, g, m, v, static_cast<__bf16*>(pb),
                     (long long)n, adam_step(lr, b1, b2, eps, step));
  return check(hipGetLastError());
}

int gx_mlp_adam_many(int32_t count, float* const* p, const float* const* g, float* const* m,
                     float* const* v, void* const* pb, const int64_t* n, float lr, float b1,
                     float b2, float eps, int64_t step, void* stream) {
  if (count < 0 || count > kAdamTensors || step < 1) return GX_EINVAL;
  if (count == 0) return GX_OK;
  if (!p || !g || !m || !v || !pb || !n) return GX_EINVAL;
  AdamTensors a{};
  long long most = 0;
  for (int k = 0; k < count; ++k) {
    if (n[k] < 0 || (n[k] > 0 && (!p[k] || !g[k] || !m[k] || !v[k]))) return GX_EINVAL;
    a.p[k] = p[k];
    a.g[k] = g[k];
    a.m[k] = m[k];
    a.v[k] = v[k];
    a.pb[k] = static_cast<__bf16*>(pb[k]);
    a.n[k] = n[k];
    if (n[k] > most) most = n[k];
  }
  if (most == 0) return GX_OK;
  const long long blocks = blocks_for(most, 256) < 4096 ? blocks_for(most, 256) : 4096;
  hipLaunchKernelGGL(k_adam_many, dim3((unsigned)blocks, (unsigned)count), dim3(256), 0,
                     (hipStream_t)stream, a, adam_step(lr, b1, b2, eps, step));
  return check(hipGetLastError());
}

int gx_mlp_huber(const float* Y, int64_t ldy, const float* T, int64_t B, float delta,
                 float scale, void* dY, int64_t ldd, double* loss, void* stream) {
  if (!Y || !T || !dY || !loss || B < 0 || ldy < 3 || ldd < 3 || !(delta > 0.f))
    return GX_EINVAL;
  if (B == 0) return GX_OK;
  if (!grid_ok(B)) return GX_EINVAL;
  hipLaunchKernelGGL(k_huber, dim3((unsigned)blocks_for(B, 256)), dim3(256), 0,
                     (hipStream_t)stream, Y, (long long)ldy, T, (long long)B, delta,
                     scale, static_cast<__bf16*>(dY), (long long)ldd, loss);
  return check(hipGetLastError());
}

int gx_sur_inputs(const double* xyz, const double* t, int32_t t_stride, double dt,
                  int64_t n, double inv_len, double omega, void* X, int64_t ldx,
                  void* stream) {
  if (!xyz || !t || !X || n < 0 || ldx < 5) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  hipLaunchKernelGGL(k_sur_inputs, dim3((unsigned)blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, xyz, t, t_stride, dt, (long long)n, inv_len,
                     omega, static_cast<__bf16*>(X), (long long)ldx);
  return check(hipGetLastError());
}

int gx_sur_targets(const double* t, int32_t t_stride, int64_t n, const double* a_full,
                   const double* a_base, double omega, double inv_scale, float* T,
                   void* stream) {
  if (!t || !a_full || !a_base || !T || n < 0) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  hipLaunchKernelGGL(k_sur_targets, dim3((unsigned)blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, t, t_stride, (long long)n, a_full, a_base, omega,
                     inv_scale, T);
  return check(hipGetLastError());
}

int gx_sur_combine(const gx_pot* base, const gx_pot* full, const double* xyz,
                   const double* t, int32_t t_stride, double dt, int64_t n,
                   const float* Y, int64_t ldy, double scale, double omega,
                   double r_max, const int32_t* flag, double* acc, void* stream) {
  if (!base || !full || !xyz || !t || !Y || !acc || n < 0 || ldy < 3) return GX_EINVAL;
  if (!base->basic || base->device != full->device) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  const dim3 grid((unsigned)blocks_for(n, 256)), blk(256);
  const bool mw = base->sig == kSigMilkyWay, rot = full->sig == kSigMilkyWayRotating;
  const auto kern = mw ? (rot ? k_sur_combine<EvalMW, EvalMilkyWayRotating>
                              : k_sur_combine<EvalMW, EvalTable<true>>)
                       : (rot ? k_sur_combine<EvalTable<false>, EvalMilkyWayRotating>
                              : k_sur_combine<EvalTable<false>, EvalTable<true>>);
  hipLaunchKernelGGL(kern, grid, blk, 0, (hipStream_t)stream, base->dev, full->dev, xyz, t,
                     t_stride, dt, (long long)n, Y, (long long)ldy, scale, omega, r_max, flag,
                     acc);
  return check(hipGetLastError());
}

int gx_sur_check(const gx_pot* full, const double* xyz, const double* t,
                 int32_t t_stride, int64_t n, const double* a_sur, double tol,
                 int32_t* flag, float* err, void* stream) {
  if (!full || !xyz || !t || !a_sur || !flag || n < 0) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  const auto kern = full->sig == kSigMilkyWayRotating ? k_sur_check<EvalMilkyWayRotating>
                                                      : k_sur_check<EvalTable<true>>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, full->dev, xyz, t, t_stride, (long long)n, a_sur,
                     tol, flag, err);
  return check(hipGetLastError());
}

int gx_method_nodes(int32_t method, double* c, int32_t cap) {
  if (method == GX_DOPRI8) {
    if (c)
      for (int i = 0; i < 13 && i < cap; ++i) c[i] = Dopri8::k.c[i];
    return 13;
  }
  if (method == GX_DOPRI5) {
    if (c)
      for (int i = 0; i < 7 && i < cap; ++i) c[i] = Dopri5::k.c[i];
    return 7;
  }
  return GX_EINVAL;
}

int gx_lockstep_stage(int32_t stage, const double* q, const double* p,
                      const double* G, int64_t n, double h, double* Q, void* stream) {
  if (stage < 0 || stage >= 13 || !q || !p || !G || !Q || n < 0) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!grid_ok(n)) return GX_EINVAL;
  hipLaunchKernelGGL(k_stage_point, dim3((unsigned)blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, (int)stage, q, p, G, (long long)n, h, Q);
  return check(hipGetLastError());
}

int gx_lockstep_update(double* q, double* p, const double* G, int64_t n, double h,
                       double* t, void* stream) {
  if (!q || !p || !G || !t || n < 0) return GX_EINVAL;
  if (!grid_ok(n)) return GX_EINVAL;
  hipLaunchKernelGGL(k_step_update, dim3((unsigned)(n > 0 ? blocks_for(n, 256) : 1)),
                     dim3(256), 0, (hipStream_t)stream, q, p, G, (long long)n, h, t);
  return check(hipGetLastError());
}

}  // extern "C"
