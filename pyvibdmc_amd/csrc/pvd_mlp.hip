// Surrogate potential: permutation-sorted inverse-distance descriptor + MLP (D -> H -> H -> H -> 1,
// SiLU) on BF16 MFMA with FP32 accumulation, for inference inside the DMC step and for
// training (forward with stored pre-activations, backward, weight gradients, Adam).
//
// MFMA formulation (v_mfma_f32_16x16x32_bf16, wave64).  Weights are the A operand
// (16 output units x 32 inputs) and activations the B operand (32 inputs x 16 walkers);
// lane l holds A[l%16][8(l/16)+j], B[8(l/16)+j][l%16] (j < 8) and D[4(l/16)+i][l%16]
// (i < 4).  A layer's accumulators therefore already hold, for walker l%16, the units
// 16m + 4(l/16) + i.  Reading the next layer's 32-wide input chunk c as
//   k = 8g + j  ->  unit 16(2c + j/4) + 4g + j%4
// makes those registers the next B operand directly, so activations never leave
// registers; the weights are stored pre-permuted to match (pvd_mlp_pack).
#include <hip/hip_runtime.h>
#include <mutex>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "../../include/pyvibdmc_amd.h"
#include "pvd_models.hpp"

namespace pvd {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int MLP_MAXD = 32;
constexpr int MLP_MAXA = 6;
constexpr int MLP_MAXP = 15;
constexpr int MLP_NQ = 1 + MLP_MAXP + MLP_MAXP * (MLP_MAXP + 1) / 2;  // 136

struct MlpNet {
  int D, H;
  const bf16x8* Wf[3];
  const bf16x8* Wt[2];  // transposed packs of layers 1 and 2
  const float* b[3];
  const float* w3;
  const float* b3;
  int na, use_range;
  float zz[MLP_MAXP];             // z_i z_j of atom pair q in order (0,1), (0,2), ..., (1,2), ...
  float cd2[MLP_MAXA];            // squared Coulomb diagonal (0.5 z_a^2.4)^2
  int cmask[MLP_MAXA];            // bit b: atom b is sorted together with atom a (0: a stays)
  int slot[MLP_MAXA][MLP_MAXA];   // position of the r-th largest-norm member of a's sublist
  int ng, gs;                     // ng > 1: ng position groups of gs positions are sorted
  int gpos[MLP_MAXA][MLP_MAXA];   // position m of group g
  float xmean[MLP_MAXD], xinv[MLP_MAXD], lo[MLP_MAXD], hi[MLP_MAXD];
  float ymean, ystd;
  float quad[MLP_NQ];  // quadratic baseline on the normalised features
};

// quadratic baseline q(x) of the NPR normalised features (FP32): constant, linear terms,
// then x_i x_j for i <= j in row order
template <int NPR>
PVD_DEV float quad_baseline(const MlpNet& M, const float* xn) {
  float q = M.quad[0];
#pragma unroll
  for (int i = 0; i < NPR; ++i) q += M.quad[1 + i] * xn[i];
  int o = 1 + NPR;
#pragma unroll
  for (int i = 0; i < NPR; ++i)
#pragma unroll
    for (int j = i; j < NPR; ++j) q += M.quad[o++] * (xn[i] * xn[j]);
  return q;
}

// SiLU and its derivative with the hardware exp2 and reciprocal (about 1 ulp each); the
// same functions serve training, backward and inference, so the network is consistent
PVD_DEV float sigmoid_f(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
PVD_DEV float silu_f(float z) { return z * sigmoid_f(z); }
PVD_DEV float dsilu_f(float z) {
  const float s = sigmoid_f(z);
  return s * (1.0f + z * (1.0f - s));
}

// unit index of element j of input chunk c for lane group g (the permuted K order)
PVD_DEV int phys_unit(int c, int g, int j) { return 16 * (2 * c + (j >> 2)) + 4 * g + (j & 3); }

// descriptor of one walker (the DistIt permutation sorting of
// simulation_utilities/tensorflow_descriptors/distance_descriptors.py:115-152): atoms are
// permuted, never pair distances, so the features stay the upper triangle of one inverse
// distance matrix.
//  1. sort key: the row norm of the Coulomb matrix (z_i z_j / r_ij, diagonal 0.5 z_i^2.4);
//  2. sorted atoms: within each sublist, position sublist[r] receives the member with the
//     r-th largest norm (ties: lower atom index first);
//  3. sorted groups: equal-size position groups are reordered by the sum of their atoms'
//     norms, largest first (ties: lower group index first);
//  4. features: 1/r of the permuted atoms for position pairs (0,1), (0,2), ..., (1,2), ...
//     (the Coulomb values divided by z_i z_j, a per-feature constant the normalisation
//     removes).
// The permutation is packed as 4-bit fields (position p holds atom (perm >> 4p) & 15), so
// no lane indexes a register array at run time; every table lookup has a compile-time index.
// With `scratch` (LDS, element q of this thread at scratch[q * step]) the pair distances are taken
// from there: 15 writes and reads instead of 225 compares and selects for six atoms.
template <typename R, int NP>
PVD_DEV void mlp_descriptor(const MlpNet& M, const R* x, float* f, float* scratch = nullptr, int step = 0) {
  constexpr int NA = NP / 3, NPR = NA * (NA - 1) / 2;
  static_assert(NA <= MLP_MAXA && NPR <= MLP_MAXP, "too many atoms");
  float dc[NPR];
  float rn2[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) rn2[a] = M.cd2[a];
  {
    int q = 0;
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = i + 1; j < NA; ++j) {
        const float d0 = (float)(x[3 * i] - x[3 * j]);
        const float d1 = (float)(x[3 * i + 1] - x[3 * j + 1]);
        const float d2 = (float)(x[3 * i + 2] - x[3 * j + 2]);
        dc[q] = 1.0f / __fsqrt_rn(d0 * d0 + d1 * d1 + d2 * d2);
        const float c = M.zz[q] * dc[q];
        rn2[i] += c * c;
        rn2[j] += c * c;
        ++q;
      }
  }
  unsigned perm = 0;
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    int r = 0;
#pragma unroll
    for (int b = 0; b < NA; ++b)
      if (b != a && ((M.cmask[a] >> b) & 1)) r += (rn2[b] > rn2[a] || (rn2[b] == rn2[a] && b < a)) ? 1 : 0;
    int p = a;
    if (M.cmask[a]) {
#pragma unroll
      for (int t = 0; t < NA; ++t)
        if (r == t) p = M.slot[a][t];
    }
    perm |= (unsigned)a << (4 * p);
  }
  if (M.ng > 1) {
    float tot[NA];
#pragma unroll
    for (int g = 0; g < NA; ++g) {
      tot[g] = 0.0f;
      if (g < M.ng) {
#pragma unroll
        for (int m = 0; m < NA; ++m) {
          if (m < M.gs) {
            const unsigned at = (perm >> (4 * M.gpos[g][m])) & 15u;
            float nrm = 0.0f;
#pragma unroll
            for (int a = 0; a < NA; ++a)
              if (at == (unsigned)a) nrm = __fsqrt_rn(rn2[a]);
            tot[g] += nrm;
          }
        }
      }
    }
    unsigned fp = perm;
#pragma unroll
    for (int g = 0; g < NA; ++g) {
      if (g < M.ng) {
        int k = 0;
#pragma unroll
        for (int h = 0; h < NA; ++h)
          if (h < M.ng && h != g) k += (tot[h] > tot[g] || (tot[h] == tot[g] && h < g)) ? 1 : 0;
#pragma unroll
        for (int m = 0; m < NA; ++m) {
          if (m < M.gs) {
            int dst = 0;
#pragma unroll
            for (int kk = 0; kk < NA; ++kk)
              if (kk == k) dst = M.gpos[kk][m];
            const unsigned src = (perm >> (4 * M.gpos[g][m])) & 15u;
            fp = (fp & ~(15u << (4 * dst))) | (src << (4 * dst));
          }
        }
      }
    }
    perm = fp;
  }
  if (scratch) {
    // pair (lo, hi) is number first(lo) + hi, with first(lo) + 1 in the nibbles of a constant
    unsigned first = 0;
#pragma unroll
    for (int a = 0; a < NA - 1; ++a) first |= (unsigned)(a * NA - a * (a + 1) / 2 - a) << (4 * a);
#pragma unroll
    for (int q = 0; q < NPR; ++q) scratch[q * step] = dc[q];
    int q = 0;
#pragma unroll
    for (int p1 = 0; p1 < NA; ++p1)
#pragma unroll
      for (int p2 = p1 + 1; p2 < NA; ++p2) {
        const unsigned a1 = (perm >> (4 * p1)) & 15u, a2 = (perm >> (4 * p2)) & 15u;
        const unsigned lo = a1 < a2 ? a1 : a2, hi = a1 < a2 ? a2 : a1;
        f[q++] = scratch[(int)(((first >> (4 * lo)) & 15u) + hi - 1u) * step];
      }
  } else {
    int q = 0;
#pragma unroll
    for (int p1 = 0; p1 < NA; ++p1)
#pragma unroll
      for (int p2 = p1 + 1; p2 < NA; ++p2) {
        const int a1 = (int)((perm >> (4 * p1)) & 15u), a2 = (int)((perm >> (4 * p2)) & 15u);
        const int lo = a1 < a2 ? a1 : a2, hi = a1 < a2 ? a2 : a1;
        const int cq = lo * NA - lo * (lo + 1) / 2 + (hi - lo - 1);
        float v = 0.0f;
#pragma unroll
        for (int s = 0; s < NPR; ++s)
          if (cq == s) v = dc[s];
        f[q++] = v;
      }
  }
#pragma unroll
  for (int k = NPR; k < MLP_MAXP; ++k) f[k] = 0.0f;
}

// ------------------------------------------------------------------------------------
// Training: forward and backward of a batch (k_mlp_fwd_bwd), the weight gradients from the BF16
// operands that it leaves (k_mlp_wgrad), and the sums of both kernels' parts (k_mlp_collect).

// What the three kernels share.  Batch element b of operand row u at [u * ld + b]; elements from n to
// np, n rounded up to 32, are zero.
struct TrainBuf {
  __bf16* x;      // the features (32 rows, zero beyond D)
  __bf16* h[2];   // silu(z_0), silu(z_1)
  __bf16* dz[3];  // dL/dz_l
  float* Y;       // network outputs
  float* B;       // per 32 batch elements: sums of dz_0, dz_1, dz_2, dy h_2 (H each), dy
  float* P;       // per batch slice: W0, W1, W2 gradients
  const float* XT;
  const float* T;
  long long n, np, ld;
};

template <int H>
constexpr int train_slice() { return H == 256 ? 512 : 256; }  // batch elements of a weight gradient part

// One workgroup takes 32 batch elements through all layers and back.  Wave w owns units 32w to
// 32w + 31 of every layer: their pre-activations stay in its registers for the backward pass, its
// share of the four packs is read once, a layer ahead, and only the BF16 operands of the next
// product travel through LDS.  Lane (g, col) holds elements 2 col and 2 col + 1 of the 32 (walker
// tiles t = 0, 1), so that its two values of a unit are one 4-byte store.
// Bound by the latency of the chain of seven products and their barriers: 8192 elements are 256
// workgroups, one to a CU.
template <int H>
__global__ __launch_bounds__(2 * H, H == 256 ? 2 : 1) void k_mlp_fwd_bwd(MlpNet M, TrainBuf D) {
  constexpr int KC = H / 32, MT = H / 16, ROW = H / 8 + 1, PROW = H + 4;
  __shared__ bf16x8 s_act[2][32 * ROW];
  __shared__ __align__(16) float s_prod[32 * PROW];
  __shared__ float s_dy[32];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const long long base = 32ll * blockIdx.x, n = D.n, ld = D.ld;
  const long long w0 = base + 2 * col;
  const bool ok[2] = {w0 < n, w0 + 1 < n};
  auto unit = [&](int m, int i) { return 32 * wv + 16 * m + 4 * g + i; };
  bf16x8 Wa[2][KC], Wb[2][KC];
  auto weights = [&](bf16x8 (&W)[2][KC], const bf16x8* pack) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int c = 0; c < KC; ++c) W[m][c] = pack[((2 * wv + m) * KC + c) * 64 + lane];
  };
  f32x4 b[3][2], w3[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int l = 0; l < 3; ++l) b[l][m][i] = M.b[l][unit(m, i)];
      w3[m][i] = M.w3[unit(m, i)];
    }
  weights(Wa, M.Wf[1]);
  f32x4 z[3][2][2];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  {  // layer 0
    bf16x8 W0[2], v[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) W0[m] = M.Wf[0][(2 * wv + m) * 64 + lane];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = 8 * g + j;
        v[t][j] = (__bf16)((ok[t] && k < M.D) ? D.XT[(long long)k * n + w0 + t] : 0.0f);
      }
#pragma unroll
      for (int m = 0; m < 2; ++m) z[0][t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W0[m], v[t], zero, 0, 0, 0) + b[0][m];
    }
    if (wv == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) *(bf16x2*)(D.x + (8 * g + j) * ld + w0) = bf16x2{v[0][j], v[1][j]};
    }
  }
  weights(Wb, M.Wf[2]);
  // a pair of batch elements of every unit to the weight gradient's operands (zero past the batch),
  // and both to the rows of the next product
  auto publish = [&](const float (&x)[2][2][4], __bf16* to, bf16x8* rows) {
    bf16x8 u[2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bf16x2 v;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          u[t][4 * m + i] = (__bf16)x[t][m][i];
          v[t] = ok[t] ? u[t][4 * m + i] : (__bf16)0.0f;
        }
        if (to) *(bf16x2*)(to + unit(m, i) * ld + w0) = v;
      }
    if (rows) {
#pragma unroll
      for (int t = 0; t < 2; ++t) rows[(16 * t + col) * ROW + 4 * wv + g] = u[t];
    }
  };
  auto product = [&](const bf16x8 (&W)[2][KC], const bf16x8* rows, f32x4 (&a)[2][2]) {
#pragma unroll
    for (int m = 0; m < 2; ++m) a[0][m] = a[1][m] = zero;
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16x8 x = rows[(16 * t + col) * ROW + 4 * c + g];
#pragma unroll
        for (int m = 0; m < 2; ++m) a[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[m][c], x, a[t][m], 0, 0, 0);
      }
  };
  float x[2][2][4];
#define PVD_EACH(expr)                                  \
  _Pragma("unroll") for (int t = 0; t < 2; ++t)         \
      _Pragma("unroll") for (int m = 0; m < 2; ++m)     \
          _Pragma("unroll") for (int i = 0; i < 4; ++i) expr
  // layers 1 and 2
  PVD_EACH(x[t][m][i] = silu_f(z[0][t][m][i]));
  publish(x, D.h[0], s_act[0]);
  __syncthreads();
  product(Wa, s_act[0], z[1]);
  weights(Wa, M.Wt[1]);
  PVD_EACH(z[1][t][m][i] = z[1][t][m][i] + b[1][m][i]);
  PVD_EACH(x[t][m][i] = silu_f(z[1][t][m][i]));
  publish(x, D.h[1], s_act[1]);
  __syncthreads();
  product(Wb, s_act[1], z[2]);
  weights(Wb, M.Wt[0]);
  PVD_EACH(z[2][t][m][i] = z[2][t][m][i] + b[2][m][i]);
  PVD_EACH(x[t][m][i] = silu_f(z[2][t][m][i]));
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      f32x4 p;
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = w3[m][i] * x[t][m][i];
      *(f32x4*)(s_prod + (16 * t + col) * PROW + 32 * wv + 16 * m + 4 * g) = p;
    }
  __syncthreads();
  // the output: four lanes to an element sum a lane group's units each, in order; then the loss
  if (tid < 128) {
    const int r = tid >> 2;
    const float* p = s_prod + r * PROW + 4 * (tid & 3);
    float s = 0.0f;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const f32x4 v = *(const f32x4*)(p + 16 * m);
#pragma unroll
      for (int i = 0; i < 4; ++i) s += v[i];
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    const long long w = base + 2 * (r & 15) + (r >> 4);
    if ((tid & 3) == 0) {
      const float y = s + M.b3[0];
      float dy = 0.0f;
      if (w < n) {
        const float e = y - D.T[w];
        dy = 2.0f * e / (float)n;
        D.Y[w] = y;
      }
      s_dy[r] = dy;
    }
  }
  __syncthreads();
  const float dy[2] = {s_dy[col], s_dy[16 + col]};
  float* B = D.B + (long long)blockIdx.x * (4 * H + 1);
  // sum of a unit's 32 elements (its 16 lanes, two each) into row k
  auto rowsum = [&](const float (&v)[2][2][4], int k) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float s = v[0][m][i] + v[1][m][i];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 64);
        if (col == 0) B[k * H + unit(m, i)] = s;
      }
  };
  PVD_EACH(x[t][m][i] = ok[t] ? dy[t] * x[t][m][i] : 0.0f);
  rowsum(x, 3);
  if (tid == 0) {
    float s = 0.0f;
    for (int r = 0; r < 32; ++r) s += s_dy[r];
    B[4 * H] = s;
  }
  // back: dz_2, dz_1, dz_0
  PVD_EACH(x[t][m][i] = ok[t] ? w3[m][i] * dy[t] * dsilu_f(z[2][t][m][i]) : 0.0f);
  publish(x, D.dz[2], s_act[0]);
  __syncthreads();
  rowsum(x, 2);
  f32x4 a[2][2];
  product(Wa, s_act[0], a);
  PVD_EACH(x[t][m][i] = ok[t] ? a[t][m][i] * dsilu_f(z[1][t][m][i]) : 0.0f);
  publish(x, D.dz[1], s_act[1]);
  __syncthreads();
  rowsum(x, 1);
  product(Wb, s_act[1], a);
  PVD_EACH(x[t][m][i] = ok[t] ? a[t][m][i] * dsilu_f(z[0][t][m][i]) : 0.0f);
  publish(x, D.dz[0], nullptr);
  rowsum(x, 0);
#undef PVD_EACH
}

// Weight gradients of a batch slice: P[o][i] = sum_b dz[o][b] hin[i][b].  A workgroup takes 64 x 64
// of a hidden layer, a wave 32 x 32 of it, or 64 rows of layer 0 (16 a wave).  Both operands are
// read as they lie, 16 bytes a lane; slices of 256 (H = 128) and 512 elements give 256 and 512
// workgroups at 8192 elements.
template <int H>
__global__ __launch_bounds__(256) void k_mlp_wgrad(int Din, TrainBuf D) {
  constexpr int TI = H / 64;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, col = lane & 15;
  // eight slices and more: all tiles of a slice on one XCD (workgroups go to the eight in turn), whose
  // L2 then reads the slice's 1.3 MB (H = 256) once, instead of each XCD every slice
  constexpr int TILES = 2 * TI * TI + TI;
  const int slices = (int)((D.np + train_slice<H>() - 1) / train_slice<H>());
  int slice = blockIdx.x / TILES, tile = blockIdx.x % TILES;
  if (slices >= 8) {
    const int i = blockIdx.x / 8;
    slice = (int)(blockIdx.x % 8) + 8 * (i / TILES);
    tile = i % TILES;
    if (slice >= slices) return;
  }
  const long long k0 = (long long)slice * train_slice<H>();
  const long long k1 = k0 + train_slice<H>() < D.np ? k0 + train_slice<H>() : D.np;
  float* P = D.P + (long long)slice * ((long long)H * Din + 2 * H * H);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if (tile < 2 * TI * TI) {
    const int l = 1 + tile / (TI * TI), ob = tile / TI % TI * 64 + 32 * (wv >> 1), ib = tile % TI * 64 + 32 * (wv & 1);
    const __bf16* pa = D.dz[l] + (ob + col) * D.ld + 8 * g;
    const __bf16* pb = D.h[l - 1] + (ib + col) * D.ld + 8 * g;
    f32x4 acc[2][2];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q >> 1][q & 1] = zero;
#pragma unroll 8
    for (long long k = k0; k < k1; k += 32) {
      bf16x8 A[2], Bv[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        A[q] = *(const bf16x8*)(pa + 16 * q * D.ld + k);
        Bv[q] = *(const bf16x8*)(pb + 16 * q * D.ld + k);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[q >> 1][q & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[q >> 1], Bv[q & 1], acc[q >> 1][q & 1], 0, 0, 0);
    }
    float* out = P + (long long)H * Din + (l - 1) * H * H;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[(ob + 16 * (q >> 1) + 4 * g + i) * H + ib + 16 * (q & 1) + col] = acc[q >> 1][q & 1][i];
    return;
  }
  const int ob = (tile - 2 * TI * TI) * 64 + 16 * wv;
  const __bf16* pa = D.dz[0] + (ob + col) * D.ld + 8 * g;
  const __bf16* pb = D.x + col * D.ld + 8 * g;
  f32x4 acc[2] = {zero, zero};
#pragma unroll 4
  for (long long k = k0; k < k1; k += 32) {
    const bf16x8 A = *(const bf16x8*)(pa + k);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, *(const bf16x8*)(pb + 16 * q * D.ld + k), acc[q], 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (16 * q + col < Din) P[(long long)(ob + 4 * g + i) * Din + 16 * q + col] = acc[q][i];
}

// Sums of the parts, in their order: weights, then the vectors (16 columns a workgroup, a sixteenth
// of the rows a thread: with 64 columns and four waves their chains of loads were the longest part,
// 10.4 us for 8192 elements at H = 256, now 5.3), then the squared error per 256 elements, then the
// loss.
template <int H>
__global__ __launch_bounds__(256) void k_mlp_collect(int Din, TrainBuf D, float* G, double* parts, double* loss) {
  __shared__ float s_f[16][17];
  __shared__ double s_d[4];
  const long long size = (long long)H * Din + 2 * H * H;
  const int wb = (int)((size + 255) / 256), vb = (4 * H + 1 + 15) / 16;
  int blk = blockIdx.x;
  if (blk < wb) {
    const long long q = blk * 256ll + threadIdx.x;
    if (q >= size) return;
    const int splits = (int)((D.np + train_slice<H>() - 1) / train_slice<H>());
    float s = 0.0f;
#pragma unroll 8
    for (int k = 0; k < splits; ++k) s += D.P[k * size + q];
    G[q < (long long)H * Din ? q : q < (long long)H * Din + H * H ? q + H : q + 2 * H] = s;
    return;
  }
  blk -= wb;
  if (blk < vb) {
    const int c = blk * 16 + (threadIdx.x & 15), part = threadIdx.x >> 4;
    const long long rows = D.np / 32;
    float s = 0.0f;
    if (c < 4 * H + 1) {
#pragma unroll 8
      for (long long r = rows * part / 16; r < rows * (part + 1) / 16; ++r) s += D.B[r * (4 * H + 1) + c];
    }
    s_f[part][threadIdx.x & 15] = s;
    __syncthreads();
    if (part == 0 && c < 4 * H + 1) {
      s = 0.0f;
#pragma unroll
      for (int k = 0; k < 16; ++k) s += s_f[k][c & 15];
      const long long b0 = (long long)H * Din;
      // b0, b1 and b2 follow their weights; w3 and b3 follow b2
      G[c < H ? b0 + c : c < 2 * H ? b0 + H * H + c : b0 + 2ll * H * H + c] = s;
    }
    return;
  }
  blk -= vb;
  const long long nb = (D.n + 255) / 256;
  const long long lo = blk < nb ? blk * 256ll : 0, hi = blk < nb ? (lo + 256 < D.n ? lo + 256 : D.n) : D.n;
  double e = 0.0;
#pragma unroll 8
  for (long long k = lo + threadIdx.x; k < hi; k += 256) {
    const float r = D.Y[k] - D.T[k];
    e += (double)r * (double)r;
  }
  e = block_sum<256>(e, s_d);
  if (threadIdx.x == 0) {
    if (blk < nb) parts[blk] = e;
    else *loss = e / (double)D.n;
  }
}

// Adam with bias correction: parameter p with moments m, v and gradient g after the step
struct AdamStep {
  float lr, b1, b2, eps, c1, c2;
  PVD_DEV float operator()(float p, float& m, float& v, float g) const {
    m = b1 * m + (1.0f - b1) * g;
    v = b2 * v + (1.0f - b2) * g * g;
    return p - lr * (m / c1) / (sqrtf(v / c2) + eps);
  }
};

// on the flat FP32 parameter vector
__global__ void k_adam(float* p, float* m, float* v, const float* g, long long size, AdamStep A) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= size) return;
  float mm = m[q], vv = v[q];
  p[q] = A(p[q], mm, vv, g[q]);
  m[q] = mm;
  v[q] = vv;
}

// FP32 master weights -> packed BF16 operands.  Forward pack of layer l (A = W_l):
// element (m, c, lane, j) = W[16m + lane%16][k], k = 8(lane/16)+j (layer 0) or the
// permuted unit (layers 1, 2).  Transposed pack (A = W_l^T): W[permuted k][16m + lane%16].
__global__ void k_mlp_pack(const float* W, int rows, int cols, int in_natural, int transpose, int MT, int KC,
                           bf16x8* out) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)MT * KC * 64;
  if (q >= total) return;
  const int lane = (int)(q % 64);
  const int c = (int)((q / 64) % KC);
  const int m = (int)(q / (64 * KC));
  const int g = lane >> 4, col = lane & 15;
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int k = in_natural ? 32 * c + 8 * g + j : phys_unit(c, g, j);
    const int r = 16 * m + col;
    float x = 0.0f;
    if (!transpose) {
      if (r < rows && k < cols) x = W[(long long)r * cols + k];
    } else {
      // A = W^T: row r is an input unit of W, k an output unit
      if (k < rows && r < cols) x = W[(long long)k * cols + r];
    }
    v[j] = (__bf16)x;
  }
  out[q] = v;
}

// Adam and the repacked operands in one pass.  A thread takes a 4 x 4 block of a hidden layer (four
// consecutive inputs, or four consecutive outputs, are 8 bytes of one pack word, so no store is
// smaller), or a word of layer 0's pack, or one of the remaining parameters.  Bound by the launch:
// 26 us a step as Adam and five pack launches (H = 128), now 7.
template <int H>
__global__ __launch_bounds__(64) void k_adam_pack(int D, float* p, float* m, float* v, const float* g, AdamStep A,
                                                  bf16x8* packs) {
  constexpr int MT = H / 16, KC = H / 32, BLK = H / 4;
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  const int HH = H * H, w1 = H * D + H;  // offset of W1; W2 follows at HH + H
  bf16x8* hidden = packs + MT * 64;
  int q = blockIdx.x * 64 + threadIdx.x;
  if (q < 2 * BLK * BLK) {
    const int layer = q / (BLK * BLK), o0 = q / BLK % BLK * 4, i0 = q % BLK * 4;
    const long long at = w1 + layer * (HH + H) + (long long)o0 * H + i0;
    f32x4 P[4], Mo[4], Vo[4], G[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      P[a] = *(const f32x4*)(p + at + a * H);
      Mo[a] = *(const f32x4*)(m + at + a * H);
      Vo[a] = *(const f32x4*)(v + at + a * H);
      G[a] = *(const f32x4*)(g + at + a * H);
    }
    bf16x4 row[4], col[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float mm = Mo[a][b], vv = Vo[a][b];
        P[a][b] = A(P[a][b], mm, vv, G[a][b]);
        Mo[a][b] = mm;
        Vo[a][b] = vv;
        row[a][b] = col[b][a] = (__bf16)P[a][b];
      }
      *(f32x4*)(p + at + a * H) = P[a];
      *(f32x4*)(m + at + a * H) = Mo[a];
      *(f32x4*)(v + at + a * H) = Vo[a];
    }
    // units k0 .. k0 + 3 of row r: half (k0 / 16) % 2 of word (r / 16, k0 / 32), lane 16 (k0 / 4 % 4) + r % 16
    auto half = [&](bf16x8* pack, int r, int k0) {
      bf16x8* w = pack + ((r >> 4) * KC + (k0 >> 5)) * 64 + 16 * ((k0 >> 2) & 3) + (r & 15);
      return (bf16x4*)w + ((k0 >> 4) & 1);
    };
    bf16x8* fwd = hidden + layer * MT * KC * 64;
    bf16x8* tr = hidden + (2 + layer) * MT * KC * 64;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      *half(fwd, o0 + a, i0) = row[a];
      *half(tr, i0 + a, o0) = col[a];
    }
    return;
  }
  q -= 2 * BLK * BLK;
  auto one = [&](long long k) {
    float mm = m[k], vv = v[k];
    const float x = A(p[k], mm, vv, g[k]);
    p[k] = x;
    m[k] = mm;
    v[k] = vv;
    return x;
  };
  if (q < MT * 64) {  // layer 0: units in natural order, zeros beyond D
    const int lane = q & 63, r = 16 * (q >> 6) + (lane & 15), k0 = 8 * (lane >> 4);
    bf16x8 w;
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = (__bf16)(k0 + j < D ? one((long long)r * D + k0 + j) : 0.0f);
    packs[q] = w;
    return;
  }
  q -= MT * 64;
  if (q < H) one((long long)H * D + q);             // b0
  else if (q < 2 * H) one(w1 + HH + q - H);         // b1
  else if (q < 4 * H + 1) one(w1 + 2ll * HH + q - H);  // b2, w3, b3
}

// descriptors of AoS walkers (n, M, 3) -> raw features F^T (D x n), float32
template <typename R, int NP>
__global__ void k_mlp_desc(MlpNet M, const R* x, long long n, float* FT) {
  const long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= n) return;
  R xx[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) xx[p] = x[w * NP + p];
  float f[MLP_MAXP];
  mlp_descriptor<R, NP>(M, xx, f);
#pragma unroll
  for (int k = 0; k < MLP_MAXP; ++k)
    if (k < M.D) FT[(long long)k * n + w] = f[k];
}

// raw features -> normalised features in place
__global__ void k_mlp_normalise(MlpNet M, long long n, float* FT) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long long)M.D * n) return;
  const int k = (int)(q / n);
  FT[q] = (FT[q] - M.xmean[k]) * M.xinv[k];
}

}  // namespace pvd

using namespace pvd;

namespace {
thread_local std::string g_merr;
int mfail(int code, const std::string& m) {
  g_merr = m;
  return code;
}
#define MHIP(x)                                                                                  \
  do {                                                                                           \
    hipError_t e_ = (x);                                                                         \
    if (e_ != hipSuccess) return mfail(8, std::string(#x) + ": " + hipGetErrorString(e_));       \
  } while (0)

long long off_W(int l, int D, int H) {
  // flat parameter order: W0 (H x D), b0, W1 (H x H), b1, W2, b2, w3, b3
  switch (l) {
    case 0: return 0;
    case 1: return (long long)H * D + H;
    default: return (long long)H * D + H + (long long)H * H + H;
  }
}
long long off_b(int l, int D, int H) { return off_W(l, D, H) + (l == 0 ? (long long)H * D : (long long)H * H); }
long long off_w3(int D, int H) { return (long long)H * D + 3ll * H + 2ll * H * H; }

// the atom-sorting tables of the descriptor from the DistIt-style specification; n_atoms = 0
// describes a network trained on given features only (no descriptor)
bool build_sorting(const pvd_mlp* m, MlpNet& N) {
  const int na = m->n_atoms;
  N.na = na;
  if (na == 0) return true;
  if (na < 2 || na > MLP_MAXA || m->D != na * (na - 1) / 2) return false;
  int q = 0;
  for (int i = 0; i < na; ++i) {
    if (m->z[i] < 1) return false;
    const double d = 0.5 * std::pow((double)m->z[i], 2.4);
    N.cd2[i] = (float)(d * d);
    for (int j = i + 1; j < na; ++j) N.zz[q++] = (float)m->z[i] * (float)m->z[j];
  }
  // sorted atoms: sublists partition the atoms (or there are none)
  if (m->n_sorted_atoms < 0 || m->n_sorted_atoms > na) return false;
  if (m->n_sorted_atoms > 0) {
    int seen = 0, o = 0;
    for (int s = 0; s < m->n_sorted_atoms; ++s) {
      const int len = m->sorted_atoms_len[s];
      if (len < 1 || o + len > na) return false;
      int mask = 0;
      for (int t = 0; t < len; ++t) {
        const int a = m->sorted_atoms[o + t];
        if (a < 0 || a >= na || ((seen >> a) & 1)) return false;
        seen |= 1 << a;
        mask |= 1 << a;
      }
      for (int t = 0; t < len; ++t) {
        const int a = m->sorted_atoms[o + t];
        N.cmask[a] = len > 1 ? (mask & ~(1 << a)) : 0;
        for (int r = 0; r < len; ++r) N.slot[a][r] = m->sorted_atoms[o + r];
      }
      o += len;
    }
    if (seen != (1 << na) - 1) return false;
  }
  // sorted groups: n_groups groups of group_size distinct positions
  N.ng = m->n_groups;
  N.gs = m->group_size;
  if (N.ng > 1) {
    if (N.gs < 1 || N.ng * N.gs > na) return false;
    int seen = 0;
    for (int g = 0; g < N.ng; ++g)
      for (int k = 0; k < N.gs; ++k) {
        const int p = m->sorted_groups[g * N.gs + k];
        if (p < 0 || p >= na || ((seen >> p) & 1)) return false;
        seen |= 1 << p;
        N.gpos[g][k] = p;
      }
  } else {
    N.ng = 0;
  }
  return true;
}

bool build_net(const pvd_mlp* m, MlpNet& N) {
  std::memset(&N, 0, sizeof(N));
  const int D = m->D, H = m->H;
  if (D < 1 || D > 32 || (H != 128 && H != 256)) return false;
  N.D = D;
  N.H = H;
  const float* p = (const float*)m->params;
  for (int l = 0; l < 3; ++l) N.b[l] = p + off_b(l, D, H);
  N.w3 = p + off_w3(D, H);
  N.b3 = N.w3 + H;
  const bf16x8* pk = (const bf16x8*)m->packs;
  const long long s0 = (long long)(H / 16) * 64, s1 = (long long)(H / 16) * (H / 32) * 64;
  N.Wf[0] = pk;
  N.Wf[1] = pk + s0;
  N.Wf[2] = pk + s0 + s1;
  N.Wt[0] = pk + s0 + 2 * s1;
  N.Wt[1] = pk + s0 + 3 * s1;
  N.use_range = m->use_range;
  if (!build_sorting(m, N)) return false;
  for (int k = 0; k < 32; ++k) {
    N.xmean[k] = m->xmean[k];
    N.xinv[k] = m->xinv[k];
    N.lo[k] = m->lo[k];
    N.hi[k] = m->hi[k];
  }
  N.ymean = m->ymean;
  for (int k = 0; k < MLP_NQ; ++k) N.quad[k] = m->quad[k];
  N.ystd = m->ystd;
  return true;
}

// ------------------------------------------------------------------------------------
// Inference on walkers, H = 128: persistent workgroups keep all three weight packs (72 KB),
// the biases and the output weights in LDS for the whole launch; each wave has its own range of
// walkers and activations never leave its registers.  A wave takes 64 walkers at a time: their
// descriptors, one lane each, then the network on two tiles of NT_E x 16 (each A fragment read
// from LDS feeds NT_E MFMAs; the biases enter as the MFMA accumulator input).  Walkers outside
// the training range get the FALLBACK_MARK bit pattern, which k_mlp_fallback replaces with the
// analytic potential.
// Bound by VALU issue (SiLU: two transcendentals of 8 cycles and three other instructions an
// activation).  With the descriptor of a walker computed by the four lanes that share its tile
// column, and workgroups taking whole chunks of 256 walkers: water, 400 000 walkers FP32 75.5 us,
// now 65.7 (k_mlp_fallback and the launches included); six atoms, 200 000 walkers FP64 133, 60.
constexpr int NT_E = 2;
constexpr int E_WAVES = 8;  // waves per workgroup sharing one LDS copy of the weights
constexpr unsigned long long FALLBACK_MARK = 0x7FF4D1CEFA11BAC4ull;  // a signalling-NaN payload
constexpr unsigned OUT_OF_RANGE = 0x7FA11BACu;                        // the same for a baseline, in FP32

template <int H>
constexpr size_t energy_lds_bytes() {
  return (size_t)((H / 16) * 64 + 2 * (H / 16) * (H / 32) * 64) * 16 + (size_t)(4 * H + 4) * 4;
}

// Normalised features of a walker as bf16 (16, the rest zero) and its quadratic baseline, or
// OUT_OF_RANGE.  `scratch`: see mlp_descriptor.
template <typename R, int NP>
PVD_DEV float energy_features(const MlpNet& M, const R* x, bf16x8 (&v)[2], float* scratch, int step) {
  constexpr int NPR = NP / 3 * (NP / 3 - 1) / 2;
  float f[MLP_MAXP];
  mlp_descriptor<R, NP>(M, x, f, scratch, step);
  bool out = false;
  if (M.use_range) {
#pragma unroll
    for (int k = 0; k < NPR; ++k) out |= !(f[k] >= M.lo[k] && f[k] <= M.hi[k]);
  }
#pragma unroll
  for (int k = 0; k < NPR; ++k) f[k] = (f[k] - M.xmean[k]) * M.xinv[k];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k >> 3][k & 7] = (__bf16)(k < NPR ? f[k < NPR ? k : 0] : 0.0f);
  return out ? __uint_as_float(OUT_OF_RANGE) : quad_baseline<NPR>(M, f);
}

// The description (a kernel's first argument), read again where it is used: kept over a kernel's
// loop its numbers would be spilled.
PVD_DEV const MlpNet& cold_net() {
  typedef const __attribute__((address_space(4))) MlpNet Cold;
  Cold* cold = (Cold*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(cold));
  return *(const MlpNet*)cold;
}

template <typename R, int NP, int H>
__global__ __launch_bounds__(64 * E_WAVES, 4) void k_mlp_energy(MlpNet M, const R* planes, long long stride,
                                                                const int* n_dev, long long n_fix, double* V) {
  extern __shared__ bf16x8 lds[];
  constexpr int MT = H / 16, KC = H / 32, NPR = NP / 3 * (NP / 3 - 1) / 2;
  bf16x8* L0 = lds;
  bf16x8* L1 = L0 + MT * 64;
  bf16x8* L2 = L1 + MT * KC * 64;
  float* lb = (float*)(L2 + MT * KC * 64);  // b0 | b1 | b2 | w3 | b3
  for (int q = threadIdx.x; q < MT * 64; q += 64 * E_WAVES) L0[q] = M.Wf[0][q];
  for (int q = threadIdx.x; q < MT * KC * 64; q += 64 * E_WAVES) {
    L1[q] = M.Wf[1][q];
    L2[q] = M.Wf[2][q];
  }
  for (int q = threadIdx.x; q < H; q += 64 * E_WAVES) {
    lb[q] = M.b[0][q];
    lb[H + q] = M.b[1][q];
    lb[2 * H + q] = M.b[2][q];
    lb[3 * H + q] = M.w3[q];
  }
  if (threadIdx.x == 0) lb[4 * H] = M.b3[0];
  __syncthreads();
  const int n = n_dev ? *n_dev : (int)n_fix;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, col = lane & 15;
  constexpr int TILE_E = 16 * NT_E;
  static_assert(TILE_E == 32, "two tiles to a batch of descriptors");
  const int tiles = (int)(((long long)n + TILE_E - 1) / TILE_E), nw = gridDim.x * E_WAVES;
  // neighbouring ranges go to different workgroups: where the tiles do not divide by the waves, the
  // longer ranges are spread over the chip
  const int wid = wave * gridDim.x + blockIdx.x;
  const int t0 = (int)((long long)tiles * wid / nw), t1 = (int)((long long)tiles * (wid + 1) / nw);
  for (int tb = t0; tb < t1; tb += 2) {
    // compiler-only barrier: the weight fragments are re-read from LDS instead of being hoisted out
    // of the loop into (spilled) registers
    asm volatile("" ::: "memory");
    bf16x8 fw[2];
    float qb;
    {
      const long long w = (long long)tb * TILE_E + lane;
      R x[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) x[p] = planes[p * stride + (w < n ? w : 0)];
      qb = energy_features<R, NP>(cold_net(), x, fw, nullptr, 0);
    }
#pragma unroll 1
    for (int s = 0; s < 2 && tb + s < t1; ++s) {
      bf16x8 bin0[NT_E], bin[NT_E][KC];
      f32x4 acc[NT_E][MT];
#pragma unroll
      for (int t = 0; t < NT_E; ++t) {
        const int from = 4 * (TILE_E * s + 16 * t + col);
        int d[4];
        int4 w0 = __builtin_bit_cast(int4, fw[0]), w1 = __builtin_bit_cast(int4, fw[1]);
        const int a0[4] = {w0.x, w0.y, w0.z, w0.w}, a1[4] = {w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int u0 = 2 * k < NPR ? __builtin_amdgcn_ds_bpermute(from, a0[k]) : 0;
          const int u1 = 8 + 2 * k < NPR ? __builtin_amdgcn_ds_bpermute(from, a1[k]) : 0;
          d[k] = g == 0 ? u0 : g == 1 ? u1 : 0;
        }
        bin0[t] = __builtin_bit_cast(bf16x8, int4{d[0], d[1], d[2], d[3]});
      }
#pragma unroll
      for (int layer = 0; layer < 3; ++layer) {
        asm volatile("" ::: "memory");
        const float* bl = lb + layer * H;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const f32x4 bias = *(const f32x4*)(bl + 16 * m + 4 * g);
          if (layer == 0) {
            const bf16x8 a = L0[m * 64 + lane];
#pragma unroll
            for (int t = 0; t < NT_E; ++t) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bin0[t], bias, 0, 0, 0);
          } else {
            const bf16x8* Wl = layer == 1 ? L1 : L2;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
              const bf16x8 a = Wl[(m * KC + c) * 64 + lane];
#pragma unroll
              for (int t = 0; t < NT_E; ++t)
                acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bin[t][c], c == 0 ? bias : acc[t][m], 0, 0, 0);
            }
          }
        }
        if (layer < 2) {
#pragma unroll
          for (int t = 0; t < NT_E; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
              for (int i = 0; i < 4; ++i) bin[t][m >> 1][(m & 1) * 4 + i] = (__bf16)silu_f(acc[t][m][i]);
        }
      }
      const float b3 = lb[4 * H];
#pragma unroll
      for (int t = 0; t < NT_E; ++t) {
        float s3 = 0.0f;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const f32x4 w3 = *(const f32x4*)(lb + 3 * H + 16 * m + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) s3 += w3[i] * silu_f(acc[t][m][i]);
        }
        s3 += __shfl_xor(s3, 16, 64);
        s3 += __shfl_xor(s3, 32, 64);
        const int r = TILE_E * s + 16 * t + col;
        const float q = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * r, __float_as_int(qb)));
        const long long w = (long long)tb * TILE_E + r;
        if (g == 0 && w < n) {
          const float y = s3 + b3;
          V[w] = __float_as_uint(q) == OUT_OF_RANGE ? __longlong_as_double((long long)FALLBACK_MARK)
                                                    : (double)(y * M.ystd + M.ymean + q);
        }
      }
    }
  }
}

// Inference on walkers, H = 256, where the packs of two hidden layers do not fit LDS together.
// Wave w of a workgroup keeps its 32 output units of both hidden layers in registers for the
// whole launch (128 registers), so no weight is read again; what travels through LDS are the
// activations (bf16, 512 bytes a walker and layer, read by every wave).  A tile of 32 walkers
// passes layer 0, layer 1, layer 2 and the output in successive rounds of one barrier each; a round
// works on four tiles at once, one per layer, so that the SiLUs of one layer cover the matrix
// products of another.  The descriptors of 512 walkers are computed at a time, one thread each.
// A layer's D registers of unit tiles 2w and 2w + 1 are word 4w + g of a walker's row: the next
// layer's B operand of input chunk w, lane group g (phys_unit).  Every sum has the order of the
// H = 128 kernel, the output's included: its 64 products a lane group go through LDS.
// Six atoms, 1 000 003 walkers FP32, fallback pass included: 878 us when the packs were staged through
// LDS for every 128 walkers, 396 now (0.68 PFLOP/s; 487 in a process's first calls, until its clock has
// risen): VALU issue 66 % of the time, matrix cores 28 %, LDS 30 %.  With H = 128
// it is slower than the kernel above (six atoms, 200 000 walkers FP64: 71 us against 60).
template <int NP, int H>
struct EnergyShape {
  static constexpr int NPR = NP / 3 * (NP / 3 - 1) / 2;
  static constexpr int NW = H / 32, NTH = 64 * NW, BT = NTH / 32;  // waves, threads, tiles per descriptor batch
  static constexpr int FW = NPR > 8 ? 2 : 1;                        // 16-byte words of a walker's features
  static constexpr int ROW = H / 8 + 1, PROW = H + 4;               // padded rows: activations (words), products (floats)
  static constexpr size_t words = 4 * 32 * (size_t)ROW + FW * NTH;
  static constexpr size_t floats = 2 * NTH + 2 * 32 * PROW + 4 * H;
  static constexpr size_t lds = words * 16 + floats * 4;
  static_assert(H == 256, "one workgroup of eight waves a CU");
};

template <typename R, int NP, int H>
__global__ __launch_bounds__(2 * H, 2) void k_mlp_energy_reg(
    MlpNet M, const R* planes, long long stride, const int* n_dev, long long n_fix, double* V) {
  using S = EnergyShape<NP, H>;
  constexpr int KC = H / 32, MT = H / 16, NPR = S::NPR;
  extern __shared__ bf16x8 lds[];
  bf16x8* act1 = lds;                                  // [2][32][ROW]
  bf16x8* act2 = act1 + 2 * 32 * S::ROW;               // [2][32][ROW]
  bf16x8* feat = act2 + 2 * 32 * S::ROW;               // [NTH][FW]
  float* s_q = (float*)(feat + S::FW * S::NTH);        // [2][NTH] baseline, or OUT_OF_RANGE
  float* s_prod = s_q + 2 * S::NTH;                    // [2][32][PROW] w3 times the last layer's activations
  float* lb = s_prod + 2 * 32 * S::PROW;               // b0 | b1 | b2 | w3
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int n = n_dev ? *n_dev : (int)n_fix;
  const int tiles = (int)(((long long)n + 31) / 32);
  const int t0 = (int)((long long)tiles * blockIdx.x / gridDim.x);
  const int nt = (int)((long long)tiles * (blockIdx.x + 1) / gridDim.x) - t0;
  if (nt == 0) return;
  bf16x8 W0[2], W1[2][KC], W2[2][KC];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    W0[m] = M.Wf[0][(2 * wv + m) * 64 + lane];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      W1[m][c] = M.Wf[1][((2 * wv + m) * KC + c) * 64 + lane];
      W2[m][c] = M.Wf[2][((2 * wv + m) * KC + c) * 64 + lane];
    }
  }
  for (int q = tid; q < H; q += S::NTH) {
    lb[q] = M.b[0][q];
    lb[H + q] = M.b[1][q];
    lb[2 * H + q] = M.b[2][q];
    lb[3 * H + q] = M.w3[q];
  }
  const float b3 = M.b3[0];
  auto descriptors = [&](int batch) {
    const long long w = 32ll * t0 + (long long)batch * S::NTH + tid;
    R x[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) x[p] = planes[p * stride + (w < n ? w : 0)];
    // scratch: the products' area that this round writes, which nobody reads any more
    static_assert(NPR * S::NTH <= 32 * S::PROW, "scratch");
    float* scratch = s_prod + 32 * (batch * S::BT & 1) * S::PROW + tid;
    bf16x8 v[2];
    s_q[(batch & 1) * S::NTH + tid] = energy_features<R, NP>(cold_net(), x, v, NP == 18 ? scratch : nullptr, S::NTH);
#pragma unroll
    for (int k = 0; k < S::FW; ++k) feat[S::FW * tid + k] = v[k];
  };
  // four units 16(2 wv + m) + 4g + i of a bias or output weight vector
  auto units = [&](const float* b, int m) { return *(const f32x4*)(b + 32 * wv + 16 * m + 4 * g); };
  // rounds past the last tile only drain the layers behind it (what the first layers make of old
  // rows is read by nobody)
  for (int it = 0; it < nt + 3; ++it) {
    if (it % S::BT == 0 && it < nt) {
      descriptors(it / S::BT);
      __syncthreads();
    }
    const int cur = it & 1, old = cur ^ 1;
    // output of tile it - 3, one wave of each SIMD, the two in turn: lane l sums the units of group l / 8, in
    // the order of the units, then the groups are added.  First in the round: at its end the other
    // waves would wait for this chain of additions
    if (it >= 3 && wv >> 2 == (it & (S::NW / 4 - 1)) && lane < 32) {
      const int t = it - 3, r = 8 * (wv & 3) + (lane & 7);
      const long long w = 32ll * (t0 + t) + r;
      const float* p = s_prod + (32 * old + r) * S::PROW + 4 * (lane >> 3);
      const float qb = s_q[t % (2 * S::BT) * 32 + r];
      f32x4 v[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) v[m] = *(const f32x4*)(p + 16 * m);
      float s = 0.0f;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) s += v[m][i];
      s += __shfl_xor(s, 8, 64);
      s += __shfl_xor(s, 16, 64);
      const float y = s + b3;
      if (lane < 8 && w < n)
        V[w] = __float_as_uint(qb) == OUT_OF_RANGE ? __longlong_as_double((long long)FALLBACK_MARK)
                                                   : (double)(y * M.ystd + M.ymean + qb);
    }
    // layer 0 of tile it, layer 1 of tile it - 1, layer 2 of tile it - 2: the matrix instructions of
    // layers 1 and 2 run between the SiLUs of the layer before (16 / KC to an input chunk's four),
    // the input chunks are read AHEAD chunks before their use
    constexpr int EL = 16 / KC, AHEAD = 2;
    f32x4 z[3][2][2];
    bf16x8 x[2 * KC][2], x0[2], u;
    auto read = [&](int k) {
      const bf16x8* rows = k < KC ? act1 + 32 * old * S::ROW : act2 + 32 * cur * S::ROW;
#pragma unroll
      for (int t = 0; t < 2; ++t) x[k][t] = rows[(16 * t + col) * S::ROW + 4 * (k % KC) + g];
    };
    auto start = [&](int layer) {
#pragma unroll
      for (int m = 0; m < 2; ++m) z[layer][0][m] = z[layer][1][m] = units(lb + layer * H, m);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      x0[t] = feat[S::FW * (it % S::BT * 32 + 16 * t + col) + (S::FW == 2 ? g & 1 : 0)];
      if (g >= S::FW) x0[t] = bf16x8{};
    }
    start(0);
    start(1);
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) read(k);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < 2; ++m) z[0][t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W0[m], x0[t], z[0][t][m], 0, 0, 0);
#pragma unroll
    for (int k = 0; k < 2 * KC; ++k) {
      const int c = k % KC, l = 1 + k / KC;
      if (k + AHEAD < 2 * KC) read(k + AHEAD);
      if (k == KC - AHEAD) start(2);
      float h[EL];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int t = q >> 1, m = q & 1;
        z[l][t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l == 1 ? W1[m][c] : W2[m][c], x[k][t], z[l][t][m], 0, 0, 0);
#pragma unroll
        for (int e = q * EL / 4; e < (q + 1) * EL / 4; ++e) {
          const int o = EL * c + e;
          h[e] = silu_f(z[l - 1][o >> 3][(o >> 2) & 1][o & 3]);
        }
      }
#pragma unroll
      for (int e = 0; e < EL; ++e) u[(EL * c + e) & 7] = (__bf16)h[e];
      if (EL * (c + 1) % 8 == 0) {
        bf16x8* out = l == 1 ? act1 + 32 * cur * S::ROW : act2 + 32 * old * S::ROW;
        out[(16 * (EL * c / 8) + col) * S::ROW + 4 * wv + g] = u;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const f32x4 w3 = units(lb + 3 * H, m);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 p;
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = w3[i] * silu_f(z[2][t][m][i]);
        *(f32x4*)(s_prod + (32 * cur + 16 * t + col) * S::PROW + 32 * wv + 16 * m + 4 * g) = p;
      }
    }
    __syncthreads();
  }
}

// analytic potential for the walkers the surrogate marked as outside its training range
template <typename R, int NP>
__global__ __launch_bounds__(256) void k_mlp_fallback(const R* planes, long long stride, const int* n_dev,
                                                      long long n_fix, double* V, PesParams fb) {
  const int n = n_dev ? *n_dev : (int)n_fix;
  for (long long w = (long long)blockIdx.x * 256 + threadIdx.x; w < n; w += (long long)gridDim.x * 256) {
    if ((unsigned long long)__double_as_longlong(V[w]) != FALLBACK_MARK) continue;
    R x[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) x[p] = planes[p * stride + w];
    V[w] = (double)pes_eval<R, NP>(fb, x);
  }
}

// Error judge: analytic potential on every `every`-th walker against the surrogate's V
// (one workgroup, fixed-order reduction); record = {step, sum of squared errors, max |error|,
// samples} in hartree.
template <typename R, int NP>
__global__ __launch_bounds__(1024) void k_mlp_judge(const R* planes, long long stride, const int* n_dev,
                                                    long long n_fix, const double* V, int every, PesParams pes,
                                                    long long step, double* rec) {
  __shared__ double s_a[16], s_b[16];
  __shared__ int s_c[16];
  const int n = n_dev ? *n_dev : (int)n_fix;
  double sse = 0.0, mx = 0.0;
  int cnt = 0;
  for (long long w = (long long)threadIdx.x * every; w < n; w += 1024ll * every) {
    R x[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) x[p] = planes[p * stride + w];
    const double d = V[w] - (double)pes_eval<R, NP>(pes, x);
    sse += d * d;
    mx = fmax(mx, fabs(d));
    ++cnt;
  }
  const int wv = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sse += __shfl_xor(sse, o, 64);
    mx = fmax(mx, __shfl_xor(mx, o, 64));
    cnt += __shfl_xor(cnt, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s_a[wv] = sse;
    s_b[wv] = mx;
    s_c[wv] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = 0.0, b = 0.0;
    int c = 0;
    for (int k = 0; k < 16; ++k) {
      a += s_a[k];
      b = fmax(b, s_b[k]);
      c += s_c[k];
    }
    rec[0] = (double)step;
    rec[1] = a;
    rec[2] = b;
    rec[3] = (double)c;
  }
}

template <typename R, int NP, int H>
int launch_energy(const MlpNet& N, const void* planes, long long stride, const int* n_dev, long long n_max,
                  double* V, const PesParams& fb, hipStream_t st) {
  int dev = 0, cus = 256;
  MHIP(hipGetDevice(&dev));
  MHIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  if constexpr (H == 128) {
    // two workgroups per CU (LDS-bound)
    const long long wgs = (n_max + 32 * E_WAVES - 1) / (32 * E_WAVES);
    const unsigned grid = (unsigned)std::max(1ll, std::min(wgs, 2ll * cus));
    const size_t lds = energy_lds_bytes<H>();
    auto k = k_mlp_energy<R, NP, H>;
    MHIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3(grid), dim3(64 * E_WAVES), lds, st, N, (const R*)planes, stride, n_dev, n_max, V);
  } else {
    using S = EnergyShape<NP, H>;
    const unsigned grid = (unsigned)std::max(1ll, std::min((n_max + 31) / 32, (long long)cus));
    auto k = k_mlp_energy_reg<R, NP, H>;
    MHIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds));
    hipLaunchKernelGGL(k, dim3(grid), dim3(S::NTH), S::lds, st, N, (const R*)planes, stride, n_dev, n_max, V);
  }
  MHIP(hipGetLastError());
  if (N.use_range) {
    const unsigned gf = (unsigned)std::max(1ll, std::min((n_max + 255) / 256, 4ll * cus));
    hipLaunchKernelGGL((k_mlp_fallback<R, NP>), dim3(gf), dim3(256), 0, st, (const R*)planes, stride, n_dev, n_max,
                       V, fb);
    MHIP(hipGetLastError());
  }
  return 0;
}

}  // namespace

extern "C" {

const char* pvd_mlp_last_error(void) { return g_merr.c_str(); }

int64_t pvd_mlp_param_count(int32_t D, int32_t H) { return off_w3(D, H) + H + 1; }

int64_t pvd_mlp_pack_bytes(int32_t H) {
  return ((int64_t)(H / 16) * 64 + 4ll * (H / 16) * (H / 32) * 64) * 16;
}

int pvd_mlp_pack(const pvd_mlp* m, void* stream) {
  if (!m || !m->params || !m->packs) return mfail(7, "null argument");
  const int D = m->D, H = m->H;
  if (H != 128 && H != 256) return mfail(7, "hidden width must be 128 or 256");
  hipStream_t st = (hipStream_t)stream;
  const float* p = (const float*)m->params;
  bf16x8* pk = (bf16x8*)m->packs;
  const int MT = H / 16, KC = H / 32;
  const long long s0 = (long long)MT * 64, s1 = (long long)MT * KC * 64;
  hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((s0 + 255) / 256)), dim3(256), 0, st, p + off_W(0, D, H), H, D, 1, 0,
                     MT, 1, pk);
  hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((s1 + 255) / 256)), dim3(256), 0, st, p + off_W(1, D, H), H, H, 0, 0,
                     MT, KC, pk + s0);
  hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((s1 + 255) / 256)), dim3(256), 0, st, p + off_W(2, D, H), H, H, 0, 0,
                     MT, KC, pk + s0 + s1);
  hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((s1 + 255) / 256)), dim3(256), 0, st, p + off_W(1, D, H), H, H, 0, 1,
                     MT, KC, pk + s0 + 2 * s1);
  hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((s1 + 255) / 256)), dim3(256), 0, st, p + off_W(2, D, H), H, H, 0, 1,
                     MT, KC, pk + s0 + 3 * s1);
  MHIP(hipGetLastError());
  return 0;
}

int pvd_mlp_descriptors(const pvd_mlp* m, int32_t precision, int32_t n_atoms, const void* coords, int64_t n,
                        int32_t normalise, float* features_t, void* stream) {
  MlpNet N;
  if (!m || !coords || !features_t || !build_net(m, N)) return mfail(7, "bad network description");
  if (n_atoms != m->n_atoms || n_atoms < 2)
    return mfail(7, "the network's descriptor is for another number of atoms");
  if (n <= 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const unsigned grid = (unsigned)((n + 255) / 256);
  const int np = n_atoms * 3;
  if (precision == PVD_FP64) {
    if (np == 9) hipLaunchKernelGGL((k_mlp_desc<double, 9>), dim3(grid), dim3(256), 0, st, N, (const double*)coords, n, features_t);
    else if (np == 18) hipLaunchKernelGGL((k_mlp_desc<double, 18>), dim3(grid), dim3(256), 0, st, N, (const double*)coords, n, features_t);
    else return mfail(7, "descriptor kernels support 3 or 6 atoms");
  } else {
    if (np == 9) hipLaunchKernelGGL((k_mlp_desc<float, 9>), dim3(grid), dim3(256), 0, st, N, (const float*)coords, n, features_t);
    else if (np == 18) hipLaunchKernelGGL((k_mlp_desc<float, 18>), dim3(grid), dim3(256), 0, st, N, (const float*)coords, n, features_t);
    else return mfail(7, "descriptor kernels support 3 or 6 atoms");
  }
  if (normalise)
    hipLaunchKernelGGL(k_mlp_normalise, dim3((unsigned)((N.D * n + 255) / 256)), dim3(256), 0, st, N, (long long)n,
                       features_t);
  MHIP(hipGetLastError());
  return 0;
}

int pvd_mlp_energy(const pvd_mlp* m, int32_t precision, int32_t n_atoms, const void* planes, int64_t stride,
                   const int32_t* n_dev, int64_t n_max, double* v_out, const pvd_pes_desc* fallback, void* stream) {
  MlpNet N;
  if (!m || !planes || !v_out || !build_net(m, N)) return mfail(7, "bad network description");
  if (n_atoms != m->n_atoms || n_atoms < 2)
    return mfail(7, "the network's descriptor is for another number of atoms");
  if (n_max <= 0) return 0;
  PesParams fb;
  std::memset(&fb, 0, sizeof(fb));
  if (fallback) std::memcpy(&fb, fallback, sizeof(fb));
  if (N.use_range && !fallback) return mfail(7, "range check needs a fallback potential");
  hipStream_t st = (hipStream_t)stream;
  const int np = n_atoms * 3;
#define PVD_E(R, NP, H) return launch_energy<R, NP, H>(N, planes, stride, n_dev, n_max, v_out, fb, st)
  if (precision == PVD_FP64) {
    if (np == 9 && N.H == 128) PVD_E(double, 9, 128);
    if (np == 9 && N.H == 256) PVD_E(double, 9, 256);
    if (np == 18 && N.H == 128) PVD_E(double, 18, 128);
    if (np == 18 && N.H == 256) PVD_E(double, 18, 256);
  } else {
    if (np == 9 && N.H == 128) PVD_E(float, 9, 128);
    if (np == 9 && N.H == 256) PVD_E(float, 9, 256);
    if (np == 18 && N.H == 128) PVD_E(float, 18, 128);
    if (np == 18 && N.H == 256) PVD_E(float, 18, 256);
  }
#undef PVD_E
  return mfail(7, "surrogate supports 3 or 6 atoms and hidden width 128 or 256");
}

int pvd_mlp_judge(const pvd_pes_desc* pes, int32_t precision, int32_t n_atoms, const void* planes, int64_t stride,
                  const int32_t* n_dev, int64_t n_max, const double* v, int32_t every, int64_t step, double* record,
                  void* stream) {
  if (!pes || !planes || !v || !record || every < 1) return mfail(7, "bad arguments");
  PesParams P;
  std::memcpy(&P, pes, sizeof(P));
  hipStream_t st = (hipStream_t)stream;
  const int np = n_atoms * 3;
#define PVD_J(R, NP)                                                                                 \
  hipLaunchKernelGGL((k_mlp_judge<R, NP>), dim3(1), dim3(1024), 0, st, (const R*)planes, stride, n_dev, n_max, v, \
                     every, P, step, record)
  if (precision == PVD_FP64) {
    if (np == 9) PVD_J(double, 9);
    else if (np == 18) PVD_J(double, 18);
    else return mfail(7, "judge supports 3 or 6 atoms");
  } else {
    if (np == 9) PVD_J(float, 9);
    else if (np == 18) PVD_J(float, 18);
    else return mfail(7, "judge supports 3 or 6 atoms");
  }
#undef PVD_J
  MHIP(hipGetLastError());
  return 0;
}

}  // extern "C"

namespace {

// The training buffers in a workspace, and their bytes (64 of them to align its start)
size_t train_layout(int D, int H, int64_t n, char* ws, TrainBuf& B) {
  // rows 320 bytes past a multiple of 4 KB: the 16 rows that a wave reads at once lie in different
  // channels (8192 elements, width 256, rows of 16 KB: weight gradients 37 us, 20 so); 320 past a
  // multiple of 512 where the rows are shorter than 4 KB, which would else take several times their bytes
  const int64_t np = (n + 31) / 32 * 32, unit = np <= 2048 ? 256 : 2048, ld = ((np + unit - 1 - 160) & ~(unit - 1)) + 160;
  const int64_t slice = H == 256 ? train_slice<256>() : train_slice<128>();
  size_t at = 0;
  auto take = [&](size_t bytes) {
    char* p = ws + at;
    at += (bytes + 63) / 64 * 64;
    return p;
  };
  B.x = (__bf16*)take(2 * 32 * (size_t)ld);
  for (auto& h : B.h) h = (__bf16*)take(2 * (size_t)H * ld);
  for (auto& d : B.dz) d = (__bf16*)take(2 * (size_t)H * ld);
  B.Y = (float*)take(4 * (size_t)np);
  B.B = (float*)take(4 * (size_t)(np / 32) * (4 * H + 1));
  B.P = (float*)take(4 * (size_t)((np + slice - 1) / slice) * ((size_t)H * D + 2 * (size_t)H * H));
  B.n = n;
  B.np = np;
  B.ld = ld;
  return at + 64;
}
int64_t train_bytes(int D, int H, int64_t n) {
  TrainBuf B;
  return n <= 0 ? 0 : (int64_t)train_layout(D, H, n, nullptr, B);
}

}  // namespace

extern "C" {

// Gradients of the mean squared error of the network on (X, T) into grads (flat, the
// parameter order), plus the loss.  ws: device workspace of pvd_mlp_workspace_bytes().
int64_t pvd_mlp_workspace_bytes(int32_t D, int32_t H, int64_t batch) {
  const int64_t n = batch;
  const int64_t splits = (n + 255) / 256;
  const int64_t P = splits * (int64_t)H * (H > D ? H : D);
  // at least what earlier versions asked for: it bounds the batches that the static scratch takes
  return std::max<int64_t>((3 * H * n * 2 + 2 * n + P + (n + 255) / 256 * 2) * 4 + 64, train_bytes(D, H, n));
}

}  // extern "C"

namespace {

// Scratch of pvd_mlp_grads_noalloc: one array per device, held until the process ends.
// Host code never uses the name `scratch` as an address: the device address comes from
// hipGetSymbolAddress, looked up once per device with that device current.
constexpr long long PVD_MLP_SCRATCH_BYTES = 32ll << 20;
static __device__ __align__(256) unsigned char scratch[PVD_MLP_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch[MAX_DEVICES];

int scratch_for_current_device(void** out) {
  int dev = 0;
  MHIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) return mfail(7, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return mfail(8, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[dev] = ptr;
  }
  *out = g_scratch[dev];
  return 0;
}

int mlp_grads(const pvd_mlp* m, const float* x_t, const float* targets, int64_t n, float* grads, float* y_out,
              double* loss_parts, double* loss, void* workspace, void* stream);

}  // namespace

extern "C" {

int pvd_mlp_loss_grads(const pvd_mlp* m, const float* x_t, const float* targets, int64_t n, float* grads, float* y_out,
                       double* loss_parts, double* loss, void* workspace, void* stream) {
  if (!workspace || !loss) return mfail(7, "bad arguments");
  return mlp_grads(m, x_t, targets, n, grads, y_out, loss_parts, loss, workspace, stream);
}

int pvd_mlp_grads(const pvd_mlp* m, const float* x_t, const float* targets, int64_t n, float* grads, float* y_out,
                  double* loss_parts, void* workspace, void* stream) {
  if (!workspace) return mfail(7, "bad arguments");
  return mlp_grads(m, x_t, targets, n, grads, y_out, loss_parts, nullptr, workspace, stream);
}

int64_t pvd_mlp_noalloc_scratch_bytes(void) { return PVD_MLP_SCRATCH_BYTES; }

int pvd_mlp_grads_noalloc(const pvd_mlp* m, const float* x_t, const float* targets, int64_t n, float* grads,
                          float* y_out, double* loss_parts, void* stream) {
  if (!m) return mfail(7, "bad arguments");
  if (n <= 0) return mfail(7, "empty batch");
  const int64_t need = pvd_mlp_workspace_bytes(m->D, m->H, n);
  if (need > PVD_MLP_SCRATCH_BYTES)
    return mfail(7, "batch too large for the static scratch: needs " + std::to_string(need) + " bytes, the maximum is " +
                        std::to_string(PVD_MLP_SCRATCH_BYTES));
  void* ws = nullptr;
  const int rc = scratch_for_current_device(&ws);
  if (rc) return rc;
  return mlp_grads(m, x_t, targets, n, grads, y_out, loss_parts, nullptr, ws, stream);
}

}  // extern "C"

namespace {

template <int H>
int launch_grads(const MlpNet& N, TrainBuf B, float* grads, double* loss_parts, double* loss, hipStream_t st) {
  const int D = N.D;
  const unsigned slices = (unsigned)((B.np + train_slice<H>() - 1) / train_slice<H>());
  hipLaunchKernelGGL(k_mlp_fwd_bwd<H>, dim3((unsigned)(B.np / 32)), dim3(2 * H), 0, st, N, B);
  const unsigned rounds = slices >= 8 ? (slices + 7) / 8 * 8 : slices;  // see k_mlp_wgrad
  hipLaunchKernelGGL(k_mlp_wgrad<H>, dim3((2 * (H / 64) * (H / 64) + H / 64) * rounds), dim3(256), 0, st, D, B);
  const long long blocks = ((long long)H * D + 2 * H * H + 255) / 256 + (4 * H + 16) / 16 + (B.n + 255) / 256 + (loss ? 1 : 0);
  hipLaunchKernelGGL(k_mlp_collect<H>, dim3((unsigned)blocks), dim3(256), 0, st, D, B, grads, loss_parts, loss);
  MHIP(hipGetLastError());
  return 0;
}

int mlp_grads(const pvd_mlp* m, const float* x_t, const float* targets, int64_t n, float* grads, float* y_out,
              double* loss_parts, double* loss, void* workspace, void* stream) {
  MlpNet N;
  if (!m || !x_t || !targets || !grads || !workspace || !build_net(m, N)) return mfail(7, "bad arguments");
  if (n <= 0) return mfail(7, "empty batch");
  hipStream_t st = (hipStream_t)stream;
  TrainBuf B;
  (void)train_layout(N.D, N.H, n, (char*)(((uintptr_t)workspace + 63) & ~(uintptr_t)63), B);
  B.XT = x_t;
  B.T = targets;
  if (y_out) B.Y = y_out;
  return N.H == 128 ? launch_grads<128>(N, B, grads, loss_parts, loss, st)
                    : launch_grads<256>(N, B, grads, loss_parts, loss, st);
}

}  // namespace

extern "C" {

int pvd_mlp_adam(float* params, float* m1, float* m2, const float* grads, int64_t size, float lr, float beta1,
                 float beta2, float eps, int64_t t, void* stream) {
  if (!params || !m1 || !m2 || !grads || size <= 0 || t <= 0) return mfail(7, "bad arguments");
  const AdamStep A{lr, beta1, beta2, eps, 1.0f - powf(beta1, (float)t), 1.0f - powf(beta2, (float)t)};
  hipLaunchKernelGGL(k_adam, dim3((unsigned)((size + 255) / 256)), dim3(256), 0, (hipStream_t)stream, params, m1, m2,
                     grads, (long long)size, A);
  MHIP(hipGetLastError());
  return 0;
}

int pvd_mlp_adam_pack(const pvd_mlp* m, float* m1, float* m2, const float* grads, float lr, float beta1, float beta2,
                      float eps, int64_t t, void* stream) {
  if (!m || !m->params || !m->packs || !m1 || !m2 || !grads || t <= 0) return mfail(7, "bad arguments");
  const int D = m->D, H = m->H;
  if (D < 1 || D > 32 || (H != 128 && H != 256)) return mfail(7, "hidden width must be 128 or 256");
  float* p = const_cast<float*>(m->params);
  // the one-pass kernel reads four parameters at a time
  if (((uintptr_t)p | (uintptr_t)m1 | (uintptr_t)m2 | (uintptr_t)grads | (uintptr_t)m->packs) & 15) {
    const int rc = pvd_mlp_adam(p, m1, m2, grads, pvd_mlp_param_count(D, H), lr, beta1, beta2, eps, t, stream);
    return rc ? rc : pvd_mlp_pack(m, stream);
  }
  const AdamStep A{lr, beta1, beta2, eps, 1.0f - powf(beta1, (float)t), 1.0f - powf(beta2, (float)t)};
  const int items = H * H / 8 + 4 * H + 4 * H + 1;
  auto k = H == 128 ? k_adam_pack<128> : k_adam_pack<256>;
  hipLaunchKernelGGL(k, dim3((unsigned)((items + 63) / 64)), dim3(64), 0, (hipStream_t)stream, D, p, m1, m2, grads, A,
                     (bf16x8*)m->packs);
  MHIP(hipGetLastError());
  return 0;
}

}  // extern "C"
