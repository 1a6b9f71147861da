// FP64 matrix-core GEMMs (v_mfma_f64_16x16x4f64) for gfx950.
//
// C[b] = alpha * op(A[b]) op(B[b]) + beta * C[b], column-major:
//   complex x complex : three real products (Gauss)
//   real x complex    : Cr += A Br, Ci += A Bi  (2 MFMA)
//   complex x real    : Cr += Ar B, Ci += Ai B  (2 MFMA)
//
// MFMA 16x16x4 f64 operand layout (lane l = 0..63):
//   A(16x4): lane l holds A[l % 16][l / 16];  B(4x16): lane l holds B[l / 16][l % 16];
//   D(16x16): lane l, register r holds D[l / 16 + 4 * r][l % 16].
#include "tg_internal.h"
#include "tg_mfma.h"

namespace {

typedef double __attribute__((ext_vector_type(4))) d4;

__device__ inline d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <typename T> struct IsC { static constexpr bool v = false; };
template <> struct IsC<cplx> { static constexpr bool v = true; };

template <int OP> __device__ inline cplx conj_op(cplx v) { return OP == OP_C ? cconj(v) : v; }
template <int OP> __device__ inline double conj_op(double v) { return v; }

template <typename T> __device__ inline T zero_v();
template <> __device__ inline double zero_v<double>() { return 0.0; }
template <> __device__ inline cplx zero_v<cplx>() { return cmk(0.0, 0.0); }

constexpr int XCDS = 8;
constexpr int KP = 2;   // k of a lane that follow each other (mfma_batched_kernel)

// One (TM x 16) x (TN x 16) tile of C per wave, operands straight from global memory
// (L1 / L2) into the matrix-core registers: a lane loads the element of op(A) and op(B)
// that it feeds, so there is no LDS, no barrier and no wave waits for another.  KS steps
// of 4 k each are in flight: a step's operands are loaded as soon as its registers are
// free, KS - 1 steps of products before they are needed.  Lane quarter lk
// takes k = 4 KP (t / KP) + KP lk + t mod KP in step t, whatever KS is, so every tile shape adds
// the products of an element in the same order: the tuner's choice, a matter of timing,
// leaves the bits alone.
// The products are formed transposed (MFMA rows = columns of C), so that lanes 0..15
// hold 16 consecutive rows of a column and loads and stores of C are unit-stride.
// Rows and columns past the edge repeat the last one and are not stored; k past the
// end is masked in the last chunk only.
// A skew product (GemmEpi) forms the tiles that reach the diagonal or lie below it, 44 of
// 77 of 48 x 32 at order 336, and stores each element at its transposed place as well.  The
// tiles above the diagonal follow those of all elements: they end at once, or, where the
// element is not skew to rounding (GemmEpi::exact), form the rest of its product.
// Complex x complex is three real products (Gauss): cr = sum Ar Br, ci = sum Ai Bi,
// c3 = sum (Ar + Ai)(Br + Bi); C = (cr - ci, c3 - cr - ci).
// Bound by the matrix cores, the load latency covered by the steps in flight and 2-4
// waves per SIMD.  The launch bound keeps the accumulators in VGPRs: without it the
// compiler parks them in AGPRs and moves every one out and back in each trip (1.4-1.9 ms
// for the first figure below).  Best tile of each, against workgroup tiles staged through
// LDS with two barriers per 16 k (48 x 48, three waves; they spent a third of their time
// waiting at barriers and for LDS):
//   225 x 336^3 complex 0.81 ms (84 TF/s, 80 % of the matrix rate at three products), 0.99
//     before; with A transposed 0.83 (0.99); real x complex 0.54 (0.64)
//   78 x 224^3 0.090 (0.136), 0.100 (0.137), 0.067 (0.092)
//   121 x 140^3 0.043 (0.065), 0.047 (0.063), 0.034 (0.039)
//   1296 x 64^3 0.046 (0.064), 0.055 (0.063), 0.038 (0.043); 49 x 24^3 0.004 (0.007)
template <typename TA, typename TB, int OPA, int OPB, int TM, int TN, int KS, int OCC>
__global__ void __launch_bounds__(256, OCC)
mfma_batched_kernel(int M, int N, int K, cplx alpha, const TA* __restrict__ A, int lda,
                    long long sA, const TB* __restrict__ B, int ldb, long long sB, cplx beta,
                    int use_beta, cplx* __restrict__ C, int ldc, long long sC, int batch,
                    int tiles_m, int tiles, int upper, int per, int divA, int divB, GemmEpi ep) {
  constexpr bool CA = IsC<TA>::v, CB = IsC<TB>::v, CC = CA && CB;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the batch * tiles (element, tile) pairs are cut into 8 contiguous runs, one per XCD
  // (workgroup ids are dealt round-robin to the XCDs), so the tiles of one element share
  // an L2 and every XCD gets the same number
  const unsigned first = XCDS * (unsigned)per;    // workgroups of the tiles counted by `tiles`
  int b, ti, tj;
  bool mirror = ep.skew != 0;
  if (blockIdx.x < first) {
    const unsigned g = (blockIdx.x % XCDS * (unsigned)per + blockIdx.x / XCDS) * 4 + w;
    if (g >= (unsigned)batch * (unsigned)tiles) return;
    b = (int)(g / (unsigned)tiles);
    const int tile = (int)(g - (unsigned)b * (unsigned)tiles);
    ti = tile % tiles_m;
    tj = tile / tiles_m;
    if (ep.skew) {        // the tiles that reach the diagonal or lie below it, by columns
      ti = tile;
      for (tj = 0; ti >= tiles_m - tj * TN / TM; ++tj) ti -= tiles_m - tj * TN / TM;
      ti += tj * TN / TM;
      if (ep.exact) mirror = ep.exact[b / ep.divExact] != 0.0;
    }
  } else {                // those above it, of products that are not skew to rounding
    const unsigned g = (blockIdx.x - first) * 4 + w;
    if (g >= (unsigned)batch * (unsigned)upper) return;
    b = (int)(g / (unsigned)upper);
    if (ep.exact[b / ep.divExact] != 0.0) return;
    mirror = false;
    ti = (int)(g - (unsigned)b * (unsigned)upper);
    for (tj = 0; ti >= tj * TN / TM; ++tj) ti -= tj * TN / TM;
  }
  const int m0 = ti * 16 * TM, n0 = tj * 16 * TN;
  const int lr = lane & 15, lk = lane >> 4;
  const TA* Ab = A + (long long)(b / divA) * sA;
  const TB* Bb = B + (long long)(b / divB) * sB;
  constexpr bool AN = OPA == OP_N, BN = OPB == OP_N;
  // element offsets of the lane's rows / columns at k = KP lk (32 bits: one matrix)
  unsigned ao[TM], bo[TN];
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    const unsigned i = min(m0 + 16 * x + lr, M - 1);
    ao[x] = AN ? i + KP * lk * (unsigned)lda : KP * lk + i * (unsigned)lda;
  }
#pragma unroll
  for (int y = 0; y < TN; ++y) {
    const unsigned j = min(n0 + 16 * y + lr, N - 1);
    bo[y] = BN ? KP * lk + j * (unsigned)ldb : j + KP * lk * (unsigned)ldb;
  }
  const long long ka = AN ? lda : 1, kb = BN ? 1 : ldb;   // elements per k
  d4 cr[TM][TN], ci[TM][TN], c3[CC ? TM : 1][CC ? TN : 1];
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) {
      cr[x][y] = d4{0.0, 0.0, 0.0, 0.0};
      ci[x][y] = d4{0.0, 0.0, 0.0, 0.0};
      if constexpr (CC) c3[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    }
  TA va[KS][TM];
  TB vb[KS][TN];
  auto load = [&](int s, int t, bool mask) {                // step t to the registers s
    const int k = t / KP * (4 * KP) + t % KP;
    const TA* pa = Ab + k * ka;
    const TB* pb = Bb + k * kb;
    const bool in = !mask || k + KP * lk < K;
#pragma unroll
    for (int x = 0; x < TM; ++x) {
      if (mask) va[s][x] = zero_v<TA>();
      if (in) va[s][x] = pa[ao[x]];
    }
#pragma unroll
    for (int y = 0; y < TN; ++y) {
      if (mask) vb[s][y] = zero_v<TB>();
      if (in) vb[s][y] = pb[bo[y]];
    }
  };
  auto multiply = [&](int s) {
#pragma unroll
    for (int x = 0; x < TM; ++x)
#pragma unroll
      for (int y = 0; y < TN; ++y) {
        const auto av = conj_op<OPA>(va[s][x]);
        const auto bv = conj_op<OPB>(vb[s][y]);
        if constexpr (CC) {
          cr[x][y] = mfma(bv.x, av.x, cr[x][y]);
          ci[x][y] = mfma(bv.y, av.y, ci[x][y]);
          c3[x][y] = mfma(bv.x + bv.y, av.x + av.y, c3[x][y]);
        } else if constexpr (CA) {
          cr[x][y] = mfma(bv, av.x, cr[x][y]);
          ci[x][y] = mfma(bv, av.y, ci[x][y]);
        } else {
          cr[x][y] = mfma(bv.x, av, cr[x][y]);
          ci[x][y] = mfma(bv.y, av, ci[x][y]);
        }
      }
  };
  // a step's registers are loaded for the step KS further on as soon as it is multiplied
  const int tf = K / (4 * KP) * KP / KS * KS;               // steps in whole chunks of KS
  const int te = (K + 4 * KP - 1) / (4 * KP) * KP;
  if (tf > 0) {
#pragma unroll
    for (int s = 0; s < KS; ++s) load(s, s, false);
#pragma unroll 1
    for (int t = KS; t < tf; t += KS) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        multiply(s);
        __builtin_amdgcn_sched_barrier(0);
        load(s, t + s, false);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) multiply(s);
  }
#pragma unroll 1
  for (int t = tf; t < te; t += KS) {
#pragma unroll
    for (int s = 0; s < KS; ++s) load(s, t + s, true);
#pragma unroll
    for (int s = 0; s < KS; ++s) multiply(s);
  }
  // lane: row lr, columns lk + 4 r of each 16 x 16 block
  cplx* Cb = C + (long long)b * sC;
  const double* add = ep.add ? ep.add + (long long)(b / ep.divAdd) * ep.sAdd : nullptr;
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    const int gi = m0 + 16 * x + lr;
    if (gi >= M) continue;
#pragma unroll
    for (int y = 0; y < TN; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = n0 + 16 * y + lk + 4 * r;
        if (gj >= N || (mirror && gi < gj)) continue;
        cplx* cp = Cb + gi + (long long)gj * ldc;
        cplx p;
        if constexpr (CC)
          p = cmk(cr[x][y][r] - ci[x][y][r], c3[x][y][r] - cr[x][y][r] - ci[x][y][r]);
        else
          p = cmk(cr[x][y][r], ci[x][y][r]);
        cplx v = cmul(alpha, p);
        if (use_beta) v = cadd(v, cmul(beta, *cp));
        if (ep.conj) v.y = -v.y;
        if (add) v.x += add[gi + (long long)gj * ldc];
        if (mirror) {
          if (gi == gj) v = cmk(0.0, 0.0);
          else Cb[gj + (long long)gi * ldc] = cmk(-v.x, -v.y);
        }
        *cp = v;
      }
  }
}

// Real FP64 GEMM on the matrix cores for the real products of the constraint
// machinery and the canonical basis (n x n, batched over states):
// C[b] = alpha op(A[b]) op(B[b]) + beta C[b].  One 16 x 16 tile of C per workgroup, a
// quarter of k per wave: few tiles (one state's matrices) and short products, so the time
// is the latency of a wave's chain, and a quarter of it with every wave's operands, 32 k
// at a time, straight in registers (mfma_batched_kernel's scheme) is the shortest one.  The
// four partial sums meet in LDS.  The transposed block is computed (D = op(B)^T op(A)^T),
// so that lane l holds rows l % 16 of four columns: the stores are unit-stride.
// One product of order 224 6.1 us, 336 14.7, medians inside a descent (32 x 32 tiles
// staged 16 k at a time through LDS: 19-23, 27).
template <int OPA, int OPB>
__global__ void __launch_bounds__(256)
mfma_dd_kernel(int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
               long long sA, const double* __restrict__ B, int ldb, long long sB, double beta,
               int use_beta, double* __restrict__ C, int ldc, long long sC, int tiles_m, int divA,
               int divB) {
  constexpr int KS = 8;                          // k steps of 4 in flight
  constexpr bool AN = OPA == OP_N, BN = OPB == OP_N;
  __shared__ double part[4][4][64];
  const int b = blockIdx.y;
  const double* Ab = A + (long long)(b / divA) * sA;
  const double* Bb = B + (long long)(b / divB) * sB;
  double* Cb = C + (long long)b * sC;
  const int m0 = (blockIdx.x % tiles_m) * 16, n0 = (blockIdx.x / tiles_m) * 16;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int kq = (K + 15) / 16 * 4;              // k of a wave
  const int kb = w * kq, ke = min(K, kb + kq);
  const long long ka = AN ? lda : 1, kc = BN ? 1 : ldb;      // elements per k
  const double* pa = Ab + (AN ? (long long)min(m0 + lr, M - 1) : (long long)min(m0 + lr, M - 1) * lda);
  const double* pb = Bb + (BN ? (long long)min(n0 + lr, N - 1) * ldb : (long long)min(n0 + lr, N - 1));
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  double va[KS], vb[KS];
  // lane quarter lk takes k = k0 + KS lk + s in step s
  auto load = [&](int s, int k0) {
    const int k = k0 + KS * lk + s;
    const bool in = k < ke;
    va[s] = in ? pa[k * ka] : 0.0;
    vb[s] = in ? pb[k * kc] : 0.0;
  };
  if (kb < ke) {
#pragma unroll
    for (int s = 0; s < KS; ++s) load(s, kb);
    for (int k0 = kb + 4 * KS; k0 < ke; k0 += 4 * KS) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        acc = mfma(vb[s], va[s], acc);
        load(s, k0);
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma(vb[s], va[s], acc);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[w][r][lane] = acc[r];
  __syncthreads();
  // wave w adds register w: C(m0 + lr, n0 + lk + 4 w)
  const int gi = m0 + lr, gj = n0 + lk + 4 * w;
  if (gi < M && gj < N) {
    double* cp = Cb + gi + (long long)gj * ldc;
    double v = alpha * ((part[0][w][lane] + part[1][w][lane]) + (part[2][w][lane] + part[3][w][lane]));
    if (use_beta) v = fma(beta, *cp, v);
    *cp = v;
  }
}

// The same for many tiles (the matrices of many states): 32 x 32 of C per workgroup, one
// 16 x 16 block per wave, both operands staged 16 k at a time through LDS, so an element is
// read for 32 rows or columns instead of 16.  The chain of its 2 K / 16 barriers sets
// its time (12.5 us at K = 224, 5 at 64) until its workgroups no longer fit the chip at once;
// mfma_dd_kernel's grows with the tiles from a few hundred on.  32 products A^T B of order 224 33.7
// against 100 us, 64 of order 140 23.8 against 51, medians inside an iteration.
template <int OPA, int OPB>
__global__ void __launch_bounds__(256)
mfma_dd_lds_kernel(int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
                   long long sA, const double* __restrict__ B, int ldb, long long sB, double beta,
                   int use_beta, double* __restrict__ C, int ldc, long long sC, int tiles_m,
                   int divA, int divB) {
  constexpr int BT = 32, BK = 16, LD = BT + 1;
  __shared__ double As[BK][LD], Bs[BK][LD];     // As[k][i] = op(A)(i,k), Bs[k][j] = op(B)(k,j)
  const int b = blockIdx.y;
  const double* Ab = A + (long long)(b / divA) * sA;
  const double* Bb = B + (long long)(b / divB) * sB;
  double* Cb = C + (long long)b * sC;
  const int m0 = (blockIdx.x % tiles_m) * BT, n0 = (blockIdx.x / tiles_m) * BT;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int wi = (w & 1) * 16, wj = (w >> 1) * 16;
  const int lr = lane & 15, lk = lane >> 4;
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < K; k0 += BK) {
    // 512 elements of each operand tile, two per thread, contiguous index fastest
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int e = t + 256 * r;
      int i, k;
      if (OPA == OP_N) { i = e % BT; k = e / BT; } else { k = e % BK; i = e / BK; }
      const int gi = m0 + i, gk = k0 + k;
      double v = 0.0;
      if (gi < M && gk < K) v = (OPA == OP_N) ? Ab[gi + (long long)gk * lda] : Ab[gk + (long long)gi * lda];
      As[k][i] = v;
      int j, k2;
      if (OPB == OP_N) { k2 = e % BK; j = e / BK; } else { j = e % BT; k2 = e / BT; }
      const int gj = n0 + j, gk2 = k0 + k2;
      double u = 0.0;
      if (gj < N && gk2 < K) u = (OPB == OP_N) ? Bb[gk2 + (long long)gj * ldb] : Bb[gj + (long long)gk2 * ldb];
      Bs[k2][j] = u;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const double av = Bs[kk + lk][wj + lr];    // D rows: columns of C
      const double bv = As[kk + lk][wi + lr];    // D columns: rows of C
      acc = mfma(av, bv, acc);
    }
    __syncthreads();
  }
  // lane l, register r: C(m0 + wi + lr, n0 + wj + lk + 4 r)
  const int gi = m0 + wi + lr;
  if (gi < M) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gj = n0 + wj + lk + 4 * r;
      if (gj < N) {
        double* cp = Cb + gi + (long long)gj * ldc;
        double v = alpha * acc[r];
        if (use_beta) v = fma(beta, *cp, v);
        *cp = v;
      }
    }
  }
}

// Grouped contraction: C(j, a) = sum_k W_g(k, j) X(k, a) for every group g; X and C hold
// a row of `ld` angles per position (angle contiguous), W_g is real, j contiguous.  The
// scheme of mfma_batched_kernel with both operands contiguous across the lanes: a wave
// takes TJ x 16 positions and TA x 16 angles of one group.  tile_group / tile_j0 list
// tiles of 64 positions, entry t for XCD t % 8 (group < 0: none); a group stays on one
// XCD, whose L2 then holds its X and W_g, and the groups are dealt to the XCDs by work.
// A unit of work is (tile, angle tile, part of the tile), four neighbouring units of an
// XCD's list per workgroup.
// Bound by the matrix cores: 225 angles x 400 groups of up to 820 positions 1.04 ms, 55
// TF/s (72 % of the FP64 matrix rate with the padding of the tiles counted), 450 angles x
// 200 groups 0.95 ms, 60 TF/s.  Through LDS with 80 x 64 tiles 1.17 and 1.07 ms; with the
// groups not kept on one XCD 1.10 and 1.06 ms; with X and W contiguous in k (each lane
// its own row) 1.46 and 1.39 ms.
struct GroupedArgs {
  int M;                       // angles
  int ld;                      // stride of a position's row (>= M)
  const cplx* X;
  cplx* C;
  const void* W;
  const GroupDesc* groups;
  const int* tile_group;
  const int* tile_j0;
  int mtiles, units;
};

template <typename TW, int TA, int TJ, int KS>
__device__ __forceinline__ void grouped_tile(const GroupedArgs& g, const GroupDesc& gd, int a0, int j0) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int s = gd.size;
  const cplx* Xb = g.X + (long long)gd.off * g.ld;
  const TW* Wb = reinterpret_cast<const TW*>(static_cast<const char*>(g.W) + gd.woff);
  unsigned xo[TA], wo[TJ];
#pragma unroll
  for (int x = 0; x < TA; ++x) xo[x] = min(a0 + 16 * x + lr, g.M - 1) + lk * g.ld;
#pragma unroll
  for (int y = 0; y < TJ; ++y) wo[y] = min(j0 + 16 * y + lr, s - 1) + lk * s;
  d4 cr[TA][TJ], ci[TA][TJ];
#pragma unroll
  for (int x = 0; x < TA; ++x)
#pragma unroll
    for (int y = 0; y < TJ; ++y) {
      cr[x][y] = d4{0.0, 0.0, 0.0, 0.0};
      ci[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    }
  cplx xv[KS][TA];
  TW wv[KS][TJ];
  auto load = [&](int q, int k0, bool mask) {
    const cplx* px = Xb + (long long)(k0 + 4 * q) * g.ld;
    const TW* pw = Wb + (long long)(k0 + 4 * q) * s;
    const bool in = !mask || k0 + 4 * q + lk < s;
#pragma unroll
    for (int x = 0; x < TA; ++x) {
      if (mask) xv[q][x] = cmk(0.0, 0.0);
      if (in) xv[q][x] = px[xo[x]];
    }
#pragma unroll
    for (int y = 0; y < TJ; ++y) {
      if (mask) wv[q][y] = (TW)0;
      if (in) wv[q][y] = pw[wo[y]];
    }
  };
  auto multiply = [&](int q) {
#pragma unroll
    for (int x = 0; x < TA; ++x)
#pragma unroll
      for (int y = 0; y < TJ; ++y) {
        cr[x][y] = mfma((double)wv[q][y], xv[q][x].x, cr[x][y]);
        ci[x][y] = mfma((double)wv[q][y], xv[q][x].y, ci[x][y]);
      }
  };
  const int kf = s / (4 * KS) * (4 * KS);
  if (kf > 0) {
#pragma unroll
    for (int q = 0; q < KS; ++q) load(q, 0, false);
#pragma unroll 1
    for (int k0 = 4 * KS; k0 < kf; k0 += 4 * KS) {
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        multiply(q);
        __builtin_amdgcn_sched_barrier(0);
        load(q, k0, false);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int q = 0; q < KS; ++q) multiply(q);
  }
  if (kf < s) {
#pragma unroll
    for (int q = 0; q < KS; ++q) load(q, kf, true);
#pragma unroll
    for (int q = 0; q < KS; ++q) multiply(q);
  }
  // lane: rows lk + 4 r (positions), column lr (angle) of each 16 x 16 block
#pragma unroll
  for (int x = 0; x < TA; ++x) {
    const int a = a0 + 16 * x + lr;
    if (a >= g.M) continue;
#pragma unroll
    for (int y = 0; y < TJ; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = j0 + 16 * y + lk + 4 * r;
        if (j < s) g.C[(long long)(gd.off + j) * g.ld + a] = cmk(cr[x][y][r], ci[x][y][r]);
      }
  }
}

template <int TA, int TJ, int KS, int OCC>
__global__ void __launch_bounds__(256, OCC)
mfma_grouped_kernel(GroupedArgs g) {
  constexpr int PARTS = 4 / TJ;
  const int u = blockIdx.x / XCDS * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (u >= g.units) return;
  const int part = u % PARTS, at = u / PARTS % g.mtiles;
  const int tile = u / (PARTS * g.mtiles) * XCDS + blockIdx.x % XCDS;
  const int grp = g.tile_group[tile];
  if (grp < 0) return;
  const GroupDesc gd = g.groups[grp];
  const int j0 = g.tile_j0[tile] + 16 * TJ * part;
  if (j0 >= gd.size) return;
  if (gd.fp32) grouped_tile<float, TA, TJ, KS>(g, gd, at * 16 * TA, j0);
  else grouped_tile<double, TA, TJ, KS>(g, gd, at * 16 * TA, j0);
}

// The same for M <= 4 angles: matrix-vector products, bound by reading W once.  A
// workgroup takes one tile of 64 positions, a lane a position; its eight waves take
// eighths of k (X elements are uniform loads) and meet in LDS.
constexpr int GV_W = 8;
template <typename TW, int M>
__device__ __forceinline__ void grouped_vec(const GroupedArgs& g, const GroupDesc& gd, int j0,
                                            cplx (&acc)[M]) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = gd.size, k0 = (int)((long long)s * w / GV_W), k1 = (int)((long long)s * (w + 1) / GV_W);
  const TW* W = reinterpret_cast<const TW*>(static_cast<const char*>(g.W) + gd.woff) + min(j0 + lane, s - 1);
  const cplx* X = g.X + (long long)gd.off * g.ld;
#pragma unroll 16
  for (int k = k0; k < k1; ++k) {
    const double v = (double)W[(long long)k * s];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const cplx x = X[(long long)k * g.ld + m];
      acc[m].x = fma(x.x, v, acc[m].x);
      acc[m].y = fma(x.y, v, acc[m].y);
    }
  }
}

template <int M>
__global__ void __launch_bounds__(64 * GV_W)
grouped_vec_kernel(GroupedArgs g) {
  __shared__ cplx part[GV_W][M][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int grp = g.tile_group[blockIdx.x];
  if (grp < 0) return;
  const GroupDesc gd = g.groups[grp];
  const int j0 = g.tile_j0[blockIdx.x];
  cplx acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = cmk(0.0, 0.0);
  if (gd.fp32) grouped_vec<float, M>(g, gd, j0, acc);
  else grouped_vec<double, M>(g, gd, j0, acc);
#pragma unroll
  for (int m = 0; m < M; ++m) part[w][m][lane] = acc[m];
  __syncthreads();
  if (w < M && j0 + lane < gd.size) {
    cplx v = part[0][w][lane];
#pragma unroll
    for (int q = 1; q < GV_W; ++q) v = cadd(v, part[q][w][lane]);
    g.C[(long long)(gd.off + j0 + lane) * g.ld + w] = v;
  }
}

template <typename TA, typename TB, int OPA, int OPB, int TM, int TN, int KS, int OCC>
int launch_batched(hipStream_t s, int M, int N, int K, cplx alpha, const TA* A, int lda,
                   long long sA, const TB* B, int ldb, long long sB, cplx beta, int use_beta,
                   cplx* C, int ldc, long long sC, int batch, int divA, int divB,
                   const GemmEpi& ep) {
  const int tiles_m = (M + 16 * TM - 1) / (16 * TM), tiles_n = (N + 16 * TN - 1) / (16 * TN);
  int tiles = tiles_m * tiles_n, upper = 0;
  if (ep.skew) {
    if (M != N || use_beta) {
      tg_set_error("mfma gemm: a skew product is square and written, not added");
      return TG_E_ARG;
    }
    tiles = 0;
    for (int j = 0; j < tiles_n; ++j) tiles += tiles_m - j * TN / TM;
    if (ep.exact) upper = tiles_m * tiles_n - tiles;
  }
  const long long wgs = ((long long)batch * tiles + 3) / 4;      // four waves, a tile each
  const long long per = (wgs + XCDS - 1) / XCDS;
  const long long grid = (long long)XCDS * per + ((long long)batch * upper + 3) / 4;
  if (grid > 0x1fffffffLL) {          // tile numbers in 32 bits
    tg_set_error("mfma gemm: grid too large");
    return TG_E_ARG;
  }
  if (grid == 0) return TG_OK;
  hipLaunchKernelGGL((mfma_batched_kernel<TA, TB, OPA, OPB, TM, TN, KS, OCC>), dim3((unsigned)grid),
                     dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, use_beta, C, ldc,
                     sC, batch, tiles_m, tiles, upper, (int)per, divA, divB, ep);
  TG_HIP(hipGetLastError());
  return TG_OK;
}

template <typename TA, typename TB, int OPA, int OPB>
int launch_variant(int variant, hipStream_t s, int M, int N, int K, cplx alpha, const TA* A,
                   int lda, long long sA, const TB* B, int ldb, long long sB, cplx beta,
                   int use_beta, cplx* C, int ldc, long long sC, int batch, int divA, int divB,
                   const GemmEpi& ep) {
#define TG_V(K_, TM, TN, KS, OCC)                                                               \
  case K_:                                                                                      \
    return launch_batched<TA, TB, OPA, OPB, TM, TN, KS, OCC>(s, M, N, K, alpha, A, lda, sA, B,  \
                                                             ldb, sB, beta, use_beta, C, ldc,   \
                                                             sC, batch, divA, divB, ep);
  switch (variant) {
    TG_V(0, 2, 2, 2, 3)
    TG_V(1, 2, 2, 4, 2)
    TG_V(2, 3, 2, 2, 2)
    TG_V(3, 2, 3, 2, 2)
    TG_V(4, 3, 2, 3, 2)
    TG_V(5, 3, 1, 3, 3)
    TG_V(6, 2, 1, 3, 4)
    TG_V(7, 2, 1, 4, 3)
    TG_V(8, 1, 1, 2, 4)
    TG_V(9, 1, 1, 4, 4)
    TG_V(10, 3, 1, 4, 2)
  }
#undef TG_V
  tg_set_error("mfma gemm: bad tile variant");
  return TG_E_ARG;
}

template <typename TA, typename TB>
int dispatch(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
             const TA* A, int lda, long long sA, const TB* B, int ldb, long long sB, cplx beta,
             int use_beta, cplx* C, int ldc, long long sC, int batch, int divA, int divB,
             const GemmEpi& ep) {
#define TG_CASE(OA, OB)                                                                        \
  if (opa == OA && opb == OB)                                                                  \
    return launch_variant<TA, TB, OA, OB>(variant, s, M, N, K, alpha, A, lda, sA, B, ldb, sB,  \
                                          beta, use_beta, C, ldc, sC, batch, divA, divB, ep);
  TG_CASE(OP_N, OP_N) TG_CASE(OP_N, OP_T) TG_CASE(OP_T, OP_N) TG_CASE(OP_T, OP_T)
  if (IsC<TA>::v) { TG_CASE(OP_C, OP_N) TG_CASE(OP_C, OP_T) }
  if (IsC<TB>::v) { TG_CASE(OP_N, OP_C) TG_CASE(OP_T, OP_C) }
  if (IsC<TA>::v && IsC<TB>::v) { TG_CASE(OP_C, OP_C) }
#undef TG_CASE
  tg_set_error("mfma gemm: unsupported op combination");
  return TG_E_ARG;
}

}  // namespace

int mfma_gemm_zz(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const cplx* A, int lda, long long sA, const cplx* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch, int divA, int divB,
                 const GemmEpi& ep) {
  return dispatch<cplx, cplx>(variant, s, opa, opb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta,
                              use_beta, C, ldc, sC, batch, divA, divB, ep);
}

int mfma_gemm_dz(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const double* A, int lda, long long sA, const cplx* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch, int divA, int divB,
                 const GemmEpi& ep) {
  if (opa == OP_C) opa = OP_T;
  return dispatch<double, cplx>(variant, s, opa, opb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta,
                                use_beta, C, ldc, sC, batch, divA, divB, ep);
}

int mfma_gemm_zd(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const cplx* A, int lda, long long sA, const double* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch, int divA, int divB,
                 const GemmEpi& ep) {
  if (opb == OP_C) opb = OP_T;
  return dispatch<cplx, double>(variant, s, opa, opb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta,
                                use_beta, C, ldc, sC, batch, divA, divB, ep);
}

int mfma_gemm_grouped(int variant, hipStream_t s, int M, const cplx* X, cplx* C, int ld,
                      const void* W, const GroupDesc* groups_dev, const int* tile_group_dev,
                      const int* tile_j0_dev, int ntiles_total) {
  if (M <= 0 || ntiles_total <= 0) return TG_OK;
  GroupedArgs g{M, ld, X, C, W, groups_dev, tile_group_dev, tile_j0_dev, 1, 0};
  if (M <= TG_GROUPED_VEC) {
    const dim3 grid(ntiles_total), th(64 * GV_W);
    if (M == 1) hipLaunchKernelGGL(grouped_vec_kernel<1>, grid, th, 0, s, g);
    else if (M == 2) hipLaunchKernelGGL(grouped_vec_kernel<2>, grid, th, 0, s, g);
    else if (M == 3) hipLaunchKernelGGL(grouped_vec_kernel<3>, grid, th, 0, s, g);
    else hipLaunchKernelGGL(grouped_vec_kernel<4>, grid, th, 0, s, g);
    TG_HIP(hipGetLastError());
    return TG_OK;
  }
#define TG_GROUPED(TA, TJ, KS, OCC)                                                            \
  do {                                                                                         \
    g.mtiles = (M + 16 * TA - 1) / (16 * TA);                                                  \
    const long long units = (long long)(4 / TJ) * (ntiles_total / XCDS) * g.mtiles;            \
    if (units > 0x3fffffffLL) {                                                                \
      tg_set_error("mfma grouped gemm: grid too large");                                       \
      return TG_E_ARG;                                                                         \
    }                                                                                          \
    g.units = (int)units;                                                                      \
    hipLaunchKernelGGL((mfma_grouped_kernel<TA, TJ, KS, OCC>),                                 \
                       dim3((unsigned)((units + 3) / 4 * XCDS)), dim3(256), 0, s, g);          \
  } while (0)
  switch (variant) {
    case 0: TG_GROUPED(3, 2, 2, 3); break;
    case 1: TG_GROUPED(3, 2, 3, 2); break;
    case 2: TG_GROUPED(2, 2, 4, 3); break;
    case 3: TG_GROUPED(2, 2, 2, 4); break;
    case 4: TG_GROUPED(1, 2, 4, 4); break;
    default:
      tg_set_error("mfma grouped gemm: bad tile variant");
      return TG_E_ARG;
  }
#undef TG_GROUPED
  TG_HIP(hipGetLastError());
  return TG_OK;
}

int mfma_gemm_dd(hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, double alpha,
                 const double* A, int lda, long long sA, const double* B, int ldb, long long sB,
                 double beta, int use_beta, double* C, int ldc, long long sC, int batch, int divA,
                 int divB) {
  if (M <= 0 || N <= 0 || batch <= 0) return TG_OK;
  const long long tiles = (long long)((M + 15) / 16) * ((N + 15) / 16) * batch;
  // Both forms were timed at orders 24 to 336 with 1 to 512 matrices, K = the order and half
  // of it.  A^T B, both read down their columns: from 750 tiles (order 224, 3 matrices 13.0 with
  // registers, 12.4 through LDS, 4: 16.6, 12.5).  A B^T, both read along their rows: registers
  // are as good at any number (order 336, 64 matrices 424, 428) but for short products (order 64,
  // 64 matrices 5.0, 5.3; 128: 6.9, 6.0).  One of each: short ones from 1000 (order 80, 32: 6.0,
  // 6.6, 48: 7.1, 6.8), long ones, whose second round of workgroups costs more, from 2000 (order
  // 224, 8: 19, 25; 16: 35, 27).
  const bool tn = opa != OP_N && opb == OP_N, nt = opa == OP_N && opb != OP_N;
  const long long most = tn ? 750 : nt ? (K <= 64 ? 1000 : tiles) : (K <= 96 ? 1000 : 2000);
  const bool many = tiles > most;
  const int bt = many ? 32 : 16, tiles_m = (M + bt - 1) / bt, tiles_n = (N + bt - 1) / bt;
  const dim3 grid(tiles_m * tiles_n, batch);
#define TG_DD(OA, OB)                                                                              \
  if (many)                                                                                        \
    hipLaunchKernelGGL((mfma_dd_lds_kernel<OA, OB>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, \
                       sA, B, ldb, sB, beta, use_beta, C, ldc, sC, tiles_m, divA, divB);           \
  else                                                                                             \
    hipLaunchKernelGGL((mfma_dd_kernel<OA, OB>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, \
                       B, ldb, sB, beta, use_beta, C, ldc, sC, tiles_m, divA, divB)
  if (opa == OP_N && opb == OP_N) { TG_DD(OP_N, OP_N); }
  else if (opa == OP_N) { TG_DD(OP_N, OP_T); }
  else if (opb == OP_N) { TG_DD(OP_T, OP_N); }
  else { TG_DD(OP_T, OP_T); }
#undef TG_DD
  TG_HIP(hipGetLastError());
  return TG_OK;
}
