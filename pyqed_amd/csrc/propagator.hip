// Liouville-space RK4 of a constant generator by powers of its step matrix.
//
// With a generator that does not change, one RK4 step of pyqed/phys.py:1051-1063 is a fixed matrix,
//   v' = v + D v,   D = z + z^2/2 + z^3/6 + z^4/24,   z = A dt,
// and 2^j steps are v + D_j v with D_{j+1} = 2 D_j + D_j D_j.  The step-by-step kernel (liouville.hip) is a
// chain of 4 nsteps dependent matrix-vector products on one workgroup; here the states of all steps are the
// rows of matrix products: rows [2^j, 2^{j+1}) are rows [0, 2^j) advanced by D_j, and once kCap rows are
// there every further launch makes kCap rows at a time from the last ones.  A quarter of the flops (one
// product per step in place of four), about nsteps / kCap + 9 launches, and every CU has tiles to form.
//
// Accuracy is that of the stepping kernels or better: D is O(dt), so what rounds in a product enters v at O(dt) of
// an ulp, a state is reached through log2(kCap) + nsteps / kCap additions instead of nsteps, and the powers, whose
// errors repeat in every product, are formed to more than FP64 (matrix_task).  Error against an extended-precision
// run relative to the stepping kernels' (states, Frobenius norm; in brackets the largest element), 30 Lindblad systems
// of d = 2..16 and Redfield oscillators of d = 3..20 with 100..1000 steps: 0.53 (0.72) on geometric mean, at most
// 0.85 (1.7); populations of 12 small hierarchies (heom.hip) 0.24 (0.37), at most 0.61 (1.0).  Powers formed in
// FP64 had 2.2 to 2.4 (1.9 to 2.9) at N = 256.  Their cost in kernel time: 400 steps of N = 256 125 -> 220 us, of which
// 8 launches of 19 to 22 us form and square matrices (the FP64 matrix cores; 8 to 10 before), 1000 steps of N = 84
// 115 -> 145, of N = 64 100 -> 125.
//
// The entries of D_j for a mode that this dt makes unstable grow like |P|^(2^j).  Such a mode may belong to a coherence
// that the state never excites, as one with a far level that nothing couples to, and steps then leave it at exactly
// zero.  0 x Inf would be NaN, so a square's components are held within 2^1000 (kHold): zero stays zero, and a mode
// that is excited still overflows, in the rows.
//
// States are rows, so the matrices are kept transposed (G_j = D_j^T): v' = v + v G.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>

#include "liouville.h"

using namespace pqa;

namespace {

constexpr int kThreads = 256;
constexpr int kCap = 64;            // largest number of steps in one power
constexpr int kDeepN = 64;          // rows of more elements are summed in short pieces (launch_power)
constexpr double kHold = 0x1p1000;
constexpr int power_threads(int split) { return split == 8 ? 512 : 256; }
constexpr int64_t kTilesFull = 1024;  // wavefront tiles that give every SIMD of the chip one
constexpr int64_t kScratchBytes = int64_t(256) << 20;  // states kept when the caller keeps none

typedef double doublex4 __attribute__((ext_vector_type(4)));

// One launch: the row task (rows s_in .. s_in + cnt - 1 of every instance times G, added to themselves, into
// rows s + shift) in workgroups [0, row_blocks), then the matrix task (out = addc * add + X B, all N x N).
struct PwParams {
  int N, cnt, n_inst, row_blocks, tile0;  // tile0: first row tile of the launch
  int64_t s_in, shift;
  const double2* G;
  const double2* v0;  // row 0 of instance i at v0 + i N
  double2* V;         // row s >= 1 at V + i strideI + (s - 1) N
  int64_t strideI;
  // matrix task: every matrix in two parts, value and remainder
  const double2* X;
  const double2* Xlo;
  const double2* B;
  const double2* Blo;
  const double2* add;
  const double2* addlo;
  double2* out;
  double2* outlo;
  double2* w;         // set when X B = zt zt: also writes w = 1/2 + zt/6 + (X B)/24
  double2* wlo;
  double addc;
  bool hold;          // keep out within kHold
};

// a value and its remainder
struct Two {
  double h, l;
};

__device__ __forceinline__ Two two_sum(double a, double b) {
  const double s = a + b, z = s - a;
  return {s, (a - (s - z)) + (b - z)};
}
__device__ __forceinline__ Two add(Two a, Two b) {
  const Two s = two_sum(a.h, b.h);
  return two_sum(s.h, s.l + (a.l + b.l));
}
__device__ __forceinline__ Two div(Two a, double n) {
  const double q = a.h / n;
  return two_sum(q, (fma(-n, q, a.h) + a.l) / n);
}

// Adding and subtracting grid_magic(max) rounds a number of magnitude up to max to kSlice bits on one grid.
// 0 (no rounding: everything stays in the first slice, an ordinary product) where squares would leave the range.
constexpr int kSlice = 23;
__device__ __forceinline__ double grid_magic(double max) {
  const int e = (int)((__double_as_longlong(max) >> 52) & 0x7ff) - 1023;
  return e > 400 || e < -400 ? 0.0 : ldexp(1.5, 52 + e + 1 - kSlice);
}

__device__ __forceinline__ const double2* row_ptr(const PwParams& p, int64_t inst, int64_t s) {
  return s == 0 ? p.v0 + inst * p.N : p.V + inst * p.strideI + (s - 1) * p.N;
}

// The matrix task: a 16 x 16 tile per workgroup, its k-blocks dealt to the SPLIT wavefronts.
//
// A power is applied many times, so what rounding leaves in it adds up over a run instead of averaging out as the
// rounding of separate steps does.  The matrices are therefore formed to about 75 bits, value and remainder, and only
// the rows round them to FP64.  Per 16-deep k-block, a row of the left operand and a column of the right one are
// each split in two: xh, the nearest multiples of a grid kSlice bits below the largest of the 16, and xl, the rest
// with the remainders.  xh bh and its sum over the block are whole multiples of one number, below 2^53 of it, so FP64
// forms them exactly; xh bl and xl b, 2^-kSlice of it, go to a second sum.  A complex product is three real ones,
//   k1 = b.x (a.x + a.y), k2 = a.x (b.y - b.x), k3 = a.y (b.x + b.y):  a b = k1 - k3 + i (k1 + k2),
// nine FP64 products of the matrix cores in place of the four of an ordinary sum.
template <int SPLIT>
__device__ __forceinline__ void matrix_task(const PwParams& p, int blk, double2* red) {
  const int tid = threadIdx.x, lane = tid & 63, gi = lane & 15, gk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, ntc = (N + 15) / 16, nkb = ntc;
  const int tr = blk / ntc * 16, tc = (blk % ntc) * 16;
  const int r = tr + (tid >> 4), q = tc + (tid & 15), e = r * N + q;  // this thread's element
  const bool in = tid < 256 && r < N && q < N;
  const double2 zero = make_double2(0.0, 0.0);
  double2 o = zero, ol = zero;
  struct Frag {
    double2 a[4], al[4], b[4], bl[4];
  };
  const int ra = min(tr + gi, N - 1) * N, j = tc + gi;
  auto load = [&](int kb, Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = 16 * kb + 4 * c + gk;
      f.a[c] = k < N ? p.X[ra + k] : zero;
      f.al[c] = k < N ? p.Xlo[ra + k] : zero;
      f.b[c] = k < N && j < N ? p.B[k * N + j] : zero;
      f.bl[c] = k < N && j < N ? p.Blo[k * N + j] : zero;
    }
  };
  doublex4 sr = {0.0, 0.0, 0.0, 0.0}, si = sr, lr = sr, li = sr, l1 = sr, l2 = sr, l3 = sr;
  struct Three {  // the factors of k1, k2, k3
    double u, v, w;
  };
  auto left = [](double2 a) { return Three{a.x + a.y, a.x, a.y}; };
  auto right = [](double2 b) { return Three{b.x, b.y - b.x, b.x + b.y}; };
  auto mul = [](const Three& x, const Three& y, doublex4& k1, doublex4& k2, doublex4& k3) __attribute__((always_inline)) {
    k1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.u, y.u, k1, 0, 0, 0);
    k2 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.v, y.v, k2, 0, 0, 0);
    k3 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.w, y.w, k3, 0, 0, 0);
  };
  auto magic = [](const double2 (&x)[4]) __attribute__((always_inline)) {  // lanes of one gi hold its 16 elements
    double m = 0.0;
#pragma unroll
    for (int c = 0; c < 4; ++c) m = fmax(m, fmax(fabs(x[c].x), fabs(x[c].y)));
    m = fmax(m, __shfl_xor(m, 16, 64));
    return grid_magic(fmax(m, __shfl_xor(m, 32, 64)));
  };
  auto multiply = [&](const Frag& f) __attribute__((always_inline)) {
    const double ga = magic(f.a), gb = magic(f.b);
    doublex4 h1 = {0.0, 0.0, 0.0, 0.0}, h2 = h1, h3 = h1;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double2 a = f.a[c], b = f.b[c];
      const double2 ah = make_double2((a.x + ga) - ga, (a.y + ga) - ga), bh = make_double2((b.x + gb) - gb, (b.y + gb) - gb);
      const double2 al = make_double2((a.x - ah.x) + f.al[c].x, (a.y - ah.y) + f.al[c].y);
      const double2 bl = make_double2((b.x - bh.x) + f.bl[c].x, (b.y - bh.y) + f.bl[c].y);
      const Three xh = left(ah);
      mul(xh, right(bh), h1, h2, h3);
      mul(xh, right(bl), l1, l2, l3);
      mul(left(al), right(b), l1, l2, l3);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const Two x = two_sum(sr[c], h1[c] - h3[c]), y = two_sum(si[c], h1[c] + h2[c]);
      sr[c] = x.h;
      si[c] = y.h;
      lr[c] += x.l;
      li[c] += y.l;
    }
  };
  Frag f;
  int kb = wv;
  if (kb < nkb) load(kb, f);
  if (in && (p.w || p.add)) {  // the epilogue's operands, behind the first block's
    o = (p.w ? p.X : p.add)[e];
    ol = (p.w ? p.Xlo : p.addlo)[e];
  }
#pragma unroll 1
  while (kb < nkb) {
    multiply(f);
    kb += SPLIT;
    if (kb < nkb) load(kb, f);
  }
  double2* low = red + SPLIT * 256;
#pragma unroll
  for (int c = 0; c < 4; ++c) {  // register c of lane (gk, gi) holds element (4 c + gk, gi)
    red[wv * 256 + (4 * c + gk) * 16 + gi] = make_double2(sr[c], si[c]);
    low[wv * 256 + (4 * c + gk) * 16 + gi] = make_double2(lr[c] + (l1[c] - l3[c]), li[c] + (l1[c] + l2[c]));
  }
  __syncthreads();
  if (!in) return;
  Two x = {red[tid].x, low[tid].x}, y = {red[tid].y, low[tid].y};
#pragma unroll
  for (int s = 1; s < SPLIT; ++s) {
    x = add(x, Two{red[s * 256 + tid].x, low[s * 256 + tid].x});
    y = add(y, Two{red[s * 256 + tid].y, low[s * 256 + tid].y});
  }
  if (p.w) {
    Two wx = add(div(Two{o.x, ol.x}, 6.0), div(x, 24.0)), wy = add(div(Two{o.y, ol.y}, 6.0), div(y, 24.0));
    if (r == q) wx = add(Two{0.5, 0.0}, wx);
    p.w[e] = make_double2(wx.h, wy.h);
    p.wlo[e] = make_double2(wx.l, wy.l);
  } else {
    x = add(x, Two{p.addc * o.x, p.addc * ol.x});
    y = add(y, Two{p.addc * o.y, p.addc * ol.y});
    // a generator with a NaN or Inf makes all of the first power NaN: that has to stay
    if (p.hold && isfinite(o.x) && isfinite(o.y)) {
      if (!(fabs(x.h) < kHold)) x = Two{copysign(kHold, x.h), 0.0};
      if (!(fabs(y.h) < kHold)) y = Two{copysign(kHold, y.h), 0.0};
    }
  }
  p.out[e] = make_double2(x.h, y.h);
  p.outlo[e] = make_double2(x.l, y.l);
}

// The row task, tiles of 16 R x 16 R per wavefront on v_mfma_f64_16x16x4_f64 (four real products per complex one),
// operands read straight from memory (L2) in the MFMA layout, one 16-deep k-block ahead.
//   SPLIT 4, 8: a workgroup is one tile, its k-blocks dealt to as many wavefronts and summed through LDS in a
//            fixed order: small launches, where the chain length counts
//   SPLIT 1: a workgroup is four tiles; R = 2 halves the operand loads per product for launches that fill
//            the chip
// MAT: the workgroups from row_blocks on hold the matrix task's tiles.
// A wavefront sums every k-block from zero (SPLIT 8): see launch_power.
template <int R, int SPLIT, bool MAT>
__global__ __launch_bounds__(power_threads(SPLIT), R == 2 || MAT ? 2 : 4) void liouville_power_kernel(PwParams p) {
  static_assert(!MAT || SPLIT > 1, "the matrix task is one tile per workgroup");
  __shared__ double2 red[SPLIT > 1 ? (MAT ? 2 : 1) * SPLIT * 256 : 1];
  if constexpr (MAT) {
    if ((int)blockIdx.x >= p.row_blocks) {
      matrix_task<SPLIT>(p, (int)blockIdx.x - p.row_blocks, red);
      return;
    }
  }
  const int tid = threadIdx.x, lane = tid & 63, gi = lane & 15, gk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, ntc = (N + 16 * R - 1) / (16 * R);
  const int wt = p.tile0 + (SPLIT > 1 ? (int)blockIdx.x : (int)blockIdx.x * 4 + wv);
  const int nrow = p.cnt * p.n_inst;
  const int tr = wt / ntc * (16 * R), tc = (wt % ntc) * (16 * R);
  if (tr >= nrow) return;  // SPLIT 1: the tail of the last workgroup
  const double2* ap[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int r = min(tr + 16 * u + gi, nrow - 1), i = (int)((unsigned)r / (unsigned)p.cnt);
    ap[u] = row_ptr(p, i, p.s_in + (r - i * p.cnt));
  }
  struct Frag {
    double2 a[4][R], b[4][R];
  };
  auto load = [&](int kb, Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = 16 * kb + 4 * c + gk;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int j = tc + 16 * u + gi;
        f.a[c][u] = k < N ? ap[u][k] : make_double2(0.0, 0.0);
        f.b[c][u] = k < N && j < N ? p.G[(unsigned)(k * N + j)] : make_double2(0.0, 0.0);
      }
    }
  };
  doublex4 sr[R][R], si[R][R];
#pragma unroll
  for (int u = 0; u < R; ++u)
#pragma unroll
    for (int v = 0; v < R; ++v) sr[u][v] = si[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](const Frag& f) __attribute__((always_inline)) {
    if constexpr (SPLIT == 8) {
      doublex4 r = {0.0, 0.0, 0.0, 0.0}, i = r;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double2 a = f.a[c][0], b = f.b[c][0];
        r = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, r, 0, 0, 0);
        i = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, i, 0, 0, 0);
        r = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, r, 0, 0, 0);
        i = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, i, 0, 0, 0);
      }
      sr[0][0] += r;
      si[0][0] += i;
      return;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < R; ++u)
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const double2 a = f.a[c][u], b = f.b[c][v];
          sr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, sr[u][v], 0, 0, 0);
          si[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, si[u][v], 0, 0, 0);
          sr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, sr[u][v], 0, 0, 0);
          si[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, si[u][v], 0, 0, 0);
        }
  };
  const int nkb = (N + 15) / 16;
  {
    Frag f0, f1;
    int kb = SPLIT > 1 ? wv : 0;
    if (kb < nkb) load(kb, f0);
#pragma unroll 1
    while (kb < nkb) {
      if (kb + SPLIT < nkb) load(kb + SPLIT, f1);
      multiply(f0);
      kb += SPLIT;
      if (kb >= nkb) break;
      if (kb + SPLIT < nkb) load(kb + SPLIT, f0);
      multiply(f1);
      kb += SPLIT;
    }
  }
  // MFMA output: register r of lane (gk, gi) holds element (4 r + gk, gi) of its 16 x 16 tile
  auto finish = [&](int r, int j, double2 v) __attribute__((always_inline)) {
    if (r >= nrow || j >= N) return;
    const int i = (int)((unsigned)r / (unsigned)p.cnt);
    const int64_t s = p.s_in + (r - i * p.cnt);
    const double2 x = row_ptr(p, i, s)[j];
    p.V[i * p.strideI + (s + p.shift - 1) * N + j] = make_double2(x.x + v.x, x.y + v.y);
  };
  if constexpr (SPLIT > 1) {
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv * 256 + (4 * r + gk) * 16 + gi] = make_double2(sr[0][0][r], si[0][0][r]);
    __syncthreads();
    if (tid >= 256) return;
    double2 v = red[tid];
#pragma unroll
    for (int s = 1; s < SPLIT; ++s) {
      v.x += red[s * 256 + tid].x;
      v.y += red[s * 256 + tid].y;
    }
    finish(tr + (tid >> 4), tc + (tid & 15), v);
  } else {
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int v = 0; v < R; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          finish(tr + 16 * u + 4 * r + gk, tc + 16 * v + gi, make_double2(sr[u][v][r], si[u][v][r]));
  }
}

// zt = dt A^T, value and remainder
__global__ __launch_bounds__(kThreads) void liouville_step_kernel(int N, const double2* A, double dt, double2* zt, double2* ztlo) {
  __shared__ double2 t[16][17];
  const int nt = (N + 15) / 16, bi = blockIdx.x / nt * 16, bj = blockIdx.x % nt * 16;
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  if (bi + r < N && bj + c < N) t[r][c] = A[(int64_t)(bi + r) * N + bj + c];
  __syncthreads();
  if (bj + r < N && bi + c < N) {
    const double2 a = t[c][r], z = make_double2(dt * a.x, dt * a.y);
    const int64_t e = (int64_t)(bj + r) * N + bi + c;
    zt[e] = z;
    ztlo[e] = make_double2(fma(dt, a.x, -z.x), fma(dt, a.y, -z.y));
  }
}

// observables of rows s = s0 .. s0 + cnt - 1 of every instance, gsz lanes (a power of two, at most 64) to a
// row: Tr(O rho) = sum_e obs[o][e] v[e]; row s goes to obs_out row t0 + s
__global__ __launch_bounds__(kThreads) void liouville_observe_kernel(PwParams p, int gsz, int n_obs, const double2* obs,
                                                                     double2* obs_out, int64_t out_rows, int64_t t0) {
  const int li = threadIdx.x % gsz;
  const int64_t per = kThreads / gsz, nr = (int64_t)p.cnt * p.n_inst;
  for (int64_t r0 = blockIdx.x * per; r0 < nr; r0 += gridDim.x * per) {  // the same trips for every lane
    const int64_t r = r0 + threadIdx.x / gsz;
    const bool live = r < nr;
    const int64_t i = live ? r / p.cnt : 0, s = live ? p.s_in + (r - i * p.cnt) : p.s_in;
    const double2* v = row_ptr(p, i, s);
    for (int o = 0; o < n_obs; ++o) {
      double re = 0.0, im = 0.0;
      for (int e = li; e < p.N; e += gsz) {
        const double2 a = obs[(int64_t)o * p.N + e], x = v[e];
        re += a.x * x.x - a.y * x.y;
        im += a.x * x.y + a.y * x.x;
      }
      for (int w = gsz / 2; w > 0; w >>= 1) {
        re += __shfl_xor(re, w, gsz);
        im += __shfl_xor(im, w, gsz);
      }
      if (live && li == 0) obs_out[(i * out_rows + t0 + s) * n_obs + o] = make_double2(re, im);
    }
  }
}

// row s of every instance into out [n_inst][N]
__global__ __launch_bounds__(kThreads) void liouville_row_kernel(PwParams p, int64_t s, double2* out) {
  for (int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x; e < (int64_t)p.n_inst * p.N; e += (int64_t)gridDim.x * kThreads) {
    const int64_t i = e / p.N;
    out[e] = row_ptr(p, i, s)[e - i * p.N];
  }
}

// the first n elements of the rows after every `every` steps, to out + slot stride (one instance)
struct Pick {
  double2* out;
  int n;
  int64_t stride, every;
};

__global__ __launch_bounds__(64) void liouville_pick_kernel(PwParams p, Pick k, int64_t t0, int64_t slot0) {
  const int64_t slot = slot0 + blockIdx.x, s = (slot + 1) * k.every - t0;  // row of the slot's step
  const double2* v = row_ptr(p, 0, s);
  for (int e = threadIdx.x; e < k.n; e += 64) k.out[slot * k.stride + e] = v[e];
}

struct Shape {
  int levels;       // powers kept: 1, 2, .. 2^(levels - 1) steps
  int64_t seg;      // states kept at a time (rows 1..seg) in the workspace; 0: in the caller's rho_out
  int64_t bytes;
};

// Is a run served here, and what does it need?  The power path pays for forming and squaring N x N matrices
// (about 8 times 3 products of N^3) and for a dozen launches, 60 to 70 us in all up to N = 64.  us, stepping against
// powers (one instance, every state kept): N = 4, 72 steps 67 / 74, 96 steps 86 / 71; N = 9, 40 steps 55 / 63, 56 steps
// 71 / 70; N = 16, 24 steps 47 / 62, 40 steps 69 / 67; N = 25, 8 steps 49 / 52, 12 steps 66 / 59 (64 instances 66 / 64);
// N = 36, 8 steps 60 / 52 (59 / 61); N = 64, 4 steps 76 / 45; N = 256, 4 steps 457 / 100; N = 1024, 4 steps 7484 / 2875.
bool power_shape(int N, int n_inst, int64_t nsteps, int n_obs, bool have_out, int64_t save_every, Shape* s) {
  if (nsteps < (N <= 4 ? 80 : N <= 9 ? 56 : N <= 16 ? 40 : N < 36 ? 14 : N < 64 ? 10 : 4)) return false;
  if (have_out && save_every != 1) return false;
  const bool traj = have_out || n_obs > 0;
  s->seg = 0;
  if (traj && !have_out)
    s->seg = std::max<int64_t>(1, std::min<int64_t>(nsteps, kScratchBytes / ((int64_t)n_inst * N * 16)));
  const int64_t span = traj ? (have_out ? nsteps : s->seg) : nsteps;  // rows, or steps, a power may cover
  s->levels = 1;
  while ((int64_t(1) << s->levels) <= std::min<int64_t>(span, kCap)) ++s->levels;
  const int64_t rows = traj ? (int64_t)n_inst * s->seg : n_inst;
  s->bytes = 16 * (power_matrix_elems(N, s->levels) + rows * N);
  // rows of a launch and its grid in 32 bits
  return (int64_t)n_inst * kCap * ((N + 15) / 16) < INT32_MAX / 2;
}

template <int R, int SPLIT, bool MAT>
int launch_form(PwParams p, int64_t row_tiles, int64_t mat_tiles, hipStream_t st) {
  constexpr int per = SPLIT > 1 ? 1 : 4;  // tiles of a workgroup
  p.row_blocks = (int)((row_tiles + per - 1) / per);
  hipLaunchKernelGGL((liouville_power_kernel<R, SPLIT, MAT>), dim3((unsigned)(p.row_blocks + mat_tiles)), dim3(power_threads(SPLIT)), 0,
                     st, p);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

// Rows of more than kDeepN elements are summed block by block over eight wavefronts.  Error of a run relative to the
// stepping kernels' with one sum per wavefront, of four: N = 100 0.4 to 0.7, 144 0.9, 256 1.0 to 1.3, 400 1.1; block by
// block 0.3 to 0.55, 0.7, 0.7 to 0.85, 0.8.  A launch for 64 rows of N = 256 takes 5.9 us (7.1), of N = 84 4.5 (4.4).
int launch_power(PwParams p, bool rows, bool mat, hipStream_t st) {
  const int64_t nrow = rows ? (int64_t)p.cnt * p.n_inst : 0;
  const int64_t c16 = (p.N + 15) / 16, c32 = (p.N + 31) / 32;
  const int64_t r16 = (nrow + 15) / 16 * c16, m16 = mat ? c16 * c16 : 0, r32 = (nrow + 31) / 32 * c32;
  const bool deep = p.N > kDeepN;
  const bool wide = !deep && p.N > 16 && r32 >= kTilesFull, many = !deep && p.N <= 32 && r16 >= kTilesFull;
  int rc = PYQED_OK;
  if (mat) {  // with the rows where they leave room
    const bool with = rows && r16 < kTilesFull;
    rc = deep ? launch_form<1, 8, true>(p, with ? r16 : 0, m16, st) : launch_form<1, 4, true>(p, with ? r16 : 0, m16, st);
    if (rc || with) return rc;
  }
  if (!rows) return rc;
  if (wide) return launch_form<2, 1, false>(p, r32, 0, st);
  if (many) return launch_form<1, 1, false>(p, r16, 0, st);
  constexpr int64_t kGrid = int64_t(1) << 22;  // workgroups of a launch: its threads in 32 bits
  for (int64_t t = 0; t < r16 && !rc; t += kGrid) {
    p.tile0 = (int)t;
    const int64_t n = std::min(kGrid, r16 - t);
    rc = deep ? launch_form<1, 8, false>(p, n, 0, st) : launch_form<1, 4, false>(p, n, 0, st);
  }
  return rc;
}

int run_power(int N, const double2* A, int n_inst, double2* rho, int64_t nsteps, double dt, int n_obs, const double2* obs,
              double2* obs_out, double2* rho_out, const Shape& sh, double2* work, hipStream_t st, const Pick* pick = nullptr) {
  const int64_t NN = (int64_t)N * N;
  double2* zt = work;
  double2* z2 = zt + NN;
  double2* w = z2 + NN;
  double2* z2lo = w + NN;
  double2* wlo = z2lo + NN;
  double2* lo[2] = {wlo + NN, wlo + 2 * NN};  // remainders of zt and, in turn, of the powers
  double2* G = wlo + 3 * NN;                  // [levels][N][N]
  double2* V = work + power_matrix_elems(N, sh.levels);
  int rc;
  PwParams p;
  std::memset(&p, 0, sizeof(p));
  p.N = N;
  p.n_inst = n_inst;
  p.cnt = 1;
  p.v0 = rho;
  const int nt = (N + 15) / 16;
  hipLaunchKernelGGL(liouville_step_kernel, dim3(nt * nt), dim3(kThreads), 0, st, N, A, dt, zt, lo[0]);
  PQA_HIP(hipGetLastError());
  p.X = p.B = zt;
  p.Xlo = p.Blo = lo[0];
  p.out = z2;
  p.outlo = z2lo;
  p.w = w;
  p.wlo = wlo;
  if ((rc = launch_power(p, false, true, st))) return rc;
  // G_0 = z + z^2 (1/2 + z/6 + z^2/24)
  p.X = z2;
  p.Xlo = z2lo;
  p.B = w;
  p.Blo = wlo;
  p.w = nullptr;
  p.add = zt;
  p.addlo = lo[0];
  p.addc = 1.0;
  p.out = G;
  p.outlo = lo[1];
  if ((rc = launch_power(p, false, true, st))) return rc;
  p.addc = 2.0;
  p.hold = true;
  // the launch that squares power j into power j + 1 also advances rows by power j
  auto level = [&](int j, bool rows, bool square) {
    p.G = G + j * NN;
    p.X = p.B = p.add = p.G;
    p.Xlo = p.Blo = p.addlo = lo[(j + 1) & 1];
    p.out = G + (j + 1) * NN;
    p.outlo = lo[j & 1];
    return launch_power(p, rows, square, st);
  };
  if (!rho_out && n_obs == 0 && !pick) {
    // final states only: nsteps = top * (most significant power) + remaining bits
    const int top = sh.levels - 1;
    double2* bufs[2] = {rho, V};
    int cur = 0;
    p.s_in = 0;
    p.shift = 1;
    p.strideI = N;
    auto step = [&](int j, bool rows, bool square) {
      p.v0 = bufs[cur];
      p.V = bufs[cur ^ 1];
      if (rows) cur ^= 1;
      return level(j, rows, square);
    };
    for (int j = 0; j < top; ++j)
      if ((rc = step(j, (nsteps >> j) & 1, true))) return rc;
    for (int64_t k = nsteps >> top; k > 0; --k)
      if ((rc = step(top, true, false))) return rc;
    if (cur) {
      p.v0 = V;
      hipLaunchKernelGGL(liouville_row_kernel, dim3((unsigned)std::min<int64_t>(((int64_t)n_inst * N + kThreads - 1) / kThreads, 2048)),
                         dim3(kThreads), 0, st, p, 0, rho);
      PQA_HIP(hipGetLastError());
    }
    return PYQED_OK;
  }
  const int64_t seg = rho_out ? nsteps : sh.seg;
  int gsz = 1;
  while (gsz < N && gsz < 64) gsz *= 2;
  int have_pow = 1;  // powers formed so far
  for (int64_t t0 = 0; t0 < nsteps; t0 += seg) {
    const int64_t S = std::min(seg, nsteps - t0);
    p.V = rho_out ? rho_out : V;
    p.strideI = (rho_out ? nsteps : seg) * N;
    int64_t have = 1;  // rows 0 .. have - 1 are in place
    for (int j = 0; have < S + 1;) {
      const int64_t step = int64_t(1) << j;  // have = step while doubling; then the last step rows advance
      const int64_t cnt = std::min(step, S + 1 - have);
      p.cnt = (int)cnt;
      p.s_in = have - step;
      p.shift = step;
      const bool up = j + 1 < sh.levels && have + cnt < S + 1;
      const bool square = up && j + 1 >= have_pow;
      if ((rc = level(j, true, square))) return rc;
      if (square) have_pow = j + 2;
      if (up) ++j;
      have += cnt;
    }
    p.s_in = t0 == 0 ? 0 : 1;
    if (n_obs) {
      p.cnt = (int)(S + 1 - p.s_in);
      const int64_t per = kThreads / gsz, nr = (int64_t)p.cnt * n_inst;
      hipLaunchKernelGGL(liouville_observe_kernel, dim3((unsigned)std::min<int64_t>((nr + per - 1) / per, 1 << 20)), dim3(kThreads), 0, st, p,
                         gsz, n_obs, obs, obs_out, nsteps + 1, t0);
      PQA_HIP(hipGetLastError());
    }
    if (pick && (t0 + S) / pick->every > t0 / pick->every) {
      const int64_t slot0 = t0 / pick->every;
      hipLaunchKernelGGL(liouville_pick_kernel, dim3((unsigned)((t0 + S) / pick->every - slot0)), dim3(64), 0, st, p, *pick, t0, slot0);
      PQA_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(liouville_row_kernel, dim3((unsigned)std::min<int64_t>(((int64_t)n_inst * N + kThreads - 1) / kThreads, 2048)),
                       dim3(kThreads), 0, st, p, S, rho);
    PQA_HIP(hipGetLastError());
  }
  return PYQED_OK;
}

// rho_k <- V rho_k V^dagger for a run of d x d matrices: a block per matrix, the three factors in LDS.  Bound by
// the states' own bytes; the caller's copy of them to the host is longer (400 states of 16 x 16, 1.6 MB: on the host
// the two products took 1.2 ms of a 1.7 ms call, here 9 us).
constexpr int kBasisD = 32, kBasisThreads = 256;

__global__ __launch_bounds__(kBasisThreads) void basis_change_kernel(int d, int64_t n, const double2* V, double2* rho) {
  __shared__ double2 sV[kBasisD * kBasisD], sR[kBasisD * kBasisD], sT[kBasisD * kBasisD];
  const int d2 = d * d;
  for (int e = threadIdx.x; e < d2; e += kBasisThreads) sV[e] = V[e];
  for (int64_t k = blockIdx.x; k < n; k += gridDim.x) {
    for (int e = threadIdx.x; e < d2; e += kBasisThreads) sR[e] = rho[k * d2 + e];
    __syncthreads();
    for (int e = threadIdx.x; e < d2; e += kBasisThreads) {
      const int i = e / d, j = e - i * d;
      double2 t = make_double2(0, 0);
      for (int q = 0; q < d; ++q) {
        const double2 a = sV[i * d + q], b = sR[q * d + j];
        t.x += a.x * b.x - a.y * b.y;
        t.y += a.x * b.y + a.y * b.x;
      }
      sT[e] = t;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < d2; e += kBasisThreads) {
      const int i = e / d, j = e - i * d;
      double2 t = make_double2(0, 0);
      for (int q = 0; q < d; ++q) {
        const double2 a = sT[i * d + q], b = sV[j * d + q];
        t.x += a.x * b.x + a.y * b.y;
        t.y += a.y * b.x - a.x * b.y;
      }
      rho[k * d2 + e] = t;
    }
    __syncthreads();  // sR and sT are free for the next matrix
  }
}

}  // namespace

namespace pqa {

int power_vector(int N, const double2* A, double2* v, int64_t nsteps, double dt, double2* out, int n_out, int64_t out_stride,
                 int64_t every, void* work, hipStream_t st) {
  Shape s;
  s.seg = std::min(nsteps, kRowSeg);
  s.levels = 1;
  while ((int64_t(1) << s.levels) <= std::min<int64_t>(out ? s.seg : nsteps, kCap)) ++s.levels;
  s.bytes = 0;
  const Pick k{out, n_out, out_stride, every};
  return run_power(N, A, 1, v, nsteps, dt, 0, nullptr, nullptr, nullptr, s, (double2*)work, st, out ? &k : nullptr);
}

}  // namespace pqa

extern "C" int pyqed_liouville_work_bytes(int32_t N, int32_t nterm, int32_t n_inst, int64_t nsteps, int32_t n_obs, int32_t keep_states,
                                          int64_t save_every, int64_t* bytes) {
  if (!bytes || N < 1 || N > 1024 || nterm < 1 || n_inst < 1 || nsteps < 0 || n_obs < 0)
    return fail(PYQED_EINVAL, "liouville_work_bytes: need 1 <= N <= 1024, nterm >= 1, n_inst >= 1, nsteps >= 0, n_obs >= 0");
  Shape s;
  if (nterm == 1 && power_shape(N, n_inst, nsteps, n_obs, keep_states != 0, save_every > 0 ? save_every : 1, &s)) {
    *bytes = s.bytes;
    return PYQED_OK;
  }
  const int64_t seg = small_fits(N, nterm, false) ? small_split(N, nterm, n_inst, nsteps, false) : 0;
  *bytes = seg ? small_split_bytes(N, nterm, n_inst, nsteps, seg, false) : 0;
  return PYQED_OK;
}

extern "C" int pyqed_liouville_run_work(int32_t N, int32_t nterm, const void* A, int32_t n_inst, void* rho, const double* field,
                                        int64_t nsteps, double dt, int32_t n_obs, const void* obs, void* obs_out, void* rho_out,
                                        int64_t save_every, void* work, int64_t work_bytes, void* stream) {
  Shape s;
  if (save_every <= 0) save_every = 1;
  const bool ok = N >= 1 && N <= 1024 && nterm >= 1 && n_inst >= 1 && A && rho && n_obs >= 0 &&
                  (n_obs == 0 || (obs && obs_out)) && nsteps >= 0 && (nterm == 1 || field) && work;
  if (!ok || nterm > 1 || !power_shape(N, n_inst, nsteps, n_obs, rho_out != nullptr, save_every, &s)) {
    const int64_t seg = ok && small_fits(N, nterm, false) ? small_split(N, nterm, n_inst, nsteps, false) : 0;
    if (seg && work_bytes >= small_split_bytes(N, nterm, n_inst, nsteps, seg, false)) {
      LiouvilleRun r = forward_run(N, nterm, A, n_inst, rho, field, nsteps, dt, n_obs, obs, obs_out, rho_out, save_every);
      r.seg = seg;
      return small_forward_split(r, work, (hipStream_t)stream);
    }
    return pyqed_liouville_run(N, nterm, A, n_inst, rho, field, nsteps, dt, n_obs, obs, obs_out, rho_out, save_every, stream);
  }
  if (work_bytes < s.bytes)
    return fail(PYQED_EINVAL, "liouville_run_work: workspace of " + std::to_string(work_bytes) + " bytes < " + std::to_string(s.bytes));
  return run_power(N, (const double2*)A, n_inst, (double2*)rho, nsteps, dt, n_obs, (const double2*)obs, (double2*)obs_out, (double2*)rho_out,
                   s, (double2*)work, (hipStream_t)stream);
}

extern "C" int pyqed_basis_change(int32_t d, int64_t n, const void* V, void* rho, void* stream) {
  if (d < 1 || d > kBasisD || n < 0 || !V || !rho) return fail(PYQED_EINVAL, "basis_change: need 1 <= d <= 32, n >= 0, V and rho");
  if (n == 0) return PYQED_OK;
  hipLaunchKernelGGL(basis_change_kernel, dim3((unsigned)std::min<int64_t>(n, 65535)), dim3(kBasisThreads), 0, (hipStream_t)stream, d, n,
                     (const double2*)V, (double2*)rho);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}
