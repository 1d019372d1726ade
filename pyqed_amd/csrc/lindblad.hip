// Lindblad master equation in matrix form, for any d (the Liouville-space kernel of liouville.hip
// holds vec(rho) and its N x N generator and serves N = d*d <= 1024):
//
//   d rho/dt = -i (Hs rho - rho Hs^dag) + sum_k c_k (rho c_k^dag),
//   Hs = Heff - sum_i f_i(step) H_i,   Heff = H0 - (i/2) sum_k c_k^dag c_k  (formed on the host),
//
// which is the reference's liouvillian (pyqed/oqs.py:697-714: -i[H, rho] + sum_k c rho c^dag
// - 1/2 {c^dag c, rho}) with the anticommutators folded into one effective Hamiltonian, stepped by
// the RK4 of pyqed/phys.py:1051-1063 in its summation order, with the drive held constant over a
// step as _lindblad_driven (oqs.py:1699-1806) evaluates it.
//
// Each RK4 stage is two launches over every instance: the products T_k = X c_k^dag, then the
// right-hand side -i H X + i X H^dag + sum_k c_k T_k with the RK4 update as its epilogue.  The output
// is cut into tiles held by single wavefronts, so one instance of d = 96 already spreads over 36
// workgroups and a large batch fills the chip; state, stage inputs and T pass through L2 / MALL.
//
// Complex FP64 products run on v_mfma_f64_16x16x4_f64 (four real products per complex one), operands
// read straight from memory in the MFMA layout, one 16-deep k-block ahead of the one being multiplied.
// The operators (H, c_k) are the same for every step and usually sparse in blocks (ladder, number and
// local operators), so a bit table made once per call marks the 16 x 16 operator blocks that hold a
// nonzero real or imaginary part; blocks, and the real products of a part, that are exactly zero are
// skipped.  A non-finite value anywhere in the inputs marks every block, so that it spreads as in the
// full product; one that a run makes on its way spreads through the marked blocks only.
//
// Measured (MI355X) against one workgroup per instance with 4 x 4 register blocks on the vector ALU, which
// left 255 CUs idle for a single instance and was bound by its LDS reads otherwise: a step of one dense
// d = 128 instance with two collapse operators 3255 -> 114 us, of one d = 96 cavity 2330 -> 42 us (about
// 5 us per launch, latency), of 256 d = 64 cavities 565 -> 180 us, of 256 dense d = 64 instances
// 830 -> 656 us (the operand loads: one wavefront per SIMD).

#include <algorithm>
#include <cstring>

#include "common.h"

namespace pqa {
namespace {

constexpr int kLThreads = 256;
constexpr int64_t kFullChip = 256;  // CUs: workgroups from which a launch fills the chip
constexpr int64_t kGridBlocks = (int64_t(1) << 32) / kLThreads - 1;  // a grid's threads are counted in 32 bits
constexpr int kScanBlocks = 64;  // workgroups of the non-finite scan

typedef double doublex4 __attribute__((ext_vector_type(4)));

struct LbParams {
  int d, nc, ndrive, n_obs;
  int nt, nw;       // 16-wide tiles per dimension, 32-bit words per tile row of a block table
  int n_inst, inst0;  // instances of this launch and the first one's index
  int stage;
  int64_t nsteps, save_every, ws_stride, step;
  double dt;
  const double2* Heff;   // [d*d]
  const double2* HeffD;  // [d*d] Heff^dag
  const double2* C;      // [nc][d*d]
  const double2* CD;     // [nc][d*d] c_k^dag
  const double2* Hd;     // [ndrive][d*d] drive operators
  const double2* HdD;    // [ndrive][d*d] their adjoints
  const double* field;   // [n_inst][nsteps][ndrive]
  double2* rho;          // [n_inst][d*d], advanced in place
  const double2* obs;    // [n_obs][d*d], O^T flattened: Tr(O rho) = sum_e obs[e] rho[e]
  double2* obs_out;      // [n_inst][nsteps+1][n_obs]
  double2* rho_out;      // [n_inst][nsteps/save_every][d*d] or NULL
  double2* ws;           // per instance (ws_stride elements): X0, X1, acc, T[nc], Hs, HsD
  // Nonzero blocks, (real, imaginary) bits: operators that multiply from the left, tab[op][row tile][word]
  // with a bit per column block, op = 0..nc-1 for C_k, nc for H; then operators that multiply from the
  // right, tab[nc + 1 + op][column tile][word] with a bit per row block.  NULL: every block counts.
  uint2* tab;
  int* flags;            // [kScanBlocks]: a workgroup of the scan met a non-finite value
  int gemm_blocks;       // workgroups that hold output tiles; the rest observe and form Hs (phase 1, stage 0)
  int side_blocks;       // per instance: observables, then parts of Hs
};

__device__ __forceinline__ double2 cmul2(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// sum over the block of one value per thread (result valid in thread 0)
__device__ __forceinline__ double2 block_sum(double2 v, double2* red) {
  __syncthreads();
  red[threadIdx.x] = v;
  __syncthreads();
  for (int h = kLThreads / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      red[threadIdx.x].x += red[threadIdx.x + h].x;
      red[threadIdx.x].y += red[threadIdx.x + h].y;
    }
    __syncthreads();
  }
  return red[0];
}

// ------------------------------------------------------------------ once per call: block tables
__device__ __forceinline__ bool finite2(double2 v) { return isfinite(v.x) && isfinite(v.y); }

// Does any input hold a NaN or Inf?  One flag per workgroup, written whole (no clearing pass).
__global__ __launch_bounds__(kLThreads) void lindblad_scan_kernel(LbParams p) {
  const int64_t d2 = (int64_t)p.d * p.d, at = blockIdx.x * (int64_t)kLThreads + threadIdx.x;
  constexpr int64_t step = (int64_t)kScanBlocks * kLThreads;
  bool bad = false;
  auto scan = [&](const double2* v, int64_t n) {
    for (int64_t e = at; e < n; e += step) bad = bad || !finite2(v[e]);
  };
  scan(p.rho, p.n_inst * d2);
  scan(p.Heff, d2);
  scan(p.HeffD, d2);
  scan(p.C, p.nc * d2);
  scan(p.CD, p.nc * d2);
  scan(p.Hd, p.ndrive * d2);
  scan(p.HdD, p.ndrive * d2);
  for (int64_t e = at; e < p.n_inst * p.nsteps * p.ndrive; e += step) bad = bad || !isfinite(p.field[e]);
  const int any = __syncthreads_or(bad ? 1 : 0);
  if (threadIdx.x == 0) p.flags[blockIdx.x] = any;
}

// Workgroup o nt + t (tile t of the table's operator row o): one bit per 16 x 16 block along the contraction.
__global__ __launch_bounds__(kLThreads) void lindblad_table_kernel(LbParams p) {
  extern __shared__ uint32_t words[];  // [2 nw]
  const int t = blockIdx.x % p.nt, o = blockIdx.x / p.nt, lane = threadIdx.x & 63, d = p.d;
  const bool right = o > p.nc;
  const int op = right ? o - p.nc - 1 : o;
  const int64_t d2 = (int64_t)d * d;
  for (int e = threadIdx.x; e < 2 * p.nw; e += kLThreads) words[e] = 0;
  const int bad = __syncthreads_or((int)threadIdx.x < kScanBlocks ? p.flags[threadIdx.x] : 0);
  for (int kb = threadIdx.x >> 6; kb < p.nt; kb += kLThreads / 64) {
    bool re = false, im = false;
    for (int q = 0; q < 4; ++q) {
      const int a = 4 * q + (lane >> 4), b = lane & 15;  // row, column within the block
      const int i = 16 * (right ? kb : t) + a, j = 16 * (right ? t : kb) + b;
      if (i < d && j < d) {
        const int64_t e = (int64_t)i * d + j;
        auto take = [&](double2 v) {
          re = re || v.x != 0.0;
          im = im || v.y != 0.0;
        };
        if (op < p.nc) {
          take((right ? p.CD : p.C)[op * d2 + e]);
        } else {
          take((right ? p.HeffD : p.Heff)[e]);
          for (int k = 0; k < p.ndrive; ++k) take((right ? p.HdD : p.Hd)[k * d2 + e]);
        }
      }
    }
    const bool r = __ballot(re) != 0 || bad, m = __ballot(im) != 0 || bad;
    if (lane == 0) {
      if (r) atomicOr(&words[2 * (kb >> 5)], 1u << (kb & 31));
      if (m) atomicOr(&words[2 * (kb >> 5) + 1], 1u << (kb & 31));
    }
  }
  __syncthreads();
  for (int w = threadIdx.x; w < p.nw; w += kLThreads)
    p.tab[((int64_t)o * p.nt + t) * p.nw + w] = make_uint2(words[2 * w], words[2 * w + 1]);
}

// ------------------------------------------------------------------ side work of a step's first launch
// Observables of the state before the step, and Hs, Hs^dag of a driven step: both read or write what no
// product of that launch touches, so they ride along as extra workgroups instead of taking launches.
__device__ __forceinline__ void side_work(const LbParams& p, int64_t inst, int part, double2* red) {
  const int64_t d2 = (int64_t)p.d * p.d;
  if (part < p.n_obs) {
    const double2* y = p.rho + inst * d2;
    const double2* O = p.obs + part * d2;
    double2 s = make_double2(0.0, 0.0);
#pragma unroll 4
    for (int64_t e = threadIdx.x; e < d2; e += kLThreads) {
      const double2 v = cmul2(O[e], y[e]);
      s.x += v.x;
      s.y += v.y;
    }
    const double2 t = block_sum(s, red);
    if (threadIdx.x == 0) p.obs_out[(inst * (p.nsteps + 1) + p.step) * p.n_obs + part] = t;
    return;
  }
  const int nhs = p.side_blocks - p.n_obs;
  double2* Hs = p.ws + inst * p.ws_stride + (3 + p.nc) * d2;
  const double* f = p.field + (inst * p.nsteps + p.step) * p.ndrive;
#pragma unroll 1
  for (int64_t e = (int64_t)(part - p.n_obs) * kLThreads + threadIdx.x; e < d2; e += (int64_t)nhs * kLThreads) {
    double2 h = p.Heff[e], hd = p.HeffD[e];
    for (int i = 0; i < p.ndrive; ++i) {
      const double2 a = p.Hd[i * d2 + e], b = p.HdD[i * d2 + e];
      h.x -= f[i] * a.x;
      h.y -= f[i] * a.y;
      hd.x -= f[i] * b.x;
      hd.y -= f[i] * b.y;
    }
    Hs[e] = h;
    Hs[d2 + e] = hd;
  }
}

__global__ __launch_bounds__(kLThreads) void lindblad_observe_kernel(LbParams p) {
  __shared__ double2 red[kLThreads];
  const int64_t b = blockIdx.x;
  side_work(p, p.inst0 + b / p.n_obs, (int)(b % p.n_obs), red);
}

// ------------------------------------------------------------------ products
// A product of the phase: left factor A, right factor B, which of them is the operator, and the
// operator's factor: 0 as it is, 1 times -i, 2 times +i.
struct Prod {
  const double2* A;
  const double2* B;
  const uint2* tab;  // the operator's table row of tile 0
  bool left;
  int scale;
};

template <int PHASE>
__device__ __forceinline__ Prod product(const LbParams& p, const double2* in, const double2* ws, int q, int k) {
  const int64_t d2 = (int64_t)p.d * p.d;
  const int64_t row = (int64_t)p.nt * p.nw;
  if (PHASE == 1) return {in, p.CD + k * d2, p.tab + (p.nc + 1 + k) * row, false, 0};
  const double2* Hs = ws + (3 + p.nc) * d2;
  if (q == 0) return {p.ndrive ? Hs : p.Heff, in, p.tab + p.nc * row, true, 1};
  if (q == 1) return {in, p.ndrive ? Hs + d2 : p.HeffD, p.tab + (2 * p.nc + 1) * row, false, 2};
  return {p.C + (q - 2) * d2, ws + (3 + (q - 2)) * d2, p.tab + (q - 2) * row, true, 0};
}

// A k-block of one product for this wavefront's tile: the operator's nonzero parts per 16-wide subtile
// (bit u) and the product it belongs to.
struct Blk {
  Prod pr;
  int kb;
  uint32_t re, im;
  bool valid;
};

// Walk over the nonzero k-blocks of the phase's products, one table word (32 blocks) at a time.
template <int PHASE, int R>
struct Walk {
  Prod pr;
  int q, w, turn;
  uint32_t bits, wre[R], wim[R];

  __device__ __forceinline__ void start(const LbParams& p, const double2* in, const double2* ws, int kop, int tr, int tc,
                                        int wv) {
    q = 0;
    w = 0;
    turn = 0;
    pr = product<PHASE>(p, in, ws, 0, kop);
    read(p, tr, tc);
  }
  __device__ __forceinline__ void read(const LbParams& p, int tr, int tc) {
    bits = 0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int t = (pr.left ? tr : tc) + u;
      uint2 v = make_uint2(0, 0);
      if (t < p.nt) {
        const uint32_t all = p.nt - 32 * w < 32 ? (1u << (p.nt - 32 * w)) - 1u : ~0u;
        v = p.tab ? pr.tab[(int64_t)t * p.nw + w] : make_uint2(all, all);
      }
      const uint32_t x = __builtin_amdgcn_readfirstlane(v.x), z = __builtin_amdgcn_readfirstlane(v.y);
      wre[u] = pr.scale ? z : x;  // +-i times the operator: the parts change places
      wim[u] = pr.scale ? x : z;
      bits |= x | z;
    }
  }
  __device__ __forceinline__ Blk next(const LbParams& p, const double2* in, const double2* ws, int kop, int tr, int tc,
                                      int wv) {
    constexpr int nsplit = R == 1 ? 4 : 1;  // R = 1: every fourth block is this wavefront's
    Blk b;
    b.valid = false;
    b.kb = 0;
    b.re = b.im = 0;
#pragma unroll 1
    for (;;) {
      if (bits == 0) {
        if (++w >= p.nw) {
          w = 0;
          if (++q >= (PHASE == 1 ? 1 : p.nc + 2)) break;
          pr = product<PHASE>(p, in, ws, q, kop);
        }
        read(p, tr, tc);
        continue;
      }
      const int j = __ffs(bits) - 1;
      bits &= bits - 1;
      const bool mine = nsplit == 1 || (turn & (nsplit - 1)) == wv;
      ++turn;
      if (!mine) continue;
      b.valid = true;
      b.kb = 32 * w + j;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        b.re |= ((wre[u] >> j) & 1u) << u;
        b.im |= ((wim[u] >> j) & 1u) << u;
      }
      break;
    }
    b.pr = pr;
    return b;
  }
};

// Fragments of a k-block: chunk c, subtile u: A[16 u + lane % 16][16 kb + 4 c + lane / 16] of the tile's
// rows and B[16 kb + 4 c + lane / 16][16 u + lane % 16] of its columns.
template <int R>
struct Frag {
  double2 a[4][R], b[4][R];
};

// PHASE 1: T_k = X c_k^dag.  PHASE 2: right-hand side and RK4 update.  A wavefront forms a 16 R x 16 R
// tile.  R = 2 (a workgroup is four wavefronts with consecutive tiles) loads each operand for two MFMA
// tiles and serves launches that fill the chip: 16 MFMAs of 64 cycles per chunk cover the L2 latency of
// the next block's loads even at one wavefront per SIMD.  R = 1 (a workgroup is one tile, its k-blocks
// dealt to the four wavefronts and summed through LDS in a fixed order) serves small ones, where the
// number of workgroups and the length of the chain count.
template <int PHASE, int R>
__global__ __launch_bounds__(kLThreads, R == 2 ? 2 : 4) void lindblad_product_kernel(LbParams p) {
  constexpr bool SPLIT = R == 1;
  __shared__ double2 red[SPLIT ? 4 * 256 : kLThreads];
  const int tid = threadIdx.x, lane = tid & 63, gi = lane & 15, gk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = p.d, nc = p.nc, nt = p.nt;
  const int64_t d2 = (int64_t)d * d;
  if (PHASE == 1 && (int)blockIdx.x >= p.gemm_blocks) {
    const int64_t b = blockIdx.x - p.gemm_blocks;
    side_work(p, p.inst0 + b / p.side_blocks, (int)(b % p.side_blocks), red);
    return;
  }
  const int ntr = (nt + R - 1) / R;  // wavefront tiles per dimension
  const int nprod = PHASE == 1 ? nc : 1;  // output matrices per instance
  const int64_t wt = SPLIT ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wv;
  const int64_t per = (int64_t)nprod * ntr * ntr;
  const int64_t li = wt / per;
  if (li >= p.n_inst) return;  // R = 2 only: the tail of the last workgroup (no barrier below for R = 2)
  const int rest = (int)(wt - li * per);
  const int kop = PHASE == 1 ? rest / (ntr * ntr) : 0;
  const int tt = rest - kop * ntr * ntr, tr = tt / ntr * R, tc = (tt % ntr) * R;  // first 16-wide subtile
  const int64_t inst = p.inst0 + li;
  double2* y = p.rho + inst * d2;
  double2* ws = p.ws + inst * p.ws_stride;
  double2* X0 = ws;
  double2* X1 = X0 + d2;
  double2* acR = X1 + d2;
  const double2* in = p.stage == 0 ? y : (p.stage == 2 ? X1 : X0);
  double2* out = p.stage == 1 ? X1 : X0;
  Walk<PHASE, R> walk;
  walk.start(p, in, ws, kop, tr, tc, wv);
  auto load = [&](const Blk& b, Frag<R>& f) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = 16 * b.kb + 4 * c + gk;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int i = 16 * (tr + u) + gi, j = 16 * (tc + u) + gi;
        f.a[c][u] = (i < d && k < d) ? b.pr.A[(int64_t)i * d + k] : make_double2(0.0, 0.0);
        f.b[c][u] = (k < d && j < d) ? b.pr.B[(int64_t)k * d + j] : make_double2(0.0, 0.0);
      }
    }
  };
  doublex4 sr[R][R], si[R][R];
#pragma unroll
  for (int u = 0; u < R; ++u)
#pragma unroll
    for (int v = 0; v < R; ++v) sr[u][v] = si[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](const Blk& b, Frag<R>& f) __attribute__((always_inline)) {
    if (b.pr.scale) {
      const double s = b.pr.scale == 1 ? 1.0 : -1.0;  // -i z = (y, -x); +i z = (-y, x)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int u = 0; u < R; ++u) {
          if (b.pr.left) f.a[c][u] = make_double2(s * f.a[c][u].y, -s * f.a[c][u].x);
          else f.b[c][u] = make_double2(s * f.b[c][u].y, -s * f.b[c][u].x);
        }
    }
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const int g = b.pr.left ? u : v;  // the operator's subtile
        if ((b.re >> g) & 1u) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const double2 a = f.a[c][u], x = f.b[c][v];
            sr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.x, sr[u][v], 0, 0, 0);
            si[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.pr.left ? a.x : a.y, b.pr.left ? x.y : x.x, si[u][v], 0, 0, 0);
          }
        }
        if ((b.im >> g) & 1u) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const double2 a = f.a[c][u], x = f.b[c][v];
            sr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, x.y, sr[u][v], 0, 0, 0);
            si[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.pr.left ? a.y : a.x, b.pr.left ? x.x : x.y, si[u][v], 0, 0, 0);
          }
        }
      }
  };
  {
    Frag<R> f0, f1;
    Blk b0 = walk.next(p, in, ws, kop, tr, tc, wv), b1;
    if (b0.valid) load(b0, f0);
#pragma unroll 1
    while (b0.valid) {
      b1 = walk.next(p, in, ws, kop, tr, tc, wv);
      if (b1.valid) load(b1, f1);
      multiply(b0, f0);
      if (!b1.valid) break;
      b0 = walk.next(p, in, ws, kop, tr, tc, wv);
      if (b0.valid) load(b0, f0);
      multiply(b1, f1);
    }
  }

  // ---- epilogue of element e with right-hand side (or product) value v
  const double dt = p.dt, dt2 = dt / 2.0;
  struct Old {
    double2 y, a;
  };
  auto fetch = [&](int64_t e) -> Old {
    Old o;
    if (PHASE == 2) {
      o.y = y[e];
      if (p.stage > 0) o.a = acR[e];
    }
    return o;
  };
  auto finish = [&](int64_t e, double2 v, const Old& o) {
    if (PHASE == 1) {
      ws[(3 + kop) * d2 + e] = v;
    } else if (p.stage == 0) {
      acR[e] = v;
      out[e] = make_double2(o.y.x + v.x * dt2, o.y.y + v.y * dt2);
    } else if (p.stage < 3) {
      acR[e] = make_double2(o.a.x + 2.0 * v.x, o.a.y + 2.0 * v.y);
      const double h = p.stage == 1 ? dt2 : dt;
      out[e] = make_double2(o.y.x + v.x * h, o.y.y + v.y * h);
    } else {
      // y is not a product input in stage 3 (its input is X0): update in place
      const double2 n = make_double2(o.y.x + (o.a.x + v.x) / 6.0 * dt, o.y.y + (o.a.y + v.y) / 6.0 * dt);
      y[e] = n;
      if (p.rho_out && (p.step + 1) % p.save_every == 0)
        p.rho_out[(inst * (p.nsteps / p.save_every) + (p.step + 1) / p.save_every - 1) * d2 + e] = n;
    }
  };
  // MFMA output: register r of lane (gk, gi) holds element (4 r + gk, gi) of its 16 x 16 tile
  if constexpr (SPLIT) {
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv * 256 + (4 * r + gk) * 16 + gi] = make_double2(sr[0][0][r], si[0][0][r]);
    const int i = 16 * tr + (tid >> 4), j = 16 * tc + (tid & 15);
    const bool ok = i < d && j < d;
    const int64_t e = (int64_t)i * d + j;
    Old o;
    if (ok) o = fetch(e);
    __syncthreads();
    if (ok) {
      double2 v = red[tid];
#pragma unroll
      for (int s = 1; s < 4; ++s) {
        v.x += red[s * 256 + tid].x;
        v.y += red[s * 256 + tid].y;
      }
      finish(e, v, o);
    }
  } else {
    Old o[R][R][4];
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int v = 0; v < R; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * (tr + u) + 4 * r + gk, j = 16 * (tc + v) + gi;
          if (i < d && j < d) o[u][v][r] = fetch((int64_t)i * d + j);
        }
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int v = 0; v < R; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * (tr + u) + 4 * r + gk, j = 16 * (tc + v) + gi;
          if (i < d && j < d) finish((int64_t)i * d + j, make_double2(sr[u][v][r], si[u][v][r]), o[u][v][r]);
        }
  }
}

// ------------------------------------------------------------------ resident form, d <= 64
// One workgroup per instance and one launch for the whole run: NT x NT wavefronts (NT = tiles per
// dimension) hold a 16 x 16 tile of rho, of the RK4 sum and of every product in registers, and the two
// matrices a product reads across tiles, the stage input X and one T_k = X c_k^dag, stand in LDS (133 KB at
// NT = 4).  Only the operators come from memory, and every workgroup reads the same ones (L2).  It wins
// where the instances give the CUs work or where eight launches per step cost more than the products:
// 256 dense d = 64 instances reach 44 TFLOP/s (FP64 matrix products reach 71 on this card), against 27 by
// launches; what bounds it there is four wavefronts per SIMD waiting on operator fragments between barriers.
template <int NT, bool DRIVEN>
__global__ __launch_bounds__(64 * NT * NT) void lindblad_resident_kernel(LbParams p) {
  constexpr int LD = 16 * NT + 1;  // row stride: the column reads of the left operand fall on different banks
  extern __shared__ __align__(16) char smem[];
  double2* X = (double2*)smem;
  double2* T = X + 16 * NT * LD;
  double2* red = T + 16 * NT * LD;     // [NT * NT]
  uint2* stab = (uint2*)(red + NT * NT);  // block table: [2 (nc + 1)][NT]
  const int tid = threadIdx.x, lane = tid & 63, gi = lane & 15, gk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = p.d, nc = p.nc, ti = wv / NT, tj = wv % NT;
  const int64_t d2 = (int64_t)d * d, inst = blockIdx.x;
  double2* rho = p.rho + inst * d2;
  const double dt = p.dt, dt2 = dt / 2.0;
  const int j = 16 * tj + gi, i0 = 16 * ti + gk;  // this lane's elements: (i0 + 4 r, j), r = 0..3
  for (int e = tid; e < 2 * (nc + 1) * NT; e += 64 * NT * NT)
    stab[e] = p.tab ? p.tab[e] : make_uint2((1u << NT) - 1u, (1u << NT) - 1u);
  double2 y[4], a[4];
  auto valid = [&](int r) { return i0 + 4 * r < d && j < d; };
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[r] = valid(r) ? rho[(i0 + 4 * r) * d + j] : make_double2(0.0, 0.0);
    X[(i0 + 4 * r) * LD + j] = y[r];
  }
  // acc += (operator) M (left) or M (operator): operator element fetch(e), rows of the operator from
  // memory, M from LDS, zero blocks skipped
  doublex4 sr, si, tr, tm;
  auto product = [&](doublex4& re, doublex4& im, bool left, int scale, const double2* M, int row, auto fetch)
                     __attribute__((always_inline)) {
    const uint2 m = stab[row * NT + (left ? ti : tj)];
    const uint32_t mx = __builtin_amdgcn_readfirstlane(m.x), my = __builtin_amdgcn_readfirstlane(m.y);
    const uint32_t br = scale ? my : mx, bi = scale ? mx : my;
    uint32_t bits = mx | my;
    auto load = [&](int kb, double2 (&f)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = 16 * kb + 4 * c + gk, o = 16 * (left ? ti : tj) + gi;
        f[c] = k < d && o < d ? fetch(left ? o * d + k : k * d + o) : make_double2(0.0, 0.0);
      }
    };
    auto multiply = [&](int kb, double2 (&f)[4]) __attribute__((always_inline)) {
      double2 x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = 16 * kb + 4 * c + gk;
        x[c] = left ? M[k * LD + j] : M[(16 * ti + gi) * LD + k];
        if (scale) f[c] = scale == 1 ? make_double2(f[c].y, -f[c].x) : make_double2(-f[c].y, f[c].x);
      }
      if ((br >> kb) & 1u) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          re = left ? __builtin_amdgcn_mfma_f64_16x16x4f64(f[c].x, x[c].x, re, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f64_16x16x4f64(x[c].x, f[c].x, re, 0, 0, 0);
          im = left ? __builtin_amdgcn_mfma_f64_16x16x4f64(f[c].x, x[c].y, im, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f64_16x16x4f64(x[c].y, f[c].x, im, 0, 0, 0);
        }
      }
      if ((bi >> kb) & 1u) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          re = left ? __builtin_amdgcn_mfma_f64_16x16x4f64(-f[c].y, x[c].y, re, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f64_16x16x4f64(x[c].y, -f[c].y, re, 0, 0, 0);
          im = left ? __builtin_amdgcn_mfma_f64_16x16x4f64(f[c].y, x[c].x, im, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f64_16x16x4f64(x[c].x, f[c].y, im, 0, 0, 0);
        }
      }
    };
    double2 f0[4], f1[4];
    auto take = [&]() __attribute__((always_inline)) {
      const int b = __ffs(bits) - 1;
      bits &= bits - 1;
      return b;
    };
    if constexpr (NT == 4) {  // four wavefronts per SIMD cover the loads; the registers of a second block spill
#pragma unroll 1
      while (bits) {
        const int kb = take();
        load(kb, f0);
        multiply(kb, f0);
      }
      return;
    }
    if (bits == 0) return;
    int k0 = take(), k1;
    load(k0, f0);
#pragma unroll 1
    for (;;) {
      if (bits == 0) {
        multiply(k0, f0);
        break;
      }
      k1 = take();
      load(k1, f1);
      multiply(k0, f0);
      if (bits == 0) {
        multiply(k1, f1);
        break;
      }
      k0 = take();
      load(k0, f0);
      multiply(k1, f1);
    }
  };
  auto observe = [&](int64_t row) {
    for (int o = 0; o < p.n_obs; ++o) {
      double2 s = make_double2(0.0, 0.0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (valid(r)) {
          const double2 v = cmul2(p.obs[o * d2 + (i0 + 4 * r) * d + j], y[r]);
          s.x += v.x;
          s.y += v.y;
        }
      for (int w = 32; w > 0; w >>= 1) {
        s.x += __shfl_xor(s.x, w, 64);
        s.y += __shfl_xor(s.y, w, 64);
      }
      if (lane == 0) red[wv] = s;
      __syncthreads();
      if (tid == 0) {
        for (int w = 1; w < NT * NT; ++w) {
          s.x += red[w].x;
          s.y += red[w].y;
        }
        p.obs_out[(inst * (p.nsteps + 1) + row) * p.n_obs + o] = s;
      }
      __syncthreads();
    }
  };
  __syncthreads();
  if (p.n_obs) observe(0);
  for (int64_t s = 0; s < p.nsteps; ++s) {
    const double* f = p.field + (inst * p.nsteps + s) * p.ndrive;
    auto driven = [&](const double2* H, const double2* D) {
      return [=](int e) {
        double2 h = H[e];
        for (int q = 0; DRIVEN && q < p.ndrive; ++q) {
          const double2 v = D[q * d2 + e];
          h.x -= f[q] * v.x;
          h.y -= f[q] * v.y;
        }
        return h;
      };
    };
#pragma unroll 1
    for (int stage = 0; stage < 4; ++stage) {
      const doublex4 zero = {0.0, 0.0, 0.0, 0.0};
      sr = si = zero;
      product(sr, si, true, 1, X, nc, driven(p.Heff, p.Hd));
      product(sr, si, false, 2, X, 2 * nc + 1, driven(p.HeffD, p.HdD));
#pragma unroll 1
      for (int k = 0; k < nc; ++k) {
        const double2* C = p.C + k * d2;
        const double2* D = p.CD + k * d2;
        tr = tm = zero;
        product(tr, tm, false, 0, X, nc + 1 + k, [=](int e) { return D[e]; });
        if (k) __syncthreads();  // T_{k-1} is no longer read
#pragma unroll
        for (int r = 0; r < 4; ++r) T[(i0 + 4 * r) * LD + j] = valid(r) ? make_double2(tr[r], tm[r]) : make_double2(0.0, 0.0);
        __syncthreads();
        product(sr, si, true, 0, T, k, [=](int e) { return C[e]; });
      }
      __syncthreads();  // every read of X (and T) is done
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double2 v = make_double2(sr[r], si[r]);
        double2 x;
        if (stage == 3) {
          x = y[r] = make_double2(y[r].x + (a[r].x + v.x) / 6.0 * dt, y[r].y + (a[r].y + v.y) / 6.0 * dt);
        } else {
          const double h = stage == 2 ? dt : dt2;
          a[r] = stage == 0 ? v : make_double2(a[r].x + 2.0 * v.x, a[r].y + 2.0 * v.y);
          x = make_double2(y[r].x + v.x * h, y[r].y + v.y * h);
        }
        X[(i0 + 4 * r) * LD + j] = valid(r) ? x : make_double2(0.0, 0.0);
      }
      __syncthreads();
    }
    if (p.n_obs) observe(s + 1);
    if (p.rho_out && (s + 1) % p.save_every == 0) {
      double2* dst = p.rho_out + (inst * (p.nsteps / p.save_every) + (s + 1) / p.save_every - 1) * d2;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (valid(r)) dst[(i0 + 4 * r) * d + j] = y[r];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (valid(r)) rho[(i0 + 4 * r) * d + j] = y[r];
}

int lb_tiles(int d) { return (d + 15) / 16; }
int lb_words(int d) { return (lb_tiles(d) + 31) / 32; }

// bytes of the block tables and scan flags, after the instances' buffers
int64_t lb_table_bytes(int d, int nc) {
  return 2 * (int64_t)(nc + 1) * lb_tiles(d) * lb_words(d) * (int64_t)sizeof(uint2) + kScanBlocks * (int64_t)sizeof(int);
}

int64_t lb_inst_elems(int d, int nc, int ndrive) { return (int64_t)(3 + nc + (ndrive > 0 ? 2 : 0)) * d * d; }

template <int NT, bool DRIVEN>
int lb_resident(const LbParams& p, hipStream_t st) {
  constexpr size_t mats = 2 * (size_t)(16 * NT) * (16 * NT + 1) * sizeof(double2) + NT * NT * sizeof(double2);
  const size_t lds = mats + 2 * (size_t)(p.nc + 1) * NT * sizeof(uint2);
  if (lds > 65536)
    PQA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&lindblad_resident_kernel<NT, DRIVEN>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL((lindblad_resident_kernel<NT, DRIVEN>), dim3((unsigned)p.n_inst), dim3(64 * NT * NT), lds, st, p);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

template <int R>
int lb_stage(const LbParams& base, int64_t blocks1, int64_t blocks2, hipStream_t st) {
  LbParams p = base;
  const int64_t side = p.stage == 0 ? (int64_t)p.side_blocks * p.n_inst : 0;
  p.gemm_blocks = (int)blocks1;
  if (blocks1 + side > 0) {
    hipLaunchKernelGGL((lindblad_product_kernel<1, R>), dim3((unsigned)(blocks1 + side)), dim3(kLThreads), 0, st, p);
    PQA_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL((lindblad_product_kernel<2, R>), dim3((unsigned)blocks2), dim3(kLThreads), 0, st, p);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

}  // namespace
}  // namespace pqa

using namespace pqa;

extern "C" int pyqed_lindblad_work_bytes(int32_t d, int32_t nc, int32_t ndrive, int32_t n_inst, int64_t* bytes) {
  if (!bytes || d < 1 || nc < 0 || ndrive < 0 || n_inst < 1)
    return fail(PYQED_EINVAL, "lindblad_work_bytes: need d >= 1, nc >= 0, ndrive >= 0, n_inst >= 1");
  *bytes = (int64_t)n_inst * lb_inst_elems(d, nc, ndrive) * (int64_t)sizeof(double2);
  return PYQED_OK;
}

extern "C" int pyqed_lindblad_table_bytes(int32_t d, int32_t nc, int64_t* bytes) {
  if (!bytes || d < 1 || nc < 0) return fail(PYQED_EINVAL, "lindblad_table_bytes: need d >= 1, nc >= 0");
  *bytes = lb_table_bytes(d, nc);
  return PYQED_OK;
}

extern "C" int pyqed_lindblad_run(int32_t d, int32_t nc, const void* Heff, const void* HeffD, const void* C,
                                  const void* CD, int32_t ndrive, const void* Hd, const void* HdD, int32_t n_inst,
                                  void* rho, const double* field, int64_t nsteps, double dt, int32_t n_obs,
                                  const void* obs, void* obs_out, void* rho_out, int64_t save_every, void* work,
                                  int64_t work_bytes, void* stream) {
  if (d < 1 || d > 46340 || nc < 0 || ndrive < 0 || n_inst < 1 || !Heff || !HeffD || !rho || !work)
    return fail(PYQED_EINVAL, "lindblad_run: need 1 <= d <= 46340, nc >= 0, ndrive >= 0, n_inst >= 1 and "
                              "Heff, HeffD, rho, work");
  if (nc > 0 && (!C || !CD)) return fail(PYQED_EINVAL, "lindblad_run: nc > 0 needs C and CD");
  if (ndrive > 0 && (!Hd || !HdD || !field)) return fail(PYQED_EINVAL, "lindblad_run: drives need Hd, HdD and a field");
  if (n_obs < 0 || (n_obs > 0 && (!obs || !obs_out))) return fail(PYQED_EINVAL, "lindblad_run: bad observables");
  if (nsteps < 0) return fail(PYQED_EINVAL, "lindblad_run: negative step count");
  int64_t need = 0;
  pyqed_lindblad_work_bytes(d, nc, ndrive, n_inst, &need);
  if (work_bytes < need)
    return fail(PYQED_EINVAL, "lindblad_run: workspace of " + std::to_string(work_bytes) + " bytes < " +
                                  std::to_string(need));
  if (nsteps == 0 && n_obs == 0) return PYQED_OK;
  LbParams p;
  std::memset(&p, 0, sizeof(p));
  p.d = d;
  p.nc = nc;
  p.ndrive = ndrive;
  p.n_obs = n_obs;
  p.nt = lb_tiles(d);
  p.nw = lb_words(d);
  p.n_inst = n_inst;
  p.nsteps = nsteps;
  p.save_every = save_every > 0 ? save_every : 1;
  p.ws_stride = lb_inst_elems(d, nc, ndrive);
  p.dt = dt;
  p.Heff = (const double2*)Heff;
  p.HeffD = (const double2*)HeffD;
  p.C = (const double2*)C;
  p.CD = (const double2*)CD;
  p.Hd = (const double2*)Hd;
  p.HdD = (const double2*)HdD;
  p.field = field;
  p.rho = (double2*)rho;
  p.obs = (const double2*)obs;
  p.obs_out = (double2*)obs_out;
  p.rho_out = (double2*)rho_out;
  p.ws = (double2*)work;
  hipStream_t st = (hipStream_t)stream;
  if (work_bytes - need >= lb_table_bytes(d, nc)) {
    p.tab = (uint2*)((char*)work + need);
    p.flags = (int*)(p.tab + 2 * (int64_t)(nc + 1) * p.nt * p.nw);
    hipLaunchKernelGGL(lindblad_scan_kernel, dim3(kScanBlocks), dim3(kLThreads), 0, st, p);
    PQA_HIP(hipGetLastError());
    hipLaunchKernelGGL(lindblad_table_kernel, dim3((unsigned)(2 * (nc + 1) * (int64_t)p.nt)), dim3(kLThreads),
                       2 * p.nw * sizeof(uint32_t), st, p);
    PQA_HIP(hipGetLastError());
  }
  // d <= 64: the resident form from the number of instances where it is the faster one, by tiles per
  // dimension.  us per step with two collapse operators, launches against resident, dense / banded operators:
  // d = 16: 30-39 / 23, 29-38 / 19; d = 32: 39 / 48, 36 / 31 for one instance, 96 / 48, 78 / 32 for 256;
  // d = 48: 98 / 138, 71 / 54 for 64, 137 / 138, 97 / 55 for 128; d = 64: 129 / 231, 82 / 75 for 64,
  // 224 / 233, 131 / 75 for 128, 368 / 233, 181 / 75 for 256.  The numbers of instances are those from which dense
  // operators are the faster; which operators a call has is known on the device alone, and banded ones would gain up
  // to a quarter by going over earlier (d = 48 and 64 from 64 instances on).
  constexpr int kResFrom[5] = {0, 1, 16, 96, 96};
  if (p.nt <= 4 && n_inst >= kResFrom[p.nt] && nc <= 256) {
    switch (p.nt) {
      case 1: return ndrive ? lb_resident<1, true>(p, st) : lb_resident<1, false>(p, st);
      case 2: return ndrive ? lb_resident<2, true>(p, st) : lb_resident<2, false>(p, st);
      case 3: return ndrive ? lb_resident<3, true>(p, st) : lb_resident<3, false>(p, st);
      default: return ndrive ? lb_resident<4, true>(p, st) : lb_resident<4, false>(p, st);
    }
  }
  // 32 x 32 wavefront tiles once they give every CU a workgroup, 16 x 16 tiles split four ways below
  const int64_t t16 = (int64_t)p.nt * p.nt, t32 = (int64_t)((p.nt + 1) / 2) * ((p.nt + 1) / 2);
  const bool big = p.nt > 1 && t32 * n_inst >= 4 * kFullChip;
  // instances per launch, so that no grid holds 2^32 threads or more
  const int64_t d2 = (int64_t)d * d;
  const int64_t hs_blocks = ndrive > 0 ? std::min<int64_t>((d2 + 4 * kLThreads - 1) / (4 * kLThreads), 64) : 0;
  if ((int64_t)n_obs + hs_blocks > INT32_MAX / 4) return fail(PYQED_EINVAL, "lindblad_run: too many observables");
  p.side_blocks = (int)(n_obs + hs_blocks);
  const int64_t tiles = std::max(nc, 1) * (big ? (t32 + 3) / 4 : t16);
  const int64_t chunk = std::max<int64_t>(1, kGridBlocks / (tiles + p.side_blocks + 1));
  for (int64_t i0 = 0; i0 < n_inst; i0 += chunk) {
    p.inst0 = (int)i0;
    p.n_inst = (int)std::min<int64_t>(chunk, n_inst - i0);
    const int64_t b1 = big ? (t32 * nc * p.n_inst + 3) / 4 : t16 * nc * p.n_inst;
    const int64_t b2 = big ? (t32 * p.n_inst + 3) / 4 : t16 * p.n_inst;
    for (int64_t s = 0; s < nsteps; ++s) {
      p.step = s;
      for (p.stage = 0; p.stage < 4; ++p.stage) {
        const int rc = big ? lb_stage<2>(p, b1, b2, st) : lb_stage<1>(p, b1, b2, st);
        if (rc) return rc;
      }
    }
    if (n_obs) {
      p.step = nsteps;
      hipLaunchKernelGGL(lindblad_observe_kernel, dim3((unsigned)(p.n_inst * (int64_t)n_obs)), dim3(kLThreads), 0, st, p);
      PQA_HIP(hipGetLastError());
    }
  }
  return PYQED_OK;
}
