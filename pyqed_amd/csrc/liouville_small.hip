// Liouville-space RK4 and its discrete adjoint for N <= 16 (up to four levels), the sizes of qubits, three-
// level Lambda systems and their optimal control.  Same equations as liouville.hip; the difference is what
// a step waits for.
//
// A group of lanes (4 for N <= 4, 16 otherwise; groups share a wavefront, a workgroup is one wavefront) owns
// one instance: lane r holds element r of every RK4 vector and row r of the step's generator
// A_0 + sum f_i A_i, formed once per step, in registers.  Only the vector a product multiplies goes through
// LDS (one write, N broadcast reads), and no barrier is needed inside a wavefront.  Against the general
// kernels of liouville.hip (a workgroup's vectors all in LDS, barriers between the stages), 4096 instances,
// 400 steps with one drive: N = 9 forward 900 -> 496 us, adjoint 6.8 -> 2.6 ms; N = 4 635 -> 278 us and
// 4.5 -> 1.3 ms; N = 16 6.8 -> 0.79 ms and 49 -> 9.0 ms.  A step is bound by the latency of its four
// dependent products (about 0.25 us each), one wavefront per SIMD.
//
// One instance still is a chain of dependent steps.  Where the instances leave the chip idle the chain is cut
// along time (small_split): every segment's propagator is formed at once (its N columns are N groups), a
// short chain over segments gives the state at every segment's start and, for gradients, the adjoint state
// at every segment's end, and then all segments run at once.  The work grows by about N + 1 but the chain
// falls from nsteps to nsteps / seg + 2 seg steps.  One N = 9 instance, 1000 driven steps: 1868 -> 137 us
// forward, 15.3 -> 0.26 ms for the gradients; 4000 steps: 7670 -> 255 us and 61.7 -> 0.49 ms.  Error
// against extended precision relative to the uncut run and sweep of liouville.hip (Lambda system, 100..1200 steps, 14
// fields, geometric mean): parameters 0.75, amplitudes 0.47, initial state 0.38; with amplitudes held for 250 steps and
// more (root mean square) final state 0.35, amplitudes 0.7, initial state 0.15.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "liouville.h"

namespace pqa {
namespace {

constexpr int kWin = 64;  // values of a group's field window in LDS
constexpr double kTame = 1e150, kHold = 0x1p1000;
constexpr int64_t kSplitBytes = int64_t(4) << 30;  // largest workspace of a cut run, 1.4% of a GPU's 288 GB

typedef cpx<double> Z;

struct SmParams {
  LiouvilleRun r;
  int64_t nsegs;
  int64_t groups;    // of this launch
  int64_t seg_buf;   // adjoint: element offset of the segment states within ckpt
  int cols;          // forward: N when the groups are propagator columns (instance, segment, column), else 1
  double2* Q;        // [n_inst][nsegs][N][N] segment propagators less the identity
  double2* lamT;     // [n_inst][nsegs][N] adjoint states at the segments' ends (split), else NULL
  double2* part;     // [n_inst][nsegs][nterm][N][N] gradient parts (split), else NULL
};

__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The group's view of a launch.
template <int NT, int G>
struct Grp {
  static constexpr int kStride = NT | 1;  // LDS row stride of the generators: rows fall on different banks
  int li;
  int64_t b, inst, seg, s0, len;
  bool live, row;  // row: this lane holds element li

  __device__ __forceinline__ void place(const SmParams& p, int64_t segs_per_inst, int cols) {
    li = threadIdx.x % G;
    b = blockIdx.x * (int64_t)(64 / G) + threadIdx.x / G;
    live = b < p.groups;
    if (!live) b = 0;
    const int64_t q = b / cols;
    inst = q / segs_per_inst;
    seg = q - inst * segs_per_inst;
    row = live && li < p.r.N;
  }
  __device__ __forceinline__ void range(const SmParams& p, int64_t sg) {
    s0 = sg * p.r.seg;
    len = min(p.r.seg, p.r.nsteps - s0);
  }
};

// Generators in LDS, zero beyond N: sA[i][r][k]
template <int NT, int G>
__device__ __forceinline__ void stage_generators(const SmParams& p, Z* sA) {
  constexpr int S = Grp<NT, G>::kStride;
  const int N = p.r.N;
  for (int e = threadIdx.x; e < p.r.nterm * NT * S; e += 64) {
    const int i = e / (NT * S), q = e - i * NT * S, r = q / S, k = q - r * S;
    Z v = mk(0.0, 0.0);
    if (r < N && k < N) {
      const double2 a = p.r.A[((int64_t)i * N + r) * N + k];
      v = mk(a.x, a.y);
    }
    sA[e] = v;
  }
}

// Row li of A_0 and A_1 and the step's combination (columns: conj(A[k][li]), for products with A^H).
template <int NT, int G, bool HT>
struct Rows {
  Z a0[NT], a1[NT], as[NT];
  const Z* base;
  int li, nterm;
  bool finite;  // every generator is finite (uniform): 0 x A_i needs no care

  static __device__ __forceinline__ Z at(const Z* sA, int i, int li, int k) {
    constexpr int S = Grp<NT, G>::kStride;
    return HT ? conjg(sA[(i * NT + k) * S + li]) : sA[(i * NT + li) * S + k];
  }
  __device__ __forceinline__ void init(const Z* sA, int li_, int nterm_) {
    base = sA;
    li = li_ < NT ? li_ : NT - 1;
    nterm = nterm_;
    const bool in = li_ < NT;
    bool ok = true;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      a0[k] = in ? at(sA, 0, li, k) : mk(0.0, 0.0);
      a1[k] = in && nterm > 1 ? at(sA, 1, li, k) : mk(0.0, 0.0);
      as[k] = a0[k];
    }
    for (int i = 1; i < nterm; ++i)
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const Z v = at(sA, i, li, k);
        ok = ok && isfinite(v.x) && isfinite(v.y);
      }
    finite = __ballot(!ok) == 0;
  }
  // as = A_0 + sum f_i A_i; a term with f_i = 0 is left out (it may hold what is not finite)
  __device__ __forceinline__ void combine(const double* f, bool in) {
    if (nterm == 1) return;
    const double f1 = in ? f[0] : 0.0;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      as[k] = a0[k];
      if (finite || f1 != 0.0) as[k] = mk(fma(f1, a1[k].x, a0[k].x), fma(f1, a1[k].y, a0[k].y));
    }
    for (int i = 2; i < nterm; ++i) {
      const double fi = in ? f[i - 1] : 0.0;
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const Z a = at(base, i, li, k);
        if (finite || fi != 0.0) as[k] = mk(fma(fi, a.x, as[k].x), fma(fi, a.y, as[k].y));
      }
    }
  }
  // (row) . x, x in LDS
  __device__ __forceinline__ Z dot(const Z* x) const {
    Z p = mk(0.0, 0.0), q = p;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      if (k & 1) cmac(q, as[k], x[k]);
      else cmac(p, as[k], x[k]);
    }
    return p + q;
  }
};

// The step's field values: a window of the group's rows in LDS, `rows` rows of nterm - 1 values.
struct Field {
  double* w;
  int64_t lo, hi;
  int rows;
};

template <int NT, int G>
__device__ __forceinline__ const double* field_row(const SmParams& p, const Grp<NT, G>& q, Field& f, int64_t s, bool down) {
  const int nt1 = p.r.nterm - 1;
  if (nt1 == 0) return nullptr;
  if (s < f.lo || s >= f.hi) {  // the groups of a wavefront walk the same local steps
    f.lo = down ? max((int64_t)0, s - f.rows + 1) : s;
    f.hi = f.lo + f.rows;
    const double* src = p.r.field + (q.inst * p.r.nsteps + q.s0 + f.lo) * nt1;
    const int64_t n = min(f.hi, q.len) - f.lo;
    wave_order();
    for (int64_t e = q.li; e < n * nt1; e += G) f.w[e] = q.live ? src[e] : 0.0;
    wave_order();
  }
  return f.w + (s - f.lo) * nt1;
}

// What one RK4 step adds to the lane's element v; x: the group's LDS vector
template <int NT, int G>
__device__ __forceinline__ Z rk4(const Rows<NT, G, false>& R, Z v, Z* x, int li, double dt) {
  const double dt2 = dt / 2.0;
  auto mul = [&](Z u) __attribute__((always_inline)) {
    if (li < NT) x[li] = u;
    wave_order();
    const Z k = R.dot(x);
    wave_order();
    return k;
  };
  const Z k1 = mul(v), k2 = mul(v + k1 * dt2), k3 = mul(v + k2 * dt2), k4 = mul(v + k3 * dt);
  const Z t = k1 + k2 * 2.0 + k3 * 2.0 + k4;
  return mk(t.x / 6.0 * dt, t.y / 6.0 * dt);
}

// LDS: [generators][per group: vector NT][per group: field window kWin or nterm - 1 values]
template <int NT, int G>
struct Carve {
  Z* sA;
  Z* x;
  double* w;
  int rows;
};
__host__ __device__ inline int win_rows(int nt1) { return nt1 < 1 ? 0 : (nt1 > kWin ? 1 : kWin / nt1); }
template <int NT, int G>
__host__ __device__ inline size_t small_lds(int nterm, int vecs) {
  return sizeof(Z) * ((size_t)nterm * NT * (NT | 1) + (size_t)(64 / G) * vecs * NT) +
         sizeof(double) * (size_t)(64 / G) * win_rows(nterm - 1) * (nterm - 1);
}
template <int NT, int G>
__device__ __forceinline__ Carve<NT, G> carve_small(char* smem, int nterm, int vecs) {
  Carve<NT, G> c;
  const int g = threadIdx.x / G;
  c.sA = (Z*)smem;
  Z* v = c.sA + nterm * NT * (NT | 1);
  c.x = v + g * vecs * NT;
  c.rows = win_rows(nterm - 1);
  c.w = (double*)(v + (64 / G) * vecs * NT) + g * c.rows * (nterm - 1);
  return c;
}

// Forward: states of whole instances or of one segment of them, or the columns of segment propagators.
template <int NT, int G, bool COLS>
__global__ __launch_bounds__(64) void small_forward_kernel(SmParams p) {
  extern __shared__ __align__(16) char smem[];
  const Carve<NT, G> c = carve_small<NT, G>(smem, p.r.nterm, 1);
  Grp<NT, G> q;
  q.place(p, p.nsegs, COLS ? p.cols : 1);
  q.range(p, q.seg);
  stage_generators<NT, G>(p, c.sA);
  __syncthreads();
  const int N = p.r.N, col = COLS ? (int)(q.b % p.cols) : 0;
  Rows<NT, G, false> R;
  R.init(c.sA, q.li, p.r.nterm);
  // columns: is everything the segment multiplies with of ordinary size?
  bool tame = true;
  if (COLS) {
    for (int e = threadIdx.x; e < p.r.nterm * NT * Grp<NT, G>::kStride; e += 64) tame = tame && fabs(c.sA[e].x) < kTame && fabs(c.sA[e].y) < kTame;
    tame = __ballot(!tame) == 0;
  }
  // Columns are summed without their unit vector: segments under one field share a propagator, and rounding of the
  // sum to the unit's ulp would repeat in each and add up.  The increment rounds to its own.
  Z v = mk(0.0, 0.0), sum = v;
  const int64_t end = p.r.ckpt ? (q.inst * (p.nsegs + 1) + q.seg) * N : q.inst * N;  // where the state comes from
  if (COLS) {
    if (q.row && q.li == col) v.x = 1.0;
  } else if (q.row) {
    const double2 s = (p.r.ckpt ? p.r.ckpt : p.r.rho)[end + q.li];
    v = mk(s.x, s.y);
  }
  auto observe = [&](int64_t row) {
    for (int o = 0; o < p.r.n_obs; ++o) {
      Z s = mk(0.0, 0.0);
      if (q.row) {
        const double2 w = p.r.obs[(int64_t)o * N + q.li];
        s = mk(w.x, w.y) * v;
      }
#pragma unroll
      for (int w = G / 2; w > 0; w >>= 1) {
        s.x += __shfl_xor(s.x, w, G);
        s.y += __shfl_xor(s.y, w, G);
      }
      if (q.live && q.li == 0) p.r.obs_out[(q.inst * (p.r.nsteps + 1) + row) * p.r.n_obs + o] = make_double2(s.x, s.y);
    }
  };
  if (!COLS && p.r.n_obs && q.seg == 0) observe(0);
  Field f{c.w, 0, 0, c.rows};
  // the longest segment of the wavefront sets the trip count; shorter ones stop changing
  for (int64_t s = 0; s < p.r.seg && s < p.r.nsteps; ++s) {
    const bool act = s < q.len;
    const double* fr = field_row<NT, G>(p, q, f, s, false);
    R.combine(fr, act);
    const Z n = rk4<NT, G>(R, v, c.x, q.li, p.r.dt);
    if (!act) continue;
    if (COLS) {
      sum = sum + n;
      v = mk((q.li == col ? 1.0 : 0.0) + sum.x, sum.y);
      for (int i = 0; i < p.r.nterm - 1; ++i) tame = tame && fabs(fr[i]) < kTame;
      continue;
    }
    v = v + n;
    const int64_t t = q.s0 + s + 1;
    if (p.r.n_obs) observe(t);
    if (p.r.rho_out && t % p.r.save_every == 0 && q.row)
      p.r.rho_out[(q.inst * (p.r.nsteps / p.r.save_every) + t / p.r.save_every - 1) * N + q.li] = make_double2(v.x, v.y);
  }
  if (COLS) {
    // A mode that this dt makes unstable and the state never excites: its column overflows, and steps would leave it
    // at exactly zero.  Held within 2^1000, zero times it stays zero.  NaN and Inf of the inputs pass.
    if (tame && !(fabs(sum.x) < kHold)) sum.x = copysign(kHold, sum.x);
    if (tame && !(fabs(sum.y) < kHold)) sum.y = copysign(kHold, sum.y);
    if (q.row) p.Q[((q.inst * p.nsegs + q.seg) * N + q.li) * N + col] = make_double2(sum.x, sum.y);
  } else if (q.row && q.seg == p.nsegs - 1) {
    p.r.rho[q.inst * N + q.li] = make_double2(v.x, v.y);
  }
}

// The chain over segments: block (instance, 0) from rho(0) forwards into ckpt, block (instance, 1) from the
// cotangent of rho(T) backwards into lamT.  The next segment's propagator is requested a segment ahead.
template <int NT, int G>
__global__ __launch_bounds__(64) void small_chain_kernel(SmParams p, int dirs) {
  __shared__ Z x[NT];
  const int li = threadIdx.x, N = p.r.N;
  const int64_t inst = blockIdx.x / dirs;
  const bool back = blockIdx.x % dirs == 1, row = li < N;
  const double2 s = row ? (back ? p.r.rhoT_bar : p.r.rho)[inst * N + li] : make_double2(0.0, 0.0);
  Z v = mk(s.x, s.y);
  const double2* Q = p.Q + inst * p.nsegs * N * N;
  auto fetch = [&](int64_t sg, Z (&q)[NT]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      double2 a = make_double2(0.0, 0.0);
      if (row && k < N) a = Q[(sg * N + (back ? k : li)) * N + (back ? li : k)];
      q[k] = mk(a.x, back ? -a.y : a.y);
    }
  };
  Z cur[NT], nxt[NT];
  fetch(back ? p.nsegs - 1 : 0, cur);
  for (int64_t j = 0; j < p.nsegs; ++j) {
    const int64_t sg = back ? p.nsegs - 1 - j : j;
    if (j + 1 < p.nsegs) fetch(back ? sg - 1 : sg + 1, nxt);
    if (row) (back ? p.lamT + (inst * p.nsegs + sg) * N : p.r.ckpt + (inst * (p.nsegs + 1) + sg) * N)[li] = make_double2(v.x, v.y);
    if (li < NT) x[li] = v;
    wave_order();
    Z a = mk(0.0, 0.0), b = a;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      if (k & 1) cmac(b, cur[k], x[k]);
      else cmac(a, cur[k], x[k]);
      cur[k] = nxt[k];
    }
    v = v + (a + b);
    wave_order();
  }
}

// Backward sweep of one segment (split) or of all segments of an instance, last to first.  Per step, with
// stage inputs X_s and kbar_s as in liouville.hip, lane r accumulates row r of O = sum_s kbar_s X_s^H:
// grad_A_i += f_i O and dJ/df_i = Re sum conj(O) A_i (elementwise), so the drives need no products of their own.
template <int NT, int G>
__global__ __launch_bounds__(64) void small_adjoint_kernel(SmParams p, int64_t segs_here) {
  extern __shared__ __align__(16) char smem[];
  // vectors: one for products, four stage inputs; then the gradient rows [nterm][NT] of every lane
  const Carve<NT, G> c = carve_small<NT, G>(smem, p.r.nterm, 5);
  Grp<NT, G> q;
  q.place(p, segs_here == 1 ? p.nsegs : 1, 1);
  const int N = p.r.N, nterm = p.r.nterm, nt1 = nterm - 1;
  Z* gA = (Z*)(smem + small_lds<NT, G>(nterm, 5)) + threadIdx.x;  // gA[(i NT + k) 64]
  stage_generators<NT, G>(p, c.sA);
  if (p.r.grad_A)
    for (int e = 0; e < nterm * NT; ++e) gA[e * 64] = mk(0.0, 0.0);
  __syncthreads();
  Rows<NT, G, false> R;
  Rows<NT, G, true> H;
  R.init(c.sA, q.li, nterm);
  H.init(c.sA, q.li, nterm);
  Z* xs = c.x + NT;  // X_1 .. X_4
  double2* buf = p.r.ckpt + p.seg_buf + q.b * p.r.seg * N;
  const double dt = p.r.dt, dt2 = dt / 2.0;
  Z lam = mk(0.0, 0.0);
  for (int64_t j = 0; j < segs_here; ++j) {
    const int64_t sg = segs_here == 1 ? q.seg : segs_here - 1 - j;
    q.range(p, sg);
    if (j == 0 && q.row) {
      const double2 s = p.lamT ? p.lamT[(q.inst * p.nsegs + sg) * N + q.li] : p.r.rhoT_bar[q.inst * N + q.li];
      lam = mk(s.x, s.y);
    }
    Z v = mk(0.0, 0.0);
    if (q.row) {
      const double2 s = p.r.ckpt[(q.inst * (p.nsegs + 1) + sg) * N + q.li];
      v = mk(s.x, s.y);
    }
    Field f{c.w, 0, 0, c.rows};
    const int64_t most = min(p.r.seg, p.r.nsteps);
    for (int64_t s = 0; s < most; ++s) {
      const bool act = s < q.len;
      if (act && q.row) buf[s * N + q.li] = make_double2(v.x, v.y);
      if (s + 1 == most) break;
      R.combine(field_row<NT, G>(p, q, f, s, false), act);
      const Z n = rk4<NT, G>(R, v, c.x, q.li, dt);
      if (act) v = v + n;
    }
    // the lane reads back its own elements only: v holds the last one, the others come a step ahead
    double2 ahead = make_double2(0.0, 0.0);
    auto fetch = [&](int64_t s) {
      if (s >= 0 && s < q.len && q.row) ahead = buf[s * N + q.li];
    };
    fetch(most - 1);
    for (int64_t s = most - 1; s >= 0; --s) {
      const bool act = s < q.len;
      const double* fr = field_row<NT, G>(p, q, f, s, true);
      R.combine(fr, act);
      H.combine(fr, act);
      const Z y = mk(ahead.x, ahead.y);
      fetch(s - 1);
      auto put = [&](int t, Z u) __attribute__((always_inline)) {
        if (q.li < NT) xs[t * NT + q.li] = u;
        wave_order();
      };
      put(0, y);
      put(1, y + R.dot(xs) * dt2);
      put(2, y + R.dot(xs + NT) * dt2);
      put(3, y + R.dot(xs + 2 * NT) * dt);
      Z O[NT];
#pragma unroll
      for (int k = 0; k < NT; ++k) O[k] = mk(0.0, 0.0);
      Z ub = lam, kb = lam * (dt / 6.0);
#pragma unroll
      for (int st = 3; st >= 0; --st) {
        if (q.li < NT) c.x[q.li] = kb;
        wave_order();
#pragma unroll
        for (int k = 0; k < NT; ++k) cmac(O[k], kb, conjg(xs[st * NT + k]));
        const Z Xb = H.dot(c.x);
        wave_order();
        ub = ub + Xb;
        if (st > 0) kb = lam * (st == 3 ? dt / 3.0 : st == 2 ? dt / 3.0 : dt / 6.0) + Xb * (st == 3 ? dt : dt2);
      }
      if (act) lam = ub;
      for (int i = 1; i < nterm; ++i) {
        double g = 0.0;
#pragma unroll
        for (int k = 0; k < NT; ++k) {
          const Z a = Rows<NT, G, false>::at(c.sA, i, R.li, k);
          g += O[k].x * a.x + O[k].y * a.y;
        }
        if (!q.row) g = 0.0;
#pragma unroll
        for (int w = G / 2; w > 0; w >>= 1) g += __shfl_xor(g, w, G);
        if (act && q.live && q.li == 0) p.r.grad_field[(q.inst * p.r.nsteps + q.s0 + s) * nt1 + (i - 1)] = g;
      }
      if (p.r.grad_A && act)
        for (int i = 0; i < nterm; ++i) {
          const double w = i == 0 ? 1.0 : fr[i - 1];
#pragma unroll
          for (int k = 0; k < NT; ++k) {
            Z& t = gA[(i * NT + k) * 64];
            t = t + O[k] * w;
          }
        }
    }
    if (p.r.rho0_bar && sg == 0 && q.row) p.r.rho0_bar[q.inst * N + q.li] = make_double2(lam.x, lam.y);
  }
  if (p.r.grad_A && q.row) {
    double2* dst = p.part ? p.part + (q.inst * p.nsegs + q.seg) * nterm * N * N : p.r.grad_A + q.inst * nterm * N * N;
    for (int i = 0; i < nterm; ++i)
      for (int k = 0; k < N; ++k) {
        const Z t = gA[(i * NT + k) * 64];
        dst[((int64_t)i * N + q.li) * N + k] = make_double2(t.x, t.y);
      }
  }
}

// grad_A = sum over segments, in order
__global__ __launch_bounds__(64) void small_reduce_kernel(SmParams p, int64_t n) {
  const int64_t e = blockIdx.x * (int64_t)64 + threadIdx.x;
  if (e >= n * p.r.n_inst) return;
  const int64_t inst = e / n, k = e - inst * n;
  double2 s = make_double2(0.0, 0.0);
#pragma unroll 4
  for (int64_t sg = 0; sg < p.nsegs; ++sg) {
    const double2 v = p.part[(inst * p.nsegs + sg) * n + k];
    s.x += v.x;
    s.y += v.y;
  }
  p.r.grad_A[e] = s;
}

// Checkpoints of an uncut adjoint: the states at the segments' starts, one chain per instance.
template <int NT, int G>
__global__ __launch_bounds__(64) void small_checkpoint_kernel(SmParams p) {
  extern __shared__ __align__(16) char smem[];
  const Carve<NT, G> c = carve_small<NT, G>(smem, p.r.nterm, 1);
  Grp<NT, G> q;
  q.place(p, 1, 1);
  q.s0 = 0;
  q.len = p.r.nsteps;
  stage_generators<NT, G>(p, c.sA);
  __syncthreads();
  const int N = p.r.N;
  Rows<NT, G, false> R;
  R.init(c.sA, q.li, p.r.nterm);
  Z v = mk(0.0, 0.0);
  if (q.row) v = mk(p.r.rho[q.inst * N + q.li].x, p.r.rho[q.inst * N + q.li].y);
  Field f{c.w, 0, 0, c.rows};
  for (int64_t s = 0; s < p.r.nsteps; ++s) {
    if (s % p.r.seg == 0 && q.row) p.r.ckpt[(q.inst * (p.nsegs + 1) + s / p.r.seg) * N + q.li] = make_double2(v.x, v.y);
    R.combine(field_row<NT, G>(p, q, f, s, false), true);
    v = v + rk4<NT, G>(R, v, c.x, q.li, p.r.dt);
  }
}

SmParams small_params(const LiouvilleRun& r) {
  SmParams p;
  std::memset(&p, 0, sizeof(p));
  p.r = r;
  p.nsegs = (r.nsteps + r.seg - 1) / r.seg;
  return p;
}

template <typename K>
int small_launch(K kernel, int64_t blocks, size_t lds, hipStream_t st, const SmParams& p) {
  if (lds > 65536)
    PQA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(64), lds, st, p);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

template <int NT, int G>
int forward_t(SmParams p, bool cols, hipStream_t st) {
  p.cols = cols ? p.r.N : 1;
  p.groups = (int64_t)p.r.n_inst * p.nsegs * p.cols;
  const int64_t blocks = (p.groups + 64 / G - 1) / (64 / G);
  const size_t lds = small_lds<NT, G>(p.r.nterm, 1);
  return cols ? small_launch(small_forward_kernel<NT, G, true>, blocks, lds, st, p)
              : small_launch(small_forward_kernel<NT, G, false>, blocks, lds, st, p);
}

template <int NT, int G>
int chain_t(const SmParams& p, int dirs, hipStream_t st) {
  hipLaunchKernelGGL((small_chain_kernel<NT, G>), dim3((unsigned)(p.r.n_inst * dirs)), dim3(64), 0, st, p, dirs);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

template <int NT, int G>
int adjoint_t(SmParams p, bool split, hipStream_t st) {
  const size_t lds1 = small_lds<NT, G>(p.r.nterm, 1);
  const size_t lds = small_lds<NT, G>(p.r.nterm, 5) + (p.r.grad_A ? sizeof(Z) * (size_t)p.r.nterm * NT * 64 : 0);
  p.groups = (int64_t)p.r.n_inst * (split ? p.nsegs : 1);
  p.seg_buf = (int64_t)p.r.n_inst * (p.nsegs + 1) * p.r.N;
  const int64_t blocks = (p.groups + 64 / G - 1) / (64 / G);
  if (!split) {
    const int rc = small_launch(small_checkpoint_kernel<NT, G>, blocks, lds1, st, p);
    if (rc) return rc;
  }
  if (lds > 65536)
    PQA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&small_adjoint_kernel<NT, G>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL((small_adjoint_kernel<NT, G>), dim3((unsigned)blocks), dim3(64), lds, st, p, split ? (int64_t)1 : p.nsegs);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

// by size: 4 lanes for N <= 4, 16 lanes beyond
#define PQA_SMALL(N, CALL4, CALL9, CALL16) ((N) <= 4 ? (CALL4) : (N) <= 9 ? (CALL9) : (CALL16))

}  // namespace

bool small_fits(int N, int nterm, bool grad_A) {
  if (N > kSmallN || nterm > 64) return false;
  const size_t nt = N <= 4 ? 4 : N <= 9 ? 9 : 16;
  const size_t lds = PQA_SMALL(N, (small_lds<4, 4>(nterm, 5)), (small_lds<9, 16>(nterm, 5)), (small_lds<16, 16>(nterm, 5))) +
                     (grad_A ? sizeof(Z) * (size_t)nterm * nt * 64 : 0);
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
    v = 65536;
  return lds <= (size_t)v;
}

int64_t small_split(int N, int nterm, int n_inst, int64_t nsteps, bool adjoint) {
  // The chain is seg steps for the propagators, nsteps / seg products of about 0.3 steps, and the sweep of
  // seg steps (forward; about three steps' time each with the adjoint): least at seg^2 = nsteps / 5 (or / 10);
  // fewer than six segments do not shorten it by enough.
  // The propagators are N times the forward work.  Once they fill the chip (4, 2, 1 wavefronts per SIMD by
  // their registers) they take `load` times the uncut forward run, whatever seg is.  Measured, uncut and cut:
  // 256 instances of N = 16 (load 1) forward 1487 and 1956 us, gradients 10.6 and 2.9 ms; 256 of N = 9 (0.28)
  // forward 1000 and 677 us, gradients 5.9 and 1.1 ms; 4096 of N = 4 (0.25) forward 278 and 317 us, gradients
  // 1.29 and 0.61 ms; 16384 of N = 4 (1) gradients 0.78 and 1.33 ms.
  const int lanes = N <= 4 ? 4 : 16, waves = N <= 4 ? 4 : N <= 9 ? 2 : 1;
  const double load = (double)n_inst * N * lanes / (65536.0 * waves);
  if (load > (adjoint ? (N <= 4 ? 0.5 : 1.5) : (N <= 4 ? 0.15 : 0.5))) return 0;
  int64_t seg = 4;
  while (seg * seg * (adjoint ? 10 : 5) < nsteps && seg < 64) ++seg;
  if ((nsteps + seg - 1) / seg < 6) return 0;
  // a cut run holds its propagators and a cut gradient every state besides, whatever checkpoints it was asked for
  return small_split_bytes(N, nterm, n_inst, nsteps, seg, adjoint) > kSplitBytes ? 0 : seg;
}

int64_t small_split_bytes(int N, int nterm, int n_inst, int64_t nsteps, int64_t seg, bool adjoint) {
  const int64_t nsegs = (nsteps + seg - 1) / seg, NN = (int64_t)N * N;
  int64_t el = n_inst * nsegs * NN + n_inst * (nsegs + 1) * N;  // propagators, segment starts
  if (adjoint) el += n_inst * nsegs * N + n_inst * nsegs * nterm * NN + n_inst * nsegs * seg * N;  // ends, gradient parts, states
  return el * (int64_t)sizeof(double2);
}

int small_forward(const LiouvilleRun& r0, hipStream_t st) {
  LiouvilleRun r = r0;
  r.seg = std::max<int64_t>(r.nsteps, 1);
  r.ckpt = nullptr;
  SmParams p = small_params(r);
  p.nsegs = 1;
  return PQA_SMALL(r.N, (forward_t<4, 4>(p, false, st)), (forward_t<9, 16>(p, false, st)), (forward_t<16, 16>(p, false, st)));
}

int small_forward_split(const LiouvilleRun& r, void* work, hipStream_t st) {
  SmParams p = small_params(r);
  p.Q = (double2*)work;
  p.r.ckpt = p.Q + (int64_t)r.n_inst * p.nsegs * r.N * r.N;
  int rc = PQA_SMALL(r.N, (forward_t<4, 4>(p, true, st)), (forward_t<9, 16>(p, true, st)), (forward_t<16, 16>(p, true, st)));
  if (rc) return rc;
  rc = PQA_SMALL(r.N, (chain_t<4, 4>(p, 1, st)), (chain_t<9, 16>(p, 1, st)), (chain_t<16, 16>(p, 1, st)));
  if (rc) return rc;
  return PQA_SMALL(r.N, (forward_t<4, 4>(p, false, st)), (forward_t<9, 16>(p, false, st)), (forward_t<16, 16>(p, false, st)));
}

int small_adjoint(const LiouvilleRun& r, hipStream_t st) {
  const SmParams p = small_params(r);
  return PQA_SMALL(r.N, (adjoint_t<4, 4>(p, false, st)), (adjoint_t<9, 16>(p, false, st)), (adjoint_t<16, 16>(p, false, st)));
}

int small_adjoint_split(const LiouvilleRun& r, void* work, hipStream_t st) {
  SmParams p = small_params(r);
  const int64_t N = r.N, NN = N * N;
  p.Q = (double2*)work;
  p.lamT = p.Q + r.n_inst * p.nsegs * NN;
  p.part = p.lamT + r.n_inst * p.nsegs * N;
  p.r.ckpt = p.part + r.n_inst * p.nsegs * r.nterm * NN;
  int rc = PQA_SMALL(r.N, (forward_t<4, 4>(p, true, st)), (forward_t<9, 16>(p, true, st)), (forward_t<16, 16>(p, true, st)));
  if (rc) return rc;
  rc = PQA_SMALL(r.N, (chain_t<4, 4>(p, 2, st)), (chain_t<9, 16>(p, 2, st)), (chain_t<16, 16>(p, 2, st)));
  if (rc) return rc;
  rc = PQA_SMALL(r.N, (adjoint_t<4, 4>(p, true, st)), (adjoint_t<9, 16>(p, true, st)), (adjoint_t<16, 16>(p, true, st)));
  if (rc || !r.grad_A) return rc;
  const int64_t n = r.nterm * NN;
  hipLaunchKernelGGL(small_reduce_kernel, dim3((unsigned)((n * r.n_inst + 63) / 64)), dim3(64), 0, st, p, n);
  PQA_HIP(hipGetLastError());
  return PYQED_OK;
}

}  // namespace pqa
