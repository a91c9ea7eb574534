// RK4 of a constant linear system dx/dt = G x on row vectors x (FP64): lime's Liouville-space
// _redfield (lime/oqs.py:373-472, rk4 over R vec(rho)) and the EOM propagator of phys.expm.
//
// One RK4 step of a constant generator is x := P x with
//   P = 1 + hG + (hG)^2/2 + (hG)^3/6 + (hG)^4/24,
// so P is formed once (three products) and a step is one product instead of four.  Steps are
// taken in blocks: with P^m (by squaring) the next m states of the trajectory are one product of the last
// m states, at most kMaxBlock of them.
//
// Rounding.  An error of the matrix comes back in every block, where step by step each step rounds anew,
// and of a state that decays by a factor q within a block the digits of q are lost if the matrix is
// held as P^m - 1 in 53 bits.  So the matrices are pairs of doubles (106 bits), in the form S + E with
// S = diag(s), s_i = 1 while |P^m_ii - 1| <= 1/2 (a slow element: x + E x rounds only what is added) and 0
// from then on (a decayed or rotated one).  Largest relative error of a record against 80 bits over
// 500 steps, step by step / P^m - 1 in 53 bits / here: uniform damping h x rate = 0.25 1.4e-14 / 2.6e-9 /
// 7.4e-16, 1.0 5.9e-14 / 1.0 / 4.0e-16; Redfield tensors of m = 4 .. 144 up to 1.9e-15 / 1.3e-14 / 1.1e-15.
//
// Stepping vec(rho) on the one-sided per-stage kernels (as column 0 of an m x m operator, m - 1
// zero columns beside it) took four launches of m^3 work per step, 44 us at m = 144.  A call of
// _redfield with one observable, on those / here: m = 144, 500 steps 22.1 / 0.49 ms, m = 256, 500 steps 35.7 /
// 0.82, m = 576, 100 steps 21.3 / 2.7, m = 1024, 20 steps 13.5 / 1.4, 300 steps 178 / 14.5 (matrices of 53 bits:
// 0.39, 0.45, 0.83, 1.4, 2.9).
#include "common.hpp"
#include "linear_rk4_decl.hpp"

namespace lime {

namespace {

// C = alpha A (B + B2)^T + beta Z  (A [rows][k], B [cols][k], Z and C [rows][cols], row-major); B2
// (the pair's low part) may be NULL, zs [cols] or NULL scales Z by columns in beta's place.
struct RowProduct {
  const double2* a;
  const double2* b;
  const double2* b2;
  const double2* z;
  const double* zs;
  double2* c;
  int rows, cols, k;
  double alpha, beta;
};

// A matrix of pairs: value h + l, |l| <= ulp(h) / 2
struct Pair {
  double2 *h, *l;
};

// C = w Z + alpha A B for m x m matrices of pairs: w = 1 or (s given) s_i + s_j, alpha a pair.  With `near`
// given, C = P - diag(near) is formed from the result T = P - diag(t), t = 1 or s.
struct ExactProduct {
  Pair a, b, z, c;
  const double* s;
  double* near;
  double alpha_h, alpha_l;
  int m;
};

constexpr int kMaxBlock = 64;
constexpr int kExactWaves = 8;
// a product: its launch, its arithmetic, and reading the m x m operand; one of pairs: its launch and latency,
// complex products a second
constexpr double kLaunchS = 6e-6, kProductRate = 2e13, kReadRate = 3e12, kExactS = 1.1e-5, kExactRate = 6e11;

__device__ __forceinline__ doublex4 mfma_f64(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

}  // namespace

// Latency-bound at the sizes it runs (m = 4 .. 256: a few to a few hundred 16 x 16 tiles, operands
// in L2), so there is no LDS staging: both operands are read by rows, 16 rows x 64 B a fragment,
// four k-steps of loads in flight.  KS = 4: a workgroup is one 16 x 16 tile whose reduction its
// four waves share (the partial sums meet in LDS in wave order: deterministic), for few tiles;
// KS = 1: four tiles, one a wave.  PAIR: B comes with its low part B2.
template <int KS, bool PAIR>
__global__ void __launch_bounds__(256) row_product(RowProduct g) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int EDGE = KS == 1 ? 32 : 16;
  const int tc = cdiv(g.cols, EDGE);
  const int row0 = ((int)blockIdx.x / tc) * EDGE + (KS == 1 ? (w >> 1) * 16 : 0);
  const int col0 = ((int)blockIdx.x % tc) * EDGE + (KS == 1 ? (w & 1) * 16 : 0);
  const int part = KS == 1 ? g.k : 4 * cdiv(g.k, 4 * KS);
  const int kb = KS == 1 ? 0 : w * part, ke = KS == 1 ? g.k : min(g.k, kb + part);
  // rows and columns beyond the operands read a valid row and are never stored
  const double2* A = g.a + (size_t)min(row0 + lr, g.rows - 1) * g.k;
  const double2* B = g.b + (size_t)min(col0 + lr, g.cols - 1) * g.k;
  const double2* B2 = PAIR ? g.b2 + (size_t)min(col0 + lr, g.cols - 1) * g.k : nullptr;
  doublex4 xx = {0, 0, 0, 0}, yy = xx, xy = xx, yx = xx;
  constexpr int U = 4;
  for (int k0 = kb; k0 < ke; k0 += 4 * U) {
    double2 a[U], b[U], d[PAIR ? U : 1];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 4 * u + lg;
      const int kc = min(k, g.k - 1);
      a[u] = A[kc];
      b[u] = B[kc];
      if constexpr (PAIR) d[u] = B2[kc];
      if (k >= ke) {
        a[u] = b[u] = make_double2(0.0, 0.0);
        if constexpr (PAIR) d[u] = a[u];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (PAIR) {
        xx = mfma_f64(a[u].x, d[u].x, xx);
        yy = mfma_f64(a[u].y, d[u].y, yy);
        xy = mfma_f64(a[u].x, d[u].y, xy);
        yx = mfma_f64(a[u].y, d[u].x, yx);
      }
      xx = mfma_f64(a[u].x, b[u].x, xx);
      yy = mfma_f64(a[u].y, b[u].y, yy);
      xy = mfma_f64(a[u].x, b[u].y, xy);
      yx = mfma_f64(a[u].y, b[u].x, yx);
    }
  }
  doublex4 re = xx - yy, im = xy + yx;
  const auto finish = [&](int r, int c, double tr, double ti) {
    const size_t o = (size_t)r * g.cols + c;
    double2 y = make_double2(g.alpha * tr, g.alpha * ti);
    if (g.z) {
      const double w = g.zs ? g.zs[c] : g.beta;
      y.x += w * g.z[o].x;
      y.y += w * g.z[o].y;
    }
    g.c[o] = y;
  };
  if constexpr (KS > 1) {
    __shared__ double2 sum[KS][16][16];
#pragma unroll
    for (int v = 0; v < 4; ++v) sum[w][lg + 4 * v][lr] = make_double2(re[v], im[v]);
    __syncthreads();
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    double2 t = sum[0][r][c];
    for (int x = 1; x < KS; ++x) {
      t.x += sum[x][r][c].x;
      t.y += sum[x][r][c].y;
    }
    if (row0 + r < g.rows && col0 + c < g.cols) finish(row0 + r, col0 + c, t.x, t.y);
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = row0 + lg + 4 * v, c = col0 + lr;   // FP64 accumulator rows: lg + 4 v
      if (r < g.rows && c < g.cols) finish(r, c, re[v], im[v]);
    }
  }
}

// ---- sums of pairs (Dekker, Knuth): exact sums and products of doubles by FMA, nothing contracted
struct DD {
  double h, l;
};
__device__ __forceinline__ DD two_sum(double a, double b) {
#pragma clang fp contract(off)
  const double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
__device__ __forceinline__ DD dd_add(DD a, DD b) {
#pragma clang fp contract(off)
  const DD s = two_sum(a.h, b.h), t = two_sum(a.l, b.l);
  const double l = s.l + t.h, h = s.h + l;
  const double r = (l - (h - s.h)) + t.l;
  return {h + r, r - ((h + r) - h)};
}
__device__ __forceinline__ DD dd_mul(DD a, DD b) {
#pragma clang fp contract(off)
  const double p = a.h * b.h;
  const double e = fma(a.h, b.l, fma(a.l, b.h, fma(a.h, b.h, -p)));
  return {p + e, e - ((p + e) - p)};
}
// acc += a b: the product's and the sum's errors are collected in acc.l
__device__ __forceinline__ void dd_fma(DD& acc, double ah, double al, double bh, double bl) {
#pragma clang fp contract(off)
  const double p = ah * bh;
  const DD s = two_sum(acc.h, p);
  acc.l += s.l + fma(al, bh, fma(ah, bl, fma(ah, bh, -p)));
  acc.h = s.h;
}

// Pairs have no matrix instruction: 48 FP64 vector instructions per complex product and sum.  An 8 x 8 tile
// of outputs a workgroup, its reduction shared by the waves (partial sums meet in LDS, in wave order), so
// that m = 144 is 324 workgroups and a lane sums 18 products.  Operands come from L2.  Issue-bound from m = 256
// on (8e11 complex products a second, the FP64 vector rate); four / eight / sixteen waves: a call at m = 144, 500
// steps 277 / 261 / 298 us, m = 100 180 / 157 / 158, m = 400 1431 / 1438 / 1610.
__global__ void __launch_bounds__(64 * kExactWaves) exact_product(ExactProduct g) {
  const int m = g.m, tiles = cdiv(m, 8);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = (int)blockIdx.x / tiles * 8 + (lane >> 3), j = (int)blockIdx.x % tiles * 8 + (lane & 7);
  const size_t ri = (size_t)min(i, m - 1) * m;       // rows and columns beyond m read the last one
  const int cj = min(j, m - 1), part = cdiv(m, kExactWaves), ke = min(m, (w + 1) * part);
  DD re = {0.0, 0.0}, im = re;
#pragma unroll 4
  for (int k = w * part; k < ke; ++k) {
    const double2 ah = g.a.h[ri + k], al = g.a.l[ri + k];
    const double2 bh = g.b.h[(size_t)k * m + cj], bl = g.b.l[(size_t)k * m + cj];
    dd_fma(re, ah.x, al.x, bh.x, bl.x);
    dd_fma(re, -ah.y, -al.y, bh.y, bl.y);
    dd_fma(im, ah.x, al.x, bh.y, bl.y);
    dd_fma(im, ah.y, al.y, bh.x, bl.x);
  }
  __shared__ DD sum[kExactWaves][64][2];
  sum[w][lane][0] = re;
  sum[w][lane][1] = im;
  __syncthreads();
  if (w > 0 || i >= m || j >= m) return;
  const size_t o = ri + j;
  const double2 zh = g.z.h[o], zl = g.z.l[o];
  double ch[2], cl[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    DD t = sum[0][lane][x];
    for (int p = 1; p < kExactWaves; ++p) t = dd_add(t, sum[p][lane][x]);
    t = dd_mul(t, DD{g.alpha_h, g.alpha_l});
    const double wt = g.s ? g.s[i] + g.s[j] : 1.0;   // 0, 1 or 2: exact
    t = dd_add(t, x == 0 ? DD{wt * zh.x, wt * zl.x} : DD{wt * zh.y, wt * zl.y});
    ch[x] = t.h;
    cl[x] = t.l;
  }
  if (g.near && i == j) {
    double near = g.s ? g.s[i] : 1.0;
    if (near != 0.0 && ch[0] * ch[0] + ch[1] * ch[1] > 0.25) {
      near = 0.0;
      const DD t = dd_add(DD{ch[0], cl[0]}, DD{1.0, 0.0});
      ch[0] = t.h;
      cl[0] = t.l;
    }
    g.near[i] = near;
  }
  g.c.h[o] = make_double2(ch[0], ch[1]);
  g.c.l[o] = make_double2(cl[0], cl[1]);
}

// c = h g as pairs
__global__ void __launch_bounds__(256) exact_scale(const double2* g, double h, Pair c, size_t count) {
#pragma clang fp contract(off)
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= count) return;
  const double2 v = g[o], p = make_double2(h * v.x, h * v.y);
  c.h[o] = p;
  c.l[o] = make_double2(fma(h, v.x, -p.x), fma(h, v.y, -p.y));
}

static void launch_rows(const RowProduct& g, hipStream_t stream) {
  // one workgroup per 16 x 16 tile while those do not fill the 256 CUs twice over
  const long long t16 = (long long)cdiv(g.rows, 16) * cdiv(g.cols, 16);
  const dim3 few((unsigned)t16), many((unsigned)(cdiv(g.rows, 32) * cdiv(g.cols, 32)));
  if (t16 <= 512) {
    if (g.b2) hipLaunchKernelGGL((row_product<4, true>), few, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((row_product<4, false>), few, dim3(256), 0, stream, g);
  } else {
    if (g.b2) hipLaunchKernelGGL((row_product<1, true>), many, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((row_product<1, false>), many, dim3(256), 0, stream, g);
  }
}

// c = alpha a b^T + z
static void product(const double2* a, const double2* b, const double2* z, double2* c, int rows, int cols, int k,
                    double alpha, hipStream_t stream) {
  launch_rows({a, b, nullptr, z, nullptr, c, rows, cols, k, alpha, 1.0}, stream);
}

static size_t round256(size_t x) { return (x + 255) & ~(size_t)255; }

// hG and two buffers for the blocks' matrices, pairs each, and two rows of s
size_t linear_workspace_bytes(int m) {
  return 6 * round256((size_t)m * m * sizeof(double2)) + 2 * round256((size_t)m * sizeof(double));
}

// Steps per block, or 0 for four products a step with G itself (few steps of a large generator,
// where three products of m x m matrices cost more than they save).  Doubling from m to 2 m steps
// is a product of matrices and one of the block's states, a block one product of its states.
static int block_steps(int m, int rows, int nsteps) {
  const double mm = 8.0 * m * (double)m;
  if (rows > m) return 1;                     // the vectors between products fit m rows
  // the products of the states: with G, and with a pair of matrices
  const auto cost = [&](double r, int parts) { return kLaunchS + parts * (mm * r / kProductRate + 2 * mm / kReadRate); };
  const double exact = kExactS + (double)m * m * m / kExactRate;
  int best = 0;
  double least = 4.0 * nsteps * cost(rows, 1);
  for (int b = 1, doublings = 0; b <= kMaxBlock && b <= nsteps; b *= 2, ++doublings) {
    const double c = 3 * exact + doublings * (exact + cost(0.5 * b * rows, 2)) + cdiv(nsteps, b) * cost((double)b * rows, 2);
    if (c < least) {
      best = b;
      least = c;
    }
  }
  return best;
}

hipError_t linear_run(const LinearArgs& a, void* work, hipStream_t stream) {
  const int m = a.m;
  const double h = a.dt;
  const size_t mm = (size_t)m * m, vec = (size_t)a.rows * m;
  unsigned char* base = static_cast<unsigned char*>(work);
  const size_t step = round256(mm * sizeof(double2)), srow = round256(m * sizeof(double));
  const auto matrix = [&](int x) { return reinterpret_cast<double2*>(base + x * step); };
  const Pair hg = {matrix(0), matrix(1)}, e[2] = {{matrix(2), matrix(3)}, {matrix(4), matrix(5)}};
  double* s[2] = {reinterpret_cast<double*>(base + 6 * step), reinterpret_cast<double*>(base + 6 * step + srow)};
  const int block = block_steps(m, a.rows, a.nsteps);
  const auto finish = [&]() {
    if (a.obs) product(a.states, a.eops, nullptr, a.obs, a.nsteps * a.rows, a.n_e, m, 1.0, stream);
    const hipError_t err = hipMemcpyAsync(a.x, a.states + (size_t)(a.nsteps - 1) * vec, vec * sizeof(double2),
                                        hipMemcpyDeviceToDevice, stream);
    return err != hipSuccess ? err : hipGetLastError();
  };
  if (block == 0) {
    // x' = x + h (x + h/2 (x + h/3 (x + h/4 x G^T) G^T) G^T) G^T
    double2 *u = matrix(0), *v = matrix(1);
    const double2* x = a.x;
    for (int s = 0; s < a.nsteps; ++s) {
      double2* y = a.states + s * vec;
      product(x, a.gen, x, u, a.rows, m, m, h / 4, stream);
      product(u, a.gen, x, v, a.rows, m, m, h / 3, stream);
      product(v, a.gen, x, u, a.rows, m, m, h / 2, stream);
      product(u, a.gen, x, y, a.rows, m, m, h, stream);
      x = y;
    }
    return finish();
  }
  const int tiles = cdiv(m, 8);
  const auto exact = [&](const Pair& x, const Pair& y, const Pair& z, const Pair& c, const double* w, double* near,
                         double alpha, double alpha_low) {
    const ExactProduct g = {x, y, z, c, w, near, alpha, alpha_low, m};
    hipLaunchKernelGGL(exact_product, dim3((unsigned)(tiles * tiles)), dim3(64 * kExactWaves), 0, stream, g);
  };
  // y := P^b x for `rows` states, P^b = diag(s) + e
  const auto advance = [&](const double2* x, double2* y, int rows, int cur) {
    launch_rows({x, e[cur].h, e[cur].l, x, s[cur], y, rows, m, m, 1.0, 0.0}, stream);
  };
  // P - 1 by Horner's rule (every factor is a polynomial of G, so the order of a product is free)
  hipLaunchKernelGGL(exact_scale, dim3((unsigned)((mm + 255) / 256)), dim3(256), 0, stream, a.gen, h, hg, mm);
  const double third = 1.0 / 3.0;
  exact(hg, hg, hg, e[0], nullptr, nullptr, 0.25, 0.0);
  exact(hg, e[0], hg, e[1], nullptr, nullptr, third, fma(-3.0, third, 1.0) / 3.0);
  exact(hg, e[1], hg, e[0], nullptr, s[0], 0.5, 0.0);
  advance(a.x, a.states, a.rows, 0);
  int have = 1, cur = 0;
  for (; have < block; have *= 2, cur ^= 1) {
    // states have .. 2 have - 1 from the first `have`, then the matrix of twice the steps:
    // (S + E)^2 = S + (s_i + s_j) E + E E
    const int more = have < a.nsteps - have ? have : a.nsteps - have;
    if (more > 0) advance(a.states, a.states + have * vec, more * a.rows, cur);
    if (2 * have < a.nsteps) exact(e[cur], e[cur], e[cur], e[cur ^ 1], s[cur], s[cur ^ 1], 1.0, 0.0);
  }
  for (int done = have; done < a.nsteps; done += block) {
    const int more = block < a.nsteps - done ? block : a.nsteps - done;
    advance(a.states + (done - block) * vec, a.states + done * vec, more * a.rows, cur);
  }
  return finish();
}

}  // namespace lime
