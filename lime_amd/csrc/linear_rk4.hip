// RK4 of a constant linear system dx/dt = G x on row vectors x (FP64): lime's Liouville-space
// _redfield (lime/oqs.py:373-472, rk4 over R vec(rho)) and the EOM propagator of phys.expm.
//
// One RK4 step of a constant generator is x += D x with
//   D = hG + (hG)^2/2 + (hG)^3/6 + (hG)^4/24,
// so D is formed once (three products) and a step is one product instead of four.  Steps are
// taken in blocks: with D_m = (1 + D)^m - 1 (doubling: D_2m = 2 D_m + D_m D_m) the next m states
// of the trajectory are one product of the last m states with D_m.  Only the increments D_m are
// rounded, not 1 + D_m, and a block is at most kMaxBlock steps, so rounding grows as in the
// step-by-step form (500 steps of a 144-dimensional Redfield tensor: 2e-14 of the state from the
// 64-bit reference, 2e-14 step by step).
//
// Stepping vec(rho) on the one-sided per-stage kernels (as column 0 of an m x m operator, m - 1
// zero columns beside it) took four launches of m^3 work per step, 47 us at m = 144.  A call of
// _redfield at m = 144, 500 steps, 3 observables went from 23.5 ms to 0.59 ms (24 products of
// ~6 us, the rest copies and host work), m = 256, 1000 steps from 71 to 0.74 ms, m = 1024, one
// step from 1.3 to 0.7 ms; phys.expm at m = 144, 20 steps from 1.33 to 0.59 ms.
#include "common.hpp"
#include "linear_rk4_decl.hpp"

namespace lime {

namespace {

// C = alpha A B^T + beta Z  (A [rows][k], B [cols][k], Z and C [rows][cols], row-major), and
// C^T in ct (square C only).
struct RowProduct {
  const double2* a;
  const double2* b;
  const double2* z;
  double2* c;
  double2* ct;
  int rows, cols, k;
  double alpha, beta;
};

constexpr int kMaxBlock = 64;
// a product: its launch, its arithmetic, and reading the m x m operand
constexpr double kLaunchS = 6e-6, kProductRate = 2e13, kReadRate = 3e12;

__device__ __forceinline__ doublex4 mfma_f64(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

}  // namespace

// Latency-bound at the sizes it runs (m = 4 .. 256: a few to a few hundred 16 x 16 tiles, operands
// in L2), so there is no LDS staging: both operands are read by rows, 16 rows x 64 B a fragment,
// four k-steps of loads in flight.  KS = 4: a workgroup is one 16 x 16 tile whose reduction its
// four waves share (the partial sums meet in LDS in wave order: deterministic), for few tiles;
// KS = 1: four tiles, one a wave.
template <int KS>
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
  doublex4 xx = {0, 0, 0, 0}, yy = xx, xy = xx, yx = xx;
  constexpr int U = 4;
  for (int k0 = kb; k0 < ke; k0 += 4 * U) {
    double2 a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 4 * u + lg;
      const int kc = min(k, g.k - 1);
      a[u] = A[kc];
      b[u] = B[kc];
      if (k >= ke) a[u] = b[u] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      xx = mfma_f64(a[u].x, b[u].x, xx);
      yy = mfma_f64(a[u].y, b[u].y, yy);
      xy = mfma_f64(a[u].x, b[u].y, xy);
      yx = mfma_f64(a[u].y, b[u].x, yx);
    }
  }
  doublex4 re = xx - yy, im = xy + yx;
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
    if (row0 + r < g.rows && col0 + c < g.cols) {
      const size_t o = (size_t)(row0 + r) * g.cols + col0 + c;
      double2 y = make_double2(g.alpha * t.x, g.alpha * t.y);
      if (g.z) {
        y.x += g.beta * g.z[o].x;
        y.y += g.beta * g.z[o].y;
      }
      g.c[o] = y;
      if (g.ct) g.ct[(size_t)(col0 + c) * g.rows + row0 + r] = y;
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = row0 + lg + 4 * v, c = col0 + lr;   // FP64 accumulator rows: lg + 4 v
      if (r >= g.rows || c >= g.cols) continue;
      const size_t o = (size_t)r * g.cols + c;
      double2 y = make_double2(g.alpha * re[v], g.alpha * im[v]);
      if (g.z) {
        y.x += g.beta * g.z[o].x;
        y.y += g.beta * g.z[o].y;
      }
      g.c[o] = y;
      if (g.ct) g.ct[(size_t)c * g.rows + r] = y;
    }
  }
}

__global__ void __launch_bounds__(256) transpose_square(const double2* __restrict__ a, double2* __restrict__ t, int m) {
  __shared__ double2 tile[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int i0 = blockIdx.y * 16, j0 = blockIdx.x * 16;
  if (i0 + ty < m && j0 + tx < m) tile[ty][tx] = a[(size_t)(i0 + ty) * m + j0 + tx];
  __syncthreads();
  if (j0 + ty < m && i0 + tx < m) t[(size_t)(j0 + ty) * m + i0 + tx] = tile[tx][ty];
}

static void product(const double2* a, const double2* b, const double2* z, double2* c, double2* ct, int rows, int cols,
                    int k, double alpha, double beta, hipStream_t stream) {
  RowProduct g = {a, b, z, c, ct, rows, cols, k, alpha, beta};
  // one workgroup per 16 x 16 tile while those do not fill the 256 CUs twice over
  const long long t16 = (long long)cdiv(rows, 16) * cdiv(cols, 16);
  if (t16 <= 512)
    hipLaunchKernelGGL(row_product<4>, dim3((unsigned)t16), dim3(256), 0, stream, g);
  else
    hipLaunchKernelGGL(row_product<1>, dim3((unsigned)(cdiv(rows, 32) * cdiv(cols, 32))), dim3(256), 0, stream, g);
}

static size_t round256(size_t x) { return (x + 255) & ~(size_t)255; }

// G^T, two buffers for the increments and two for their transposes
size_t linear_workspace_bytes(int m) { return 5 * round256((size_t)m * m * sizeof(double2)); }

// Steps per block, or 0 for four products a step with G itself (few steps of a large generator,
// where three products of m x m matrices cost more than they save).  Doubling from m to 2 m steps
// is a product of matrices and one of the block's states, a block one product of its states.
static int block_steps(int m, int rows, int nsteps) {
  const double mm = 8.0 * m * (double)m;
  if (rows > m) return 1;                     // the vectors between products fit m rows
  const auto cost = [&](double r) { return kLaunchS + mm * r / kProductRate + 2 * mm / kReadRate; };
  int best = 0;
  double least = 4.0 * nsteps * cost(rows);
  for (int b = 1, doublings = 0; b <= kMaxBlock && b <= nsteps; b *= 2, ++doublings) {
    const double c = 3 * cost(m) + doublings * (cost(m) + cost(0.5 * b * rows)) + cdiv(nsteps, b) * cost((double)b * rows);
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
  const size_t step = round256(mm * sizeof(double2));
  double2* gt = reinterpret_cast<double2*>(base);
  double2* d[2] = {reinterpret_cast<double2*>(base + step), reinterpret_cast<double2*>(base + 2 * step)};
  double2* dt[2] = {reinterpret_cast<double2*>(base + 3 * step), reinterpret_cast<double2*>(base + 4 * step)};
  const int block = block_steps(m, a.rows, a.nsteps);
  const auto finish = [&]() {
    if (a.obs)
      product(a.states, a.eops, nullptr, a.obs, nullptr, a.nsteps * a.rows, a.n_e, m, 1.0, 0.0, stream);
    const hipError_t e = hipMemcpyAsync(a.x, a.states + (size_t)(a.nsteps - 1) * vec, vec * sizeof(double2),
                                        hipMemcpyDeviceToDevice, stream);
    return e != hipSuccess ? e : hipGetLastError();
  };
  if (block == 0) {
    // x' = x + h (x + h/2 (x + h/3 (x + h/4 x G^T) G^T) G^T) G^T
    const double2* x = a.x;
    for (int s = 0; s < a.nsteps; ++s) {
      double2* y = a.states + s * vec;
      product(x, a.gen, x, d[0], nullptr, a.rows, m, m, h / 4, 1.0, stream);
      product(d[0], a.gen, x, d[1], nullptr, a.rows, m, m, h / 3, 1.0, stream);
      product(d[1], a.gen, x, d[0], nullptr, a.rows, m, m, h / 2, 1.0, stream);
      product(d[0], a.gen, x, y, nullptr, a.rows, m, m, h, 1.0, stream);
      x = y;
    }
    return finish();
  }
  // D by Horner's rule (every factor is a polynomial of G, so the order of a product is free):
  // T2 = G + h/4 G G, T3 = G + h/3 T2 G, D = h G + h^2/2 T3 G
  hipLaunchKernelGGL(transpose_square, dim3(cdiv(m, 16), cdiv(m, 16)), dim3(256), 0, stream, a.gen, gt, m);
  product(a.gen, gt, a.gen, d[1], nullptr, m, m, m, h / 4, 1.0, stream);
  product(d[1], gt, a.gen, dt[1], nullptr, m, m, m, h / 3, 1.0, stream);
  product(dt[1], gt, a.gen, d[0], dt[0], m, m, m, h * h / 2, h, stream);
  product(a.x, d[0], a.x, a.states, nullptr, a.rows, m, m, 1.0, 1.0, stream);
  int have = 1, cur = 0;
  for (; have < block; have *= 2, cur ^= 1) {
    // states have .. 2 have - 1 from the first `have`, then the increment of twice the steps
    const int more = have < a.nsteps - have ? have : a.nsteps - have;
    if (more > 0)
      product(a.states, d[cur], a.states, a.states + have * vec, nullptr, more * a.rows, m, m, 1.0, 1.0, stream);
    if (2 * have < a.nsteps)
      product(d[cur], dt[cur], d[cur], d[cur ^ 1], dt[cur ^ 1], m, m, m, 1.0, 2.0, stream);
  }
  for (int s = have; s < a.nsteps; s += block) {
    const int more = block < a.nsteps - s ? block : a.nsteps - s;
    product(a.states + (s - block) * vec, d[cur], a.states + (s - block) * vec, a.states + s * vec, nullptr,
            more * a.rows, m, m, 1.0, 1.0, stream);
  }
  return finish();
}

}  // namespace lime
