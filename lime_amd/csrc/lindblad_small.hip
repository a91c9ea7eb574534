// Lindblad RK4 for the smallest operators (n <= 16): the resident kernel's algorithm with one
// lane per matrix element and the products on the vector units.
//
// A 16 x 16 MFMA tile spends 16 x 16 x 4 products on what an n = 8 operator needs a quarter of,
// and its lane owns 4 elements, half of them padding, so one wave issues 512 cycles of MFMA and
// four elements' FP64 epilogue in a row: 1760 cycles a stage.  Here n <= 8 is one wave with one
// element a lane (64 FMAs of k, 256 cycles), n <= 4 four operators a wave, n <= 16 four waves.
// Rows i and j of H_eff stay in registers; S is exchanged through two LDS buffers (one barrier a
// stage, none across waves for n <= 8).
//
// The order of the products is the resident kernel's: the FP32 MFMA adds its four products one
// after the other, each rounded like an FMA, so the results are the same bits as on the tiles.  The FP64 trace
// of a renormalisation too: its elements lie on other lanes for n <= 8, but pair up in the same tree
// (n = 1 .. 8, with and without, against a build that ran them on the tiles).
#include "common.hpp"
#include "lindblad_resident_decl.hpp"

namespace lime {

namespace {

template <int NS>
struct Small {
  static constexpr int LPO = NS * NS;                 // lanes per operator
  static constexpr int T = LPO < 64 ? 64 : LPO;       // threads per workgroup
  static constexpr int OPS = T / LPO;                 // operators per workgroup
  static constexpr int P = NS + 2;                    // row pitch: even, so rows are read in 16 bytes
  static constexpr int MAT = NS * P;
};

// Sum over the lanes of one operator, to every lane of its wave's part (n <= 8: the operator).
template <int NS>
__device__ __forceinline__ double op_sum(double x) {
  if constexpr (NS == 4) {
    x += dpp_f64<0xB1>(x);
    x += dpp_f64<0x4E>(x);
    x += dpp_f64<0x141>(x);
    x += dpp_f64<0x140>(x);
    return x;
  } else {
    return wave_sum(x);
  }
}

// x[k] = M[r][k], k < NS, a row in LDS (two elements a read)
template <int NS>
__device__ __forceinline__ void lds_row(float2 (&x)[NS], const float2* row) {
#pragma unroll
  for (int k = 0; k < NS; k += 2) {
    const float4 v = *reinterpret_cast<const float4*>(row + k);
    x[k] = make_float2(v.x, v.y);
    x[k + 1] = make_float2(v.z, v.w);
  }
}

}  // namespace

template <int NS, bool DENSE, bool DRV>
__global__ void __launch_bounds__(Small<NS>::T) lindblad_rk4_small(ResidentArgs a) {
  using G = Small<NS>;
  constexpr int P = G::P, MAT = G::MAT;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x;
  const int q = tid / G::LPO, e = tid % G::LPO;       // operator of the workgroup, element
  const int i = e / NS, j = e % NS;
  const int n = a.n, nn = n * n;
  const int b0 = xcd_block() * G::OPS + q;
  const bool valid = b0 < a.batch;
  const int b = valid ? b0 : a.batch - 1;
  const bool act = i < n && j < n, own = act && valid;
  const int set = b / a.group, o = act ? i * n + j : 0;
  const int mats = DENSE ? a.n_dense * (a.rops ? 2 : 1) : 0;
  // LDS: per operator S twice (then T twice and the dense operands), then its observables when
  // they are staged; then the waves' partial sums
  const int per = (DENSE ? 4 + mats : 2) * MAT;
  float2* sS = reinterpret_cast<float2*>(lds_raw) + (size_t)q * per;
  float2* sT = sS + 2 * MAT;
  float2* sL = sS + 4 * MAT;
  double2* sE0 = reinterpret_cast<double2*>(reinterpret_cast<float2*>(lds_raw) + (size_t)G::OPS * per);
  double2* sE = sE0 + (size_t)q * a.op_pitch * nn;    // op_pitch: observables staged per operator
  double2* sRed = sE0 + (size_t)G::OPS * a.op_pitch * nn;

  for (int x = tid; x < G::OPS * per; x += G::T) reinterpret_cast<float2*>(lds_raw)[x] = make_float2(0.f, 0.f);
  __syncthreads();
  const double2* E = a.eops_t + (size_t)(b / a.eop_group) * a.n_eops * nn;
  if (act) {
    for (int x = 0; x < a.op_pitch; ++x) sE[x * nn + o] = E[(size_t)x * nn + o];
    for (int m = 0; m < mats; ++m) {
      const float2* src = m < a.n_dense ? a.lops + ((size_t)set * a.n_dense + m) * nn
                                        : a.rops + ((size_t)set * a.n_dense + m - a.n_dense) * nn;
      sL[m * MAT + i * P + j] = src[o];
    }
  }

  float2 hi[NS], hj[NS];                              // rows i and j of H_eff
  const auto load_h = [&](const float2* H, float2 (&u)[NS], float2 (&v)[NS]) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const bool in = act && k < n;
      u[k] = in ? H[i * n + k] : make_float2(0.f, 0.f);
      v[k] = in ? H[j * n + k] : make_float2(0.f, 0.f);
    }
  };
  const float2* H0 = a.heff + (size_t)set * nn;
  load_h(H0, hi, hj);
  double2 rho = make_double2(0.0, 0.0);
  if (act) rho = a.rho[(size_t)b * nn + o];
  const bool has_d = a.dmat != nullptr;
  const float2 d = has_d && act ? a.dmat[(size_t)set * nn + o] : make_float2(0.f, 0.f);
  float2 inc = make_float2(0.f, 0.f);
  float2 sv = make_float2((float)rho.x, (float)rho.y);
  if (act) sS[i * P + j] = sv;
  __syncthreads();

  const double dt = a.dt;
  const bool renorm = (a.flags & 1) != 0;
  const bool record_any = a.nout > 0 && (a.obs != nullptr || a.states != nullptr);
  int ph = 0;
  for (int s = 0; s < a.nsteps; ++s) {
    float2 hin[DRV ? NS : 1], hjn[DRV ? NS : 1];      // the next step's generator, on its way
    if constexpr (DRV) {
      if (s + 1 < a.nsteps) load_h(H0 + (size_t)(s + 1) * a.heff_step, hin, hjn);
    }
#pragma unroll 1
    for (int st = 0; st < 4; ++st) {
      const float2* S = sS + ph * MAT;
      float2 y[NS], z[NS];                            // S[k][j], S[i][k]
#pragma unroll
      for (int k = 0; k < NS; ++k) y[k] = S[k * P + j];
      lds_row<NS>(z, S + i * P);
      // the accumulators of the resident kernel: (cr, ci) with D o S added at the end, or with
      // dense operators the split-sign ones (cr - dr, ci - di) with D o S as start values
      float cr = 0.f, ci = 0.f, dr = 0.f, di = 0.f;
      if constexpr (DENSE) {
        cr = -fmaf(d.x, sv.y, d.y * sv.x);
        ci = fmaf(d.x, sv.x, -(d.y * sv.y));
      }
#pragma unroll
      for (int kb = 0; kb < NS; kb += 4) {
        if (kb >= n) break;
        const auto each = [&](float& c, float sign, auto u, auto v) {
#pragma unroll
          for (int k = kb; k < kb + 4; ++k) c = fmaf(sign * u(k), v(k), c);
        };
        const auto xx = [&](int k) { return hi[k].x; };
        const auto xy = [&](int k) { return hi[k].y; };
        const auto yx = [&](int k) { return y[k].x; };
        const auto yy = [&](int k) { return y[k].y; };
        const auto zx = [&](int k) { return z[k].x; };
        const auto zy = [&](int k) { return z[k].y; };
        const auto hx = [&](int k) { return hj[k].x; };
        const auto hy = [&](int k) { return hj[k].y; };
        if constexpr (DENSE) {
          each(cr, 1.f, xx, yx);
          each(ci, 1.f, xx, yy);
          each(dr, 1.f, xy, yy);
          each(di, 1.f, zy, hx);
          each(ci, 1.f, xy, yx);
          each(dr, 1.f, zx, hx);
          each(ci, 1.f, zx, hy);
          each(dr, 1.f, zy, hy);
        } else {
          each(cr, 1.f, xx, yx);
          each(ci, 1.f, xx, yy);
          each(cr, -1.f, xy, yy);
          each(ci, 1.f, xy, yx);
          each(cr, -1.f, zx, hx);
          each(ci, 1.f, zx, hy);
          each(cr, -1.f, zy, hy);
          each(ci, -1.f, zy, hx);
        }
      }
      if constexpr (DENSE) {
        cr -= dr;
        ci -= di;
        for (int m = 0; m < a.n_dense; ++m) {
          // T = L S, exchanged through one of two buffers; C += i T R^dag
          float2 l[NS];
          lds_row<NS>(l, sL + m * MAT + i * P);
          float tr = 0.f, ti = 0.f;
#pragma unroll
          for (int kb = 0; kb < NS; kb += 4) {
            if (kb >= n) break;
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) tr = fmaf(l[k].x, y[k].x, tr);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) ti = fmaf(l[k].x, y[k].y, ti);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) tr = fmaf(-l[k].y, y[k].y, tr);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) ti = fmaf(l[k].y, y[k].x, ti);
          }
          float2* Tm = sT + (m & 1) * MAT;
          if (act) Tm[i * P + j] = make_float2(tr, ti);
          __syncthreads();
          float2 t[NS];
          lds_row<NS>(t, Tm + i * P);
          lds_row<NS>(l, sL + (a.rops ? a.n_dense + m : m) * MAT + j * P);
#pragma unroll
          for (int kb = 0; kb < NS; kb += 4) {
            if (kb >= n) break;
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) cr = fmaf(t[k].x, l[k].y, cr);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) ci = fmaf(t[k].x, l[k].x, ci);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) cr = fmaf(-t[k].y, l[k].x, cr);
#pragma unroll
            for (int k = kb; k < kb + 4; ++k) ci = fmaf(t[k].y, l[k].y, ci);
          }
        }
      } else if (has_d) {
        ci += d.x * sv.x - d.y * sv.y;
        cr -= d.x * sv.y + d.y * sv.x;
      }

      const float cacc = (float)((st == 0 || st == 3) ? dt / 6.0 : dt / 3.0);
      const float keep = (st == 0) ? 0.f : 1.f;       // the increment restarts at stage 0
      const float kr = ci, ki = -cr;
      float2* N = sS + (ph ^ 1) * MAT;
      if (st < 3) {
        const double cnext = (st == 2) ? dt : 0.5 * dt;
        inc.x = fmaf(cacc, kr, keep * inc.x);
        inc.y = fmaf(cacc, ki, keep * inc.y);
        sv = make_float2((float)(rho.x + cnext * (double)kr), (float)(rho.y + cnext * (double)ki));
        if (act) N[i * P + j] = sv;
        __syncthreads();
        ph ^= 1;
        continue;
      }
      rho.x += (double)fmaf(cacc, kr, inc.x);
      rho.y += (double)fmaf(cacc, ki, inc.y);

      // ---------------- end of step: optional trace renormalisation, records
      if (renorm) {
        double t = op_sum<NS>(act && i == j ? rho.x : 0.0);
        if constexpr (NS == 16) {
          if ((tid & 63) == 0) sRed[tid >> 6].x = t;
          __syncthreads();
          t = (sRed[0].x + sRed[1].x) + (sRed[2].x + sRed[3].x);   // the tiles' order of the diagonal
        }
        const double inv = 1.0 / t;
        rho.x *= inv;
        rho.y *= inv;
      }
      sv = make_float2((float)rho.x, (float)rho.y);
      if (act) N[i * P + j] = sv;
      const int g = a.step_offset + s + 1;
      const bool rec_now = record_any && (g % a.nout) == 0 && (g / a.nout - 1) < a.rec_capacity;
      const int rec = rec_now ? g / a.nout - 1 : 0;
      if (rec_now) {
        if (a.obs != nullptr) {
#pragma unroll 2
          for (int x = 0; x < a.n_eops; ++x) {
            double2 ev = make_double2(0.0, 0.0);
            if (act) {
              if (a.op_pitch > 0) ev = sE[x * nn + o];
              else ev = E[(size_t)x * nn + o];
            }
            const double pr = op_sum<NS>(ev.x * rho.x - ev.y * rho.y);
            const double pi = op_sum<NS>(ev.x * rho.y + ev.y * rho.x);
            if constexpr (NS == 16) {
              if ((tid & 63) == 0) sRed[4 * (1 + x) + (tid >> 6)] = make_double2(pr, pi);
            } else if (e == 0 && valid) {
              a.obs[((size_t)b * a.rec_capacity + rec) * a.n_eops + x] = make_double2(pr, pi);
            }
          }
        }
        if (a.states != nullptr && own) a.states[((size_t)b * a.rec_capacity + rec) * nn + o] = rho;
      }
      if constexpr (DRV) {
        if (s + 1 < a.nsteps) {
#pragma unroll
          for (int k = 0; k < NS; ++k) {
            hi[k] = hin[k];
            hj[k] = hjn[k];
          }
        }
      }
      __syncthreads();   // S of the next step (and the record partials) are complete
      ph ^= 1;
      if constexpr (NS == 16) {
        if (rec_now && a.obs != nullptr) {
          for (int x = tid; x < a.n_eops; x += G::T) {
            double2 t = make_double2(0.0, 0.0);
            for (int w = 0; w < 4; ++w) {
              t.x += sRed[4 * (1 + x) + w].x;
              t.y += sRed[4 * (1 + x) + w].y;
            }
            a.obs[((size_t)b * a.rec_capacity + rec) * a.n_eops + x] = t;
          }
        }
      }
    }
  }
  if (own) a.rho[(size_t)b * nn + o] = rho;
}

namespace {

constexpr size_t kLdsMax = 160 * 1024;
constexpr int kCUs = 256;

template <int NS>
size_t small_lds(int n, int n_dense, int n_eops, bool rops, int staged) {
  using G = Small<NS>;
  const size_t per = (n_dense > 0 ? 4 + (size_t)n_dense * (rops ? 2 : 1) : 2) * G::MAT * sizeof(float2);
  const size_t red = NS == 16 ? 4 * (1 + (size_t)n_eops) * sizeof(double2) : 0;
  return G::OPS * (per + (size_t)staged * n * n * sizeof(double2)) + red;
}

template <int NS, bool DENSE>
hipError_t small_launch_ns(ResidentArgs a, hipStream_t stream) {
  using G = Small<NS>;
  const int groups = cdiv(a.batch, G::OPS);
  // observables are staged in LDS when the workgroups the batch puts on a CU still fit
  const size_t with = small_lds<NS>(a.n, a.n_dense, a.n_eops, a.rops != nullptr, a.n_eops);
  a.op_pitch = with * cdiv(groups, kCUs) <= kLdsMax ? a.n_eops : 0;
  const size_t lds = a.op_pitch > 0 ? with : small_lds<NS>(a.n, a.n_dense, a.n_eops, a.rops != nullptr, 0);
  auto k = a.heff_step > 0 ? lindblad_rk4_small<NS, DENSE, true> : lindblad_rk4_small<NS, DENSE, false>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3(groups), dim3(G::T), lds, stream, a);
  return hipGetLastError();
}

}  // namespace

// n <= 8 beats the tiles at every batch as long as its operands leave the CU its workgroups (one
// wave each): all of the batch's, or at least 10.  n = 9 .. 16 takes four waves an operator and wins
// by latency alone: with one operator per CU, or four without dense operators.  us per RK4 step,
// tiles / here: n = 8 3.30 / 1.56 (one operator), 59.9 / 18.4 (32768), 4 jump operators 10.4 / 6.4 and
// 277 / 86; n = 4 2.65 / 1.12 and 42 / 3.8; n = 16 4.60 / 2.75 (one), 5.6 / 5.5 (1024), 7.7 / 9.5
// (2048), 4 jump operators 17.0 / 13.8 (one), 17.6 / 14.5 (256), 19.1 / 29.8 (1024).
bool small_eligible(const ResidentArgs& a) {
  if (a.n > 16) return false;
  const bool rops = a.rops != nullptr;
  const size_t lds = a.n <= 4 ? small_lds<4>(a.n, a.n_dense, a.n_eops, rops, 0)
                   : a.n <= 8 ? small_lds<8>(a.n, a.n_dense, a.n_eops, rops, 0)
                              : small_lds<16>(a.n, a.n_dense, a.n_eops, rops, 0);
  if (lds > kLdsMax) return false;
  if (a.n > 8) return a.batch <= (a.n_dense > 0 ? 1 : 4) * kCUs && lds * cdiv(a.batch, kCUs) <= kLdsMax;
  const int groups = a.n <= 4 ? cdiv(a.batch, Small<4>::OPS) : a.batch, fit = (int)(kLdsMax / lds);
  return fit >= 10 || cdiv(groups, kCUs) <= fit;
}

hipError_t small_launch(const ResidentArgs& a, hipStream_t stream) {
  if (a.n <= 4) return a.n_dense > 0 ? small_launch_ns<4, true>(a, stream) : small_launch_ns<4, false>(a, stream);
  if (a.n <= 8) return a.n_dense > 0 ? small_launch_ns<8, true>(a, stream) : small_launch_ns<8, false>(a, stream);
  return a.n_dense > 0 ? small_launch_ns<16, true>(a, stream) : small_launch_ns<16, false>(a, stream);
}

}  // namespace lime
