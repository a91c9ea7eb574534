// Lindblad RK4 with dense jump operators for sizes just past a multiple of 16: n = 16 M + r,
// r = 1..4 (a chain of 16 M sites and its ground state), one workgroup per operator.
//
// Padded to 16 (M + 1), n = 33 spends 9 tiles of MFMA on a 2 x 2 core and one row and column: one
// SIMD issues three tiles in a row, 23 of the 36 us that an RK4 step took.  Here the M x M core
// tiles stay on MFMA, one wave each, and the r (2 * 16 M + r) outputs of the last rows and columns
// are summed one per lane on the vector units by waves of their own, beside the MFMAs.  H_eff, S
// (two buffers), T_k = L_k S (two buffers) and every jump operator stay in LDS, so a stage needs
// one barrier and one more per jump operator; on the core H_eff S, S H_eff^dag and L_0 S share one
// loop and the fragments of S.  What bounds it: the core's MFMAs, 4600 of 9400 cycles a stage at
// n = 33; the rest is the edge chains' excess over them, two barriers and the FP64 epilogue.
//
// us per RK4 step, padded / here, one jump operator: n = 17 12.6 / 7.6, n = 20 12.2 / 8.1, n = 33
// 36.3 / 15.9, n = 34 36.3 / 18.5, n = 36 36.5 / 19.6; four: n = 17 30.9 / 16.5, n = 33 93 / 38,
// n = 36 94 / 46; 4096 operators with one: n = 17 108 / 55, n = 20 106 / 73, n = 33 580 / 255, n = 36
// 585 / 319.  At n = 49..52 the padded kernel has 16 tiles for 9 here (4 and 3 a SIMD), and the 16
// waves leave 128 registers, which spill.
//
// The order of the products is that of the resident kernel's tiles (the FP32 MFMA adds its four
// products one after the other, each rounded like an FMA), so the results are the same bits.
#include "common.hpp"
#include "lindblad_resident_decl.hpp"

namespace lime {

namespace {

constexpr int kEdge = 4;   // most rows past the core: the reduction's last MFMA step

template <int M>
struct Edge {
  static constexpr int NC = 16 * M, KE = NC + kEdge;   // core size; reduction length
  static constexpr int P = KE + 1;                     // row pitch (odd)
  static constexpr int MAT = KE * P;
  static constexpr int CORE = M * M;                   // waves holding a core tile
  static constexpr int NEXT = M == 1 ? 3 : 2;                       // elements of the next H_eff a lane holds (driven)
};

// What an edge wave sums for its 64 outputs: the real part of C, the imaginary part, T = L S.  These
// are separate chains of FMAs.  Core of 32: a wave for each (one wave for all three took 8400 cycles
// beside the core's 4200: n = 33 19.8 us per RK4 step, three parts 15.9); 4 rows past it need 5 waves a
// part, and one wave sums both parts of C (21.2 / 19.6).  Core of 16: three parts fill the four SIMDs
// at n = 17 (one 8.1, three 7.6); past that one wave a part of the outputs sums everything (n = 20 three
// 9.3, one 8.1; 4096 operators 145 / 73).
constexpr int kRe = 1, kIm = 2, kT = 4;

struct EdgeWaves {
  int core, part, parts;   // core waves; waves per part; parts
  __host__ __device__ int state() const { return core + part * (parts == 3 ? 2 : 1); }   // waves holding state
  __host__ __device__ int all() const { return core + part * parts; }
};
__host__ __device__ inline EdgeWaves edge_waves(int m, int n) {
  const int nc = 16 * m, r = n - nc, part = (r * (n + nc) + 63) / 64;
  return {m * m, part, m == 1 ? (r == 1 ? 3 : 1) : m * m + 3 * part <= 16 ? 3 : 2};
}

// LDS bytes: H_eff, two S, two T, the jump operators, the diagonal, the record partials and (cached
// observables) E^T
size_t edge_lds(int n, int n_dense, bool rops, int n_eops, bool eops_cached) {
  const int m = n / 16, ke = 16 * m + kEdge;
  size_t bytes = (size_t)(5 + n_dense * (rops ? 2 : 1)) * ke * (ke + 1) * sizeof(float2);
  bytes += (size_t)ke * sizeof(double) + (size_t)n_eops * edge_waves(m, n).all() * sizeof(double2);
  if (eops_cached) bytes += (size_t)n_eops * n * n * sizeof(double2);
  return bytes;
}

template <int M>
struct EdgeLds {
  float2 *h, *s0, *s1, *t0, *t1, *l, *r;
  double* diag;
  double2 *red, *e;
  __device__ EdgeLds(const ResidentArgs& a, float2* lds, int waves) {
    constexpr int MAT = Edge<M>::MAT;
    h = lds;
    s0 = h + MAT;
    s1 = s0 + MAT;
    t0 = s1 + MAT;
    t1 = t0 + MAT;
    l = t1 + MAT;
    r = l + (a.rops ? a.n_dense * MAT : 0);
    diag = reinterpret_cast<double*>(r + a.n_dense * MAT);
    red = reinterpret_cast<double2*>(diag + Edge<M>::KE);
    e = red + (a.obs ? a.n_eops * waves : 0);
  }
};

__device__ __forceinline__ float2 edge_cmul(float2 d, float2 s) {
  return make_float2(fmaf(d.x, s.x, -(d.y * s.y)), fmaf(d.x, s.y, d.y * s.x));
}

// acc += sum over k < 4 of a_k b_k, one FMA after the other
__device__ __forceinline__ void chain(float& acc, const float (&a)[4], const float (&b)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = fmaf(a[q], b[q], acc);
}
__device__ __forceinline__ void chain_neg(float& acc, const float (&a)[4], const float (&b)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = fmaf(-a[q], b[q], acc);
}

// four elements p[q step] as separate real and imaginary parts
struct Four {
  float x[4], y[4];
  __device__ __forceinline__ void load(const float2* p, int step) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float2 v = p[q * step];
      x[q] = v.x;
      y[q] = v.y;
    }
  }
};

// ---- core tiles: C += H_eff S - S H_eff^dag and T = L S in one loop (row fragments at ri, columns at cj)
template <int M>
__device__ __forceinline__ void core_hl(const float2* sH, const float2* sS, const float2* sL, int ri, int cj, int lg,
                                        floatx4& cr, floatx4& ci, floatx4& tr, floatx4& ti) {
  using G = Edge<M>;
  constexpr int P = G::P;
  floatx4 dr = {0.f, 0.f, 0.f, 0.f}, di = dr;
  tr = ti = dr;
  const float2 *pH = sH + ri * P + lg, *pY = sS + lg * P + cj, *pZ = sS + ri * P + lg, *pG = sH + cj * P + lg,
               *pL = sL + ri * P + lg;
#pragma unroll
  for (int k0 = 0; k0 < G::KE; k0 += 4) {
    const float2 x = pH[k0], y = pY[k0 * P], z = pZ[k0], h = pG[k0], l = pL[k0];
    cr = mfma_f32(x.x, y.x, cr);
    ci = mfma_f32(x.x, y.y, ci);
    dr = mfma_f32(x.y, y.y, dr);
    di = mfma_f32(z.y, h.x, di);
    tr = mfma_f32(l.x, y.x, tr);
    ti = mfma_f32(l.x, y.y, ti);
    ci = mfma_f32(x.y, y.x, ci);
    dr = mfma_f32(z.x, h.x, dr);
    tr = mfma_f32(-l.y, y.y, tr);
    ti = mfma_f32(l.y, y.x, ti);
    ci = mfma_f32(z.x, h.y, ci);
    dr = mfma_f32(z.y, h.y, dr);
  }
  cr -= dr;
  ci -= di;
}

// C += i T R^dag and, with a next operator, U = L S
template <int M, bool NEXT>
__device__ __forceinline__ void core_tr(const float2* sT, const float2* sR, const float2* sL, const float2* sS, int ri,
                                        int cj, int lg, floatx4& cr, floatx4& ci, floatx4& tr, floatx4& ti) {
  using G = Edge<M>;
  constexpr int P = G::P;
  if (NEXT) tr = ti = floatx4{0.f, 0.f, 0.f, 0.f};
  const float2 *pT = sT + ri * P + lg, *pR = sR + cj * P + lg, *pL = sL + ri * P + lg, *pS = sS + lg * P + cj;
#pragma unroll
  for (int k0 = 0; k0 < G::KE; k0 += 4) {
    const float2 x = pT[k0], y = pR[k0];
    cr = mfma_f32(x.x, y.y, cr);
    ci = mfma_f32(x.x, y.x, ci);
    if constexpr (NEXT) {
      const float2 l = pL[k0], h = pS[k0 * P];
      tr = mfma_f32(l.x, h.x, tr);
      ti = mfma_f32(l.x, h.y, ti);
      cr = mfma_f32(-x.y, y.x, cr);
      ci = mfma_f32(x.y, y.y, ci);
      tr = mfma_f32(-l.y, h.y, tr);
      ti = mfma_f32(l.y, h.x, ti);
    } else {
      cr = mfma_f32(-x.y, y.x, cr);
      ci = mfma_f32(x.y, y.y, ci);
    }
  }
}

// ---- edge outputs: the same chains, for the parts in ROLE
template <int M, int ROLE>
__device__ __forceinline__ void edge_h(const float2* sH, const float2* sS, int i, int j, float& cr, float& ci) {
  using G = Edge<M>;
  constexpr int P = G::P;
  float dr = 0.f, di = 0.f;
#pragma unroll 3
  for (int k0 = 0; k0 < G::KE; k0 += 4) {
    Four x, y, z, h;
    x.load(sH + i * P + k0, 1);
    y.load(sS + k0 * P + j, P);
    z.load(sS + i * P + k0, 1);
    h.load(sH + j * P + k0, 1);
    if constexpr (ROLE & kRe) {
      chain(cr, x.x, y.x);
      chain(dr, x.y, y.y);
      chain(dr, z.x, h.x);
      chain(dr, z.y, h.y);
    }
    if constexpr (ROLE & kIm) {
      chain(ci, x.x, y.y);
      chain(di, z.y, h.x);
      chain(ci, x.y, y.x);
      chain(ci, z.x, h.y);
    }
  }
  cr -= dr;
  ci -= di;
}
template <int M>
__device__ __forceinline__ float2 edge_l(const float2* sL, const float2* sS, int i, int j) {
  using G = Edge<M>;
  constexpr int P = G::P;
  float tr = 0.f, ti = 0.f;
#pragma unroll 3
  for (int k0 = 0; k0 < G::KE; k0 += 4) {
    Four l, y;
    l.load(sL + i * P + k0, 1);
    y.load(sS + k0 * P + j, P);
    chain(tr, l.x, y.x);
    chain(ti, l.x, y.y);
    chain_neg(tr, l.y, y.y);
    chain(ti, l.y, y.x);
  }
  return make_float2(tr, ti);
}
template <int M, int ROLE>
__device__ __forceinline__ void edge_tr(const float2* sT, const float2* sR, int i, int j, float& cr, float& ci) {
  using G = Edge<M>;
  constexpr int P = G::P;
#pragma unroll 3
  for (int k0 = 0; k0 < G::KE; k0 += 4) {
    Four x, y;
    x.load(sT + i * P + k0, 1);
    y.load(sR + j * P + k0, 1);
    if constexpr (ROLE & kRe) {
      chain(cr, x.x, y.y);
      chain_neg(cr, x.y, y.x);
    }
    if constexpr (ROLE & kIm) {
      chain(ci, x.x, y.x);
      chain(ci, x.y, y.y);
    }
  }
}

// The run of one wave: a core tile (ROLE 0) or the parts in ROLE of 64 edge outputs.  The forms are
// different code with the same number of barriers (one, then 4 (n_dense + 1) a step and one more with
// renormalisation).  A wave of Re C holds the imaginary part of the state and one of Im C the
// real part (k = -i C).
template <int M, bool DRV, bool REC, int ROLE>
__device__ __forceinline__ void edge_run(const ResidentArgs& a, int b, int tid, int w, int e0, const EdgeLds<M>& m,
                                         const EdgeWaves& waves, bool eops_cached) {
  using G = Edge<M>;
  constexpr int P = G::P, NC = G::NC, NV = ROLE == 0 ? 4 : 1;
  constexpr bool CORE = ROLE == 0, STATE = CORE || (ROLE & (kRe | kIm)) != 0, EDGE_T = (ROLE & kT) != 0, X = CORE || (ROLE & kIm) != 0, Y = CORE || (ROLE & kRe) != 0;
  const int n = a.n, nn = n * n, T = blockDim.x, W = waves.all(), lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int set = b / a.group;

  // the lane's outputs: rows i0 + v, column j; ri: the row whose products it reads
  int i0, j, ri;
  bool own = true;
  if constexpr (CORE) {
    ri = w / M * 16 + lr;
    j = w % M * 16 + lr;
    i0 = w / M * 16 + 4 * lg;
  } else {
    const int r = n - NC, rows = r * n, e = e0 + lane;
    own = e < rows + r * NC;   // lanes past the last output repeat it and store nothing
    const int f = own ? e : rows + r * NC - 1;
    i0 = f < rows ? NC + f / n : (f - rows) % NC;
    j = f < rows ? f % n : NC + (f - rows) / NC;
    ri = i0;
  }

  double rx[NV], ry[NV];
  float ix[NV], iy[NV];
  float2 dc[NV];
  floatx4 cr, ci, tr, ti;        // core
  float er = 0.f, ei = 0.f;      // edge: C
  const auto get_r = [&](int v) { return CORE ? cr[v] : er; };
  const auto get_i = [&](int v) { return CORE ? ci[v] : ei; };
  // the next stage's operand; the core's D o S starts its accumulators here (the edge waves hold one
  // component each and form it from LDS when the stage begins)
  const auto put_s = [&](float2* S, int v, float sx, float sy) {
    float* o = reinterpret_cast<float*>(S + (i0 + v) * P + j);
    if (own && X && Y) S[(i0 + v) * P + j] = make_float2(sx, sy);
    else if (own && X) o[0] = sx;
    else if (own && Y) o[1] = sy;
    if constexpr (CORE) {
      const float2 p = edge_cmul(dc[v], make_float2(sx, sy));
      cr[v] = -p.y;
      ci[v] = p.x;
    }
  };
  if constexpr (STATE) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int o = (i0 + v) * n + j;
      const double2 x = a.rho[(size_t)b * nn + o];
      rx[v] = x.x;
      ry[v] = x.y;
      ix[v] = iy[v] = 0.f;
      dc[v] = a.dmat ? a.dmat[(size_t)set * nn + o] : make_float2(0.f, 0.f);
      put_s(m.s0, v, (float)rx[v], (float)ry[v]);
    }
  }
  wave_barrier();

  const double dt = a.dt;
  int ph = 0;
  for (int s = 0; s < a.nsteps; ++s) {
#pragma unroll 1
    for (int st = 0; st < 4; ++st) {
      const float2* sS = ph ? m.s1 : m.s0;
      float2* sN = ph ? m.s0 : m.s1;
      // opaque copies: addresses of the records and the next H_eff are formed where they are used
      // instead of being held (or spilled) across the step
      int otid = tid, oel = i0 * n + j;
      asm volatile("" : "+v"(otid), "+v"(oel));
      const auto put_t = [&](float2* Tk) {
#pragma unroll
        for (int v = 0; v < 4; ++v) Tk[(i0 + v) * P + j] = make_float2(tr[v], ti[v]);
      };
      if constexpr (CORE) {
        core_hl<M>(m.h, sS, m.l, ri, j, lg, cr, ci, tr, ti);
        put_t(m.t0);
      }
      if constexpr (!CORE && STATE) {
        const float2 p = edge_cmul(dc[0], sS[i0 * P + j]);
        er = -p.y;
        ei = p.x;
        edge_h<M, ROLE>(m.h, sS, ri, j, er, ei);
      }
      if constexpr (EDGE_T) {
        const float2 t = edge_l<M>(m.l, sS, ri, j);
        if (own) m.t0[i0 * P + j] = t;
      }
      wave_barrier();
      // driven: every wave is past its products with H_eff; the next step's loads leave here and
      // are stored after the step's last products
      float2 hn[G::NEXT];
      if constexpr (DRV) {
        if (st == 3) {
          const float2* H = a.heff + (size_t)min(s + 1, a.nsteps - 1) * a.heff_step + (size_t)set * nn;
#pragma unroll
          for (int i = 0; i < G::NEXT; ++i) hn[i] = H[min(otid + i * T, nn - 1)];
        }
      }
      int kk = 0;
      for (; kk + 1 < a.n_dense; ++kk) {
        const float2 *Tk = kk & 1 ? m.t1 : m.t0, *R = m.r + kk * G::MAT, *L = m.l + (kk + 1) * G::MAT;
        float2* Tn = kk & 1 ? m.t0 : m.t1;
        if constexpr (CORE) {
          core_tr<M, true>(Tk, R, L, sS, ri, j, lg, cr, ci, tr, ti);
          put_t(Tn);
        }
        if constexpr (!CORE && STATE) edge_tr<M, ROLE>(Tk, R, ri, j, er, ei);
        if constexpr (EDGE_T) {
          const float2 t = edge_l<M>(L, sS, ri, j);
          if (own) Tn[i0 * P + j] = t;
        }
        wave_barrier();
      }
      const float2 *Tk = kk & 1 ? m.t1 : m.t0, *R = m.r + kk * G::MAT;
      if constexpr (CORE) core_tr<M, false>(Tk, R, nullptr, nullptr, ri, j, lg, cr, ci, tr, ti);
      else if constexpr (STATE) edge_tr<M, ROLE>(Tk, R, ri, j, er, ei);

      // k = -i C; the RK4 combination as in the resident kernel
      const float cacc = (float)((st == 0 || st == 3) ? dt / 6.0 : dt / 3.0);
      const float keep = (st == 0) ? 0.f : 1.f;
      if (st < 3) {
        if constexpr (STATE) {
          const double cnext = (st == 2) ? dt : 0.5 * dt;
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            const float kr = get_i(v), ki = -get_r(v);
            ix[v] = fmaf(cacc, kr, keep * ix[v]);
            iy[v] = fmaf(cacc, ki, keep * iy[v]);
            put_s(sN, v, (float)(rx[v] + cnext * (double)kr), (float)(ry[v] + cnext * (double)ki));
          }
        }
        wave_barrier();
        ph ^= 1;
        continue;
      }
      if constexpr (DRV) {
#pragma unroll
        for (int i = 0; i < G::NEXT; ++i) {
          const int idx = otid + i * T, row = idx / n;
          if (idx < nn) m.h[row * P + idx - row * n] = hn[i];
        }
      }
      if constexpr (STATE) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          rx[v] += (double)fmaf(cacc, get_i(v), ix[v]);
          ry[v] += (double)fmaf(cacc, -get_r(v), iy[v]);
        }
      }
      if (a.flags & 1) {
        // trace: the diagonal tiles' sums in the resident kernel's order (a tile's element d on the
        // lane that owns it there)
        if constexpr (STATE && X) {
#pragma unroll
          for (int v = 0; v < NV; ++v)
            if (own && i0 + v == j) m.diag[j] = rx[v];
        }
        wave_barrier();
        if constexpr (STATE) {
          double tot = 0.0;
#pragma unroll
          for (int t = 0; t <= M; ++t) {
            const int d = 16 * t + lr;
            tot += wave_sum(lg == lr >> 2 && d < n ? m.diag[d] : 0.0);
          }
          const double inv = 1.0 / tot;
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            rx[v] *= inv;
            ry[v] *= inv;
          }
        }
      }
      if constexpr (STATE) {
#pragma unroll
        for (int v = 0; v < NV; ++v) put_s(sN, v, (float)rx[v], (float)ry[v]);
      }

      bool rec_now = false;
      int rec = 0;
      if constexpr (REC) {
        const int g = a.step_offset + s + 1;
        rec_now = (g % a.nout) == 0 && (g / a.nout - 1) < a.rec_capacity;
        rec = g / a.nout - 1;
        if constexpr (STATE) {
          if (rec_now && a.obs != nullptr) {
            const double2* Eg = a.eops_t + (size_t)(b / a.eop_group) * a.n_eops * nn;
            for (int e = 0; e < a.n_eops; ++e) {
              double pr = 0.0, pi = 0.0;
#pragma unroll
              for (int v = 0; v < NV; ++v) {
                const int o = e * nn + oel + v * n;
                double2 ev;
                if (eops_cached) ev = m.e[o];
                else ev = Eg[o];
                if (X) pr += ev.x * rx[v], pi += ev.y * rx[v];
                if (Y) pr -= ev.y * ry[v], pi += ev.x * ry[v];
              }
              pr = wave_sum(own ? pr : 0.0);
              pi = wave_sum(own ? pi : 0.0);
              if (lane == 0) m.red[e * W + w] = make_double2(pr, pi);
            }
          }
          if (rec_now && a.states != nullptr) {
            double2* Sg = a.states + ((size_t)b * a.rec_capacity + rec) * nn;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
              double* o = reinterpret_cast<double*>(Sg + oel + v * n);
              if (own && X) o[0] = rx[v];
              if (own && Y) o[1] = ry[v];
            }
          }
        }
      }
      wave_barrier();   // S (and H_eff) of the next step and the record partials are complete
      ph ^= 1;
      // the record's sums go to the last wave (at three parts it holds no state)
      if constexpr (REC && EDGE_T) {
        if (rec_now && a.obs != nullptr && w == W - 1) {
          for (int e = lane; e < a.n_eops; e += 64) {
            double2 t = make_double2(0.0, 0.0);
            for (int x = 0; x < waves.state(); ++x) {
              t.x += m.red[e * W + x].x;
              t.y += m.red[e * W + x].y;
            }
            a.obs[((size_t)b * a.rec_capacity + rec) * a.n_eops + e] = t;
          }
        }
      }
    }
  }
  if constexpr (STATE) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      double* o = reinterpret_cast<double*>(a.rho + (size_t)b * nn + (i0 + v) * n + j);
      if (own && X) o[0] = rx[v];
      if (own && Y) o[1] = ry[v];
    }
  }
}

}  // namespace

template <int M, bool DRV, bool REC>
__global__ void __launch_bounds__(M == 1 ? 640 : 1024) lindblad_rk4_edge(ResidentArgs a, int eops_cached) {
  using G = Edge<M>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  float2* lds = reinterpret_cast<float2*>(lds_raw);
  const int b = xcd_block();
  if (b >= a.batch) return;
  const int tid = threadIdx.x, T = blockDim.x, n = a.n, nn = n * n, set = b / a.group;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const EdgeWaves waves = edge_waves(M, n);
  const EdgeLds<M> m(a, lds, waves.all());
  // H_eff, zeroed S and T, the jump operators: zero beyond n
  const int mats = a.n_dense * (a.rops ? 2 : 1);
  for (int idx = tid; idx < (5 + mats) * G::MAT; idx += T) {
    const int mat = idx / G::MAT, e = idx - mat * G::MAT, i = e / G::P, j = e - i * G::P;
    const float2* src = mat == 0 ? a.heff + (size_t)set * nn
                        : mat < 5 ? nullptr
                        : mat < 5 + a.n_dense ? a.lops + ((size_t)set * a.n_dense + mat - 5) * nn
                                              : a.rops + ((size_t)set * a.n_dense + mat - 5 - a.n_dense) * nn;
    lds[idx] = src && i < n && j < n ? src[i * n + j] : make_float2(0.f, 0.f);
  }
  if (REC && eops_cached) {
    const double2* E = a.eops_t + (size_t)(b / a.eop_group) * a.n_eops * nn;
    for (int idx = tid; idx < a.n_eops * nn; idx += T) m.e[idx] = E[idx];
  }
  __syncthreads();
  const bool cached = eops_cached != 0;
  const int x = w - waves.core, part = x / waves.part, e0 = (x - part * waves.part) * 64;
  if (x < 0) edge_run<M, DRV, REC, 0>(a, b, tid, w, 0, m, waves, cached);
  else if (M == 1 && waves.parts == 1) edge_run<M, DRV, REC, M == 1 ? kRe | kIm | kT : kT>(a, b, tid, w, e0, m, waves, cached);
  else if (part == waves.parts - 1) edge_run<M, DRV, REC, kT>(a, b, tid, w, e0, m, waves, cached);
  else if (M == 2 && waves.parts == 2) edge_run<M, DRV, REC, M == 2 ? kRe | kIm : kT>(a, b, tid, w, e0, m, waves, cached);
  else if (part == 0) edge_run<M, DRV, REC, kRe>(a, b, tid, w, e0, m, waves, cached);
  else edge_run<M, DRV, REC, kIm>(a, b, tid, w, e0, m, waves, cached);
}

namespace {

constexpr size_t kLdsMax = 160 * 1024;
constexpr int kCUs = 256;

template <int M>
hipError_t edge_launch_m(const ResidentArgs& a, hipStream_t stream) {
  const bool rec = a.nout > 0 && (a.obs != nullptr || a.states != nullptr);
  const int ne = rec && a.obs ? a.n_eops : 0, per_cu = cdiv(a.batch, kCUs);
  // E^T in LDS where the batch's workgroups per CU still fit
  const bool cached = ne > 0 && edge_lds(a.n, a.n_dense, a.rops != nullptr, ne, true) * per_cu <= kLdsMax;
  const size_t lds = edge_lds(a.n, a.n_dense, a.rops != nullptr, ne, cached);
  void (*k)(ResidentArgs, int) = a.heff_step > 0 ? (rec ? lindblad_rk4_edge<M, true, true> : lindblad_rk4_edge<M, true, false>)
                                 : rec           ? lindblad_rk4_edge<M, false, true>
                                                 : lindblad_rk4_edge<M, false, false>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3(a.batch), dim3(edge_waves(M, a.n).all() * 64), lds, stream, a, (int)cached);
  return hipGetLastError();
}

}  // namespace

// Every size it is built for, at every batch (above: faster from 1 to 4096 operators), while the
// operands of one operator fit the LDS.
bool edge_eligible(const ResidentArgs& a) {
  const int m = a.n / 16, r = a.n - 16 * m;
  if (a.n_dense < 1 || m < 1 || m > 2 || r < 1 || r > kEdge) return false;
  return edge_lds(a.n, a.n_dense, a.rops != nullptr, a.obs ? a.n_eops : 0, false) <= kLdsMax;
}

hipError_t edge_launch(const ResidentArgs& a, hipStream_t stream) {
  return a.n < 32 ? edge_launch_m<1>(a, stream) : edge_launch_m<2>(a, stream);
}

}  // namespace lime
