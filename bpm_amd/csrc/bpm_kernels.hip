// Split-step beam propagation on gfx950: fused row/column FFT passes.
//
// One propagation step z-1 -> z of the reference loop (bpm/bpm/bpm_3d.py:283-382;
// bpm/bpmclass/_bpm3d_ocl.py:100-126) is
//     u_z = screen_z( IFFT2( H . FFT2(u_{z-1}) ) )
// and is executed as two passes over the (Ny,Nx) complex64 plane that stays
// in HBM between them, holding F_x u (the plane transformed along x only):
//   column pass (one work-group per tile of COLS columns):
//       FFT_y -> multiply by H (table or on-the-fly formula) -> IFFT_y
//   row pass (one work-group per LINES rows):
//       IFFT_x -> 1/(NxNy) -> phase screen dn[z] and taper -> outputs
//       (field/intensity slice, running sum of |u|^2) -> FFT_x
// so each step reads and writes the plane twice and reads dn[z] once.  The
// default mean_mode "weighted" of bpm_3d needs the k-space reduction of
// bpm_3d.py:302-303 before H, so its column pass is split in two (A: FFT_y
// and per-column partial sums; B: H(n0+dn0) and IFFT_y).
#include "items.hpp"
#include "loop_adj.hpp"

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

// ----------------------------------------------------------------------------
// error reporting
// ----------------------------------------------------------------------------
static thread_local std::string g_err;

int bpmh_set_error(int code, const char* msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                        \
  do {                                                                       \
    hipError_t e_ = (expr);                                                  \
    if (e_ != hipSuccess) {                                                  \
      char b_[256];                                                          \
      snprintf(b_, sizeof b_, "%s: %s", #expr, hipGetErrorString(e_));       \
      return bpmh_set_error(BPMH_ERR_HIP, b_);                               \
    }                                                                        \
  } while (0)

extern "C" const char* bpmh_last_error(void) { return g_err.c_str(); }
extern "C" int bpmh_version(void) { return BPMH_VERSION; }

// ----------------------------------------------------------------------------
// row pass
// ----------------------------------------------------------------------------
template <int NX, int V, int EE>
__global__ void __launch_bounds__((RowCfg<NX, V, EE>::THREADS))
k_row(RowArgs a) {
  using Cfg = RowCfg<NX, V, EE>;
  constexpr int E = Cfg::E, T = Cfg::T, LINES = Cfg::LINES;
  // a line of at most 64 threads lies inside one wavefront (T divides 64)
  constexpr bool WAVE = T <= 64;
  __shared__ float2 lds[LINES][Cfg::ROW_LINE];
  const int line = threadIdx.x / T;
  const int t = threadIdx.x - line * T;
  const int row = blockIdx.x * LINES + line;  // in [0, batch*ny)
  const int b = row / a.ny;
  const int y = row - b * a.ny;
  float2* p = a.plane + (size_t)row * NX;
  const size_t plane_off = (size_t)y * NX;

  // Every global load of the pass is issued here, before the first barrier,
  // so their latencies overlap instead of adding up behind the transforms.
  float2 v[E];
#pragma unroll
  for (int m = 0; m < E; ++m) v[m] = ld_stream(p + t + m * T);
  Twiddles<NX, E> tw;
  const bool forward = b < a.fwd_items;  // uniform: a work-group's rows are one item's
  if (a.inverse || forward) tw.load(t, a.tw);
  float2 d[E];
  if (a.screen) {
    const size_t slice = ((size_t)a.z * a.ny + y) * NX + (size_t)dn_volume(a, b) * a.dn_bstride;
#pragma unroll
    for (int m = 0; m < E; ++m) d[m] = load_dn(a.dn, a.dn_kind, slice + t + m * T);
  }
  float accv[E];
  float* acc_row = a.acc ? a.acc + (size_t)b * a.ny * NX + plane_off : nullptr;
  if (acc_row && !a.acc_init) {
#pragma unroll
    for (int m = 0; m < E; ++m) accv[m] = acc_row[t + m * T];
  }
  float2 ua[E];
  if (a.adjoint) {
    const float2* u = a.useg + (size_t)b * a.useg_bstride + (size_t)a.useg_z * a.ny * NX + plane_off;
#pragma unroll
    for (int m = 0; m < E; ++m) ua[m] = u[t + m * T];
  }

  if (a.inverse) {
    line_fft<NX, E, true, SwzLayout<4>, WAVE>(v, lds[line], t, tw);
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = c_scale(v[m], a.inv_n);
  }

  if (a.screen) {
    float dn0 = 0.f;
    if (a.dn0_mode == BPMH_MEAN_SIMPLE) dn0 = a.dn0_arr[a.z];
    else if (a.dn0_mode == BPMH_MEAN_WEIGHTED) dn0 = a.dn0_item[b];
    row_screen<NX, E, true>(a, b, y, t, dn0, d, ua, v);
  }

  row_outputs<NX, E>(a, a.z, b, plane_off, t, v);
  if (acc_row) {
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const float i2 = v[m].x * v[m].x + v[m].y * v[m].y;
      acc_row[t + m * T] = a.acc_init ? i2 : accv[m] + i2;
    }
  }

  if (forward) line_fft<NX, E, false, SwzLayout<4>, WAVE>(v, lds[line], t, tw);
#pragma unroll
  for (int m = 0; m < E; ++m) st_stream(p + t + m * T, v[m]);
}

// ----------------------------------------------------------------------------
// column pass
// ----------------------------------------------------------------------------
// PHASE 0: FFT_y, H, IFFT_y.  PHASE 1: FFT_y, weighted partials, store.
// PHASE 2: weighted dn0, H(n0+dn0), IFFT_y.
// Adjoint of a weighted step (X = F G_v, the k-space gradient):
// PHASE 3: FFT_y, per-column partials of sum Im(conj(X) H U)/beta, store X.
// PHASE 4: dL/ddn0 from the partials, conj(H) X plus the term of dn0's
//          dependence on |U|, the weight-slice gradient, IFFT_y (simple mean:
//          conj(H) X, IFFT_y, dL/ddn0 stored).
// PHASE 5: PHASE 0 with H evaluated on the fly (hmode 1, the simple mean),
//          half the rows per thread as in PHASE 2.
template <int NY, int V, int PHASE, int EE>
__global__ void __launch_bounds__((ColCfg<NY, V, EE>::THREADS))
k_col(ColArgs a) {
  using Cfg = ColCfg<NY, V, EE>;
  constexpr int E = Cfg::E, T = Cfg::T, COLS = Cfg::COLS;
  constexpr bool FWD = PHASE == 0 || PHASE == 1 || PHASE == 3 || PHASE == 5;  // forward FFT_y
  constexpr bool INV = PHASE == 0 || PHASE == 2 || PHASE == 4 || PHASE == 5;  // H, inverse FFT_y
  constexpr bool ADJW = PHASE == 3 || PHASE == 4;
  // each thread holds P adjacent columns; the LC lane columns of a 16-lane
  // group are the LDS lines it touches together
  constexpr int P = Cfg::P, LC = Cfg::LC;
  constexpr bool SPLIT = Cfg::SPLIT;
  // swizzled lines 16/LC float2 apart, or padded lines 9 float2 longer
  // than padded: either way the LC lines a 16-lane group touches together
  // start in different LDS banks.  Two lane columns swizzle when each
  // thread holds two columns (1 % faster than padding at 1024^2 in batches)
  // and pad otherwise (the swizzle was slower there).
  constexpr bool SWZ = LC >= 4 || (P == 2 && LC >= 2);
  static_assert(COLS <= 16, "at most 16 columns per tile");
  constexpr int LINE = SWZ ? NY + 16 / LC : Cfg::COL_LINE;
  __shared__ float2 lds[COLS][LINE];
  using CL = std::conditional_t<SWZ, SwzLayout<4 - ilog2c(LC)>, PadLayout<Cfg::COL_SH>>;
  const int ntiles = a.nx / COLS;
  const int bx = blockIdx.x;
  // adjacent tiles share cache lines: keep them on one XCD (blocks are
  // dealt round-robin over the 8 XCDs)
  const int tile = (ntiles % 8 == 0) ? (bx & 7) * (ntiles >> 3) + (bx >> 3) : bx;
  const int b = blockIdx.y;
  const int c = threadIdx.x % LC;
  const int t = threadIdx.x / LC;
  const int x0 = tile * COLS + c * P;  // the thread's columns x0 .. x0+P-1
  float2* p = a.plane + (size_t)b * NY * a.nx + x0;

  // all global loads first (plane, twiddles, the propagator quadrant); with
  // P = 2 and 16-byte accesses the host guarantees a 16-byte aligned plane
  // (x0 and nx are even)
  float2 v[P][E];
  Twiddles<NY, E> tw;
  WeightParts wparts;
  if constexpr (PHASE == 2) weighted_parts_load(a.wpart + (size_t)b * a.nx, a.nx, wparts);
  // split columns: the twiddles first, so waiting for the first column's
  // data (loads complete in issue order) does not wait for the second's
  if constexpr (SPLIT) tw.load(t, a.tw);
  if constexpr (SPLIT) {
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int m = 0; m < E; ++m) v[q][m] = p[(size_t)(t + m * T) * a.nx + q];
  } else {
#pragma unroll
    for (int m = 0; m < E; ++m) {
      float2* r = p + (size_t)(t + m * T) * a.nx;
      if constexpr (P == 2) {
        const float4 w = *reinterpret_cast<const float4*>(r);
        v[0][m] = make_float2(w.x, w.y);
        v[1][m] = make_float2(w.z, w.w);
      } else {
        v[0][m] = *r;
      }
    }
  }
  if constexpr (!SPLIT) tw.load(t, a.tw);
  // H depends on kx^2 and ky^2 only, so H[j][i] = H[(ny-j)%ny][(nx-i)%nx]
  // holds bit for bit; reading the quadrant j<=ny/2, i<=nx/2 keeps the
  // table's footprint at a quarter (L2-resident per XCD strip).
  // adjoint: the forward k-space plane U (and the weight slice) of the step
  float2 uv[P][E];
  float dv[P][E];
  if constexpr (ADJW) {
    const float2* uk = a.uk + (size_t)b * a.uk_bstride + x0;
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int m = 0; m < E; ++m) uv[q][m] = uk[(size_t)(t + m * T) * a.nx + q];
    if constexpr (PHASE == 4) {
      const size_t s0 = (size_t)b * a.dn_bstride + x0;
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < E; ++m)
          dv[q][m] = a.dn ? load_dn(a.dn, a.dn_kind, s0 + (size_t)(t + m * T) * a.nx + q).x : 0.f;
    }
  }
  float2 hv[P][E];
  if (INV && a.hmode == 0) {
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int qx = min(x0 + q, a.nx - x0 - q);
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int ky = t + m * T;
        hv[q][m] = a.H[(size_t)min(ky, NY - ky) * a.nx + qx];
      }
    }
  }

  float dn0w = 0.f;
  if constexpr (PHASE == 2) {
    __shared__ float dn0_slot[2];
    dn0w = weighted_dn0_group(a.wpart + (size_t)b * a.nx, a.nx, wparts, dn0_slot);
    if (bx == 0 && threadIdx.x == 0) {
      a.dn0_item[b] = dn0w;
      if (a.rec_c) {
        a.rec_c[b] = dn0w;
        a.rec_w[b] = dn0_slot[1];
      }
    }
  }
  if constexpr (ADJW) dn0w = a.simple ? 0.f : a.cz[b];  // the forward's dn0 of this step
  // the step's refractive index: weighted n0 + dn0 (as PHASE 2), simple n_eff[z]
  float n_adj = 0.f;
  if constexpr (ADJW) n_adj = a.simple ? a.n_eff[a.z] : f_add(a.n0, dn0w);
  float cgrad = 0.f, inv_w = 0.f, n_pts = 0.f;
  if constexpr (PHASE == 4) {
    // dL/ddn0 = -sum_x (screen gradient) + dz (n0+dn0) k0^2 / N sum_k Im(conj(X) H U)/beta
    __shared__ float cg_slot[2];
    const float2 sums = group_sum_pair(a.s1part + (size_t)b * NY, NY, a.s2part + (size_t)b * a.nx,
                                       a.nx, cg_slot);
    n_pts = (float)a.nx * (float)NY;
    cgrad = adjoint_cgrad(sums.x, sums.y, a.dz, n_adj, a.k0, n_pts);
    if (a.simple) {
      if (bx == 0 && threadIdx.x == 0) a.cg_out[b] = cgrad;
    } else {
      inv_w = 1.f / a.wz[b];
    }
  }

  if constexpr (FWD) {
#pragma unroll
    for (int q = 0; q < P; ++q) line_fft<NY, E, false, CL>(v[q], lds[q * LC + c], t, tw);
  }
  if constexpr (PHASE == 0 || PHASE == 5) {
    // forward recorded for the adjoint: U = F u of this step, before H
    if (a.kout) {
      float2* ko = a.kout + (size_t)b * a.kout_bstride + x0;
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < E; ++m) ko[(size_t)(t + m * T) * a.nx + q] = v[q][m];
    }
  }

#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int x = x0 + q;
    float2* line = lds[q * LC + c];
    if constexpr (PHASE == 1) {
      const size_t s0 = (size_t)b * a.dn_bstride;
      float d[E];
#pragma unroll
      for (int m = 0; m < E; ++m)
        d[m] = a.dn ? load_dn(a.dn, a.dn_kind, s0 + (size_t)(t + m * T) * a.nx + x).x : 0.f;
      const float2 acc = col_weight_sums<NY, E>(v[q], d, t, line);
      if (t == 0) a.wpart[(size_t)b * a.nx + x] = acc;
    } else if constexpr (PHASE == 3) {
      // dH/ddn0 = H * (-i dz (n0+dn0) k0^2 / beta): collect Im(conj(X) H U)/beta
      const float an = n_term_f32(n_adj, a.k0);
      const float kx2 = kcomp2_f32(x, a.nx, a.dx);
      float2 h[E];
      float bt[E];
      col_hb_fly<NY, E>(kx2, an, a.dy, a.dz, t, line, h, bt);
      const float tot = col_beta_sum<NY, E>(v[q], h, uv[q], bt, t, line);
      if (t == 0) a.s2part[(size_t)b * a.nx + x] = tot;
    } else {
      float an = 0.f, kx2 = 0.f;
      if (a.hmode != 0) {
        float n = ADJW ? n_adj : (a.hmode == 1) ? a.n_eff[a.z] : f_add(a.n0, dn0w);
        an = n_term_f32(n, a.k0);
        kx2 = kcomp2_f32(x, a.nx, a.dx);
      }
      if constexpr (PHASE == 2 || PHASE == 4 || PHASE == 5) {
        // H(n0 + dn0) (weighted pass B, its adjoint) or H(n_eff[z]) (simple
        // mean, its adjoint) on the fly for every row
        float2 h[E];
        col_h_fly<NY, E>(kx2, an, a.dy, a.dz, t, line, h);
#pragma unroll
        for (int m = 0; m < E; ++m)
          v[q][m] = c_mul_fused(v[q][m], make_float2(h[m].x, a.conj_h ? -h[m].y : h[m].y));
      } else {
#pragma unroll
        for (int m = 0; m < E; ++m) {
          const int ky = t + m * T;
          const float2 h =
              (a.hmode == 0) ? hv[q][m] : prop_f32(kx2, kcomp2_f32(ky, NY, a.dy), an, a.dz);
          v[q][m] = c_mul_fused(v[q][m], make_float2(h.x, a.conj_h ? -h.y : h.y));
        }
      }
      if (PHASE == 4 && !a.simple) {
        float* gd = a.gd_item + (size_t)b * NY * a.nx + x;
#pragma unroll
        for (int m = 0; m < E; ++m)
          gd[(size_t)(t + m * T) * a.nx] +=
              adjoint_weight_term(v[q][m], uv[q][m], dv[q][m], dn0w, cgrad, inv_w, n_pts);
      }
      if (a.sw) col_scatter<NY, E>(a, a.z, b, x, t, line, v[q]);
    }
  }
  if constexpr (PHASE == 1) {
    // weighted forward recorded for the adjoint: U = F u of this step
    if (a.kout) {
      float2* ko = a.kout + (size_t)b * a.kout_bstride + x0;
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < E; ++m) ko[(size_t)(t + m * T) * a.nx + q] = v[q][m];
    }
  }
  if constexpr (SPLIT) {
    // each column stored as soon as its inverse transform is done
#pragma unroll
    for (int q = 0; q < P; ++q) {
      if constexpr (INV) line_fft<NY, E, true, CL>(v[q], lds[q * LC + c], t, tw);
#pragma unroll
      for (int m = 0; m < E; ++m) p[(size_t)(t + m * T) * a.nx + q] = v[q][m];
    }
  } else {
    if constexpr (INV) {
#pragma unroll
      for (int q = 0; q < P; ++q) line_fft<NY, E, true, CL>(v[q], lds[q * LC + c], t, tw);
    }
#pragma unroll
    for (int m = 0; m < E; ++m) {
      float2* r = p + (size_t)(t + m * T) * a.nx;
      if constexpr (P == 2)
        *reinterpret_cast<float4*>(r) = make_float4(v[0][m].x, v[0][m].y, v[1][m].x, v[1][m].y);
      else
        *r = v[0][m];
    }
  }
}

// ----------------------------------------------------------------------------
// propagator tables and small helpers
// ----------------------------------------------------------------------------
// kind F32: compute_propagator (bpm_3d_kernels.cl:408-432), float32 formula.
// kind F64: host float64 propagator (bpm_3d.py:163-181, bpmclass/bpm3d.py:88-107)
//           rounded to complex64.
__global__ void k_prop_table(float2* H, int nx, int ny, int kind, double dx, double dy,
                             double dz, double n0, double lam) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= nx) return;
  const double k0 = 2. * M_PI / lam;
  float2 h;
  if (kind == BPMH_H_F32) {
    const float an = n_term_f32((float)n0, (float)k0);
    h = prop_f32(kcomp2_f32(i, nx, (float)dx), kcomp2_f32(j, ny, (float)dy), an, (float)dz);
  } else {
    // numpy: 2*pi*fftfreq(n,d) = 2*pi*(m * (1/(n*d)))
    const int mi = (i < (nx - 1) / 2 + 1) ? i : i - nx;
    const int mj = (j < (ny - 1) / 2 + 1) ? j : j - ny;
    const double kx = (2. * M_PI) * ((double)mi * (1.0 / (nx * dx)));
    const double ky = (2. * M_PI) * ((double)mj * (1.0 / (ny * dy)));
    const double tmp = (n0 * n0) * (k0 * k0) - kx * kx - ky * ky;
    if (tmp < 0.) {
      h = make_float2(0.f, 0.f);
    } else {
      double s, c;
      sincos(-dz * sqrt(tmp), &s, &c);
      h = make_float2((float)c, (float)s);
    }
  }
  H[(size_t)j * nx + i] = h;
}

__global__ void k_scatter_final(const float2* spart, float* out, int nz, int nparts) {
  const int z = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (z >= nz) return;
  float2 s = make_float2(0.f, 0.f);
  if (z > 0) {
    const float2* q = spart + ((size_t)b * nz + z) * nparts;
    for (int i = 0; i < nparts; ++i) s = c_add(s, q[i]);
  }
  out[((size_t)b * nz + z) * 2 + 0] = s.x;
  out[((size_t)b * nz + z) * 2 + 1] = s.y;
}

// ----------------------------------------------------------------------------
// plans
// ----------------------------------------------------------------------------
// Kernel kinds timed by the optional HIP-event instrumentation.
enum { TK_ROW = 0, TK_COL = 1, TK_COL_A = 2, TK_COL_B = 3, TK_N = 4 };

// One captured launch sequence of bpmh_propagate: its argument key, the
// executable graph, and an event recorded after its latest launch (an
// executable is destroyed only once that event has completed, so a replay
// still running on some stream is never destroyed under it).
struct GraphEntry {
  std::vector<unsigned char> key;
  hipGraphExec_t exec;
  hipEvent_t done;
  unsigned long long used;  // recency stamp for eviction
};

// Executables kept per plan (least recently used is evicted).
constexpr int kGraphCache = 4;

struct bpmh_plan_s {
  int nx, ny;
  // stage-major twiddles of both radix schedules (index ealt), on the host
  // and their device copies
  std::vector<float2> htw_x[2], htw_y[2];
  float2* tw_x[2];
  float2* tw_y[2];
  void* work;                        // step scratch (allocated on demand)
  size_t work_bytes;
  int device;
  // timing: events recorded around every launch of bpmh_propagate
  int timing;
  std::vector<hipEvent_t> ev;   // pairs (start, stop)
  std::vector<int> ev_kind;     // kind of each pair
  size_t ev_used;               // pairs recorded since the last read-out
  // graph mode: the launch sequence of bpmh_propagate is captured once per
  // distinct argument list and replayed with hipGraphLaunch
  int row_v, col_v;             // launch-shape variants (autotuned)
  int graph_mode;
  hipStream_t cap_stream;
  std::vector<GraphEntry> graphs;
  unsigned long long graph_clock;
  int loop_mode;                // bpmh_plan_set_loop
  long long loop_calls;         // z-loops run as one launch
};

// Wait for an entry's latest replay, then release it.
static int graph_release(GraphEntry& g) {
  hipError_t e1 = hipEventSynchronize(g.done);
  hipError_t e2 = hipGraphExecDestroy(g.exec);
  hipError_t e3 = hipEventDestroy(g.done);
  g.exec = nullptr;
  g.done = nullptr;
  hipError_t e = e1 != hipSuccess ? e1 : (e2 != hipSuccess ? e2 : e3);
  if (e != hipSuccess) return bpmh_set_error(BPMH_ERR_HIP, hipGetErrorString(e));
  return BPMH_OK;
}

static int graph_release_all(bpmh_plan p) {
  int rc = BPMH_OK;
  for (GraphEntry& g : p->graphs) {
    const int r = graph_release(g);
    if (r && !rc) rc = r;
  }
  p->graphs.clear();
  return rc;
}

static bool pow2_in_range(int n) { return n >= 16 && n <= 4096 && (n & (n - 1)) == 0; }

// Twiddles exp(-2 pi i m/N).  Angles are reduced to the first octant so the
// symmetric values (m = 0, N/8, N/4, ...) are exact; among the float32
// neighbours of (cos, sin) the pair with |w|^2 closest to 1 is kept, since
// a magnitude error of a twiddle is applied again on every step.
static void make_twiddles(int N, std::vector<float2>& tw) {
  tw.resize(N);
  for (int m = 0; m < N; ++m) {
    // exact octant reduction of the angle 2 pi m / N
    const long long M = 8LL * m;  // angle in units of 2*pi/(8N): octant = M / N
    const int oct = (int)(M / N);
    const double frac = (double)(M - (long long)oct * N) / N;  // in [0,1)
    double c, s;
    const double phi = frac * (M_PI / 4.0);
    const double cp = cos(phi), sp = sin(phi), cq = cos(M_PI / 4.0 - phi), sq = sin(M_PI / 4.0 - phi);
    switch (oct & 7) {  // cos/sin of oct*pi/4 + phi
      case 0: c = cp; s = sp; break;
      case 1: c = sq; s = cq; break;
      case 2: c = -sp; s = cp; break;
      case 3: c = -cq; s = sq; break;
      case 4: c = -cp; s = -sp; break;
      case 5: c = -sq; s = -cq; break;
      case 6: c = sp; s = -cp; break;
      default: c = cq; s = -sq; break;
    }
    if (frac == 0.0) {  // exact multiples of pi/4
      const double r = sqrt(0.5);
      const double cc[8] = {1, r, 0, -r, -1, -r, 0, r};
      const double ss[8] = {0, r, 1, r, 0, -r, -1, -r};
      c = cc[oct & 7];
      s = ss[oct & 7];
    }
    const float c0 = (float)c, s0 = (float)-s;
    float bc = c0, bs = s0;
    double best = 1e300;
    for (int dc = -1; dc <= 1; ++dc) {
      for (int ds = -1; ds <= 1; ++ds) {
        const float cf = dc == 0 ? c0 : nextafterf(c0, dc > 0 ? 2.f : -2.f);
        const float sf = ds == 0 ? s0 : nextafterf(s0, ds > 0 ? 2.f : -2.f);
        const double mag = fabs((double)cf * cf + (double)sf * sf - 1.0);
        const double ang = fabs(atan2((double)sf, (double)cf) - atan2(-s, c));
        const double score = mag + 0.25 * ang;
        if (score < best) { best = score; bc = cf; bs = sf; }
      }
    }
    tw[m] = make_float2(bc, bs);
  }
}

// Stage-major twiddles for the line FFT of N points with E elements per
// thread (fft.hpp: Twiddles::load), built from the natural-order table.
static void make_stage_twiddles(int N, int E, std::vector<float2>& out) {
  std::vector<float2> full;
  make_twiddles(N, full);
  int n = 0, e = 0;
  while ((1 << n) < N) ++n;
  while ((1 << e) < E) ++e;
  const int S = n / e, R0 = 1 << (n - S * e);
  int ns = R0 > 1 ? R0 : E;
  const int nst = R0 > 1 ? S : S - 1;
  out.clear();
  for (int s = 0; s < nst; ++s) {
    for (int r = 1; r < E; ++r)
      for (int k = 0; k < ns; ++k) out.push_back(full[(size_t)r * k * (N / (ns * E))]);
    ns *= E;
  }
  if (out.empty()) out.push_back(make_float2(1.f, 0.f));
}

static int plan_upload(bpmh_plan p);

// plans alive (guarded by g_loop_mu); the last one frees the buffers below
static std::mutex g_loop_mu;
static int g_plans = 0;
static void loop_bufs_free();

extern "C" int bpmh_plan_create(int nx, int ny, bpmh_plan* out) {
  if (!out) return bpmh_set_error(BPMH_ERR_INVALID, "null plan pointer");
  *out = nullptr;
  if (!pow2_in_range(nx) || !pow2_in_range(ny))
    return bpmh_set_error(BPMH_ERR_UNSUPPORTED,
                          "grid sizes must be powers of two in [16, 4096]");
  bpmh_plan p = new bpmh_plan_s();
  p->nx = nx;
  p->ny = ny;
  p->work = nullptr;
  p->work_bytes = 0;
  p->timing = 0;
  p->ev_used = 0;
  p->row_v = 1;
  p->col_v = 1;
  p->graph_mode = 0;
  p->cap_stream = nullptr;
  p->graph_clock = 0;
  p->loop_mode = 0;
  p->loop_calls = 0;
  p->device = -1;
  for (int e = 0; e < 2; ++e) {
    p->tw_x[e] = p->tw_y[e] = nullptr;
    make_stage_twiddles(nx, row_e_of(nx, e), p->htw_x[e]);
    make_stage_twiddles(ny, col_e_of(ny, e), p->htw_y[e]);
  }
  // device copies now when a device is present (on a machine without one
  // the plan stays host-only: its argument checks still run)
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0) {
    const int rc = plan_upload(p);
    if (rc) {
      delete p;
      return rc;
    }
  } else {
    (void)hipGetLastError();
  }
  {
    std::lock_guard<std::mutex> lock(g_loop_mu);
    ++g_plans;
  }
  *out = p;
  return BPMH_OK;
}

// Device copies of the twiddle tables on the current device, which becomes
// the plan's device (made at plan creation, or at the first propagation of a
// plan created without a device).
static int plan_upload(bpmh_plan p) {
  if (p->tw_x[0]) return BPMH_OK;
  HIP_TRY(hipGetDevice(&p->device));
  auto release = [p] {
    for (int e = 0; e < 2; ++e) {
      (void)hipFree(p->tw_x[e]);
      (void)hipFree(p->tw_y[e]);
      p->tw_x[e] = p->tw_y[e] = nullptr;
    }
  };
  for (int e = 0; e < 2; ++e) {
    if (hipMalloc(&p->tw_x[e], p->htw_x[e].size() * sizeof(float2)) != hipSuccess ||
        hipMalloc(&p->tw_y[e], p->htw_y[e].size() * sizeof(float2)) != hipSuccess) {
      release();
      return bpmh_set_error(BPMH_ERR_NOMEM, "hipMalloc failed for twiddles");
    }
    if (hipMemcpy(p->tw_x[e], p->htw_x[e].data(), p->htw_x[e].size() * sizeof(float2),
                  hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->tw_y[e], p->htw_y[e].data(), p->htw_y[e].size() * sizeof(float2),
                  hipMemcpyHostToDevice) != hipSuccess) {
      release();
      return bpmh_set_error(BPMH_ERR_HIP, "hipMemcpy failed for twiddles");
    }
  }
  return BPMH_OK;
}

extern "C" int bpmh_plan_destroy(bpmh_plan p) {
  if (!p) return BPMH_OK;
  for (int e = 0; e < 2; ++e) {
    (void)hipFree(p->tw_x[e]);
    (void)hipFree(p->tw_y[e]);
  }
  if (p->work) (void)hipFree(p->work);
  for (hipEvent_t e : p->ev) (void)hipEventDestroy(e);
  (void)graph_release_all(p);
  if (p->cap_stream) (void)hipStreamDestroy(p->cap_stream);
  delete p;
  std::lock_guard<std::mutex> lock(g_loop_mu);
  if (--g_plans == 0) loop_bufs_free();
  return BPMH_OK;
}

extern "C" int bpmh_plan_set_graph(bpmh_plan p, int enable) {
  if (!p) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  p->graph_mode = enable != 0;
  if (!p->graph_mode) return graph_release_all(p);
  return BPMH_OK;
}

extern "C" int bpmh_plan_set_timing(bpmh_plan p, int enable) {
  if (!p) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  p->timing = enable != 0;
  p->ev_used = 0;
  return BPMH_OK;
}

extern "C" int bpmh_plan_kernel_times(bpmh_plan p, float* ms, int* counts) {
  if (!p || !ms || !counts) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  for (int k = 0; k < TK_N; ++k) {
    ms[k] = 0.f;
    counts[k] = 0;
  }
  for (size_t i = 0; i < p->ev_used; ++i) {
    float t = 0.f;
    HIP_TRY(hipEventSynchronize(p->ev[2 * i + 1]));
    HIP_TRY(hipEventElapsedTime(&t, p->ev[2 * i], p->ev[2 * i + 1]));
    ms[p->ev_kind[i]] += t;
    counts[p->ev_kind[i]] += 1;
  }
  p->ev_used = 0;
  return BPMH_OK;
}

// Reserve event pairs for n more timed launches (outside any stream capture).
static int timing_reserve(bpmh_plan p, size_t n) {
  const size_t need = 2 * (p->ev_used + n);
  while (p->ev.size() < need) {
    hipEvent_t e;
    HIP_TRY(hipEventCreate(&e));
    p->ev.push_back(e);
  }
  if (p->ev_kind.size() < need / 2) p->ev_kind.resize(need / 2);
  return BPMH_OK;
}

// Plan scratch of at least `bytes` (grown, never shrunk).
static int plan_scratch(bpmh_plan p, size_t bytes, void** ptr) {
  if (bytes > p->work_bytes) {
    if (p->work) {
      HIP_TRY(hipDeviceSynchronize());
      HIP_TRY(hipFree(p->work));
      p->work = nullptr;
      p->work_bytes = 0;
    }
    bytes = (bytes + 255) & ~(size_t)255;
    if (hipMalloc(&p->work, bytes) != hipSuccess)
      return bpmh_set_error(BPMH_ERR_NOMEM, "hipMalloc failed for plan scratch");
    p->work_bytes = bytes;
  }
  *ptr = p->work;
  return BPMH_OK;
}

extern "C" int bpmh_propagator_table(int nx, int ny, int kind, double dx, double dy, double dz,
                                     double n0, double lam, float* H_, void* stream) {
  float2* H = (float2*)H_;
  if (!H) return bpmh_set_error(BPMH_ERR_INVALID, "null H");
  if (nx <= 0 || ny <= 0) return bpmh_set_error(BPMH_ERR_INVALID, "bad grid");
  if (kind != BPMH_H_F32 && kind != BPMH_H_F64)
    return bpmh_set_error(BPMH_ERR_INVALID, "unknown propagator kind");
  dim3 grid((nx + 255) / 256, ny);
  hipLaunchKernelGGL(k_prop_table, grid, dim3(256), 0, (hipStream_t)stream, H, nx, ny, kind, dx,
                     dy, dz, n0, lam);
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}

// ----------------------------------------------------------------------------
// launchers
// ----------------------------------------------------------------------------
typedef void (*row_fn)(const RowArgs&, int batch, hipStream_t);
typedef void (*col_fn)(const ColArgs&, int batch, hipStream_t);

template <int N, int V, int E>
static void launch_row(const RowArgs& a, int batch, hipStream_t s) {
  const int rows = batch * a.ny;
  hipLaunchKernelGGL((k_row<N, V, E>), dim3(rows / RowCfg<N, V, E>::LINES),
                     dim3(RowCfg<N, V, E>::THREADS), 0, s, a);
}
template <int N, int V, int PHASE, int E>
static void launch_col(const ColArgs& a, int batch, hipStream_t s) {
  hipLaunchKernelGGL((k_col<N, V, PHASE, E>), dim3(a.nx / ColCfg<N, V, E>::COLS, batch),
                     dim3(ColCfg<N, V, E>::THREADS), 0, s, a);
}

#define BPMH_SIZES(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)

// Row launcher of variant v = V + 3*ealt for rows of N points.
template <int N>
static row_fn pick_row_n(int v) {
  constexpr int E0 = row_e_of(N, 0), E1 = row_e_of(N, 1);
  switch (v) {
    case 0: return launch_row<N, 0, E0>;
    case 2: return launch_row<N, 2, E0>;
    case 3: return launch_row<N, 0, E1>;
    case 4: return launch_row<N, 1, E1>;
    case 5: return launch_row<N, 2, E1>;
    default: return launch_row<N, 1, E0>;
  }
}

static row_fn pick_row(int n, int v) {
#define ROW_CASE(N) \
  case N:           \
    return pick_row_n<N>(v);
  switch (n) { BPMH_SIZES(ROW_CASE) }
#undef ROW_CASE
  return nullptr;
}

// Column launcher of variant v = V + 5*ealt for columns of N points.
template <int N, int PHASE>
static col_fn pick_col_n(int v) {
  constexpr int E0 = col_e_of(N, 0), E1 = col_e_of(N, 1);
  switch (v) {
    case 0: return launch_col<N, 0, PHASE, E0>;
    case 2: return launch_col<N, 2, PHASE, E0>;
    case 3: return launch_col<N, 3, PHASE, E0>;
    case 4: return launch_col<N, 4, PHASE, E0>;
    case 5: return launch_col<N, 0, PHASE, E1>;
    case 6: return launch_col<N, 1, PHASE, E1>;
    case 7: return launch_col<N, 2, PHASE, E1>;
    case 8: return launch_col<N, 3, PHASE, E1>;
    case 9: return launch_col<N, 4, PHASE, E1>;
    default: return launch_col<N, 1, PHASE, E0>;
  }
}

// Column phases of the weighted adjoint: one launch shape (V = 1) in the
// radix schedule of column variant v (its twiddle table is the plan's).
template <int PHASE>
static col_fn pick_col_adj(int n, int v) {
#define COLA_CASE(N)                                                                   \
  case N:                                                                              \
    return v >= kColShapes ? launch_col<N, 1, PHASE, col_e_of(N, 1)>                  \
                           : launch_col<N, 1, PHASE, col_e_of(N, 0)>;
  switch (n) { BPMH_SIZES(COLA_CASE) }
#undef COLA_CASE
  return nullptr;
}

template <int PHASE>
static col_fn pick_col(int n, int v) {
#define COL_CASE(N) \
  case N:           \
    return pick_col_n<N, PHASE>(v);
  switch (n) { BPMH_SIZES(COL_CASE) }
#undef COL_CASE
  return nullptr;
}

template <int N>
static int col_cols_n(int v) {
  constexpr int E0 = col_e_of(N, 0), E1 = col_e_of(N, 1);
  switch (v) {
    case 0: return ColCfg<N, 0, E0>::COLS;
    case 2: return ColCfg<N, 2, E0>::COLS;
    case 3: return ColCfg<N, 3, E0>::COLS;
    case 4: return ColCfg<N, 4, E0>::COLS;
    case 5: return ColCfg<N, 0, E1>::COLS;
    case 6: return ColCfg<N, 1, E1>::COLS;
    case 7: return ColCfg<N, 2, E1>::COLS;
    case 8: return ColCfg<N, 3, E1>::COLS;
    case 9: return ColCfg<N, 4, E1>::COLS;
    default: return ColCfg<N, 1, E0>::COLS;
  }
}

template <int N>
static int row_lines_n(int v) {
  constexpr int E0 = row_e_of(N, 0), E1 = row_e_of(N, 1);
  switch (v) {
    case 0: return RowCfg<N, 0, E0>::LINES;
    case 2: return RowCfg<N, 2, E0>::LINES;
    case 3: return RowCfg<N, 0, E1>::LINES;
    case 4: return RowCfg<N, 1, E1>::LINES;
    case 5: return RowCfg<N, 2, E1>::LINES;
    default: return RowCfg<N, 1, E0>::LINES;
  }
}

static int col_tiles(int nx, int ny, int v) {
#define TILE_CASE(N) \
  case N:            \
    return nx / col_cols_n<N>(v);
  switch (ny) { BPMH_SIZES(TILE_CASE) }
#undef TILE_CASE
  return 0;
}

// Column variants with V = 3 load and store 16 bytes per column pair: a
// plane that is only 8-byte aligned (a view at an odd element offset) runs
// V = 0 of the same radix schedule (one column per thread), which gives the
// same bits.
static int col_variant_for(int cv, const float2* plane) {
  return (cv % kColShapes == 3 && (reinterpret_cast<uintptr_t>(plane) & 15)) ? cv - 3 : cv;
}

static void variant_shape(int nx, int ny, int rv, int cv, int* lines, int* cols, int* row_e,
                          int* col_e) {
#define SHAPE_CASE(N)                 \
  case N:                             \
    *lines = row_lines_n<N>(rv);      \
    *row_e = row_e_of(N, rv / kRowShapes); \
    break;
  switch (nx) { BPMH_SIZES(SHAPE_CASE) }
#undef SHAPE_CASE
#define CE_CASE(N)                    \
  case N:                             \
    *col_e = col_e_of(N, cv / kColShapes); \
    break;
  switch (ny) { BPMH_SIZES(CE_CASE) }
#undef CE_CASE
  *cols = nx / col_tiles(nx, ny, cv);
}

extern "C" int bpmh_plan_set_variant(bpmh_plan p, int row_variant, int col_variant) {
  if (!p) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  if (row_variant < 0 || row_variant >= 2 * kRowShapes || col_variant < 0 ||
      col_variant >= 2 * kColShapes)
    return bpmh_set_error(BPMH_ERR_INVALID, "row variants are 0 to 5; column variants 0 to 9");
  __atomic_store_n(&p->row_v, row_variant, __ATOMIC_RELAXED);
  __atomic_store_n(&p->col_v, col_variant, __ATOMIC_RELAXED);
  return BPMH_OK;
}

// The variants of one call.  A call reads them once and takes its kernels and
// its twiddle tables from this copy: another host thread may set the plan's
// while the call enqueues (the plans of a grid size are shared), and kernels
// of one radix schedule on the tables of the other give wrong fields.
struct Variant {
  int row, col;
  int row_alt() const { return row / kRowShapes; }  // radix schedules, as ealt
  int col_alt() const { return col / kColShapes; }
};
static Variant plan_variant(bpmh_plan p) {
  return {__atomic_load_n(&p->row_v, __ATOMIC_RELAXED), __atomic_load_n(&p->col_v, __ATOMIC_RELAXED)};
}

extern "C" int bpmh_plan_get_variant(bpmh_plan p, int* row_variant, int* col_variant,
                                     int* lines_per_group, int* cols_per_group, int* row_elems,
                                     int* col_elems) {
  if (!p || !row_variant || !col_variant || !lines_per_group || !cols_per_group || !row_elems ||
      !col_elems)
    return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  const Variant var = plan_variant(p);
  *row_variant = var.row;
  *col_variant = var.col;
  variant_shape(p->nx, p->ny, var.row, var.col, lines_per_group, cols_per_group, row_elems,
                col_elems);
  return BPMH_OK;
}

// Validated arguments of one bpmh_propagate call.
struct PropCall {
  int batch, nz;
  float2* plane;
  const void* dn;
  int dn_kind;
  long long dn_bstride, dn_numel;
  int mean_mode;
  const float2* H;
  const float* n_eff;
  const float* dn0;
  float n0, k0, dx, dy, dz, unit_k;
  int absorb;
  float2* out_field;
  float* out_intens;
  long long out_numel;
  float* out_sum;
  const float* scat_w;
  const float* g_w;
  const float2* plain;
  float* out_scat;
};

static int prop_validate(bpmh_plan plan, const PropCall& c) {
  char b[256];
  if (!plan) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  if (!c.plane) return bpmh_set_error(BPMH_ERR_INVALID, "null plane");
  if (c.batch < 1 || c.nz < 1) return bpmh_set_error(BPMH_ERR_INVALID, "batch and nz must be >= 1");
  if (c.dn_kind < BPMH_DN_NONE || c.dn_kind > BPMH_DN_C64)
    return bpmh_set_error(BPMH_ERR_INVALID, "unknown dn kind");
  if (c.dn_kind != BPMH_DN_NONE && !c.dn) return bpmh_set_error(BPMH_ERR_INVALID, "null dn");
  if (c.dn_bstride < 0) return bpmh_set_error(BPMH_ERR_INVALID, "dn batch stride must be >= 0");
  if (c.mean_mode < BPMH_MEAN_IGNORE || c.mean_mode > BPMH_MEAN_WEIGHTED)
    return bpmh_set_error(BPMH_ERR_INVALID, "unknown mean mode");
  if (c.mean_mode == BPMH_MEAN_IGNORE && !c.H)
    return bpmh_set_error(BPMH_ERR_INVALID, "mean_mode ignore needs a propagator table");
  if (c.mean_mode == BPMH_MEAN_SIMPLE && (!c.n_eff || !c.dn0))
    return bpmh_set_error(BPMH_ERR_INVALID, "mean_mode simple needs n_eff and dn0 arrays");
  if (c.absorb < 0) return bpmh_set_error(BPMH_ERR_INVALID, "absorbing width must be >= 0");
  if (c.out_scat && (!c.scat_w || !c.g_w || !c.plain))
    return bpmh_set_error(BPMH_ERR_INVALID, "scattering output needs weights and plane-wave array");
  // the column grid's y extent is the batch (at most 65535)
  if (c.batch > 65535 || (long long)c.batch * plan->ny > (1LL << 30))
    return bpmh_set_error(BPMH_ERR_INVALID, "batch too large");
  const long long n = (long long)plan->nx * plan->ny;
  if (c.dn_kind != BPMH_DN_NONE) {
    // planes 0..nz-1 of every item (slice 0 also feeds the weighted mean)
    const long long need = (long long)(c.batch - 1) * c.dn_bstride + (long long)c.nz * n;
    if (c.dn_numel < need) {
      snprintf(b, sizeof b, "dn holds %lld elements; %d planes of %d item(s) at stride %lld read %lld",
               c.dn_numel, c.nz, c.batch, c.dn_bstride, need);
      return bpmh_set_error(BPMH_ERR_INVALID, b);
    }
  }
  if (c.out_field || c.out_intens) {
    const long long need = (long long)c.batch * c.nz * n;
    if (c.out_numel < need) {
      snprintf(b, sizeof b, "output volume holds %lld elements; %d item(s) x %d planes write %lld",
               c.out_numel, c.batch, c.nz, need);
      return bpmh_set_error(BPMH_ERR_INVALID, b);
    }
  }
  return BPMH_OK;
}

// Scratch of one call: weighted dn0 per item (batch floats), weighted
// per-column partials (batch*nx float2) and scattering per-column partials
// (batch*nz*nx float2, only with out_scat).
struct StepScratch {
  float2* wpart;
  float2* spart;
  float* dn0;
};

// 0 when the call needs none (no weighted mean, no scattering sums).
static size_t prop_scratch_bytes(bpmh_plan plan, const PropCall& c) {
  if (c.mean_mode != BPMH_MEAN_WEIGHTED && !c.out_scat) return 0;
  const size_t n_w = (size_t)c.batch * plan->nx;
  const size_t n_s = c.out_scat ? (size_t)c.batch * c.nz * plan->nx : 0;
  return (n_w + n_s) * sizeof(float2) + (((size_t)c.batch * 4 + 255) & ~(size_t)255);
}

static StepScratch prop_scratch_carve(bpmh_plan plan, const PropCall& c, void* base) {
  StepScratch r;
  const size_t n_w = (size_t)c.batch * plan->nx;
  const size_t n_s = c.out_scat ? (size_t)c.batch * c.nz * plan->nx : 0;
  const size_t seg = ((size_t)c.batch * 4 + 255) & ~(size_t)255;
  char* p = (char*)base;
  r.dn0 = (float*)p;
  r.wpart = (float2*)(p + seg);
  r.spart = r.wpart + n_w;
  (void)n_s;
  return r;
}

// ----------------------------------------------------------------------------
// one-launch z-loop (loop.hpp): when it runs, and its synchronisation state
// ----------------------------------------------------------------------------
// Synchronisation words of the calls in flight, per device: a call takes a
// buffer whose last user ran on the same stream (stream order protects it) or
// has completed, so calls on several streams and host threads never share
// one.  At most kLoopBufs buffers, each for the largest call (388 KiB), so none
// is ever replaced while calls are in flight; beyond that a call's stream
// waits for the buffer used longest ago.  They are freed with the last plan.
constexpr int kLoopBufs = 16;
struct LoopBuf {
  unsigned* ptr = nullptr;
  hipEvent_t last = nullptr;
  hipStream_t stream = nullptr;
  unsigned long long used = 0;  // 0: never
  unsigned calls = 0;
  bool zero = false;            // the words are zero, once what is enqueued has run
};
static LoopBuf g_loop_buf[64][kLoopBufs];
// per device, in host memory: set by a call whose waits gave up
static unsigned* g_loop_failed[64];
static unsigned long long g_loop_clock = 0;

// Called with g_loop_mu held; -1 when none can be had.
static int loop_buf_take(int dev, hipStream_t s) {
  LoopBuf* b = g_loop_buf[dev];
  int pick = -1;
  for (int i = 0; i < kLoopBufs && pick < 0; ++i)
    if (b[i].used && b[i].stream == s) pick = i;
  for (int i = 0; i < kLoopBufs && pick < 0; ++i)
    if (!b[i].used || hipEventQuery(b[i].last) == hipSuccess) pick = i;
  if (pick < 0) {
    pick = 0;
    for (int i = 1; i < kLoopBufs; ++i)
      if (b[i].used < b[pick].used) pick = i;
  }
  LoopBuf& p = b[pick];
  // (also on the same handle: another stream may have got a destroyed one's)
  if (p.used && hipEventQuery(p.last) != hipSuccess && hipStreamWaitEvent(s, p.last, 0) != hipSuccess)
    pick = -1;
  (void)hipGetLastError();  // hipEventQuery's "not ready"
  if (pick < 0) return -1;
  if (!p.ptr && hipMalloc(&p.ptr, loop_words(kLoopTeams) * sizeof(unsigned)) != hipSuccess) p.ptr = nullptr;
  if (!p.last && hipEventCreateWithFlags(&p.last, hipEventDisableTiming) != hipSuccess) p.last = nullptr;
  if (p.ptr && p.last) return pick;
  (void)hipGetLastError();
  return -1;
}

static void loop_bufs_free() {
  for (auto& dev : g_loop_buf)
    for (LoopBuf& b : dev) {
      if (b.used) (void)hipEventSynchronize(b.last);
      if (b.ptr) (void)hipFree(b.ptr);
      if (b.last) (void)hipEventDestroy(b.last);
      b = LoopBuf();
    }
  for (unsigned*& w : g_loop_failed) {
    if (w) (void)hipHostFree(w);
    w = nullptr;
  }
}

// Reports, once, that a one-launch call on the device gave up (g_loop_mu held).
static int loop_failure(int dev) {
  if (dev < 0 || dev >= 64 || !g_loop_failed[dev] || !__atomic_exchange_n(g_loop_failed[dev], 0u, __ATOMIC_RELAXED))
    return BPMH_OK;
  return bpmh_set_error(BPMH_ERR_HIP,
                        "an earlier one-launch z-loop gave up waiting for its work-groups; its results are NaN");
}

extern "C" int bpmh_loop_check(void) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return BPMH_OK;
  std::lock_guard<std::mutex> lock(g_loop_mu);
  return loop_failure(dev);
}

__global__ void k_fill_zero(float* __restrict__ p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// After every one-launch call: its synchronisation words are zero again for the
// next one, and if one of its waits gave up all that it writes becomes NaN and
// the host's word is set.
constexpr int kLoopOuts = 9;
struct LoopDone {
  unsigned* sync;
  unsigned words, call;
  unsigned* failed;
  float* out[kLoopOuts];  // null: not written by this call
  size_t n[kLoopOuts];
};
constexpr int kDoneThreads = 256;
__global__ void __launch_bounds__(kDoneThreads) k_loop_done(LoopDone d) {
  const unsigned i = blockIdx.x * kDoneThreads + threadIdx.x;
  const unsigned failed = d.sync[kLoopFailed];  // (under way beside the stores)
  if (i < d.words && i != kLoopFailed) d.sync[i] = 0u;
  if (failed != d.call) return;
#pragma unroll
  for (int k = 0; k < kLoopOuts; ++k)
    if (d.out[k])
      for (size_t j = i; j < d.n[k]; j += (size_t)gridDim.x * kDoneThreads)
        d.out[k][j] = __uint_as_float(0x7fc00000u);
  if (i == 0) __hip_atomic_store(d.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

static LoopDone loop_done(const LoopCall& c, int points, int nz, size_t words, unsigned* failed) {
  const size_t plane = (size_t)c.la.batch * points, steps = (size_t)c.la.batch * (nz - 1);
  const size_t comps = c.ra.dn_kind == BPMH_DN_C64 ? 2 : 1;
  return {c.la.sync, (unsigned)words, c.la.call, failed,
          {(float*)c.ra.plane, c.ra.acc, (float*)c.ra.out_field, c.ra.out_intens,
           c.ca.sw ? (float*)c.ca.spart : nullptr, c.ca.gd_item, c.ra.gitem, c.ca.rec_c, c.ca.cg_out},
          {2 * plane, plane, 2 * plane * nz, plane * nz, 2 * (size_t)c.la.batch * nz * c.ca.nx, plane,
           steps * points * comps, steps, steps}};
}

static bool loop_size(bpmh_plan plan) {
  return plan->nx >= 64 && plan->ny >= 64 && plan->nx <= 512 && plan->ny <= 512;
}

// Whether a call of this grid, batch and schedule (er, ec points per thread of
// rows and columns) runs as one launch.  By size: everywhere from 64^2 to
// 512 x 256 (1.3 to 2.6 times faster, loop.hpp), except batches beyond 16 with
// 1024-thread groups (512 x 256 at 4.4, batch 50: 83 against 70 us per step);
// at 512^2, 32 CUs are too few for a field alone (batch 1: 14.0 against 12.5),
// only 8.8 fits two groups a CU (batch 2: 14.3 against 15.7; 16: 27.8 against
// 40; at 4.8 and batch 17 52 against 49.5), and eight fields take a round of
// 14 us, so not when one or two are left over for the last of three or more
// (batch 17: 40.9 against 39.8, 20: 41.9 against 45.7, 33: 69 against 64); with
// the weighted mean's registers a round takes 23.5 us, so it stops at four
// (batch 32: 94 against 96, 40: 117 against 116, 64: 188 against 169).
static bool loop_wanted(bpmh_plan plan, int mode, int batch, int nz, int er, int ec) {
  const int nx = plan->nx, ny = plan->ny;
  if (plan->loop_mode == 1 || nz < 2 || !loop_size(plan)) return false;
  if (!((er == 4 && ec == 4) || (er == 4 && ec == 8) || (er == 8 && ec == 8))) return false;  // not built
  // fields of the records: 20 bits each for field, plane and sequence
  if (nz >= (1 << 20) || (long long)batch * (nz / kLoopStepsPart + 2) >= (1 << 20)) return false;
  if (plan->loop_mode >= 2) return true;
  if (nx * ny == 512 * 512)
    return er == 8 && batch >= 2 && (batch <= 16 || (batch - 1) % 8 > 1) &&
           (mode != BPMH_MEAN_WEIGHTED || batch <= 32);
  if (loop_points(nx, ny) == 4096 && ec == 4) return batch <= 16;
  return true;
}

// us of a step of `fields` fields as one launch and as launches per pass, to
// about 15 % from 64^2 to 512^2 and 1 to 256 fields (the launches rather too
// low).  The loop takes rounds of the fields whose teams an XCD holds at once.
constexpr double kLoopCallUs = 15;  // a loop's start and end
static double loop_step_us(bpmh_plan plan, int ec, int fields) {
  const int nx = plan->nx, ny = plan->ny, slots = loop_slots(nx, ny);
  const int threads = loop_points(nx, ny) / ec;
  const double pts = (double)nx * ny;
  int at_once = 32 * (1024 / threads) / slots;
  if (at_once > loop_teams(slots)) at_once = loop_teams(slots);
  if (at_once < 1) at_once = 1;
  auto round = [&](int k) {
    return (4.2 + 4.1e-5 * pts + 2.5e-5 * pts * (k - 1)) * (threads == 1024 ? 1.3 : 1.);
  };
  const int per_xcd = (fields + 7) / 8, full = per_xcd / at_once, rest = per_xcd % at_once;
  return full * round(at_once) + (rest ? round(rest) : 0.);
}
static double launch_step_us(bpmh_plan plan, int fields) {
  const double v = (double)plan->nx * plan->ny * fields, one = 8.6e-6 * v, many = 5 + 5.9e-6 * v;
  return 8 + (plan->nx >= 512 && many < one ? many : one);  // (many: passes of several items)
}

// The same for the adjoint of a segment of nz planes.  Not built for rows of
// more than one wavefront; the reduction's grid has a block row per plane.
// Without a mean correction a step is short beside the forward planes it reads
// and the screen gradients it writes, so from 512 x 256 on only while the
// teams take the batch in one round (512^2 at 8.8, batch 8: 34.2 against 34.5
// us per step, 16: 68 against 53; 512 x 256, batch 1: 16.3 against 15.7, 16: 33
// against 35, 50: 112 against 80; 256^2, batch 50: 37 against 55).  With one
// it is 1.1 to 2.1 times faster throughout (512^2 at 8.8, batch 8: 81 against
// 116, 50: 546 against 591).
static bool loop_adj_wanted(bpmh_plan plan, int mode, int batch, int nz, int er, int ec) {
  const long long pts = (long long)plan->nx * plan->ny;
  if (!loop_wanted(plan, BPMH_MEAN_IGNORE, batch, nz, er, ec) || plan->nx / er > 64 || nz > 65536) return false;
  if (plan->loop_mode >= 2 || mode != BPMH_MEAN_IGNORE || pts < 512 * 256) return true;
  return batch >= 2 && batch * pts <= 8LL * 512 * 512;
}

// Enqueue the z-loop of a call (adj: the adjoint of a segment of nz planes) as
// one launch.  Returns 1 when done, 0 when this call runs as launches per pass
// (size, schedule, or a stream that is being captured: the synchronisation
// buffer must not be replayed), or an error.
static int loop_run(bpmh_plan plan, Variant var, int mode, int batch, int nz, const LoopCall& call0,
                    hipStream_t s, bool adj = false) {
  const int nx = plan->nx, ny = plan->ny;
  const int er = row_e_of(nx, var.row_alt()), ec = col_e_of(ny, var.col_alt());
  if (!(adj ? loop_adj_wanted(plan, mode, batch, nz, er, ec)
            : loop_wanted(plan, mode, batch, nz, er, ec)))
    return 0;
  loop_launch_fn launch = nx == 64    ? (adj ? bpmh_loop_adj_nx64 : bpmh_loop_nx64)
                          : nx == 128 ? (adj ? bpmh_loop_adj_nx128 : bpmh_loop_nx128)
                          : nx == 256 ? (adj ? bpmh_loop_adj_nx256 : bpmh_loop_nx256)
                                      : (adj ? bpmh_loop_adj_nx512 : bpmh_loop_nx512);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return 0;
  }
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev != plan->device || dev < 0 || dev >= 64) return 0;
  LoopCall call = call0;
  const int slots = loop_slots(nx, ny);
  // teams per XCD: one per field up to what the XCD's 32 CUs hold
  int teams = (batch + 7) / 8;
  const int most = loop_teams(slots);
  if (teams > most) teams = most;
  call.la.batch = batch;
  call.la.teams = teams;
  const size_t words = loop_words(teams);
  std::lock_guard<std::mutex> lock(g_loop_mu);
  const int rc = loop_failure(dev);
  if (rc) return rc;
  unsigned*& failed = g_loop_failed[dev];
  if (!failed) {
    if (hipHostMalloc((void**)&failed, sizeof(unsigned), hipHostMallocPortable | hipHostMallocMapped) !=
        hipSuccess) {
      failed = nullptr;
      (void)hipGetLastError();
      return 0;
    }
    *failed = 0;
  }
  const int i = loop_buf_take(dev, s);
  if (i < 0) return 0;
  LoopBuf& b = g_loop_buf[dev][i];
  call.la.sync = b.ptr;
  if (++b.calls == 0) b.calls = 1;
  call.la.call = b.calls;
  call.la.lost = plan->loop_mode == 4;
  if (!b.zero) {
    const size_t all = loop_words(kLoopTeams);
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)((all + 255) / 256)), dim3(256), 0, s, (float*)b.ptr, all);
  }
  const int groups = 8 * teams * slots;
  const bool ok = launch(ny, er, ec, mode, call, plan->loop_mode == 3 ? groups / 4 : groups, s);
  if (ok)
    hipLaunchKernelGGL(k_loop_done, dim3((unsigned)((words + kDoneThreads - 1) / kDoneThreads)),
                       dim3(kDoneThreads), 0, s,
                       loop_done(call, nx * ny, nz, words, failed));
  const hipError_t le = hipGetLastError();
  const hipError_t re = hipEventRecord(b.last, s);
  if (re != hipSuccess) (void)hipStreamSynchronize(s);  // no event tells when the buffer is free
  b.zero = ok && le == hipSuccess;
  b.stream = s;
  b.used = ++g_loop_clock;
  if (!ok) return 0;
  if (le != hipSuccess || re != hipSuccess)
    return bpmh_set_error(BPMH_ERR_HIP, hipGetErrorString(le != hipSuccess ? le : re));
  ++plan->loop_calls;
  return 1;
}

extern "C" int bpmh_plan_set_loop(bpmh_plan p, int mode) {
  if (!p) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  if (mode < 0 || mode > 4) return bpmh_set_error(BPMH_ERR_INVALID, "loop mode is 0 to 4");
  p->loop_mode = mode;
  return BPMH_OK;
}

extern "C" int bpmh_plan_loop_calls(bpmh_plan p, long long* calls) {
  if (!p || !calls) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  std::lock_guard<std::mutex> lock(g_loop_mu);
  *calls = p->loop_calls;
  return BPMH_OK;
}

// ----------------------------------------------------------------------------
// passes of several items per work-group (items.hpp)
// ----------------------------------------------------------------------------
// They run from kItemsRows/kItemsCols points of a call on.  us per step with
// the one-item passes / with these (each pass alone; running sum kept):
//   1024^2  batch 2: 36.0 / 34.4 (rows 35.4, columns 34.4)
//           batch 3: 49.0 / 40.5 (44.1, 44.7);  4: 62.1 / 45.9;  16: 191 / 139
//   2048^2  batch 1: 81.1 / 63.7 (73.5, 72.3);  4: 274 / 164
//   512 x 1024  batch 16: 118 / 80;   1024 x 512  batch 16: 90 / 69
// Below, their registers leave too few wavefronts to hide a short call's
// latencies: rows of 2 M points 33.4 against 32.2 (2048 x 64, batch 16), of
// 1 M 24.3 against 21.7 (1024^2, batch 1); columns of 1 M points 27.9 against
// 24.9 (256 x 2048, batch 2).  Lines of 512, 1024 and 2048 points have them;
// there is none for 4096 and shorter lines and the weighted column passes.
constexpr long long kItemsRows = 5 << 19, kItemsCols = 2 << 20;
constexpr long long kItemsThreads = 256 << 10;  // 16 wavefronts a CU

// Items per work-group: as many as leave 16 wavefronts a CU, at most 8.
static int items_per(long long threads, int batch) {
  const long long most = threads / kItemsThreads;
  const int per = (int)(most < 1 ? 1 : (most > 8 ? 8 : most));
  const int chunks = (batch + per - 1) / per;
  return (batch + chunks - 1) / chunks;
}

template <int NX, int E>
static void launch_row_items(const RowArgs& a, int batch, hipStream_t s) {
  constexpr int T = NX / E, LINES = T >= 256 ? 1 : 256 / T, W = E == 4 ? 5 : 3;
  const bool shared = a.ngroups == 0 && a.dn_bstride == 0 && a.dn0_mode != BPMH_MEAN_WEIGHTED;
  const int per = shared || !a.screen ? items_per((long long)batch * a.ny * T, batch) : 1;
  const dim3 g(a.ny / LINES, (batch + per - 1) / per), b(T * LINES);
  if (a.adjoint) hipLaunchKernelGGL((k_row_items<NX, E, LINES, W, true>), g, b, 0, s, a, batch, per);
  else hipLaunchKernelGGL((k_row_items<NX, E, LINES, W, false>), g, b, 0, s, a, batch, per);
}
template <int NY, int E>
static void launch_col_items(const ColArgs& a, int batch, hipStream_t s) {
  constexpr int T = NY / E, LC = T >= 512 ? 2 : (T >= 128 ? 4 : 8);
  const int per = items_per((long long)batch * a.nx * T, batch);
  const dim3 g(a.nx / LC, (batch + per - 1) / per), b(T * LC);
  if (a.hmode == 0) hipLaunchKernelGGL((k_col_items<NY, E, LC, 4, false>), g, b, 0, s, a, batch, per);
  else hipLaunchKernelGGL((k_col_items<NY, E, LC, 4, true>), g, b, 0, s, a, batch, per);
}
template <int N>
static void run_row_items(int ealt, const RowArgs& a, int batch, hipStream_t s) {
  if (ealt) launch_row_items<N, row_e_of(N, 1)>(a, batch, s);
  else launch_row_items<N, row_e_of(N, 0)>(a, batch, s);
}
template <int N>
static void run_col_items(int ealt, const ColArgs& a, int batch, hipStream_t s) {
  if (ealt) launch_col_items<N, col_e_of(N, 1)>(a, batch, s);
  else launch_col_items<N, col_e_of(N, 0)>(a, batch, s);
}

// One row pass of a call; row: its one-item pass.
static void run_row(bpmh_plan plan, Variant var, row_fn row, const RowArgs& a, int batch, hipStream_t s) {
  const int nx = plan->nx, ealt = var.row_alt();
  if ((nx == 512 || nx == 1024 || nx == 2048) && (long long)batch * nx * plan->ny >= kItemsRows &&
      (!a.adjoint || a.screen)) {
    if (nx == 512) run_row_items<512>(ealt, a, batch, s);
    else if (nx == 1024) run_row_items<1024>(ealt, a, batch, s);
    else run_row_items<2048>(ealt, a, batch, s);
  } else {
    row(a, batch, s);
  }
}

// One column pass with H of a table or of n_eff[z].
static void run_col(bpmh_plan plan, Variant var, col_fn col, const ColArgs& a, int batch, hipStream_t s) {
  const int ny = plan->ny, ealt = var.col_alt();
  if ((ny == 512 || ny == 1024 || ny == 2048) && (long long)batch * ny * plan->nx >= kItemsCols &&
      !a.sw) {
    if (ny == 512) run_col_items<512>(ealt, a, batch, s);
    else if (ny == 1024) run_col_items<1024>(ealt, a, batch, s);
    else run_col_items<2048>(ealt, a, batch, s);
  } else {
    col(a, batch, s);
  }
}

// Enqueue (or capture and replay) the whole z-loop of one call on stream s.
// may_allocate false: plain launches only (no graph capture or timing
// events, which create runtime objects).
static int prop_run(bpmh_plan plan, const PropCall& c, const StepScratch& sc, hipStream_t s,
                    bool may_allocate) {
  const int nx = plan->nx, ny = plan->ny;
  const int batch = c.batch, nz = c.nz;
  const Variant var = plan_variant(plan);
  const row_fn row = pick_row(nx, var.row);
  const int cv = col_variant_for(var.col, c.plane);
  // the simple mean's propagator is evaluated in the column pass (PHASE 5)
  const col_fn col0 =
      c.mean_mode == BPMH_MEAN_SIMPLE ? pick_col<5>(ny, cv) : pick_col<0>(ny, cv);
  const col_fn colA = pick_col<1>(ny, cv);
  const col_fn colB = pick_col<2>(ny, cv);

  RowArgs ra;
  memset(&ra, 0, sizeof ra);
  ra.plane = c.plane;
  ra.tw = plan->tw_x[var.row_alt()];
  ra.dn = c.dn;
  ra.dn_bstride = c.dn_bstride;
  ra.dn_kind = c.dn_kind;
  ra.ny = ny;
  ra.nz = nz;
  ra.unit_k = c.unit_k;
  ra.inv_n = 1.0f / ((float)nx * (float)ny);
  ra.absorb = c.absorb;
  ra.dn0_mode = (c.dn_kind == BPMH_DN_NONE) ? 0 : c.mean_mode;
  ra.dn0_arr = c.dn0;
  ra.dn0_item = sc.dn0;
  ra.out_field = c.out_field;
  ra.out_intens = c.out_intens;
  ra.acc = c.out_sum;

  ColArgs ca;
  memset(&ca, 0, sizeof ca);
  ca.plane = c.plane;
  ca.tw = plan->tw_y[cv / kColShapes];
  ca.nx = nx;
  ca.nz = nz;
  ca.hmode = c.mean_mode;  // 0 table, 1 n_eff array, 2 weighted
  ca.H = c.H;
  ca.n_eff = c.n_eff;
  ca.n0 = c.n0;
  ca.k0 = c.k0;
  ca.dx = c.dx;
  ca.dy = c.dy;
  ca.dz = c.dz;
  ca.dn = c.dn;
  ca.dn_bstride = c.dn_bstride;
  ca.dn_kind = c.dn_kind;
  ca.wpart = sc.wpart;
  ca.dn0_item = sc.dn0;
  ca.sw = c.out_scat ? c.scat_w : nullptr;
  ca.gw = c.g_w;
  ca.pw = c.plain;
  ca.spart = sc.spart;

  const bool timing = may_allocate && plan->timing;
  if (may_allocate && !timing) {
    LoopCall call;
    memset(&call, 0, sizeof call);
    call.ra = ra;
    call.ca = ca;
    const int rc = loop_run(plan, var, c.mean_mode, batch, nz, call, s);
    if (rc < 0) return rc;
    if (rc == 1) {
      if (c.out_scat)
        hipLaunchKernelGGL(k_scatter_final, dim3((nz + 63) / 64, batch), dim3(64), 0, s, sc.spart,
                           c.out_scat, nz, nx);
      HIP_TRY(hipGetLastError());
      return BPMH_OK;
    }
  }
  if (timing) {
    const int rc = timing_reserve(plan, (size_t)nz * 3 + 1);
    if (rc) return rc;
  }
  const bool use_graph = may_allocate && plan->graph_mode && !plan->timing;
  const hipStream_t user = s;
  std::vector<unsigned char> key;
  if (use_graph) {
    auto put = [&key](const void* v, size_t n) {
      const unsigned char* q = (const unsigned char*)v;
      key.insert(key.end(), q, q + n);
    };
    put(&ra, sizeof ra);
    put(&ca, sizeof ca);
    put(&batch, sizeof batch);
    put(&nz, sizeof nz);
    put(&c.mean_mode, sizeof c.mean_mode);
    put(&c.out_scat, sizeof c.out_scat);
    put(&var, sizeof var);
    for (GraphEntry& g : plan->graphs) {
      if (g.key == key) {
        HIP_TRY(hipGraphLaunch(g.exec, user));
        HIP_TRY(hipEventRecord(g.done, user));
        g.used = ++plan->graph_clock;
        return BPMH_OK;
      }
    }
    if (!plan->cap_stream) HIP_TRY(hipStreamCreateWithFlags(&plan->cap_stream, hipStreamNonBlocking));
    HIP_TRY(hipStreamBeginCapture(plan->cap_stream, hipStreamCaptureModeThreadLocal));
    s = plan->cap_stream;
  }
  auto timed = [&](int kind, auto&& launch) {
    if (!timing) {
      launch();
      return;
    }
    const size_t i = plan->ev_used++;
    plan->ev_kind[i] = kind;
    (void)hipEventRecord(plan->ev[2 * i], s);
    launch();
    (void)hipEventRecord(plan->ev[2 * i + 1], s);
  };

  // plane 0: outputs of u0, then FFT_x
  ra.z = 0;
  ra.acc_init = 1;
  ra.inverse = 0;
  ra.screen = 0;
  ra.fwd_items = nz > 1 ? batch : 0;
  timed(TK_ROW, [&] { run_row(plan, var, row, ra, batch, s); });
  ra.acc_init = 0;
  ra.inverse = 1;
  ra.screen = c.dn_kind != BPMH_DN_NONE;
  for (int z = 1; z < nz; ++z) {
    ca.z = z;
    if (c.mean_mode == BPMH_MEAN_WEIGHTED) {
      timed(TK_COL_A, [&] { colA(ca, batch, s); });
      timed(TK_COL_B, [&] { colB(ca, batch, s); });
    } else {
      timed(TK_COL, [&] { run_col(plan, var, col0, ca, batch, s); });
    }
    ra.z = z;
    ra.fwd_items = z < nz - 1 ? batch : 0;
    timed(TK_ROW, [&] { run_row(plan, var, row, ra, batch, s); });
  }
  if (c.out_scat) {
    hipLaunchKernelGGL(k_scatter_final, dim3((nz + 63) / 64, batch), dim3(64), 0, s, sc.spart,
                       c.out_scat, nz, nx);
  }
  if (use_graph) {
    hipGraph_t g = nullptr;
    hipError_t le = hipGetLastError();
    hipError_t ce = hipStreamEndCapture(plan->cap_stream, &g);
    if (le != hipSuccess || ce != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return bpmh_set_error(BPMH_ERR_HIP, hipGetErrorString(le != hipSuccess ? le : ce));
    }
    GraphEntry e;
    e.key = std::move(key);
    e.exec = nullptr;
    e.done = nullptr;
    hipError_t ie = hipGraphInstantiate(&e.exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess) return bpmh_set_error(BPMH_ERR_HIP, hipGetErrorString(ie));
    hipError_t ee = hipEventCreateWithFlags(&e.done, hipEventDisableTiming);
    if (ee != hipSuccess) {
      (void)hipGraphExecDestroy(e.exec);
      return bpmh_set_error(BPMH_ERR_HIP, hipGetErrorString(ee));
    }
    if ((int)plan->graphs.size() >= kGraphCache) {
      size_t lru = 0;
      for (size_t i = 1; i < plan->graphs.size(); ++i)
        if (plan->graphs[i].used < plan->graphs[lru].used) lru = i;
      const int rc = graph_release(plan->graphs[lru]);
      plan->graphs.erase(plan->graphs.begin() + lru);
      if (rc) {
        (void)hipGraphExecDestroy(e.exec);
        (void)hipEventDestroy(e.done);
        return rc;
      }
    }
    e.used = ++plan->graph_clock;
    plan->graphs.push_back(std::move(e));
    GraphEntry& ne = plan->graphs.back();
    HIP_TRY(hipGraphLaunch(ne.exec, user));
    HIP_TRY(hipEventRecord(ne.done, user));
    return BPMH_OK;
  }
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}

// ----------------------------------------------------------------------------
// memory floor of a step: the two passes' global loads and stores in their
// launch shapes, without the transforms
// ----------------------------------------------------------------------------
// Row pattern: each line of the row pass read and written with streaming
// accesses and its dn row read (20 B per voxel), one multiply in between.
template <int NX, int V, int EE>
__global__ void __launch_bounds__((RowCfg<NX, V, EE>::THREADS))
k_floor_row(float2* __restrict__ plane, const float* __restrict__ dn, int ny, int z) {
  using Cfg = RowCfg<NX, V, EE>;
  constexpr int E = Cfg::E, T = Cfg::T, LINES = Cfg::LINES;
  const int line = threadIdx.x / T;
  const int t = threadIdx.x - line * T;
  const int row = blockIdx.x * LINES + line;
  const int y = row % ny;
  float2* p = plane + (size_t)row * NX;
  const float* d = dn + ((size_t)z * ny + y) * NX;
  float2 v[E];
  float dv[E];
#pragma unroll
  for (int m = 0; m < E; ++m) v[m] = ld_stream(p + t + m * T);
#pragma unroll
  for (int m = 0; m < E; ++m) dv[m] = d[t + m * T];
#pragma unroll
  for (int m = 0; m < E; ++m) st_stream(p + t + m * T, c_scale(v[m], 1.f + dv[m]));
}

// Column pattern: the column pass's tiles (XCD-aware tile order, P columns
// per thread with 16-byte accesses when P = 2) read and written, 16 B per
// voxel.
template <int NY, int V, int EE>
__global__ void __launch_bounds__((ColCfg<NY, V, EE>::THREADS)) k_floor_col(float2* __restrict__ plane,
                                                                          int nx) {
  using Cfg = ColCfg<NY, V, EE>;
  constexpr int E = Cfg::E, T = Cfg::T, COLS = Cfg::COLS, P = Cfg::P, LC = Cfg::LC;
  const int ntiles = nx / COLS;
  const int bx = blockIdx.x;
  const int tile = (ntiles % 8 == 0) ? (bx & 7) * (ntiles >> 3) + (bx >> 3) : bx;
  const int c = threadIdx.x % LC;
  const int t = threadIdx.x / LC;
  float2* p = plane + (size_t)blockIdx.y * NY * nx + tile * COLS + c * P;
  constexpr bool WIDE = P == 2 && !Cfg::SPLIT;  // 16-byte accesses, as the pass
  float2 v[P][E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    float2* r = p + (size_t)(t + m * T) * nx;
    if constexpr (WIDE) {
      const float4 w = *reinterpret_cast<const float4*>(r);
      v[0][m] = make_float2(w.x, w.y);
      v[1][m] = make_float2(w.z, w.w);
    } else {
#pragma unroll
      for (int q = 0; q < P; ++q) v[q][m] = r[q];
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) {
    float2* r = p + (size_t)(t + m * T) * nx;
    if constexpr (WIDE) {
      *reinterpret_cast<float4*>(r) = make_float4(-v[0][m].x, v[0][m].y, -v[1][m].x, v[1][m].y);
    } else {
#pragma unroll
      for (int q = 0; q < P; ++q) r[q] = make_float2(-v[q][m].x, v[q][m].y);
    }
  }
}

template <int N, int V, int E>
static void launch_floor_row(float2* plane, const float* dn, int batch, int ny, int z,
                             hipStream_t s) {
  hipLaunchKernelGGL((k_floor_row<N, V, E>), dim3(batch * ny / RowCfg<N, V, E>::LINES),
                     dim3(RowCfg<N, V, E>::THREADS), 0, s, plane, dn, ny, z);
}

template <int N, int V, int E>
static void launch_floor_col(float2* plane, int batch, int nx, hipStream_t s) {
  hipLaunchKernelGGL((k_floor_col<N, V, E>), dim3(nx / ColCfg<N, V, E>::COLS, batch),
                     dim3(ColCfg<N, V, E>::THREADS), 0, s, plane, nx);
}

typedef void (*floor_row_fn)(float2*, const float*, int, int, int, hipStream_t);
typedef void (*floor_col_fn)(float2*, int, int, hipStream_t);

template <int N>
static floor_row_fn pick_floor_row_n(int v) {
  constexpr int E0 = row_e_of(N, 0), E1 = row_e_of(N, 1);
  switch (v) {
    case 0: return launch_floor_row<N, 0, E0>;
    case 2: return launch_floor_row<N, 2, E0>;
    case 3: return launch_floor_row<N, 0, E1>;
    case 4: return launch_floor_row<N, 1, E1>;
    case 5: return launch_floor_row<N, 2, E1>;
    default: return launch_floor_row<N, 1, E0>;
  }
}

template <int N>
static floor_col_fn pick_floor_col_n(int v) {
  constexpr int E0 = col_e_of(N, 0), E1 = col_e_of(N, 1);
  switch (v) {
    case 0: return launch_floor_col<N, 0, E0>;
    case 2: return launch_floor_col<N, 2, E0>;
    case 3: return launch_floor_col<N, 3, E0>;
    case 4: return launch_floor_col<N, 4, E0>;
    case 5: return launch_floor_col<N, 0, E1>;
    case 6: return launch_floor_col<N, 1, E1>;
    case 7: return launch_floor_col<N, 2, E1>;
    case 8: return launch_floor_col<N, 3, E1>;
    case 9: return launch_floor_col<N, 4, E1>;
    default: return launch_floor_col<N, 1, E0>;
  }
}

extern "C" int bpmh_floor_steps(bpmh_plan plan, int batch, int nz, float* plane_, const float* dn,
                                long long dn_numel, void* stream) {
  if (!plan || !plane_ || !dn) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  if (batch < 1 || nz < 1 || batch > 65535 || (long long)batch * plan->ny > (1LL << 30))
    return bpmh_set_error(BPMH_ERR_INVALID, "bad batch or depth");
  const int nx = plan->nx, ny = plan->ny;
  if (dn_numel < (long long)nz * nx * ny)
    return bpmh_set_error(BPMH_ERR_INVALID, "dn holds fewer than nz planes");
  float2* plane = (float2*)plane_;
  const Variant var = plan_variant(plan);
  const int cv = col_variant_for(var.col, plane);
  floor_row_fn fr = nullptr;
  floor_col_fn fc = nullptr;
#define FLOOR_CASE(N)                          \
  case N:                                      \
    fr = pick_floor_row_n<N>(var.row);         \
    break;
  switch (nx) { BPMH_SIZES(FLOOR_CASE) }
#undef FLOOR_CASE
#define FLOOR_CASE(N)                  \
  case N:                              \
    fc = pick_floor_col_n<N>(cv);      \
    break;
  switch (ny) { BPMH_SIZES(FLOOR_CASE) }
#undef FLOOR_CASE
  if (!fr || !fc) return bpmh_set_error(BPMH_ERR_UNSUPPORTED, "grid size");
  hipStream_t s = (hipStream_t)stream;
  for (int z = 1; z < nz; ++z) {
    fc(plane, batch, nx, s);
    fr(plane, dn, batch, ny, z, s);
  }
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}

extern "C" int bpmh_propagate(bpmh_plan plan, int batch, int nz, float* plane, const void* dn,
                              int dn_kind, long long dn_batch_stride, long long dn_numel,
                              int mean_mode, const float* H, const float* n_eff, const float* dn0,
                              float n0, float k0, float dx, float dy, float dz, float unit_k,
                              int absorb, float* out_field, float* out_intens,
                              long long out_numel, float* out_sum, const float* scat_w,
                              const float* g_w, const float* plain, float* out_scat,
                              void* stream) {
  PropCall c;
  c.batch = batch;
  c.nz = nz;
  c.plane = (float2*)plane;
  c.dn = dn;
  c.dn_kind = dn_kind;
  c.dn_bstride = dn_batch_stride;
  c.dn_numel = dn_numel;
  c.mean_mode = mean_mode;
  c.H = (const float2*)H;
  c.n_eff = n_eff;
  c.dn0 = dn0;
  c.n0 = n0;
  c.k0 = k0;
  c.dx = dx;
  c.dy = dy;
  c.dz = dz;
  c.unit_k = unit_k;
  c.absorb = absorb;
  c.out_field = (float2*)out_field;
  c.out_intens = out_intens;
  c.out_numel = out_numel;
  c.out_sum = out_sum;
  c.scat_w = scat_w;
  c.g_w = g_w;
  c.plain = (const float2*)plain;
  c.out_scat = out_scat;
  int rc = prop_validate(plan, c);
  if (rc) return rc;
  rc = plan_upload(plan);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  StepScratch sc = {nullptr, nullptr, nullptr};
  const size_t sb = prop_scratch_bytes(plan, c);
  if (sb) {
    void* scr = nullptr;
    rc = plan_scratch(plan, sb, &scr);
    if (rc) return rc;
    sc = prop_scratch_carve(plan, c, scr);
  }
  return prop_run(plan, c, sc, s, true);
}

// ----------------------------------------------------------------------------
// ragged batch: groups of fields with their own dn volumes and depths
// ----------------------------------------------------------------------------
// How a ragged batch runs as one-launch loops: the number of them, in ends[r]
// the first (deepest) group of loop r, loop 0 holding the shallowest groups; 0:
// as launches per pass.  Without events it is one loop.  With events a group's
// fires at the end of its loop, while the launches, which carry all groups
// side by side, finish a group after its own depth.  So the groups are cut into
// the loops that end first among those in which, by the step times above, no
// group ends later than it would with the launches.  Measured, us until the
// shallowest / the last group is done: so, as launches, one loop per group:
//   128^2, 6 jobs of 8 angles x 200 planes   1360 / 1380, 3060 / 3070, 930 / 5450
//   128^2, 24 x 193, 17 x 150, 9 x 77         400 / 1600, 1240 / 2790, 390 / 2190
//   256^2, the same                          2310 / 5290, 3180 / 6790, 620 / 5890
//   256^2, 3 jobs of 1 angle, 200, 150, 100  (launches)   1110 / 2190, 620 / 2740
//   512^2, 8 x 100, 8 x 80, 8 x 60           2260 / 3900, 3120 / 4530, 930 / 3880
static int groups_runs(bpmh_plan plan, Variant var, int n, const int* items, const int* nzs, bool events,
                       int* ends) {
  const int er = row_e_of(plan->nx, var.row_alt()), ec = col_e_of(plan->ny, var.col_alt());
  auto wanted = [&](int lo, int hi) {  // groups [lo, hi) as one loop
    int fields = 0;
    for (int g = lo; g < hi; ++g) fields += items[g];
    return loop_wanted(plan, BPMH_MEAN_IGNORE, fields, nzs[lo], er, ec);
  };
  if (!events || n == 1) {
    ends[0] = 0;
    return wanted(0, n) ? 1 : 0;
  }
  int runs = 0;
  if (plan->loop_mode >= 2) {  // a loop for each depth
    for (int lo = n, hi = n; lo > 0; hi = lo) {
      for (--lo; lo > 0 && nzs[lo - 1] == nzs[hi - 1];) --lo;
      if (!wanted(lo, hi)) return runs;
      ends[runs++] = lo;
    }
    return runs;
  }
  // us of the steps that carry groups [lo, hi), and until group g is done
  // (launches: lo = 0, hi = n)
  auto until = [&](int lo, int hi, int g, auto&& step) {
    double us = 0;
    int fields = 0;
    for (int k = lo; k < hi; ++k) fields += items[k];
    for (int k = hi - 1, z = 1; k >= g; fields -= items[k--])
      if (nzs[k] > z) us += (nzs[k] - z) * step(fields), z = nzs[k];
    return us;
  };
  double best[BPMH_MAX_GROUPS + 1];  // groups [lo, n) done, over their best cut
  int cut[BPMH_MAX_GROUPS + 1];      // the end of the first group's loop
  best[n] = 0;
  for (int lo = n - 1; lo >= 0; --lo) {
    best[lo] = -1;
    for (int hi = lo + 1; hi <= n; ++hi) {
      if (best[hi] < 0 || !wanted(lo, hi)) continue;
      const double us = best[hi] + kLoopCallUs +
                        until(lo, hi, lo, [&](int f) { return loop_step_us(plan, ec, f); });
      const double most = until(0, n, hi - 1, [&](int f) { return launch_step_us(plan, f); });
      if (us - kLoopCallUs > .95 * most || (best[lo] >= 0 && us >= best[lo])) continue;
      best[lo] = us;
      cut[lo] = hi;
    }
  }
  if (best[0] < 0) return 0;
  for (int lo = 0; lo < n; lo = cut[lo]) ++runs;
  for (int lo = 0, r = runs; lo < n; lo = cut[lo]) ends[--r] = lo;
  return runs;
}

// The launches per pass of a ragged batch: group g of items[g] fields, depth
// nzs[g]; events as in bpmh_propagate_groups.
static int groups_launches(bpmh_plan plan, Variant var, row_fn row, col_fn col, RowArgs ra, ColArgs ca,
                           int dn_kind, int n_groups, const int* items, const int* nzs, int total,
                           void** group_done, hipStream_t s) {
  // items still propagating at plane z (and, for the forward transform, past
  // it): a prefix, the groups being in order of non-increasing depth
  auto items_deeper = [&](int z) {
    int c = 0;
    for (int g = 0; g < n_groups; ++g)
      if (nzs[g] > z) c += items[g];
    return c;
  };
  auto mark_done = [&](int z) -> int {  // groups whose last plane is z
    if (!group_done) return BPMH_OK;
    for (int g = 0; g < n_groups; ++g)
      if (nzs[g] - 1 == z && group_done[g]) HIP_TRY(hipEventRecord((hipEvent_t)group_done[g], s));
    return BPMH_OK;
  };
  ra.z = 0;
  ra.acc_init = 1;
  ra.inverse = 0;
  ra.screen = 0;
  ra.fwd_items = items_deeper(1);
  run_row(plan, var, row, ra, total, s);
  int rc = mark_done(0);
  if (rc) return rc;
  ra.acc_init = 0;
  ra.inverse = 1;
  ra.screen = dn_kind != BPMH_DN_NONE;
  for (int z = 1; z < nzs[0]; ++z) {
    const int active = items_deeper(z);
    ca.z = z;
    run_col(plan, var, col, ca, active, s);
    ra.z = z;
    ra.fwd_items = items_deeper(z + 1);
    run_row(plan, var, row, ra, active, s);
    rc = mark_done(z);
    if (rc) return rc;
  }
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}

extern "C" int bpmh_propagate_groups(bpmh_plan plan, int n_groups, const int* items,
                                     const int* nzs, float* plane_, const void* dn, int dn_kind,
                                     long long dn_group_stride, long long dn_numel,
                                     const float* H_, float unit_k, int absorb, float* out_sum,
                                     void** group_done, void* stream) {
  float2* plane = (float2*)plane_;
  const float2* H = (const float2*)H_;
  char b[256];
  if (!plan) return bpmh_set_error(BPMH_ERR_INVALID, "null plan");
  if (!plane || !H) return bpmh_set_error(BPMH_ERR_INVALID, "null plane or propagator");
  if (n_groups < 1 || n_groups > BPMH_MAX_GROUPS || !items || !nzs)
    return bpmh_set_error(BPMH_ERR_INVALID, "1 to 16 groups with item and depth arrays");
  if (dn_kind != BPMH_DN_NONE && dn_kind != BPMH_DN_F32 && dn_kind != BPMH_DN_F16 &&
      dn_kind != BPMH_DN_C64)
    return bpmh_set_error(BPMH_ERR_INVALID, "unknown dn kind");
  if (dn_kind != BPMH_DN_NONE && !dn) return bpmh_set_error(BPMH_ERR_INVALID, "null dn");
  if (dn_group_stride < 0 || absorb < 0)
    return bpmh_set_error(BPMH_ERR_INVALID, "negative stride or absorbing width");
  const int nx = plan->nx, ny = plan->ny;
  const long long n = (long long)nx * ny;
  int total = 0;
  for (int g = 0; g < n_groups; ++g) {
    if (items[g] < 1 || nzs[g] < 1)
      return bpmh_set_error(BPMH_ERR_INVALID, "every group needs >= 1 item and >= 1 plane");
    if (g > 0 && nzs[g] > nzs[g - 1])
      return bpmh_set_error(BPMH_ERR_INVALID, "groups must come in order of non-increasing depth");
    if (dn_kind != BPMH_DN_NONE &&
        (long long)g * dn_group_stride + (long long)nzs[g] * n > dn_numel) {
      snprintf(b, sizeof b, "dn holds %lld elements; group %d reads %d planes at offset %lld",
               dn_numel, g, nzs[g], (long long)g * dn_group_stride);
      return bpmh_set_error(BPMH_ERR_INVALID, b);
    }
    total += items[g];
    if (total > 65535) return bpmh_set_error(BPMH_ERR_INVALID, "batch too large");
  }
  if ((long long)total * ny > (1LL << 30)) return bpmh_set_error(BPMH_ERR_INVALID, "batch too large");
  int rc = plan_upload(plan);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const Variant var = plan_variant(plan);
  const row_fn row = pick_row(nx, var.row);
  const int cv = col_variant_for(var.col, plane);
  const col_fn col = pick_col<0>(ny, cv);

  RowArgs ra;
  memset(&ra, 0, sizeof ra);
  ra.plane = plane;
  ra.tw = plan->tw_x[var.row_alt()];
  ra.dn = dn;
  ra.dn_bstride = dn_group_stride;
  ra.dn_kind = dn_kind;
  ra.ngroups = n_groups;
  for (int g = 0, e = 0; g < n_groups; ++g) ra.gend[g] = (e += items[g]);
  ra.ny = ny;
  ra.nz = nzs[0];
  ra.unit_k = unit_k;
  ra.inv_n = 1.0f / ((float)nx * (float)ny);
  ra.absorb = absorb;
  ra.acc = out_sum;

  ColArgs ca;
  memset(&ca, 0, sizeof ca);
  ca.plane = plane;
  ca.tw = plan->tw_y[cv / kColShapes];
  ca.nx = nx;
  ca.nz = nzs[0];
  ca.hmode = 0;
  ca.H = H;

  // As one-launch loops, each over a run of groups of neighbouring depths, the
  // shallowest first; all in one without events.
  int ends[BPMH_MAX_GROUPS];
  const int runs = groups_runs(plan, var, n_groups, items, nzs, group_done != nullptr, ends);
  const size_t dn_size = dn_kind == BPMH_DN_F16 ? 2 : (dn_kind == BPMH_DN_C64 ? 8 : 4);
  int left = n_groups;  // groups [0, left) are still to be run
  for (int r = 0; r < runs; ++r) {
    const int lo = ends[r];  // the run is groups [lo, left)
    int first = 0, fields = 0;
    for (int g = 0; g < lo; ++g) first += items[g];
    LoopCall call;
    memset(&call, 0, sizeof call);
    call.ra = ra;
    call.ca = ca;
    call.ra.plane = call.ca.plane = plane + (size_t)first * n;
    call.ra.acc = out_sum ? out_sum + (size_t)first * n : nullptr;
    if (dn) call.ra.dn = (const char*)dn + (size_t)lo * dn_group_stride * dn_size;
    call.ra.ngroups = left - lo;
    for (int g = lo; g < left; ++g) {
      call.ra.gend[g - lo] = (fields += items[g]);
      call.la.gnz[g - lo] = nzs[g];
    }
    call.ra.nz = call.ca.nz = nzs[lo];
    rc = loop_run(plan, var, BPMH_MEAN_IGNORE, fields, nzs[lo], call, s);
    if (rc < 0) return rc;
    if (rc == 0) break;
    for (int g = left - 1; g >= lo && group_done; --g)
      if (group_done[g]) HIP_TRY(hipEventRecord((hipEvent_t)group_done[g], s));
    left = lo;
    total = first;
  }
  if (left == 0) return BPMH_OK;
  return groups_launches(plan, var, row, col, ra, ca, dn_kind, left, items, nzs, total, group_done, s);
}

// ----------------------------------------------------------------------------
// allocation-free variant of bpmh_propagate
// ----------------------------------------------------------------------------
// Its step scratch (weighted-mean and scattering partials, weighted dn0) is
// this fixed device array instead of plan memory.  Each GPU holds its own
// copy for the life of the process.  In host code `scratch` names a
// host-side stand-in, not device memory: the device address comes from
// hipGetSymbolAddress, once per device, and only that address is used.
constexpr size_t kNoAllocScratchBytes = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_noalloc_mu;
static void* g_noalloc_ptr[64] = {};  // per device

// Device address of this device's `scratch`, resolved on the first call on
// the device (with that device current) and kept.
static int noalloc_scratch(void** out) {
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return bpmh_set_error(BPMH_ERR_UNSUPPORTED, "device index above 63");
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      char b[256];
      snprintf(b, sizeof b, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
               hipGetErrorString(e));
      return bpmh_set_error(BPMH_ERR_HIP, b);
    }
    g_noalloc_ptr[dev] = p;
  }
  *out = g_noalloc_ptr[dev];
  return BPMH_OK;
}

extern "C" int bpmh_propagate_noalloc(bpmh_plan plan, int batch, int nz, float* plane,
                                      const void* dn, int dn_kind, long long dn_batch_stride,
                                      long long dn_numel, int mean_mode, const float* H,
                                      const float* n_eff, const float* dn0, float n0, float k0,
                                      float dx, float dy, float dz, float unit_k, int absorb,
                                      float* out_field, float* out_intens, long long out_numel,
                                      float* out_sum, const float* scat_w, const float* g_w,
                                      const float* plain, float* out_scat, void* stream) {
  PropCall c;
  c.batch = batch;
  c.nz = nz;
  c.plane = (float2*)plane;
  c.dn = dn;
  c.dn_kind = dn_kind;
  c.dn_bstride = dn_batch_stride;
  c.dn_numel = dn_numel;
  c.mean_mode = mean_mode;
  c.H = (const float2*)H;
  c.n_eff = n_eff;
  c.dn0 = dn0;
  c.n0 = n0;
  c.k0 = k0;
  c.dx = dx;
  c.dy = dy;
  c.dz = dz;
  c.unit_k = unit_k;
  c.absorb = absorb;
  c.out_field = (float2*)out_field;
  c.out_intens = out_intens;
  c.out_numel = out_numel;
  c.out_sum = out_sum;
  c.scat_w = scat_w;
  c.g_w = g_w;
  c.plain = (const float2*)plain;
  c.out_scat = out_scat;
  int rc = prop_validate(plan, c);
  if (rc) return rc;
  if (!plan->tw_x[0])
    return bpmh_set_error(BPMH_ERR_INVALID,
                          "plan has no device tables: create it with a device present");
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev != plan->device) return bpmh_set_error(BPMH_ERR_INVALID, "plan belongs to another device");
  StepScratch sc = {nullptr, nullptr, nullptr};
  const size_t sb = prop_scratch_bytes(plan, c);
  if (sb > kNoAllocScratchBytes) {
    char b[256];
    snprintf(b, sizeof b, "this call needs %zu bytes of scratch; the fixed scratch holds %zu "
             "(fewer items or planes with scattering sums)", sb, kNoAllocScratchBytes);
    return bpmh_set_error(BPMH_ERR_INVALID, b);
  }
  if (sb) {
    void* p = nullptr;
    rc = noalloc_scratch(&p);
    if (rc) return rc;
    sc = prop_scratch_carve(plan, c, p);
  }
  return prop_run(plan, c, sc, (hipStream_t)stream, false);
}

// ----------------------------------------------------------------------------
// adjoint (gradient of a loss on the last plane with respect to dn)
// ----------------------------------------------------------------------------
// Per plane p: grad[p][i] += sum_b gitem[p][b][i] in item order (deterministic),
// then, with cg, (sum_b cg[p][b]) * inv_n: dL/ddn0 of a simple-mean step spread
// over the plane that dn0 is the mean of.  n counts floats (one per voxel for
// real dn, two for complex dn).
__global__ void k_grad_reduce(const float* __restrict__ gitem, float* __restrict__ grad, int batch,
                              size_t n, const float* __restrict__ cg, float inv_n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t p = blockIdx.y;
  float s = grad[p * n + i];
  for (int b = 0; b < batch; ++b) s += gitem[(p * batch + b) * n + i];
  if (cg) {
    float c = 0.f;
    for (int b = 0; b < batch; ++b) c += cg[p * batch + b];
    s += c * inv_n;
  }
  grad[p * n + i] = s;
}

static void launch_grad_reduce(const float* gitem, float* grad, int batch, size_t n, int planes,
                               const float* cg, float inv_n, hipStream_t s) {
  hipLaunchKernelGGL(k_grad_reduce, dim3((unsigned)((n + 255) / 256), planes), dim3(256), 0, s, gitem,
                     grad, batch, n, cg, inv_n);
}

static int adjoint_segment(bpmh_plan plan, int batch, int z_lo, int z_hi, float* g_,
                           const float* u_seg_, long long u_seg_numel, const void* dn, int dn_kind,
                           long long dn_numel, const float* H_, float unit_k, int absorb,
                           float* grad_dn, float* gitem, long long work_numel, void* stream) {
  float2* g = (float2*)g_;
  const float2* u_seg = (const float2*)u_seg_;
  const float2* H = (const float2*)H_;
  if (!plan || !g || !u_seg || !dn || !H || !grad_dn || !gitem)
    return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  if (dn_kind != BPMH_DN_F32 && dn_kind != BPMH_DN_C64)
    return bpmh_set_error(BPMH_ERR_UNSUPPORTED, "the adjoint takes float32 or complex64 dn");
  if (batch < 1 || z_lo < 0 || z_hi < z_lo) return bpmh_set_error(BPMH_ERR_INVALID, "bad range");
  if (batch > 65535 || (long long)batch * plan->ny > (1LL << 30))
    return bpmh_set_error(BPMH_ERR_INVALID, "batch too large");
  if (absorb < 0) return bpmh_set_error(BPMH_ERR_INVALID, "absorbing width must be >= 0");
  const int nx = plan->nx, ny = plan->ny;
  const int nseg = z_hi - z_lo + 1;
  const long long n2 = (long long)nx * ny;
  char b[256];
  if (dn_numel < (long long)(z_hi + 1) * n2) {
    snprintf(b, sizeof b, "dn and grad_dn hold %lld elements; planes up to %d need %lld",
             dn_numel, z_hi, (long long)(z_hi + 1) * n2);
    return bpmh_set_error(BPMH_ERR_INVALID, b);
  }
  if (u_seg_numel < (long long)batch * nseg * n2) {
    snprintf(b, sizeof b, "u_seg holds %lld elements; %d item(s) x %d planes need %lld",
             u_seg_numel, batch, nseg, (long long)batch * nseg * n2);
    return bpmh_set_error(BPMH_ERR_INVALID, b);
  }
  if (z_hi == z_lo) return BPMH_OK;
  const int urc = plan_upload(plan);
  if (urc) return urc;
  hipStream_t s = (hipStream_t)stream;
  const Variant var = plan_variant(plan);
  const row_fn row = pick_row(nx, var.row);
  const int cv = col_variant_for(var.col, g);
  const col_fn col0 = pick_col<0>(ny, cv);
  const int comps = dn_kind == BPMH_DN_C64 ? 2 : 1;  // floats of gradient per voxel

  RowArgs ra;
  memset(&ra, 0, sizeof ra);
  ra.plane = g;
  ra.tw = plan->tw_x[var.row_alt()];
  ra.dn = dn;
  ra.dn_kind = dn_kind;
  ra.ny = ny;
  ra.nz = z_hi + 1;
  ra.unit_k = unit_k;
  ra.inv_n = 1.0f / ((float)nx * (float)ny);
  ra.absorb = absorb;
  ra.adjoint = 1;
  ra.useg = u_seg;
  ra.useg_bstride = (long long)nseg * ny * nx;
  ra.gitem = gitem;

  ColArgs ca;
  memset(&ca, 0, sizeof ca);
  ca.plane = g;
  ca.tw = plan->tw_y[cv / kColShapes];
  ca.nx = nx;
  ca.hmode = 0;
  ca.H = H;
  ca.conj_h = 1;

  const size_t n = (size_t)n2 * comps;
  // one launch when every step's per-item gradients fit the workspace
  if (work_numel >= (long long)(nseg - 1) * batch * (long long)n) {
    LoopCall call;
    memset(&call, 0, sizeof call);
    call.ra = ra;
    call.ra.dn = (const char*)dn + (size_t)z_lo * n * sizeof(float);
    call.ra.nz = nseg;
    call.ca = ca;
    const int rc = loop_run(plan, var, BPMH_MEAN_IGNORE, batch, nseg, call, s, true);
    if (rc < 0) return rc;
    if (rc == 1) {
      launch_grad_reduce(gitem, grad_dn + (size_t)(z_lo + 1) * n, batch, n, nseg - 1, nullptr, 0.f, s);
      HIP_TRY(hipGetLastError());
      return BPMH_OK;
    }
  }
  for (int z = z_hi; z > z_lo; --z) {
    ra.z = z;
    ra.useg_z = z - z_lo;
    ra.inverse = z != z_hi;
    ra.screen = 1;
    ra.fwd_items = batch;
    run_row(plan, var, row, ra, batch, s);
    launch_grad_reduce(gitem, grad_dn + (size_t)z * n, batch, n, 1, nullptr, 0.f, s);
    run_col(plan, var, col0, ca, batch, s);
  }
  // back to real space: the gradient with respect to u[z_lo]
  ra.adjoint = 0;
  ra.screen = 0;
  ra.inverse = 1;
  ra.fwd_items = 0;
  run_row(plan, var, row, ra, batch, s);
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}

extern "C" int bpmh_adjoint_segment(bpmh_plan plan, int batch, int z_lo, int z_hi, float* g,
                                    const float* u_seg, long long u_seg_numel, const void* dn,
                                    int dn_kind, long long dn_numel, const float* H, float unit_k,
                                    int absorb, float* grad_dn, float* gitem, void* stream) {
  return adjoint_segment(plan, batch, z_lo, z_hi, g, u_seg, u_seg_numel, dn, dn_kind, dn_numel, H,
                         unit_k, absorb, grad_dn, gitem, 0, stream);
}

extern "C" int bpmh_adjoint_segment_work(bpmh_plan plan, int batch, int z_lo, int z_hi, int dn_kind,
                                         long long* numel) {
  if (!plan || !numel) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  if (batch < 1 || z_lo < 0 || z_hi < z_lo) return bpmh_set_error(BPMH_ERR_INVALID, "bad range");
  const long long n = (long long)plan->nx * plan->ny * (dn_kind == BPMH_DN_C64 ? 2 : 1);
  const Variant var = plan_variant(plan);
  const bool loop = loop_adj_wanted(plan, BPMH_MEAN_IGNORE, batch, z_hi - z_lo + 1,
                                    row_e_of(plan->nx, var.row_alt()), col_e_of(plan->ny, var.col_alt()));
  *numel = n * batch * (loop ? z_hi - z_lo : 1);
  return BPMH_OK;
}

extern "C" int bpmh_adjoint_segment_ws(bpmh_plan plan, int batch, int z_lo, int z_hi, float* g,
                                       const float* u_seg, long long u_seg_numel, const void* dn,
                                       int dn_kind, long long dn_numel, const float* H,
                                       float unit_k, int absorb, float* grad_dn, float* work,
                                       long long work_numel, void* stream) {
  if (plan && batch >= 1 &&
      work_numel < (long long)batch * plan->nx * plan->ny * (dn_kind == BPMH_DN_C64 ? 2 : 1))
    return bpmh_set_error(BPMH_ERR_INVALID, "work holds less than one plane per item");
  return adjoint_segment(plan, batch, z_lo, z_hi, g, u_seg, u_seg_numel, dn, dn_kind, dn_numel, H,
                         unit_k, absorb, grad_dn, work, work_numel, stream);
}

// ----------------------------------------------------------------------------
// mean-corrected (weighted or simple) segment of the differentiable form
// ----------------------------------------------------------------------------
// out[r] = sum of row r (nx floats) of g; one wavefront per row, fixed order
__global__ void __launch_bounds__(256) k_row_sums(const float* __restrict__ g,
                                                  float* __restrict__ out, int rows, int nx) {
  const int r = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;  // whole wavefront
  const float* p = g + (size_t)r * nx;
  float sum = 0.f;
  for (int i = lane; i < nx; i += 64) sum += p[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (lane == 0) out[r] = sum;
}

// Workspace of bpmh_mean_segment, in floats (each part 256-byte aligned).
struct WsegLayout {
  size_t wpart, dn0, fplane, useg, kseg, recc, recw, s1, s2, gitem, gd, cg, total;
};

// whole: with the screen gradients of every step, which the adjoint as one
// launch takes; else of one step.
static WsegLayout wseg_layout(bpmh_plan plan, int batch, int nseg, bool adjoint, bool whole) {
  const int nx = plan->nx, ny = plan->ny;
  WsegLayout L;
  memset(&L, 0, sizeof L);
  size_t o = 0;
  auto take = [&o](size_t n) {
    const size_t r = o;
    o += (n + 63) & ~(size_t)63;
    return r;
  };
  const size_t n2 = (size_t)nx * ny, B = (size_t)batch, S = (size_t)nseg;
  L.wpart = take(2 * B * nx);
  L.dn0 = take(B);
  if (adjoint) {
    L.fplane = take(2 * B * n2);
    L.useg = take(2 * B * S * n2);
    L.kseg = take(2 * B * (S - 1) * n2);
    L.recc = take((S - 1) * B);
    L.recw = take((S - 1) * B);
    L.s1 = take(B * ny);
    L.s2 = take(B * nx);
    L.gitem = take(whole ? B * (S - 1) * n2 : B * n2);
    L.gd = take(B * n2);
    L.cg = take(B * S);
  }
  L.total = o;
  return L;
}

// Whether the adjoint of a mean-corrected segment runs as one launch (of either
// mean) when its workspace allows.
static bool wseg_whole(bpmh_plan plan, Variant var, int batch, int nseg) {
  return loop_adj_wanted(plan, BPMH_MEAN_WEIGHTED, batch, nseg, row_e_of(plan->nx, var.row_alt()),
                         col_e_of(plan->ny, var.col_alt()));
}

extern "C" int bpmh_mean_segment_work(bpmh_plan plan, int batch, int z_lo, int z_hi,
                                      int adjoint, long long* numel) {
  if (!plan || !numel) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  if (batch < 1 || z_lo < 0 || z_hi < z_lo) return bpmh_set_error(BPMH_ERR_INVALID, "bad range");
  const int nseg = z_hi - z_lo + 1;
  *numel = (long long)wseg_layout(plan, batch, nseg, adjoint != 0,
                                  adjoint == 1 && wseg_whole(plan, plan_variant(plan), batch, nseg)).total;
  return BPMH_OK;
}

extern "C" int bpmh_mean_segment(bpmh_plan plan, int mean_mode, int batch, int z_lo, int z_hi,
                                 float* plane_, const float* dn, long long dn_numel,
                                 const float* n_eff, const float* dn0_arr, float n0, float k0,
                                 float dx, float dy, float dz, float unit_k, int absorb, float* g_,
                                 float* grad_dn, float* work, long long work_numel, void* stream) {
  if (!plan || !plane_ || !dn || !work) return bpmh_set_error(BPMH_ERR_INVALID, "null argument");
  if (mean_mode != BPMH_MEAN_SIMPLE && mean_mode != BPMH_MEAN_WEIGHTED)
    return bpmh_set_error(BPMH_ERR_INVALID, "mean_mode must be simple or weighted");
  const bool simple = mean_mode == BPMH_MEAN_SIMPLE;
  if (simple && (!n_eff || !dn0_arr))
    return bpmh_set_error(BPMH_ERR_INVALID, "mean_mode simple needs n_eff and dn0 arrays");
  const bool adjoint = g_ != nullptr;
  if (adjoint && !grad_dn) return bpmh_set_error(BPMH_ERR_INVALID, "the adjoint needs grad_dn");
  if (batch < 1 || z_lo < 0 || z_hi < z_lo) return bpmh_set_error(BPMH_ERR_INVALID, "bad range");
  if (batch > 65535 || (long long)batch * plan->ny > (1LL << 30))
    return bpmh_set_error(BPMH_ERR_INVALID, "batch too large");
  if (absorb < 0) return bpmh_set_error(BPMH_ERR_INVALID, "absorbing width must be >= 0");
  const int nx = plan->nx, ny = plan->ny;
  const int nseg = z_hi - z_lo + 1;
  const long long n2 = (long long)nx * ny;
  char msg[256];
  if (dn_numel < (long long)(z_hi + 1) * n2) {
    snprintf(msg, sizeof msg, "dn holds %lld elements; planes up to %d need %lld", dn_numel, z_hi,
             (long long)(z_hi + 1) * n2);
    return bpmh_set_error(BPMH_ERR_INVALID, msg);
  }
  const Variant var = plan_variant(plan);
  bool whole = adjoint && wseg_whole(plan, var, batch, nseg);
  // (the workspace may have been asked for at another variant or loop mode)
  if (whole && work_numel < (long long)wseg_layout(plan, batch, nseg, adjoint, true).total) whole = false;
  const WsegLayout L = wseg_layout(plan, batch, nseg, adjoint, whole);
  if (work_numel < (long long)L.total) {
    snprintf(msg, sizeof msg, "work holds %lld floats; this segment needs %lld", work_numel,
             (long long)L.total);
    return bpmh_set_error(BPMH_ERR_INVALID, msg);
  }
  if (nseg == 1) return BPMH_OK;
  const int urc = plan_upload(plan);
  if (urc) return urc;
  hipStream_t s = (hipStream_t)stream;
  const row_fn row = pick_row(nx, var.row);
  float2* plane = (float2*)plane_;
  float2* fp = adjoint ? (float2*)(work + L.fplane) : plane;
  const int cv = col_variant_for(var.col, fp);
  const col_fn col0 = simple ? pick_col<5>(ny, cv) : pick_col<0>(ny, cv);
  const col_fn colA = pick_col<1>(ny, cv);
  const col_fn colB = pick_col<2>(ny, cv);
  const size_t B = (size_t)batch, S = (size_t)nseg;
  float2* useg = (float2*)(work + L.useg);
  float2* kseg = (float2*)(work + L.kseg);
  if (adjoint)
    HIP_TRY(hipMemcpyAsync(fp, plane, B * n2 * sizeof(float2), hipMemcpyDeviceToDevice, s));

  // forward z_lo -> z_hi (recorded when the adjoint follows); the weights
  // read slice 0 of the whole volume, the screens dn[z_lo + z]
  RowArgs ra;
  memset(&ra, 0, sizeof ra);
  ra.plane = fp;
  ra.tw = plan->tw_x[var.row_alt()];
  ra.dn = dn + (size_t)z_lo * n2;
  ra.dn_kind = BPMH_DN_F32;
  ra.ny = ny;
  ra.nz = nseg;
  ra.unit_k = unit_k;
  ra.inv_n = 1.0f / ((float)nx * (float)ny);
  ra.absorb = absorb;
  ra.dn0_mode = mean_mode;
  ra.dn0_item = work + L.dn0;
  ra.dn0_arr = simple ? dn0_arr + z_lo : nullptr;  // per plane, indexed by the segment's z
  ra.out_field = adjoint ? useg : nullptr;

  ColArgs ca;
  memset(&ca, 0, sizeof ca);
  ca.plane = fp;
  ca.tw = plan->tw_y[cv / kColShapes];
  ca.nx = nx;
  ca.nz = nseg;
  ca.hmode = mean_mode;
  ca.n_eff = simple ? n_eff + z_lo : nullptr;
  ca.n0 = n0;
  ca.k0 = k0;
  ca.dx = dx;
  ca.dy = dy;
  ca.dz = dz;
  ca.dn = dn;
  ca.dn_kind = BPMH_DN_F32;
  ca.wpart = (float2*)(work + L.wpart);
  ca.dn0_item = work + L.dn0;

  int looped = 0;
  {
    LoopCall call;
    memset(&call, 0, sizeof call);
    call.ra = ra;
    call.ca = ca;
    if (adjoint) {
      call.ca.kout = kseg;
      call.ca.kout_bstride = (long long)(S - 1) * n2;
      call.ca.rec_c = work + L.recc;
      call.ca.rec_w = work + L.recw;
      call.la.kout_zstride = n2;
    }
    looped = loop_run(plan, var, mean_mode, batch, nseg, call, s);
    if (looped < 0) return looped;
  }
  ra.z = 0;
  ra.fwd_items = batch;
  if (!looped) run_row(plan, var, row, ra, batch, s);
  ra.inverse = 1;
  ra.screen = 1;
  for (int z = 1; z < nseg && !looped; ++z) {
    ca.z = z;
    if (adjoint) {
      ca.kout = kseg + (size_t)(z - 1) * n2;
      ca.kout_bstride = (long long)(S - 1) * n2;
      ca.rec_c = work + L.recc + (size_t)(z - 1) * B;
      ca.rec_w = work + L.recw + (size_t)(z - 1) * B;
    }
    if (simple) {
      run_col(plan, var, col0, ca, batch, s);
    } else {
      colA(ca, batch, s);
      colB(ca, batch, s);
    }
    ra.z = z;
    ra.fwd_items = z < nseg - 1 ? batch : 0;
    run_row(plan, var, row, ra, batch, s);
  }
  if (!adjoint) {
    HIP_TRY(hipGetLastError());
    return BPMH_OK;
  }

  // adjoint z_hi -> z_lo
  float2* g = (float2*)g_;
  float* gitem = work + L.gitem;
  float* gd = work + L.gd;
  const size_t nn = (size_t)n2;
  const unsigned fill_blocks = (unsigned)((B * nn + 255) / 256);
  hipLaunchKernelGGL(k_fill_zero, dim3(fill_blocks), dim3(256), 0, s, gd, B * nn);
  const col_fn col3 = pick_col_adj<3>(ny, cv);
  const col_fn col4 = pick_col_adj<4>(ny, cv);
  RowArgs rb = ra;
  rb.plane = g;
  rb.out_field = nullptr;
  rb.adjoint = 1;
  rb.useg = useg;
  rb.useg_bstride = (long long)S * n2;
  rb.gitem = gitem;
  rb.screen = 1;
  rb.fwd_items = batch;
  ColArgs cb;
  memset(&cb, 0, sizeof cb);
  cb.plane = g;
  cb.tw = ca.tw;
  cb.nx = nx;
  cb.nz = nseg;
  cb.hmode = mean_mode;
  cb.simple = simple;
  cb.n_eff = simple ? n_eff + z_lo : nullptr;
  cb.cg_out = work + L.cg;
  cb.conj_h = 1;
  cb.n0 = n0;
  cb.k0 = k0;
  cb.dx = dx;
  cb.dy = dy;
  cb.dz = dz;
  cb.dn = dn;
  cb.dn_kind = BPMH_DN_F32;
  cb.uk_bstride = (long long)(S - 1) * n2;
  cb.s2part = work + L.s2;
  cb.s1part = work + L.s1;
  cb.gd_item = gd;
  if (whole) {
    LoopCall call;
    memset(&call, 0, sizeof call);
    call.ra = rb;
    call.ra.fwd_items = 0;
    call.ca = cb;
    call.ca.uk = kseg;
    call.ca.cz = work + L.recc;
    call.ca.wz = work + L.recw;
    const int rc = loop_run(plan, var, mean_mode, batch, nseg, call, s, true);
    if (rc < 0) return rc;
    if (rc == 1) {
      launch_grad_reduce(gitem, grad_dn + (size_t)(z_lo + 1) * nn, batch, nn, nseg - 1,
                         simple ? work + L.cg : nullptr, 1.f / (float)nn, s);
      if (!simple) launch_grad_reduce(gd, grad_dn, batch, nn, 1, nullptr, 0.f, s);
      HIP_TRY(hipGetLastError());
      return BPMH_OK;
    }
  }
  for (int z = nseg - 1; z >= 1; --z) {
    rb.z = z;
    rb.useg_z = z;
    rb.inverse = z != nseg - 1;
    if (!simple) rb.dn0_item = work + L.recc + (size_t)(z - 1) * B;
    run_row(plan, var, row, rb, batch, s);
    hipLaunchKernelGGL(k_row_sums, dim3((unsigned)((B * ny + 3) / 4)), dim3(256), 0, s, gitem,
                       work + L.s1, (int)(B * ny), nx);
    cb.z = z;
    cb.uk = kseg + (size_t)(z - 1) * n2;
    cb.cz = work + L.recc + (size_t)(z - 1) * B;
    cb.wz = work + L.recw + (size_t)(z - 1) * B;
    col3(cb, batch, s);
    col4(cb, batch, s);
    // (simple: dn0 of this step is the mean of plane z, dL/ddn0 / N on every voxel)
    launch_grad_reduce(gitem, grad_dn + (size_t)(z_lo + z) * nn, batch, nn, 1,
                       simple ? work + L.cg : nullptr, 1.f / (float)nn, s);
  }
  rb.adjoint = 0;
  rb.screen = 0;
  rb.inverse = 1;
  rb.fwd_items = 0;
  run_row(plan, var, row, rb, batch, s);
  // the weight slice is slice 0 of the volume
  if (!simple)
    launch_grad_reduce(gd, grad_dn, batch, nn, 1, nullptr, 0.f, s);
  HIP_TRY(hipGetLastError());
  return BPMH_OK;
}
