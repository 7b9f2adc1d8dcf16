// Line configurations, argument records and the per-line work of the split-step
// passes, shared by the two-launch step (bpm_kernels.hip) and the
// one-launch z-loop (loop.hpp): both run the same operations in the same
// order on every line, so their results agree bit for bit.
#pragma once
#include "common.hpp"
#include "fft.hpp"
#include "bpm_hip.h"

#include <type_traits>

using namespace bpmfft;

// ----------------------------------------------------------------------------
// per-size launch configurations: variant V in {0,1,2} scales the default
// number of lines (rows) or columns per work-group by 1/2, 1, 2, clamped to
// 1..16 lines, 1024 threads and 128 KiB of LDS (gfx950 has 160 KiB per CU);
// the autotuner picks V per size.
// ----------------------------------------------------------------------------
constexpr int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
constexpr int pow2floor(int v) { return v < 2 ? 1 : 2 * pow2floor(v / 2); }
constexpr int scale_v(int base, int V) { return V == 0 ? base / 2 : (V == 1 ? base : base * 2); }

// Elements per thread of a line.  Rows: 4 up to N = 1024 (twice the
// wavefronts of E = 8 for the same data, so loads, transforms and stores of
// different wavefronts overlap better; measured 5-13 % faster per z-step at
// 64^2..1024^2, batch 1), 8 above.  Columns: 8 (4-column tiles of 8-element
// threads; E = 4 measured slower at 1024^2, also with 4-column tiles of
// 1024 threads, and at 256^2..512^2 in batches).
constexpr int row_e(int n) { return n <= 1024 ? 4 : 8; }
constexpr int col_e(int n) { return n <= 32 ? 4 : 8; }
// The other radix schedule of a size, which the autotuner times against the
// default: 8 elements per thread instead of 4 (when the line still holds two
// radix-8 stages, N >= 64), or 4 instead of 8.  ealt selects it.
constexpr int alt_e(int e, int n) { return e == 4 ? (n >= 64 ? 8 : 4) : 4; }
constexpr int row_e_of(int n, int ealt) { return ealt ? alt_e(row_e(n), n) : row_e(n); }
constexpr int col_e_of(int n, int ealt) { return ealt ? alt_e(col_e(n), n) : col_e(n); }
// Variant numbers: row variant = V + 3*ealt (V = 0, 1, 2), column variant =
// V + 5*ealt (V = 0..4).
constexpr int kRowShapes = 3, kColShapes = 5;
#define BPMH_MAX_GROUPS 16


template <int N, int E_>
struct Base {
  static constexpr int E = E_;
  static constexpr int T = N / E;
  // LDS (layouts of fft.hpp): a row line is N float2 in the swizzled
  // exchange layout (8 more when lines of fewer than 16 threads share a
  // 16-lane group, so those lines start in different banks).  Column tiles
  // of 4 or more columns use the swizzled layout for C = COLS lines per
  // 16-lane group, lines N + 16/COLS apart; narrower tiles keep lines padded
  // one per 32 and 9 float2 longer (the swizzle measured slower there).
  // COL_LINE, the padded length, bounds both.
  static constexpr int ROW_LINE = N + (T < 16 ? 8 : 0);
  static constexpr int COL_SH = 5;
  static constexpr int COL_LINE = N + (N >> COL_SH) + 9;  // float2 per column line
  static constexpr int LDS_LINE = COL_LINE * 8;        // bytes per column line
};

template <int N, int V, int E_ = row_e(N)>
struct RowCfg : Base<N, E_> {
  using Base<N, E_>::T;
  static constexpr int L0 = clampi(256 / T, 1, 16);
  // at least one full wavefront per work-group (the cross-lane reductions
  // use all 64 lanes), at most 16 lines and 1024 threads
  static constexpr int LMIN = 64 / T < 1 ? 1 : 64 / T;
  static constexpr int LINES =
      clampi(clampi(scale_v(L0, V), LMIN, 16), 1, (1024 / T) < 1 ? 1 : 1024 / T);
  static constexpr int THREADS = LINES * T;
};

template <int N, int V, int E_ = col_e(N)>
struct ColCfg : Base<N, E_> {
  using Base<N, E_>::T;
  using Base<N, E_>::LDS_LINE;
  static constexpr int C0 = N >= 4096 ? 1 : clampi(512 / T, 2, 16);
  static constexpr int CMAX0 = 131072 / LDS_LINE < 1 ? 1 : 131072 / LDS_LINE;
  // <= 512 threads with 8 elements per thread (1024 spilled), <= 1024 with 4
  static constexpr int TMAX = (E_ <= 4 ? 1024 : 512) / T < 1 ? 1 : (E_ <= 4 ? 1024 : 512) / T;
  static constexpr int CMAX = pow2floor(clampi(CMAX0 < TMAX ? CMAX0 : TMAX, 1, 16));
  static constexpr int CMIN = 64 / T < 1 ? 1 : 64 / T;  // >= one full wavefront
  // V = 3: the work-group of V = 0 with P = 2 adjacent columns per thread
  // (tiles twice as wide), so a row of a column pair is one 16-byte load and
  // store.  V = 4: the same with each column's loads and stores issued
  // separately (8-byte accesses), the first column's loads first, so its
  // transform can start while the second column's loads are in flight.
  // Used for columns of 256-1024 points (where they were measured);
  // elsewhere they are V = 0.
  static constexpr bool PAIRED = (V == 3 || V == 4) && N >= 256 && N <= 1024;
  static constexpr int P = PAIRED ? 2 : 1;
  static constexpr bool SPLIT = PAIRED && V == 4;
  static constexpr int LC = clampi(scale_v(C0, V >= 3 ? 0 : V), CMIN, CMAX);  // lane columns
  static constexpr int COLS = LC * P;
  static constexpr int THREADS = LC * T;
};

// ----------------------------------------------------------------------------
// device helpers
// ----------------------------------------------------------------------------
BPMH_DEV float2 load_dn(const void* dn, int kind, size_t idx) {
  if (kind == BPMH_DN_F32) return make_float2(((const float*)dn)[idx], 0.f);
  if (kind == BPMH_DN_F16) return make_float2(__half2float(((const __half*)dn)[idx]), 0.f);
  return ((const float2*)dn)[idx];
}

// FFTFREQ(i,N,d) of bpm_3d_kernels.cl:6 in float32
BPMH_DEV float fftfreq_f32(int i, int N, float d) {
  const int half = (N - 1) / 2 + 1;
  const float num = (i < half) ? (float)i : (float)((i - half) - N / 2);
  return f_div(f_div(num, (float)N), d);
}

BPMH_DEV float kcomp2_f32(int i, int N, float d) {
  const float k = f_mul(2.f * BPMH_PI_F, fftfreq_f32(i, N, d));
  return f_mul(k, k);
}

// H for one (kx^2, ky^2) with a = ((n*n)*k0)*k0, as compute_propagator
// (bpm_3d_kernels.cl:419-430): (tmp>=0) * exp(-i dz sqrt(tmp)).
BPMH_DEV float2 prop_f32(float kx2, float ky2, float a, float dz) {
  const float tmp = f_sub(f_sub(a, kx2), ky2);
  const float h0 = tmp < 0.f ? 0.f : __fsqrt_rn(tmp);
  const float2 cs = sincos_f32_via_f64(f_mul(-dz, h0));
  return tmp >= 0.f ? cs : make_float2(0.f, 0.f);
}

BPMH_DEV float n_term_f32(float n, float k0) { return f_mul(f_mul(f_mul(n, n), k0), k0); }

// prop_f32 (the same operations, so the same H) that also returns
// beta = sqrt(a - kx^2 - ky^2), 0 where the component does not propagate
// (H = 0 there, and its derivative with respect to dn0 is taken as 0).
BPMH_DEV float2 prop_f32_beta(float kx2, float ky2, float a, float dz, float* beta) {
  const float tmp = f_sub(f_sub(a, kx2), ky2);
  const float h0 = tmp < 0.f ? 0.f : __fsqrt_rn(tmp);
  const float2 cs = sincos_f32_via_f64(f_mul(-dz, h0));
  *beta = tmp > 0.f ? h0 : 0.f;
  return tmp >= 0.f ? cs : make_float2(0.f, 0.f);
}

// Weighted mean (bpm_3d.py:149-159,302-303): dn0 = dn_sum/u_sum over the nx
// per-column partials of item b (x = dn part, y = u part) that column pass A
// wrote.  Column pass B forms it once per work-group: lane p of the first
// wavefront sums partials p, p+64, ... and an xor butterfly completes the
// sum (a fixed order, so every work-group gets the same bits); the result is
// broadcast through LDS, and the work-group of tile 0 stores it for the row
// pass.  The kernel boundary after pass A orders the partials' stores before
// these loads.
// The first 1024 partials are loaded before the work-group's plane (loads
// complete in order: behind the plane's, the sum waited for all of it, and its
// loop for one partial after another), those past the end as zeros: weighted
// steps of 1024^2 34.9 -> 31.0 us (batch 1), 243 -> 207 (16), of 2048^2 123 ->
// 114.  (Pass A's weight slice loaded before its transform likewise: 193 at
// batch 16, but 2048^2 121 and 512^2 18.6 -> 19.3, so it is read after it.)
struct WeightParts {
  float2 w[16];
};
BPMH_DEV void weighted_parts_load(const float2* wp, int nparts, WeightParts& r) {
  if (threadIdx.x >= 64) return;
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float2*>(wp), (short)0, nparts * 8, 0x00020000);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)threadIdx.x * 8, k * 512, 0);
    r.w[k] = make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
  }
}
// slot[0] receives dn0, slot[1] the weight sum sum|U| (the adjoint needs it).
BPMH_DEV float weighted_dn0_group(const float2* __restrict__ wp, int nparts, const WeightParts& r,
                                  float* slot) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    float sd = 0.f, su = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      sd += r.w[k].x;
      su += r.w[k].y;
    }
    for (int p = 1024 + lane; p < nparts; p += 64) {
      const float2 v = wp[p];
      sd += v.x;
      su += v.y;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      sd += __shfl_xor(sd, o, 64);
      su += __shfl_xor(su, o, 64);
    }
    if (lane == 0) {
      slot[0] = sd / su;
      slot[1] = su;
    }
  }
  __syncthreads();
  return slot[0];
}

// Sum of n1 floats at p1 and of n2 floats at p2 by the first wavefront in a
// fixed order (lane l takes elements l, l+64, ..., then an xor butterfly),
// so every work-group of an item gets the same bits; returned to all
// threads through slot[0..1].
BPMH_DEV float2 group_sum_pair(const float* __restrict__ p1, int n1, const float* __restrict__ p2,
                               int n2, float* slot) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    float s1 = 0.f, s2 = 0.f;
    for (int i = lane; i < n1; i += 64) s1 += p1[i];
    for (int i = lane; i < n2; i += 64) s2 += p2[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      s1 += __shfl_xor(s1, o, 64);
      s2 += __shfl_xor(s2, o, 64);
    }
    if (lane == 0) {
      slot[0] = s1;
      slot[1] = s2;
    }
  }
  __syncthreads();
  return make_float2(slot[0], slot[1]);
}

// Sum over the T threads of each column of a tile, in a fixed binary-tree
// order that depends only on T (not on how many columns share the
// work-group), so per-column partial sums are identical for every launch
// shape.  Uses the tile's LDS lines as scratch; returns the sum in t == 0.
template <int T>
BPMH_DEV float2 column_sum2(float2 v, float2* __restrict__ col_lds, int t) {
  __syncthreads();  // the FFT's last reads of col_lds are done
  col_lds[t] = v;
  __syncthreads();
#pragma unroll
  for (int s = T / 2; s > 0; s >>= 1) {
    if (t < s) col_lds[t] = c_add(col_lds[t], col_lds[t + s]);
    __syncthreads();
  }
  return col_lds[0];
}

// ----------------------------------------------------------------------------
// row pass
// ----------------------------------------------------------------------------
struct RowArgs {
  float2* plane;           // (rows = batch*ny, nx)
  const float2* tw;        // stage-major twiddles of the nx-point transform
  const void* dn;          // (nz, ny, nx) per batch item, kind dn_kind
  long long dn_bstride;    // elements between batch items' (or groups') dn (0: shared)
  // ragged batch: items [gend[g-1], gend[g]) read dn volume g; ngroups = 0:
  // item b reads volume b
  int ngroups;
  int gend[BPMH_MAX_GROUPS];
  int dn_kind;
  int ny, nz, z;
  float unit_k;            // float32(k0*dz)
  float inv_n;             // 1/(nx*ny)
  int absorb;
  int dn0_mode;            // BPMH_MEAN_*: 0 none, 1 per-plane array, 2 weighted
  const float* dn0_arr;    // simple mode: float32 dn0 per plane
  const float* dn0_item;   // weighted: dn0 of this step per item (column pass A)
  float2* out_field;       // (batch, nz, ny, nx) or null
  float* out_intens;       // (batch, nz, ny, nx) or null
  float* acc;              // (batch, ny, nx) or null: sum_z |u_z|^2
  int acc_init;
  int inverse;             // input is F_x u: inverse FFT first
  int screen;              // apply dn[z] screen
  int fwd_items;           // items b < fwd_items get the forward FFT_x before storing
  // adjoint step: v is the gradient G_z (torch convention, 2 dL/du*); the
  // row pass writes unit_k*Im(conj(G_z) u_z) per item and multiplies by the
  // conjugate screen
  int adjoint;
  const float2* useg;      // forward planes of the segment (batch, nseg, ny, nx)
  long long useg_bstride;  // elements between items in useg
  int useg_z;              // plane of z inside the segment
  float* gitem;            // (batch, ny, nx) per-item gradient of dn[z] (2 floats per voxel for complex dn)
};

// dn volume of item b: b itself, or in a ragged batch the group holding b
// (a few scalar compares; b is uniform over a work-group).
BPMH_DEV int dn_volume(const RowArgs& a, int b) {
  if (a.ngroups == 0) return b;
  int g = 0;
  while (g + 1 < a.ngroups && b >= a.gend[g]) ++g;
  return g;
}

// a*b with its two roundings fixed (the compiler may fuse either product of
// c_mul), for the multiplies that the launches per pass and the one-launch
// z-loop both compile.
BPMH_DEV float2 c_mul_fused(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -f_mul(a.y, b.y)), fmaf(a.x, b.y, f_mul(a.y, b.x)));
}

// a*conj(b) likewise.
BPMH_DEV float2 c_mulc_fused(float2 a, float2 b) { return c_mul_fused(a, make_float2(b.x, -b.y)); }

// conj(g) u: its imaginary and real part are the screen gradients in Re dn
// and Im dn (times k0 dz).
BPMH_DEV float2 adjoint_pair(float2 g, float2 u) {
  return make_float2(fmaf(g.x, u.x, f_mul(g.y, u.y)), fmaf(g.x, u.y, -f_mul(g.y, u.x)));
}

// Taper 1/2 (1 - cos(pi dist / width)) of a voxel `dist` from the border.
BPMH_DEV float taper_factor(int dist, int width) {
  const float arg = f_div(f_mul(BPMH_PI_F, (float)dist), (float)width);
  return f_mul(0.5f, f_sub(1.f, (float)cos((double)arg)));
}

// The phase screen exp(-i k0 dz (d - dn0)) and the taper on the elements v of
// row y of item b, d the row's refractive-index values.  ADJ: compiled with
// the adjoint step (a.adjoint), which also takes the forward field ua.
template <int NX, int E, bool ADJ>
BPMH_DEV void row_screen(const RowArgs& a, int b, int y, int t, float dn0, const float2 (&d)[E],
                         const float2 (&ua)[E], float2 (&v)[E]) {
  constexpr int T = NX / E;
  const int disty = min(a.ny - y - 1, y);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int x = t + m * T;
    if (a.dn_kind == BPMH_DN_C64) {
      // cexp((0,-k)*(dn - dn0)) = e^{k Im} (cos(-k Re), sin(-k Re)), no taper
      const float re = f_mul(a.unit_k, d[m].y);
      const float im = f_mul(-a.unit_k, f_sub(d[m].x, dn0));
      float s, c;
      sincos_fast(im, &s, &c);
      const float mag = expf(re);
      if (ADJ && a.adjoint) {
        // u = s v with s = e^{k Im dn} e^{-i k Re dn}: dL/dRe dn = k Im(conj(G) u),
        // dL/dIm dn = k Re(conj(G) u), and G_v = conj(s) G
        const float2 w = adjoint_pair(v[m], ua[m]);
        reinterpret_cast<float2*>(a.gitem)[((size_t)b * a.ny + y) * NX + x] =
            make_float2(a.unit_k * w.y, a.unit_k * w.x);
        v[m] = c_mulc_fused(v[m], make_float2(mag * c, mag * s));
      } else {
        v[m] = c_mul_fused(v[m], make_float2(mag * c, mag * s));
      }
    } else {
      const float ph = f_mul(-a.unit_k, f_sub(d[m].x, dn0));
      float s, c;
      sincos_fast(ph, &s, &c);
      float2 r;
      if (ADJ && a.adjoint) {
        a.gitem[((size_t)b * a.ny + y) * NX + x] = a.unit_k * adjoint_pair(v[m], ua[m]).y;
        r = c_mulc_fused(v[m], make_float2(c, s));
      } else {
        r = c_mul_fused(v[m], make_float2(c, s));
      }
      if (a.absorb > 0) {  // uniform: no taper work at all without one
        const int dist = min(min(NX - x - 1, x), disty);
        if (dist < a.absorb) {
          const float tp = taper_factor(dist, a.absorb);
          r = make_float2(r.x * tp, r.y * tp);
        }
      }
      v[m] = r;
    }
  }
}

// Output slices of plane z: field and/or intensity.
template <int NX, int E>
BPMH_DEV void row_outputs(const RowArgs& a, int z, int b, size_t plane_off, int t,
                          const float2 (&v)[E]) {
  constexpr int T = NX / E;
  if (a.out_field) {
    float2* o = a.out_field + ((size_t)b * a.nz + z) * a.ny * NX + plane_off;
#pragma unroll
    for (int m = 0; m < E; ++m) st_stream(o + t + m * T, v[m]);
  }
  if (a.out_intens) {
    float* o = a.out_intens + ((size_t)b * a.nz + z) * a.ny * NX + plane_off;
#pragma unroll
    for (int m = 0; m < E; ++m) st_stream(o + t + m * T, v[m].x * v[m].x + v[m].y * v[m].y);
  }
}

// ----------------------------------------------------------------------------
// column pass
// ----------------------------------------------------------------------------
struct ColArgs {
  float2* plane;           // (batch, ny, nx)
  const float2* tw;        // stage-major twiddles of the ny-point transform
  int nx, nz, z;
  int hmode;               // 0: table H, 1: formula with n_eff[z], 2: formula with n0+weighted dn0
  const float2* H;         // (ny, nx)
  const float* n_eff;      // per plane, float32
  float n0, k0, dx, dy, dz;
  const void* dn;          // weighted: slice 0 of each item's dn is the weight
  long long dn_bstride;
  int dn_kind;
  float2* wpart;           // weighted per-column partials (batch, nx)
  float* dn0_item;         // weighted: dn0 per item, stored by pass B for the row pass
  const float* sw;         // scattering weights (ny, nx) or null
  const float* gw;
  const float2* pw;        // plane-wave DC per plane (nz)
  float2* spart;           // scattering per-column partials (batch, nz, nx)
  int conj_h;              // adjoint: multiply by conj(H)
  // forward recorded for the adjoint (null: nothing recorded): PHASE 1, and
  // PHASE 0 before H, also store U = F u of this step (item stride
  // kout_bstride); PHASE 2 stores this step's dn0 and sum|U| per item
  float2* kout;
  long long kout_bstride;
  float* rec_c;
  float* rec_w;
  // weighted adjoint (PHASE 3, 4) of the step whose forward k-space plane is
  // U (uk, item stride uk_bstride) with dn0 c = cz[b] and sum|U| = wz[b]
  const float2* uk;
  long long uk_bstride;
  const float* cz;
  const float* wz;
  float* s2part;           // (batch, nx): per column sum Im(conj(X) H U) / beta
  const float* s1part;     // (batch, ny): per row sum of the screen gradient
  float* gd_item;          // (batch, ny, nx): += dL/d(weight slice) per item
  // simple mean (PHASE 3, 4): dn0 = mean(dn[z]) does not depend on the
  // field: n = n_eff[z], no |U| term, and PHASE 4 stores dL/ddn0 per item
  int simple;
  float* cg_out;
};

// Weighted mean, one column x of item b: sum over ky of |U| d and |U| (valid
// in every thread), d the weight slice at the thread's rows.
template <int NY, int E>
BPMH_DEV float2 col_weight_sums(const float2 (&v)[E], const float (&d)[E], int t, float2* line) {
  float2 acc = make_float2(0.f, 0.f);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const float au = hypotf(v[m].x, v[m].y);
    acc.x += au * d[m];
    acc.y += au;
  }
  return column_sum2<NY / E>(acc, line, t);
}

// H of the step's index for every row of a column (an = ((n*n)*k0)*k0).
// H(ky) == H(NY - ky) bit for bit (kcomp2_f32 of both rows is the same
// float), and the rows of thread t mirror those of thread T - t (element m
// <-> E-1-m; thread 0 mirrors its own, m <-> E-m, and holds row NY/2 alone),
// so each thread evaluates its first E/2 rows (thread 0 also row NY/2) and
// takes the others from its partner through the column's LDS line (free
// before the inverse transform).
template <int NY, int E>
BPMH_DEV void col_h_fly(float kx2, float an, float dy, float dz, int t, float2* line,
                        float2 (&h)[E]) {
  constexpr int T = NY / E;
#pragma unroll
  for (int m = 0; m < E / 2; ++m) h[m] = prop_f32(kx2, kcomp2_f32(t + m * T, NY, dy), an, dz);
  if (t == 0) h[E / 2] = prop_f32(kx2, kcomp2_f32(NY / 2, NY, dy), an, dz);
  __syncthreads();  // earlier users of the line are done with it
#pragma unroll
  for (int m = 0; m < E / 2; ++m) line[m * T + t] = h[m];
  __syncthreads();
  const int pt = T - t;
#pragma unroll
  for (int m = E / 2; m < E; ++m) {
    if (t == 0) {
      if (m > E / 2) h[m] = h[E - m];
    } else {
      h[m] = line[(E - 1 - m) * T + pt];
    }
  }
  __syncthreads();  // before the line is written again
}

// Scattering reductions of bpm_3d.py:243-247,335-341 on the k-space plane
// after H: per-column sums of w |U - delta_{k,0} plain|^2.
template <int NY, int E>
BPMH_DEV void col_scatter(const ColArgs& a, int z, int b, int x, int t, float2* line,
                          const float2 (&v)[E]) {
  constexpr int T = NY / E;
  float2 acc = make_float2(0.f, 0.f);
  const float2 pl = a.pw[z];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int ky = t + m * T;
    float2 f = v[m];
    if (ky == 0 && x == 0) f = c_sub(f, pl);
    const float af = hypotf(f.x, f.y);
    const float a2 = af * af;
    const size_t k = (size_t)ky * a.nx + x;
    acc.x += a.sw[k] * a2;
    acc.y += a.gw[k] * a2;
  }
  acc = column_sum2<T>(acc, line, t);
  if (t == 0) a.spart[((size_t)b * a.nz + z) * a.nx + x] = acc;
  __syncthreads();  // the line is the inverse transform's exchange buffer
}

// Mean-corrected adjoint, one column: H and beta = the axial wavenumber (0
// where nothing propagates) of every row, as col_h_fly; and the column's sum
// of Im(conj(X) H U) / beta (valid in every thread).
template <int NY, int E>
BPMH_DEV void col_hb_fly(float kx2, float an, float dy, float dz, int t, float2* line, float2 (&h)[E],
                         float (&bt)[E]) {
  constexpr int T = NY / E;
#pragma unroll
  for (int m = 0; m < E / 2; ++m)
    h[m] = prop_f32_beta(kx2, kcomp2_f32(t + m * T, NY, dy), an, dz, &bt[m]);
  if (t == 0) h[E / 2] = prop_f32_beta(kx2, kcomp2_f32(NY / 2, NY, dy), an, dz, &bt[E / 2]);
  __syncthreads();  // earlier users of the line are done with it
#pragma unroll
  for (int m = 0; m < E / 2; ++m) {
    line[m * T + t] = h[m];
    line[NY / 2 + m * T + t] = make_float2(bt[m], 0.f);
  }
  __syncthreads();
#pragma unroll
  for (int m = E / 2; m < E; ++m) {
    if (t == 0) {
      if (m > E / 2) {
        h[m] = h[E - m];
        bt[m] = bt[E - m];
      }
    } else {
      h[m] = line[(E - 1 - m) * T + T - t];
      bt[m] = line[NY / 2 + (E - 1 - m) * T + T - t].x;
    }
  }
}

template <int NY, int E>
BPMH_DEV float col_beta_sum(const float2 (&v)[E], const float2 (&h)[E], const float2 (&uv)[E],
                            const float (&bt)[E], int t, float2* line) {
  float acc = 0.f;  // (column_sum2 waits for every reader of the line)
#pragma unroll
  for (int m = 0; m < E; ++m) {
    if (bt[m] > 0.f) {
      const float2 hu = c_mul_fused(h[m], uv[m]);
      acc += fmaf(v[m].x, hu.y, -f_mul(v[m].y, hu.x)) / bt[m];
    }
  }
  return column_sum2<NY / E>(make_float2(acc, 0.f), line, t).x;
}

// dL/ddn0 = -sum_x (screen gradient) + dz (n0+dn0) k0^2 / N sum_k Im(conj(X) H U)/beta
BPMH_DEV float adjoint_cgrad(float s1, float s2, float dz, float n, float k0, float n_pts) {
  const float c = f_div(f_mul(f_mul(f_mul(dz, n), k0), k0), n_pts);
  return fmaf(c, s2, -s1);
}

// dn0 = sum|U| d / sum|U| depends on U through |U|: the k-space gradient v
// gains dL/ddn0 (d - dn0) / W * U/|U| (times N: X is N G_V); returns
// dL/dd = dL/ddn0 |U| / W.
BPMH_DEV float adjoint_weight_term(float2& v, float2 u, float d, float dn0, float cgrad, float inv_w,
                                   float n_pts) {
  const float au = hypotf(u.x, u.y);
  if (au > 0.f) {
    const float coef = f_div(f_mul(f_mul(f_mul(n_pts, cgrad), f_sub(d, dn0)), inv_w), au);
    v.x = fmaf(coef, u.x, v.x);
    v.y = fmaf(coef, u.y, v.y);
  }
  return f_mul(f_mul(cgrad, au), inv_w);
}
