// The row and column pass of large calls: a work-group does the same line (or
// column tile) of several items in turn, the next item's loads in flight while
// it transforms this one's.
//
// What bounds the one-item passes at 1024^2, batch 16 (107 us a column pass, 91
// a row pass; a copy of the plane's bytes takes 37): the column pass makes 15.6 M
// L2 requests of which two thirds are propagator and twiddles, both passes
// alternate between waiting for memory and transforming, and half the row
// pass's vector instructions of a field are the same for every field (screen
// phases) or addresses.  Here the propagator, twiddles and screen factors stay
// in registers over the items, planes are addressed as buffers, and accesses
// are plain: streaming hints, which paid when a line was touched once per
// launch, cost 10 (rows, columns reading after streaming stores) to 20 us
// (columns) of 122.  1024^2, batch 16: 62 us a column pass, 58 a row pass,
// 139 us a step with the running sum against 191; 2048^2, batch 4: 164 against
// 274 (4.8 TB/s of its reads and writes, what a copy beyond the Infinity Cache
// reaches).  4-column tiles of 8-point threads without spills (114 registers)
// and two work-groups a CU are best at 1024 (two columns a thread 67 to 72 us,
// 8-column tiles 67, 4-point threads 91), 8-column tiles at 512 (16 against 18
// us, batch 16); rows of 4 points a thread to 1024 (8 points: 58 to 64), 8 at
// 2048 (62 against 89, batch 4).
#pragma once
#include "passes.hpp"

typedef unsigned items_u2 __attribute__((ext_vector_type(2)));

// A plane as a buffer: one per-thread byte offset for all its accesses, the
// element's part in a scalar register (64-bit addresses for each element took
// 16 to 32 more vector registers).
BPMH_DEV __amdgpu_buffer_rsrc_t items_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}
BPMH_DEV float2 items_ld(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  const items_u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0);
  return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}
BPMH_DEV void items_st(__amdgpu_buffer_rsrc_t r, int off, int soff, float2 v) {
  const items_u2 w = {__float_as_uint(v.x), __float_as_uint(v.y)};
  __builtin_amdgcn_raw_buffer_store_b64(w, r, off, soff, 0);
}
BPMH_DEV float items_ld1(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
}
BPMH_DEV void items_st1(__amdgpu_buffer_rsrc_t r, int off, int soff, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, soff, 0);
}

// Items b0 = blockIdx.y * per to b0 + per - 1 (below batch) of row
// blockIdx.x * LINES + line.  Items that share a work-group share the dn
// volume and dn0 (per = 1 otherwise).  ADJ: the adjoint step (no running sum).
template <int NX, int E, int LINES, int W, bool ADJ>
__global__ void __launch_bounds__((NX / E * LINES), W)
k_row_items(RowArgs a, int batch, int per) {
  constexpr int T = NX / E;
  constexpr bool WAVE = T <= 64;
  __shared__ float2 lds[LINES][Base<NX, E>::ROW_LINE];
  __shared__ float taper[LINES][NX];  // each thread's own elements
  const int line = threadIdx.x / T, t = threadIdx.x - line * T;
  const int y = blockIdx.x * LINES + line;
  const int b0 = blockIdx.y * per, b1 = min(batch, b0 + per);
  const size_t n2 = (size_t)a.ny * NX;
  const int bytes = (int)n2 * 8;
  const int o8 = (y * NX + t) * 8, o4 = o8 / 2;

  float2 next[E], unext[E];
  float anext[E];
  auto load = [&](int b) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rp = items_rsrc(a.plane + b * n2, bytes);
#pragma unroll
    for (int m = 0; m < E; ++m) next[m] = items_ld(rp, o8, m * T * 8);
    if constexpr (ADJ) {
      const __amdgpu_buffer_rsrc_t ru =
          items_rsrc(a.useg + (size_t)b * a.useg_bstride + (size_t)a.useg_z * n2, bytes);
#pragma unroll
      for (int m = 0; m < E; ++m) unext[m] = items_ld(ru, o8, m * T * 8);
    } else if (a.acc && !a.acc_init) {
      const __amdgpu_buffer_rsrc_t rc = items_rsrc(a.acc + b * n2, bytes / 2);
#pragma unroll
      for (int m = 0; m < E; ++m) anext[m] = items_ld1(rc, o4, m * T * 4);
    }
  };
  load(b0);
  Twiddles<NX, E> tw;
  tw.load(t, a.tw);

  // the screen with 1/n of the inverse transform (a power of two, so folding
  // it in is exact), and the taper
  float2 sc[E];
  const float scale = a.inverse ? a.inv_n : 1.f;
  const bool cplx = a.dn_kind == BPMH_DN_C64;
  const bool tapered = a.absorb > 0 && !cplx && a.screen;
  if (a.screen) {
    const size_t at = ((size_t)a.z * a.ny + y) * NX + (size_t)dn_volume(a, b0) * a.dn_bstride + t;
    if (a.dn_kind == BPMH_DN_F32) {
#pragma unroll
      for (int m = 0; m < E; ++m) sc[m] = make_float2(((const float*)a.dn)[at + m * T], 0.f);
    } else if (cplx) {
#pragma unroll
      for (int m = 0; m < E; ++m) sc[m] = ((const float2*)a.dn)[at + m * T];
    } else {
#pragma unroll
      for (int m = 0; m < E; ++m) sc[m] = make_float2(__half2float(((const __half*)a.dn)[at + m * T]), 0.f);
    }
    float dn0 = 0.f;
    if (a.dn0_mode == BPMH_MEAN_SIMPLE) dn0 = a.dn0_arr[a.z];
    else if (a.dn0_mode == BPMH_MEAN_WEIGHTED) dn0 = a.dn0_item[b0];
    float mag[E];
#pragma unroll
    for (int m = 0; m < E; ++m) mag[m] = scale;
    if (cplx) {
#pragma unroll
      for (int m = 0; m < E; ++m) mag[m] = expf(f_mul(a.unit_k, sc[m].y)) * scale;
    }
#pragma unroll
    for (int m = 0; m < E; ++m) {
      float sn, cs;
      sincos_fast(f_mul(-a.unit_k, f_sub(sc[m].x, dn0)), &sn, &cs);
      sc[m] = make_float2(mag[m] * cs, mag[m] * sn);
    }
    if (tapered) {
      const int disty = min(a.ny - y - 1, y);
#pragma unroll 1
      for (int m = 0; m < E; ++m) {
        const int x = t + m * T, dist = min(min(NX - x - 1, x), disty);
        taper[line][x] = dist < a.absorb ? taper_factor(dist, a.absorb) : 1.f;
      }
    }
  }

#pragma unroll 1
  for (int b = b0; b < b1; ++b) {
    float2 v[E], ua[E];
    float av[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      v[m] = next[m];
      if constexpr (ADJ) ua[m] = unext[m];
      else av[m] = anext[m];
    }
    if (b + 1 < b1) load(b + 1);
    if (a.inverse) line_fft<NX, E, true, SwzLayout<4>, WAVE>(v, lds[line], t, tw);
    if constexpr (ADJ) {
      // screen gradient (unit_k times 1/n: exact, as above), conjugate screen
      const float uk = a.unit_k * scale;
      const __amdgpu_buffer_rsrc_t rg =
          items_rsrc(a.gitem + b * n2 * (cplx ? 2 : 1), cplx ? bytes : bytes / 2);
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const float2 w = adjoint_pair(v[m], ua[m]);
        if (cplx) items_st(rg, o8, m * T * 8, make_float2(uk * w.y, uk * w.x));
        else items_st1(rg, o4, m * T * 4, uk * w.y);
        v[m] = c_mulc_fused(v[m], sc[m]);
      }
    } else if (a.screen) {
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = c_mul_fused(v[m], sc[m]);
    } else if (a.inverse) {
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = c_scale(v[m], scale);
    }
    if (tapered) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const float tp = taper[line][t + m * T];
        v[m] = make_float2(v[m].x * tp, v[m].y * tp);
      }
    }
    if constexpr (!ADJ) {
      const size_t out = ((size_t)b * a.nz + a.z) * n2;
      if (a.out_field) {
        const __amdgpu_buffer_rsrc_t ro = items_rsrc(a.out_field + out, bytes);
#pragma unroll
        for (int m = 0; m < E; ++m) items_st(ro, o8, m * T * 8, v[m]);
      }
      if (a.out_intens) {
        const __amdgpu_buffer_rsrc_t ro = items_rsrc(a.out_intens + out, bytes / 2);
#pragma unroll
        for (int m = 0; m < E; ++m) items_st1(ro, o4, m * T * 4, v[m].x * v[m].x + v[m].y * v[m].y);
      }
      if (a.acc) {
        const __amdgpu_buffer_rsrc_t rc = items_rsrc(a.acc + b * n2, bytes / 2);
#pragma unroll
        for (int m = 0; m < E; ++m) {
          const float i2 = v[m].x * v[m].x + v[m].y * v[m].y;
          items_st1(rc, o4, m * T * 4, a.acc_init ? i2 : av[m] + i2);
        }
      }
    }
    if (b < a.fwd_items) line_fft<NX, E, false, SwzLayout<4>, WAVE>(v, lds[line], t, tw);
    const __amdgpu_buffer_rsrc_t rp = items_rsrc(a.plane + b * n2, bytes);
#pragma unroll
    for (int m = 0; m < E; ++m) items_st(rp, o8, m * T * 8, v[m]);
  }
}

// FFT_y, H, IFFT_y of items b0 .. b0 + per - 1 of a tile of LC columns, H (of
// the table or, FLY, of n_eff[z]: evaluated once here) and twiddles in registers.
template <int NY, int E, int LC, int W, bool FLY>
__global__ void __launch_bounds__((NY / E * LC), W)
k_col_items(ColArgs a, int batch, int per) {
  constexpr int T = NY / E;
  constexpr bool SWZ = LC >= 4;
  constexpr int LINE = SWZ ? NY + 16 / LC : Base<NY, E>::COL_LINE;
  __shared__ float2 lds[LC][LINE];
  using CL = std::conditional_t<SWZ, SwzLayout<4 - ilog2c(LC)>, PadLayout<Base<NY, E>::COL_SH>>;
  // adjacent tiles share cache lines: keep them on one XCD
  const int ntiles = a.nx / LC, bx = blockIdx.x;
  const int tile = (ntiles % 8 == 0) ? (bx & 7) * (ntiles >> 3) + (bx >> 3) : bx;
  const int c = threadIdx.x % LC, t = threadIdx.x / LC;
  const int x = tile * LC + c;
  const int b0 = blockIdx.y * per, b1 = min(batch, b0 + per);
  const size_t n2 = (size_t)NY * a.nx;
  const int bytes = (int)n2 * 8, o8 = (t * a.nx + x) * 8, step = a.nx * T * 8;

  float2 next[E];
  auto load = [&](int b) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rp = items_rsrc(a.plane + b * n2, bytes);
#pragma unroll
    for (int m = 0; m < E; ++m) next[m] = items_ld(rp, o8, m * step);
  };
  float2 h[E];
  if constexpr (FLY)
    col_h_fly<NY, E>(kcomp2_f32(x, a.nx, a.dx), n_term_f32(a.n_eff[a.z], a.k0), a.dy, a.dz, t, lds[c], h);
  load(b0);
  Twiddles<NY, E> tw;
  tw.load(t, a.tw);
  if constexpr (!FLY) {
    const int qx = min(x, a.nx - x);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int ky = t + m * T;
      h[m] = a.H[(size_t)min(ky, NY - ky) * a.nx + qx];
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) h[m].y = a.conj_h ? -h[m].y : h[m].y;

#pragma unroll 1
  for (int b = b0; b < b1; ++b) {
    float2 v[E];
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = next[m];
    if (b + 1 < b1) load(b + 1);
    line_fft<NY, E, false, CL>(v, lds[c], t, tw);
    if (a.kout) {  // recorded for the adjoint: U = F u of this step
      const __amdgpu_buffer_rsrc_t rk = items_rsrc(a.kout + (size_t)b * a.kout_bstride, bytes);
#pragma unroll
      for (int m = 0; m < E; ++m) items_st(rk, o8, m * step, v[m]);
    }
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = c_mul_fused(v[m], h[m]);
    line_fft<NY, E, true, CL>(v, lds[c], t, tw);
    const __amdgpu_buffer_rsrc_t rp = items_rsrc(a.plane + b * n2, bytes);
#pragma unroll
    for (int m = 0; m < E; ++m) items_st(rp, o8, m * step, v[m]);
  }
}
