// The adjoint z-loop of small grids in one launch: the gradient planes of a
// batch carried back through a recorded segment by the teams of loop.hpp, one
// field per team.  Phase k works on plane z = nz - 1 - k of the segment:
//   row phase: (IFFT_x) -> screen gradient of the plane, per field, into
//              gvol -> conjugate screen -> FFT_x (plane 0: IFFT_x alone)
//   column phase: FFT_y -> conj(H) -> IFFT_y; with a mean correction FFT_y and
//              the per-column sums, then dL/ddn0, conj(H) and the term of dn0's
//              dependence on the field, IFFT_y -- the columns, H and the
//              forward plane stay in registers between the two.
// The fields' screen gradients are summed in field order by one kernel over
// the whole segment afterwards.  The operations are those of the launches per
// pass (bpmh_adjoint_segment, bpmh_mean_segment), so the bits are too.
//
// Measured (segments of 16 steps), us per step against the launches: without a
// mean correction the adjoint step, with the weighted mean the recorded forward
// step and the adjoint step.
//   64^2   batch 1: 4.8 against 10.8, weighted 16.8 against 32.4
//          batch 50: 6.7 against 23.9,         20.6 against 41.8
//   128^2  batch 1: 5.5 against 11.9,          19.2 against 37.7
//          batch 50: 10.7 against 31.7,        33.5 against 73.5
//   256^2  batch 1: 8.0 against 12.4,          24.6 against 39.8
//          batch 8: 8.8 against 18.8,          25.1 against 52.9
//          batch 50: 37.6 against 54.7,        136 against 173
//   512^2  batch 8: 34.2 against 34.5,         81 against 116
// A mean-corrected step is 6 phases (3 of them adjoint) and the float64 sines
// of its propagator; what bounds a phase is as in loop.hpp.
#pragma once
#include "loop.hpp"

// Sum over a row of NX values held by T threads of E (element t + m*T in
// w[m]), in the order of k_row_sums: lane l of 64 adds elements l, l + 64, ...,
// then an xor butterfly.  T <= 64; the result is in every thread of the row.
template <int NX, int E>
BPMH_DEV float loop_row_sum(const float (&w)[E]) {
  constexpr int T = NX / E, J = 64 / T;  // J lanes' worth of elements per thread
  float s[J];
#pragma unroll
  for (int j = 0; j < J; ++j) s[j] = 0.f;
#pragma unroll
  for (int m = 0; m < E; ++m) s[m % J] += w[m];
#pragma unroll
  for (int h = J / 2; h > 0; h >>= 1)
#pragma unroll
    for (int j = 0; j < h; ++j) s[j] += s[j + h];
  float r = s[0];
#pragma unroll
  for (int o = T / 2; o > 0; o >>= 1) r += __shfl_xor(r, o, 64);
  return r;
}

// MODE: BPMH_MEAN_IGNORE, _SIMPLE or _WEIGHTED.  ra: plane = the gradients,
// dn at the segment's first plane, nz = the segment's planes, useg, gitem =
// gvol (nz-1, batch, ny, nx) floats (float2 for complex dn); ca as the column
// phases 3 and 4 of k_col, uk at the segment's first step.
template <int NX, int NY, int ER, int EC, int MODE, bool LOST = false>
__global__ void __launch_bounds__((LoopCfg<NX, NY, ER, EC>::TH), (LoopCfg<NX, NY, ER, EC>::WAVES))
k_loop_adj(LoopCall) {
  using C = LoopCfg<NX, NY, ER, EC>;
  static_assert(C::WAVE, "rows of one wavefront");
  constexpr int SLOTS = C::SLOTS, QR = C::QR, TR = C::TR, TC = C::TC;
  constexpr bool MEAN = MODE != BPMH_MEAN_IGNORE;
  using RL = SwzLayout<4>;
  using CL = std::conditional_t<C::SWZ, SwzLayout<4 - ilog2c(C::SWZ ? C::LC : 1)>,
                                PadLayout<Base<NY, EC>::COL_SH>>;
  __shared__ __align__(16) float2 lds[C::LDS];
  __shared__ unsigned long long sh_rec;
  __shared__ unsigned sh_u[2];
  __shared__ float sh_f[2];
  constexpr int HALF = (NX < NY ? NX : NY) / 2;
  __shared__ float sh_taper[HALF];
  __shared__ float sh_g[MODE == BPMH_MEAN_WEIGHTED && C::E != 4 ? C::PTS : 1];
  const int tid0 = threadIdx.x;

  LoopTeam<C, LOST> tm;
  if (!tm.join(sh_u)) return;
  {
    const int w = min(loop_args().ra.absorb, HALF);
    for (int d = tid0; d < w; d += C::TH) sh_taper[d] = taper_factor(d, loop_args().ra.absorb);
    __syncthreads();
  }
  int held = -1;
  float2 v[EC], h[EC], uv[EC];  // columns, H and forward plane between phases 3 and 4
  // gradient of the weight slice, over a complete team's steps (8-point
  // threads keep it in LDS)
  constexpr bool GKEEP = C::E == 4;
  float gacc[EC];
  float2 upre[QR][ER];          // forward plane and dn of the next row phase
  float dpre[QR][ER];

  while (tm.next(&sh_rec)) {
    const int field = tm.field, me = tm.me, M = tm.M;
    const bool whole = tm.whole;
    const int top = [&] { const LoopCall& c = loop_args(); return loop_nz(c.ra, c.la, field) - 1; }();

    auto load_row = [&](const RowArgs& ra, int s, int z, int line, int tr) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < QR; ++q) {
        const int o = (s * C::LR + q * C::LRP + line) * NX + tr;
        const float2* u = ra.useg + (size_t)field * ra.useg_bstride + (size_t)z * C::POINTS + o;
#pragma unroll
        for (int m = 0; m < ER; ++m) upre[q][m] = u[m * TR];
        if (ra.dn_kind == BPMH_DN_F32) {
          const float* p = (const float*)ra.dn + (size_t)z * C::POINTS + o;
#pragma unroll
          for (int m = 0; m < ER; ++m) dpre[q][m] = p[m * TR];
        }
      }
    };

    if (MODE == BPMH_MEAN_WEIGHTED && whole && held != field) {
      const LoopCall& call = loop_args();
      const int tid = loop_opaque(tid0);
      const __amdgpu_buffer_rsrc_t rg = loop_rsrc(call.ca.gd_item + (size_t)field * C::POINTS, C::POINTS * 4);
#pragma unroll
      for (int m = 0; m < EC; ++m)
        (GKEEP ? gacc[m] : sh_g[m * C::TH + tid]) = loop_ld1(rg, ((tid / C::LC) * NX + tid % C::LC) * 4, (me * C::LC + m * TC * NX) * 4);
      held = field;
    }

    auto row_phase = [&](int k, bool first) __attribute__((always_inline)) {
      const int z = top - k;
      const RowArgs& ra = loop_args().ra;
      Twiddles<NX, ER> tw;
      tw.load(loop_opaque(tid0) % TR, ra.tw);
      tm.enter(first, sh_u);
      if (tm.dead) return;
      const __amdgpu_buffer_rsrc_t rp = loop_rsrc(ra.plane + (size_t)field * C::POINTS, C::POINTS * 8);
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int line = tid / TR, tr = tid - line * TR;
        const int off = (line * NX + tr) * 8;
        float2 g[QR][ER];
#pragma unroll
        for (int q = 0; q < QR; ++q)
#pragma unroll
          for (int m = 0; m < ER; ++m)
            g[q][m] = loop_ld(rp, off, ((s * C::LR + q * C::LRP) * NX + m * TR) * 8);
        if (z > 0 && (first || !whole)) load_row(ra, s, z, line, tr);
        float dn0 = 0.f;
        if (MODE == BPMH_MEAN_SIMPLE && z > 0) dn0 = ra.dn0_arr[z];
        if (MODE == BPMH_MEAN_WEIGHTED && z > 0) {
          const LoopCall& call = loop_args();
          dn0 = call.ca.cz[(size_t)(z - 1) * call.la.batch + field];
        }
#pragma unroll
        for (int q = 0; q < QR; ++q) {
          const int y = s * C::LR + q * C::LRP + line;
          float2* const ln = lds + (q * C::LRP + line) * C::ROW_LINE;
          if (k > 0) {
            line_fft<NX, ER, true, RL, true>(g[q], ln, tr, tw);
#pragma unroll
            for (int m = 0; m < ER; ++m) g[q][m] = c_scale(g[q][m], ra.inv_n);
          }
          if (z > 0) {
            const size_t o = ((size_t)(z - 1) * loop_args().la.batch + field) * C::POINTS +
                             (size_t)(y * NX + tr);
            if (!MEAN && ra.dn_kind == BPMH_DN_C64) {
              // phases and magnitudes through the thread's slots of its line,
              // in a rolled loop (as loop_screen)
              const float2* dc = (const float2*)ra.dn + (size_t)z * C::POINTS + (size_t)(y * NX + tr);
#pragma unroll
              for (int m = 0; m < ER; ++m) {
                const float2 w = adjoint_pair(g[q][m], upre[q][m]);
                st_stream(reinterpret_cast<float2*>(ra.gitem) + o + m * TR,
                          make_float2(ra.unit_k * w.y, ra.unit_k * w.x));
                const float2 d = dc[m * TR];
                ln[tr + m * TR] = make_float2(f_mul(-ra.unit_k, f_sub(d.x, dn0)), f_mul(ra.unit_k, d.y));
              }
#pragma unroll 1
              for (int m = 0; m < ER; ++m) {
                const float2 w = ln[tr + m * TR];
                float sn, cs;
                sincos_fast(w.x, &sn, &cs);
                const float mag = expf(w.y);
                ln[tr + m * TR] = make_float2(mag * cs, mag * sn);
              }
#pragma unroll
              for (int m = 0; m < ER; ++m) g[q][m] = c_mulc_fused(g[q][m], ln[tr + m * TR]);
            } else {
              float w[ER];
              bool far = false;
#pragma unroll
              for (int m = 0; m < ER; ++m) {
                w[m] = f_mul(ra.unit_k, adjoint_pair(g[q][m], upre[q][m]).y);
                st_stream(ra.gitem + o + m * TR, w[m]);
                far |= !(fabsf(f_mul(-ra.unit_k, f_sub(dpre[q][m], dn0))) <= kSincosNear);
              }
              if constexpr (MEAN) {
                const float sum = loop_row_sum<NX, ER>(w);
                if (tr == 0) const_cast<float*>(loop_args().ca.s1part)[(size_t)field * NY + y] = sum;
              }
              if (__any(far)) {
#pragma unroll
                for (int m = 0; m < ER; ++m) ln[tr + m * TR].x = f_mul(-ra.unit_k, f_sub(dpre[q][m], dn0));
#pragma unroll 1
                for (int m = 0; m < ER; ++m) {
                  float sn, cs;
                  sincos_fast(ln[tr + m * TR].x, &sn, &cs);
                  ln[tr + m * TR] = make_float2(cs, sn);
                }
#pragma unroll
                for (int m = 0; m < ER; ++m) g[q][m] = c_mulc_fused(g[q][m], ln[tr + m * TR]);
              } else {
#pragma unroll
                for (int m = 0; m < ER; ++m) {
                  float sn, cs;
                  sincos_near(f_mul(-ra.unit_k, f_sub(dpre[q][m], dn0)), &sn, &cs);
                  g[q][m] = c_mulc_fused(g[q][m], make_float2(cs, sn));
                }
              }
              if (ra.absorb > 0) {
                const int disty = min(NY - y - 1, y);
#pragma unroll
                for (int m = 0; m < ER; ++m) {
                  const int x = tr + m * TR;
                  const int dist = min(min(NX - x - 1, x), disty);
                  if (dist < ra.absorb) {
                    const float tp = sh_taper[dist];
                    g[q][m] = make_float2(g[q][m].x * tp, g[q][m].y * tp);
                  }
                }
              }
            }
            line_fft<NX, ER, false, RL, true>(g[q], ln, tr, tw);
          }
#pragma unroll
          for (int m = 0; m < ER; ++m)
            loop_st(rp, off, ((s * C::LR + q * C::LRP) * NX + m * TR) * 8, g[q][m]);
        }
        tm.leave(s);
      }
      tm.at += 1;
    };

    // back through the propagator from plane z = top - k to z - 1 (k >= 0)
    auto col_phase = [&](int k, bool first) __attribute__((always_inline)) {
      const int z = top - k;
      const LoopCall& call = loop_args();
      const ColArgs& ca = call.ca;
      Twiddles<NY, EC> tw;
      tw.load(loop_opaque(tid0) / C::LC, ca.tw);
      tm.enter(first, sh_u);
      if (tm.dead) return;
      const __amdgpu_buffer_rsrc_t rp = loop_rsrc(ca.plane + (size_t)field * C::POINTS, C::POINTS * 8);
      // refractive index and dn0 of the step
      float dn0 = 0.f, n_adj = 0.f;
      if constexpr (MEAN) {
        dn0 = MODE == BPMH_MEAN_SIMPLE ? 0.f : ca.cz[(size_t)(z - 1) * call.la.batch + field];
        n_adj = MODE == BPMH_MEAN_SIMPLE ? ca.n_eff[z] : f_add(ca.n0, dn0);
      }
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int cl = tid % C::LC, tc = tid / C::LC;
        float2* const ln = lds + cl * C::COL_LINE;
        const int off = (tc * NX + cl) * 8;
        const int x = s * C::LC + cl;
#pragma unroll
        for (int m = 0; m < EC; ++m) v[m] = loop_ld(rp, off, (s * C::LC + m * TC * NX) * 8);
        if constexpr (!MEAN) {
          const int qx = min(x, NX - x);
#pragma unroll
          for (int m = 0; m < EC; ++m) {
            const int ky = tc + m * TC;
            h[m] = ca.H[min(ky, NY - ky) * NX + qx];
          }
          line_fft<NY, EC, false, CL>(v, ln, tc, tw);
#pragma unroll
          for (int m = 0; m < EC; ++m) v[m] = c_mul_fused(v[m], make_float2(h[m].x, -h[m].y));
          if (whole && z > 1) load_row(call.ra, s, z - 1, tid / TR, tid % TR);
          line_fft<NY, EC, true, CL>(v, ln, tc, tw);
#pragma unroll
          for (int m = 0; m < EC; ++m) loop_st(rp, off, (s * C::LC + m * TC * NX) * 8, v[m]);
        } else {
          const float2* uk = ca.uk + (size_t)field * ca.uk_bstride + (size_t)(z - 1) * C::POINTS + x;
#pragma unroll
          for (int m = 0; m < EC; ++m) uv[m] = uk[(tc + m * TC) * NX];
          line_fft<NY, EC, false, CL>(v, ln, tc, tw);
          float bt[EC];
          col_hb_fly<NY, EC>(kcomp2_f32(x, NX, ca.dx), n_term_f32(n_adj, ca.k0), ca.dy, ca.dz, tc, ln,
                             h, bt);
          const float tot = col_beta_sum<NY, EC>(v, h, uv, bt, tc, ln);
          if (tc == 0) ca.s2part[(size_t)field * NX + x] = tot;
          if (!whole) {
#pragma unroll
            for (int m = 0; m < EC; ++m) loop_st(rp, off, (s * C::LC + m * TC * NX) * 8, v[m]);
          }
        }
        tm.leave(s);
      }
      tm.at += 1;
      if constexpr (MEAN) {
        // (read again: over the sums before they only took registers)
        tw.load(loop_opaque(tid0) / C::LC, ca.tw);
        tm.enter(false, sh_u);
        if (tm.dead) return;
        if (tid0 < 64) {  // both sums in the order of group_sum_pair
          const int lane = loop_opaque(tid0);
          const __amdgpu_buffer_rsrc_t r1 = loop_rsrc(ca.s1part + (size_t)field * NY, NY * 4);
          const __amdgpu_buffer_rsrc_t r2 = loop_rsrc(ca.s2part + (size_t)field * NX, NX * 4);
          float s1 = 0.f, s2 = 0.f;
#pragma unroll
          for (int i = 0; i < NY; i += 64) s1 += loop_ld1(r1, lane * 4, i * 4);
#pragma unroll
          for (int i = 0; i < NX; i += 64) s2 += loop_ld1(r2, lane * 4, i * 4);
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) {
            s1 += __shfl_xor(s1, o, 64);
            s2 += __shfl_xor(s2, o, 64);
          }
          if (tid0 == 0) {
            sh_f[0] = s1;
            sh_f[1] = s2;
          }
        }
        __syncthreads();
        const float n_pts = (float)NX * (float)NY;
        const float cgrad = adjoint_cgrad(sh_f[0], sh_f[1], ca.dz, n_adj, ca.k0, n_pts);
        float inv_w = 0.f;
        if (MODE == BPMH_MEAN_WEIGHTED) inv_w = 1.f / ca.wz[(size_t)(z - 1) * call.la.batch + field];
        for (int s = me; s < SLOTS; s += M) {
          const int tid = loop_opaque(tid0);
          const int cl = tid % C::LC, tc = tid / C::LC;
          float2* const ln = lds + cl * C::COL_LINE;
          const int off = (tc * NX + cl) * 8;
          const int x = s * C::LC + cl;
          if (MODE == BPMH_MEAN_SIMPLE && s == 0 && tid == 0)
            ca.cg_out[(size_t)(z - 1) * call.la.batch + field] = cgrad;
          if (!whole) {
#pragma unroll
            for (int m = 0; m < EC; ++m) v[m] = loop_ld(rp, off, (s * C::LC + m * TC * NX) * 8);
            const float2* uk = ca.uk + (size_t)field * ca.uk_bstride + (size_t)(z - 1) * C::POINTS + x;
#pragma unroll
            for (int m = 0; m < EC; ++m) uv[m] = uk[(tc + m * TC) * NX];
            col_h_fly<NY, EC>(kcomp2_f32(x, NX, ca.dx), n_term_f32(n_adj, ca.k0), ca.dy, ca.dz, tc, ln, h);
          }
#pragma unroll
          for (int m = 0; m < EC; ++m) v[m] = c_mul_fused(v[m], make_float2(h[m].x, -h[m].y));
          if constexpr (MODE == BPMH_MEAN_WEIGHTED) {
            const __amdgpu_buffer_rsrc_t rg =
                loop_rsrc(ca.gd_item + (size_t)field * C::POINTS, C::POINTS * 4);
            const int goff = (tc * NX + cl) * 4;
#pragma unroll
            for (int m = 0; m < EC; ++m) {
              const float d = ca.dn ? load_dn(ca.dn, ca.dn_kind,
                                              (size_t)field * ca.dn_bstride +
                                                  (size_t)((tc + m * TC) * NX + x)).x
                                    : 0.f;
              const float w = adjoint_weight_term(v[m], uv[m], d, dn0, cgrad, inv_w, n_pts);
              const int goffs = (s * C::LC + m * TC * NX) * 4;
              float& mine = GKEEP ? gacc[m] : sh_g[m * C::TH + tid];
              const float sum = (whole ? mine : loop_ld1(rg, goff, goffs)) + w;
              if (whole) mine = sum;
              if (!whole || z == 1)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum), rg, goff, goffs, 0);
            }
          }
          if (whole && z > 1) load_row(call.ra, s, z - 1, tid / TR, tid % TR);
          line_fft<NY, EC, true, CL>(v, ln, tc, tw);
#pragma unroll
          for (int m = 0; m < EC; ++m) loop_st(rp, off, (s * C::LC + m * TC * NX) * 8, v[m]);
          tm.leave(s);
        }
        tm.at += 1;
      }
    };

    // a chunk's planes z0 (done) to z1 count the phases k; phase 0 is a row
    // phase alone
    const int kb = tm.z0 == 0 ? 0 : tm.z0 + 1;
    for (int k = kb; k <= tm.z1 && !tm.dead; ++k) {
      if (k > 0) col_phase(k - 1, k == kb);
      if (!tm.dead) row_phase(k, k == 0);
    }
    if (tm.dead) {
      tm.give_up();
      return;
    }
  }
}

bool bpmh_loop_adj_nx64(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_adj_nx128(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_adj_nx256(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_adj_nx512(int, int, int, int, const LoopCall&, int, hipStream_t);

template <int NX, int NY, int ER, int EC, bool LOST>
static bool loop_adj_launch_m(int mode, const LoopCall& c, int groups, hipStream_t s) {
  const dim3 g((unsigned)groups), b(LoopCfg<NX, NY, ER, EC>::TH);
  switch (mode) {
    case BPMH_MEAN_IGNORE:
      hipLaunchKernelGGL((k_loop_adj<NX, NY, ER, EC, BPMH_MEAN_IGNORE, LOST>), g, b, 0, s, c);
      return true;
    case BPMH_MEAN_SIMPLE:
      hipLaunchKernelGGL((k_loop_adj<NX, NY, ER, EC, BPMH_MEAN_SIMPLE, LOST>), g, b, 0, s, c);
      return true;
    case BPMH_MEAN_WEIGHTED:
      hipLaunchKernelGGL((k_loop_adj<NX, NY, ER, EC, BPMH_MEAN_WEIGHTED, LOST>), g, b, 0, s, c);
      return true;
  }
  return false;
}

template <int NX, int NY, int ER, int EC>
static bool loop_adj_launch_e(int mode, const LoopCall& c, int groups, hipStream_t s) {
  if constexpr (!LoopCfg<NX, NY, ER, EC>::WAVE) {
    return false;
  } else {
    if (!c.la.lost) return loop_adj_launch_m<NX, NY, ER, EC, false>(mode, c, groups, s);
    if constexpr (kLoopLost<NX, NY, ER, EC>) return loop_adj_launch_m<NX, NY, ER, EC, true>(mode, c, groups, s);
    return false;
  }
}

template <int NX, int NY>
static bool loop_adj_launch_n(int er, int ec, int mode, const LoopCall& c, int groups, hipStream_t s) {
  if (er == 4 && ec == 4) return loop_adj_launch_e<NX, NY, 4, 4>(mode, c, groups, s);
  if (er == 4 && ec == 8) return loop_adj_launch_e<NX, NY, 4, 8>(mode, c, groups, s);
  if (er == 8 && ec == 8) return loop_adj_launch_e<NX, NY, 8, 8>(mode, c, groups, s);
  return false;
}

template <int NX>
static bool loop_adj_launch_nx(int ny, int er, int ec, int mode, const LoopCall& c, int groups,
                               hipStream_t s) {
  switch (ny) {
    case 64: return loop_adj_launch_n<NX, 64>(er, ec, mode, c, groups, s);
    case 128: return loop_adj_launch_n<NX, 128>(er, ec, mode, c, groups, s);
    case 256: return loop_adj_launch_n<NX, 256>(er, ec, mode, c, groups, s);
    case 512: return loop_adj_launch_n<NX, 512>(er, ec, mode, c, groups, s);
  }
  return false;
}
