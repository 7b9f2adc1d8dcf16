// The whole z-loop of small grids in one launch.
//
// A field of up to 512 x 512 points (2 MiB) fits the 4 MiB L2 of one XCD, so
// a team of work-groups on one XCD propagates it through all its steps: the
// plane goes from the row phase to the column phase and back through that L2,
// and the phases are separated by flags in it instead of by kernel
// boundaries.  What bounds the two-launch step at these sizes is the boundary
// (4.7 us per launch at 64^2 as at 256^2, batch 1); a phase here costs 0.6 us
// of synchronisation and 0.5 us of L2 latency (256^2, 32 work-groups,
// measured without the transforms).  Batches run one team per field, so the
// planes stay in eight L2s instead of crossing the XCDs twice per step.
//
// Teams.  Every work-group reads its XCD's number and registers there (an
// atomic in the XCD's L2).  Rank r belongs to team r / SLOTS of its XCD as
// member r % SLOTS; member 0 leads.  A team's work is cut into SLOTS equal
// slots of rows and of columns.  The leader announces the work in records
// (field, first plane, number of members M, a power of two), a chunk of up to
// kLoopSteps steps each (few while the team is incomplete), and member m < M does the slots m, m + M, ...: all of
// its own slot when the team is complete, more while some of its work-groups
// have not started (the GPU may be shared with other streams' kernels).  A
// work-group therefore waits only for others that are already running,
// whatever is resident; no co-residency is assumed and nothing depends on how
// the dispatcher deals work-groups to XCDs.  The fields are claimed from one
// counter by the leaders, deepest first.  Every wait is bounded: should one give
// up, the kernel after this one (which clears the synchronisation words, as a
// kernel before it would) turns the call's results into NaN and tells the host.
//
// Memory.  Within an XCD the L2 is the point where all its CUs' accesses
// meet: stores are written through the CU's L1 to it, and loads with the sc1
// bit skip the L1.  A phase ends with every wavefront waiting for its stores
// (vmcnt 0), then the slot's flag; the next phase starts when every slot's
// flag is seen.  Data that other CUs write (the plane, per-column partial
// sums, flags, records) is read with sc1; tables, dn and a slot's own values
// are read as usual.  (A cache invalidate per phase instead of sc1 loads
// costs 1.6 us per phase.)  No two XCDs touch the same field.
//
// A complete team's member keeps its columns of the propagator (4-point
// threads) and its rows of the running intensity sum over all steps, in
// registers or LDS, and loads its dn row of a step while the column phase
// before it is under way.
//
// Measured, us per step against the launches per pass (65 planes, running
// sum kept; 4.4, 4.8, 8.8: points per thread of rows and columns):
//   64^2   batch 1: 4.0 (4.4) against 8.5;   batch 50: 4.4 against 9.6
//   128^2  batch 1: 4.9 (4.4) against 9.6;   batch 50: 7.2 against 16.6
//   256^2  batch 1: 6.8 (4.4) against 10.1;  8: 6.7 against 13.7;
//          batch 16: 8.4 against 18.8;       50: 25.1 (8.8) against 37.4
//   512^2  batch 1: 14.0 (8.8) against 12.5; 2: 14.3 against 15.7;
//          batch 8: 14.2 against 30.9;       50: 94.9 against 100.6
// What bounds a phase now: at 64^2 its chain of L2, LDS and flag latencies
// (2.0 us), at 512^2 the transforms' instruction issue on the XCD's 32 CUs
// (a field-step of 512^2 on one XCD is about 9 us of issue).
#pragma once
#include "passes.hpp"

#include <cstddef>

constexpr int kLoopSteps = 64;      // z-steps per record
constexpr int kLoopStepsPart = 4;   // the same while the team is not complete
constexpr int kLoopXcds = 16;       // XCD numbers are 4 bits
constexpr int kLoopTeamWords = 192; // 128 flags, the record, padding
constexpr int kLoopHead = 64 + 64 * kLoopXcds;  // claim counter, failure, registrations
constexpr int kLoopFailed = 32;  // word (in a line of its own): number of the last call a wait of which gave up
constexpr unsigned kLoopLimit = 1u << 25;  // polls after which a wait gives up (> 10 s)

// Points of a slot: a 32nd of the plane (one slot per CU of an XCD), at least
// 512 (two wavefronts of 4-point threads) and at most 4096 (1024 threads).
constexpr int loop_points(int nx, int ny) {
  const int p = nx * ny / 32;
  return p < 512 ? 512 : (p > 4096 ? 4096 : p);
}
constexpr int loop_slots(int nx, int ny) { return nx * ny / loop_points(nx, ny); }
// Teams per XCD of `slots` members: what its 32 CUs hold of the smallest
// members (two wavefronts), at most kLoopTeams.
constexpr int loop_teams(int slots) { return 256 / slots < 1 ? 1 : 256 / slots; }
constexpr int kLoopTeams = loop_teams(loop_slots(64, 64));
// 32-bit words of synchronisation state for `teams` teams per XCD
constexpr size_t loop_words(int teams) {
  return (size_t)kLoopHead + (size_t)kLoopXcds * teams * kLoopTeamWords;
}

struct LoopArgs {
  unsigned* sync;               // loop_words(teams) words, zero at launch (but kLoopFailed)
  int batch;                    // fields
  int teams;                    // teams per XCD
  int gnz[BPMH_MAX_GROUPS];     // planes of each group of a ragged batch
  long long kout_zstride;       // recorded forward: between two steps' k-space planes
  unsigned call;                // number of this call on `sync`, from 1
  int lost;                     // tests: every wait gives up (host: which kernel)
};

// The kernel's one argument.  It is read through the kernel-argument segment
// at the start of each phase (loop_args below), not held in registers.
struct LoopCall {
  RowArgs ra;
  ColArgs ca;
  LoopArgs la;
};

template <int NX, int NY, int ER, int EC>
struct LoopCfg {
  static constexpr int POINTS = NX * NY;
  static constexpr int PTS = loop_points(NX, NY), SLOTS = loop_slots(NX, NY);
  static constexpr int E = EC;                  // points per thread
  static constexpr int TH = PTS / E;
  static constexpr int TR = NX / ER, TC = NY / EC;  // threads of a row, of a column
  static constexpr int QR = E / ER;             // rows per thread (one column)
  static constexpr int LR = PTS / NX, LC = PTS / NY;  // rows, columns of a slot
  static constexpr int LRP = LR / QR;           // rows side by side
  static constexpr bool WAVE = TR <= 64;
  static constexpr int WAVES = 4;  // wavefronts per SIMD compiled for: two 512-thread groups a CU
  static constexpr int ROW_LINE = Base<NX, ER>::ROW_LINE;
  static constexpr bool SWZ = LC >= 4;
  static constexpr int COL_LINE = SWZ ? NY + 16 / LC : Base<NY, EC>::COL_LINE;
  static constexpr int LDS = LR * ROW_LINE > LC * COL_LINE ? LR * ROW_LINE : LC * COL_LINE;
  static_assert(EC >= ER && LRP >= 1 && LC >= 1 && LC <= 16 && TH >= 64 && TH <= 1024, "loop shape");
  static_assert(LRP * TR == TH && LC * TC == TH, "every thread works in both phases");
  static_assert(SLOTS <= 128, "flags of a team");
};

typedef unsigned loop_u2 __attribute__((ext_vector_type(2)));
constexpr int kSc1 = 16;  // cache policy bits of the buffer loads: sc1

BPMH_DEV __amdgpu_buffer_rsrc_t loop_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}
// off: per-thread byte offset, soff: uniform byte offset (a scalar operand)
BPMH_DEV float2 loop_ld(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  const loop_u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, kSc1);
  return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}
BPMH_DEV void loop_st(__amdgpu_buffer_rsrc_t r, int off, int soff, float2 v) {
  const loop_u2 w = {__float_as_uint(v.x), __float_as_uint(v.y)};
  __builtin_amdgcn_raw_buffer_store_b64(w, r, off, soff, 0);
}
BPMH_DEV float loop_ld1(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, soff, kSc1));
}

// The kernel's argument, as a pointer the compiler cannot trace back: what a
// phase reads from it is loaded (scalar loads) in that phase.  Held over the
// whole loop the 130 argument words took all scalar registers, and addresses
// formed from them most vector registers (225 to 256, with 187 scalar
// spills, at 256^2).
BPMH_DEV const LoopCall& loop_args() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const LoopCall*)p;
}
BPMH_DEV int loop_opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Record: sequence 20 bits, end 1, log2 of the members 3, field 20, plane 20.
BPMH_DEV unsigned long long loop_pack(unsigned seq, bool end, int mlog, int field, int z) {
  return ((unsigned long long)seq << 44) | ((unsigned long long)end << 43) |
         ((unsigned long long)mlog << 40) | ((unsigned long long)field << 20) | (unsigned)z;
}

// One wavefront waits until the n flags are all at least `need`.  LOST: it gives
// up at once.  (A template argument: a limit or switch held in a register or
// read at each wait cost 50 ns of a phase.)
template <bool LOST>
BPMH_DEV bool loop_wait(const unsigned* flags, int n, unsigned need) {
  if constexpr (LOST) return false;
  const __amdgpu_buffer_rsrc_t r = loop_rsrc(flags, 128 * 4);
  const int lane = loop_opaque(threadIdx.x & 63);
  for (unsigned k = 0; k < kLoopLimit; ++k) {
    bool ok = true;
    for (int i = lane; i < n; i += 64)
      ok &= __builtin_amdgcn_raw_buffer_load_b32(r, i * 4, 0, kSc1) >= need;
    asm volatile("" ::: "memory");
    if (__all(ok)) return true;
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

// dn volume (group) and depth of a field, looked up once per record (15 compares
// and selects per phase cost 1 to 3 %).  The group tables are read at
// constant indices: a kernel argument indexed at run time would be copied to
// scratch memory whole.
BPMH_DEV int loop_volume(const RowArgs& ra, int field) {
  if (ra.ngroups == 0) return field;
  int g = 0;
#pragma unroll
  for (int k = 0; k + 1 < BPMH_MAX_GROUPS; ++k) g += k + 1 < ra.ngroups && field >= ra.gend[k];
  return g;
}
BPMH_DEV int loop_nz(const RowArgs& ra, const LoopArgs& la, int field) {
  if (ra.ngroups == 0) return ra.nz;
  int nz = la.gnz[0];
#pragma unroll
  for (int k = 0; k + 1 < BPMH_MAX_GROUPS; ++k)
    if (k + 1 < ra.ngroups && field >= ra.gend[k]) nz = la.gnz[k + 1];
  return nz;
}

// A work-group's place in its team, and the work that the team is at.
template <class C, bool LOST>
struct LoopTeam {
  unsigned* flags;
  int group, me;
  unsigned xcd;
  unsigned seq;          // last record seen
  unsigned at;           // value of the flags once the phases so far are done
  int lead_field, lead_z;
  bool dead;             // a wait gave up
  int M, field, z0, z1;  // members; the field and its planes z0 (done) to z1
  int volume;            // the field's dn volume
  bool whole, last;      // M == SLOTS; z1 is the field's last plane

  // Registers this work-group; false when there is no team for it.
  BPMH_DEV bool join(unsigned* sh) {
    const LoopArgs& la = loop_args().la;
    if (threadIdx.x == 0) {
      const unsigned x = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & (kLoopXcds - 1);  // XCC_ID
      sh[0] = __hip_atomic_fetch_add(la.sync + 64 + 64 * x, 1u, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
      sh[1] = x;
    }
    __syncthreads();
    const unsigned rank = __builtin_amdgcn_readfirstlane(sh[0]);
    xcd = __builtin_amdgcn_readfirstlane(sh[1]);
    group = (int)(rank / C::SLOTS);
    me = (int)(rank % C::SLOTS);
    flags = la.sync + kLoopHead + ((size_t)xcd * la.teams + group) * kLoopTeamWords;
    seq = at = 0;
    lead_field = -1;
    lead_z = 0;
    dead = false;
    return group < la.teams;
  }

  // Member 0, one wavefront: the previous chunk is complete, announce the next.
  BPMH_DEV void announce() {
    bool end = seq != 0 && !loop_wait<LOST>(flags, C::SLOTS, at);
    if (threadIdx.x != 0) return;
    if (end) failed();
    const LoopCall& call = loop_args();
    // the first time, up to ~20 us for the team to come together
    const __amdgpu_buffer_rsrc_t reg = loop_rsrc(call.la.sync, kLoopHead * 4);
    int n = 0;
    for (int k = 0; k < 64; ++k) {
      n = (int)__builtin_amdgcn_raw_buffer_load_b32(reg, (64 + 64 * xcd) * 4, 0, kSc1) -
          group * C::SLOTS;
      asm volatile("" ::: "memory");
      if (n >= C::SLOTS || seq != 0) break;
      __builtin_amdgcn_s_sleep(8);
    }
    n = n > C::SLOTS ? C::SLOTS : (n < 1 ? 1 : n);
    if (lead_field < 0 || lead_z >= loop_nz(call.ra, call.la, lead_field) - 1) {
      lead_field = (int)__hip_atomic_fetch_add(call.la.sync, 1u, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
      lead_z = 0;
    }
    end |= lead_field >= call.la.batch;
    const unsigned long long rec =
        loop_pack(seq + 1, end, 31 - __clz(n), end ? 0 : lead_field, lead_z);
    if (!end)
      lead_z = min(lead_z + (n == C::SLOTS ? kLoopSteps : kLoopStepsPart),
                   loop_nz(call.ra, call.la, lead_field) - 1);
    publish(rec);
  }
  BPMH_DEV void publish(unsigned long long rec) {
    __hip_atomic_store((unsigned long long*)(flags + 128), rec, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
  }

  // The next chunk that counts this work-group in; false at the end.
  BPMH_DEV bool next(unsigned long long* sh) {
    if (threadIdx.x < 64) {
      if (me == 0) announce();
      const __amdgpu_buffer_rsrc_t team = loop_rsrc(flags, kLoopTeamWords * 4);
      for (unsigned k = 0;; ++k) {
        if (k >= kLoopLimit) {  // the leader stopped
          if (threadIdx.x == 0) {
            failed();
            *sh = 1ull << 43;
          }
          break;
        }
        const loop_u2 w = __builtin_amdgcn_raw_buffer_load_b64(team, 128 * 4, 0, kSc1);
        asm volatile("" ::: "memory");
        const unsigned hi = __builtin_amdgcn_readfirstlane(w.y);
        const unsigned lo = __builtin_amdgcn_readfirstlane(w.x);
        const unsigned s = hi >> 12;
        if (s != seq) {
          seq = s;
          k = 0;
          if (((hi >> 11) & 1) || me < (1 << ((hi >> 8) & 7))) {
            if (threadIdx.x == 0) *sh = ((unsigned long long)hi << 32) | lo;
            break;
          }
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    __syncthreads();
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(*sh >> 32));
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)*sh);
    if ((hi >> 11) & 1) return false;
    seq = hi >> 12;
    at = seq << 8;
    M = 1 << ((hi >> 8) & 7);
    field = (int)(((hi & 0xffu) << 12) | (lo >> 20));
    z0 = (int)(lo & 0xfffffu);
    whole = M == C::SLOTS;
    const LoopCall& call = loop_args();
    const int nz = loop_nz(call.ra, call.la, field);
    z1 = min(z0 + (whole ? kLoopSteps : kLoopStepsPart), nz - 1);
    last = z1 == nz - 1;
    volume = __builtin_amdgcn_readfirstlane(loop_volume(call.ra, field));
    return true;
  }

  // Before a phase: every slot of the phase before it is done.  (The first
  // phase of a chunk: the leader saw that before it wrote the record.)
  BPMH_DEV void enter(bool first, unsigned* sh) {
    if (first) return;
    // To 32 slots every wavefront reads the flags itself: 2 to 4 % a step less
    // than one wavefront and a barrier (64^2 4.17 -> 4.03 us, 256^2 weighted
    // 9.9 -> 9.6); at 512^2's 64 slots the reads of 8 wavefronts cost 3 % more.
    if constexpr (C::SLOTS <= 32) {
      dead |= !loop_wait<LOST>(flags, C::SLOTS, at);
      return;
    }
    if (threadIdx.x < 64) {
      const bool ok = loop_wait<LOST>(flags, C::SLOTS, at);
      if (threadIdx.x == 0) sh[0] = ok;
    }
    __syncthreads();
    dead |= __builtin_amdgcn_readfirstlane(sh[0]) == 0;
  }
  // Slot s of the phase is done (the caller adds 1 to `at` after its slots).
  BPMH_DEV void leave(int s) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(flags + s, at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }

  // A wait gave up (a member of the team stopped): the kernel after this one
  // marks what the call wrote.  The wavefront ends (barriers then count the
  // others), and the leader ends the team.
  BPMH_DEV void failed() {
    const LoopArgs& la = loop_args().la;
    __hip_atomic_store(la.sync + kLoopFailed, la.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  BPMH_DEV void give_up() {
    if ((threadIdx.x & 63) == 0) failed();
    if (me == 0 && threadIdx.x == 0) publish(loop_pack(seq + 1, true, 0, 0, 0));
  }
};

// row_screen of a forward step, the same operations, for a kernel that keeps
// state in registers around it: one element after another, the taper from a
// table in LDS, and the rare or heavy forms (a phase beyond pi/4 in any lane
// of the wavefront, complex dn) in a rolled loop through the thread's own
// slots of its LDS line instead of inlined once per element.
template <int NX, int E, bool WAVE>
BPMH_DEV void loop_screen(const RowArgs& a, int ny, int y, int t, float dn0, const float (&dre)[E],
                          const float2* dc, float2* ln, const float* taper, float2 (&v)[E]) {
  constexpr int T = NX / E;
  const bool cplx = a.dn_kind == BPMH_DN_C64;
  bool rolled = cplx;
  if (WAVE && !cplx) {
    bool far = false;
#pragma unroll
    for (int m = 0; m < E; ++m) far |= !(fabsf(f_mul(-a.unit_k, f_sub(dre[m], dn0))) <= kSincosNear);
    rolled = __any(far);
  }
  if (rolled) {
    // (a line shared by wavefronts may still be read by the others)
    if (!WAVE) __syncthreads();
#pragma unroll
    for (int m = 0; m < E; ++m) {
      if (cplx) {
        const float2 w = dc[m * T];
        ln[t + m * T] = make_float2(f_mul(-a.unit_k, f_sub(w.x, dn0)), f_mul(a.unit_k, w.y));
      } else {
        ln[t + m * T] = make_float2(f_mul(-a.unit_k, f_sub(dre[m], dn0)), 0.f);
      }
    }
#pragma unroll 1
    for (int m = 0; m < E; ++m) {
      const float2 w = ln[t + m * T];
      float sn, cs;
      sincos_fast(w.x, &sn, &cs);
      const float mag = cplx ? expf(w.y) : 1.f;
      ln[t + m * T] = make_float2(mag * cs, mag * sn);
    }
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = c_mul_fused(v[m], ln[t + m * T]);
    if (!WAVE) __syncthreads();
    if (cplx) return;
  }
  if (!rolled) {
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const float ph = f_mul(-a.unit_k, f_sub(dre[m], dn0));
      float sn, cs;
      if (WAVE) sincos_near(ph, &sn, &cs);
      else sincos_fast(ph, &sn, &cs);
      v[m] = c_mul_fused(v[m], make_float2(cs, sn));
    }
  }
  if (a.absorb > 0) {
    const int disty = min(ny - y - 1, y);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int x = t + m * T;
      const int dist = min(min(NX - x - 1, x), disty);
      if (dist < a.absorb) {
        const float tp = taper[dist];
        v[m] = make_float2(v[m].x * tp, v[m].y * tp);
      }
    }
  }
}

// MODE: BPMH_MEAN_IGNORE (propagator table), BPMH_MEAN_SIMPLE, BPMH_MEAN_WEIGHTED.
template <int NX, int NY, int ER, int EC, int MODE, bool LOST = false>
__global__ void __launch_bounds__((LoopCfg<NX, NY, ER, EC>::TH), (LoopCfg<NX, NY, ER, EC>::WAVES))
k_loop(LoopCall) {
  using C = LoopCfg<NX, NY, ER, EC>;
  constexpr bool HKEEP = C::E == 4;
  constexpr int SLOTS = C::SLOTS, QR = C::QR, TR = C::TR, TC = C::TC;
  using RL = SwzLayout<4>;
  using CL = std::conditional_t<C::SWZ, SwzLayout<4 - ilog2c(C::SWZ ? C::LC : 1)>,
                                PadLayout<Base<NY, EC>::COL_SH>>;
  __shared__ __align__(16) float2 lds[C::LDS];
  __shared__ unsigned long long sh_rec;
  __shared__ unsigned sh_u[2];
  __shared__ float sh_f[2];
  constexpr int HALF = (NX < NY ? NX : NY) / 2;  // largest distance from the border, plus one
  __shared__ float sh_taper[HALF];
  __shared__ float sh_acc[HKEEP ? 1 : C::PTS];  // a complete team's running |u|^2 sums, [element][thread]
  const int tid0 = threadIdx.x;

  LoopTeam<C, LOST> tm;
  if (!tm.join(sh_u)) return;
  {
    const int w = min(loop_args().ra.absorb, HALF);
    for (int d = tid0; d < w; d += C::TH) sh_taper[d] = taper_factor(d, loop_args().ra.absorb);
    __syncthreads();
  }

  // state that a member of a complete team keeps over the steps of a field
  int held = -1;
  float2 hk[EC];      // propagator (4-point columns)
  float accv[QR][ER];     // running |u|^2 sums (4-point threads; 8-point ones keep them in LDS)
  float wd[EC];       // weight slice (weighted mean)
  float2 v[EC];       // columns (kept from phase A to phase B of the weighted mean)
  float dpre[QR][ER];     // dn of the next row phase (real dn)

  while (tm.next(&sh_rec)) {
    const int field = tm.field, me = tm.me, M = tm.M;
    const int z0 = tm.z0, z1 = tm.z1;
    const bool whole = tm.whole, last = tm.last;
    auto load_h = [&](float2 (&hv)[EC], const ColArgs& ca, int s, int tid) __attribute__((always_inline)) {
      const int cl = tid % C::LC, tc = tid / C::LC;
      const int x = s * C::LC + cl;
      const int qx = min(x, NX - x);
#pragma unroll
      for (int m = 0; m < EC; ++m) {
        const int ky = tc + m * TC;
        hv[m] = ca.H[min(ky, NY - ky) * NX + qx];
      }
    };
    auto load_w = [&](const ColArgs& ca, int s, int tid) __attribute__((always_inline)) {
      const int cl = tid % C::LC, tc = tid / C::LC;
#pragma unroll
      for (int m = 0; m < EC; ++m)
        wd[m] = ca.dn ? load_dn(ca.dn, ca.dn_kind,
                                (size_t)field * ca.dn_bstride +
                                    (size_t)((tc + m * TC) * NX + s * C::LC + cl)).x
                      : 0.f;
    };
    // element index in ra.dn of row q of slot s at the thread's first point
    auto dn_at = [&](const RowArgs& ra, int s, int q, int z, int line, int tr) __attribute__((always_inline)) {
      return (size_t)tm.volume * ra.dn_bstride + (size_t)z * (NX * NY) +
             (size_t)((s * C::LR + q * C::LRP + line) * NX + tr);
    };
    auto load_dpre = [&](const RowArgs& ra, int s, int z, int line, int tr) __attribute__((always_inline)) {
      if (ra.dn_kind == BPMH_DN_F32) {
#pragma unroll
        for (int q = 0; q < QR; ++q) {
          const float* p = (const float*)ra.dn + dn_at(ra, s, q, z, line, tr);
#pragma unroll
          for (int m = 0; m < ER; ++m) dpre[q][m] = p[m * TR];
        }
      } else if (ra.dn_kind == BPMH_DN_F16) {
#pragma unroll
        for (int q = 0; q < QR; ++q) {
          const __half* p = (const __half*)ra.dn + dn_at(ra, s, q, z, line, tr);
#pragma unroll
          for (int m = 0; m < ER; ++m) dpre[q][m] = __half2float(p[m * TR]);
        }
      }
    };
    auto load_cols = [&](float2 (&v)[EC], __amdgpu_buffer_rsrc_t rp, int s, int cl, int tc) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < EC; ++m)
        v[m] = loop_ld(rp, (tc * NX + cl) * 8, (s * C::LC + m * TC * NX) * 8);
    };
    auto store_cols = [&](const float2 (&v)[EC], __amdgpu_buffer_rsrc_t rp, int s, int cl, int tc) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < EC; ++m)
        loop_st(rp, (tc * NX + cl) * 8, (s * C::LC + m * TC * NX) * 8, v[m]);
    };
    auto record = [&](const float2 (&v)[EC], const LoopCall& call, int s, int z, int cl, int tc) __attribute__((always_inline)) {
      // U = F u of this step, for the adjoint
      float2* ko = call.ca.kout + (size_t)field * call.ca.kout_bstride +
                   (size_t)(z - 1) * call.la.kout_zstride + s * C::LC + cl;
#pragma unroll
      for (int m = 0; m < EC; ++m) ko[(tc + m * TC) * NX] = v[m];
    };

    if (whole && held != field) {
      const LoopCall& call = loop_args();
      const int tid = loop_opaque(tid0);
      if (MODE == BPMH_MEAN_IGNORE && HKEEP) load_h(hk, call.ca, me, tid);
      if (MODE == BPMH_MEAN_WEIGHTED && HKEEP) load_w(call.ca, me, tid);
      if (call.ra.acc && z0 > 0) {
        const __amdgpu_buffer_rsrc_t rac =
            loop_rsrc(call.ra.acc + (size_t)field * NX * NY, NX * NY * 4);
#pragma unroll
        for (int q = 0; q < QR; ++q)
#pragma unroll
          for (int m = 0; m < ER; ++m)
            (HKEEP ? accv[q][m] : sh_acc[(q * ER + m) * C::TH + tid]) =
                loop_ld1(rac, ((tid / TR) * NX + tid % TR) * 4,
                         ((me * C::LR + q * C::LRP) * NX + m * TR) * 4);
      }
      held = field;
    }

    auto row_phase = [&](int z, bool first) __attribute__((always_inline)) {
      const RowArgs& ra = loop_args().ra;
      Twiddles<NX, ER> tw;
      tw.load(loop_opaque(tid0) % TR, ra.tw);
      tm.enter(first, sh_u);
      if (tm.dead) return;
      const __amdgpu_buffer_rsrc_t rp = loop_rsrc(ra.plane + (size_t)field * NX * NY, NX * NY * 8);
      const bool screened = z > 0 && ra.dn_kind != BPMH_DN_NONE;
      const bool end = last && z == z1;  // the field's last plane: no forward transform
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int line = tid / TR, tr = tid - line * TR;
        const int off = (line * NX + tr) * 8;
        float2 u[QR][ER];
#pragma unroll
        for (int q = 0; q < QR; ++q)
#pragma unroll
          for (int m = 0; m < ER; ++m)
            u[q][m] = loop_ld(rp, off, ((s * C::LR + q * C::LRP) * NX + m * TR) * 8);
        if (screened && !whole) load_dpre(ra, s, z, line, tr);
        float dn0 = 0.f;
        if (MODE == BPMH_MEAN_SIMPLE && screened) dn0 = ra.dn0_arr[z];
        if (MODE == BPMH_MEAN_WEIGHTED && screened) dn0 = loop_ld1(loop_rsrc(ra.dn0_item + field, 4), 0, 0);
#pragma unroll
        for (int q = 0; q < QR; ++q) {
          const int y = s * C::LR + q * C::LRP + line;
          float2* const ln = lds + (q * C::LRP + line) * C::ROW_LINE;
          const int plane_off = y * NX;
          if (z > 0) {
            line_fft<NX, ER, true, RL, C::WAVE>(u[q], ln, tr, tw);
#pragma unroll
            for (int m = 0; m < ER; ++m) u[q][m] = c_scale(u[q][m], ra.inv_n);
            if (screened)
              loop_screen<NX, ER, C::WAVE>(ra, NY, y, tr, dn0, dpre[q],
                                           (const float2*)ra.dn + dn_at(ra, s, q, z, line, tr), ln,
                                           sh_taper, u[q]);
          }
          row_outputs<NX, ER>(ra, z, field, plane_off, tr, u[q]);
          if (ra.acc) {
            const __amdgpu_buffer_rsrc_t rac = loop_rsrc(ra.acc + (size_t)field * NX * NY, NX * NY * 4);
#pragma unroll
            for (int m = 0; m < ER; ++m) {
              float& mine = HKEEP ? accv[q][m] : sh_acc[(q * ER + m) * C::TH + tid];
              const int at4 = (plane_off + tr) * 4;
              float sum = u[q][m].x * u[q][m].x + u[q][m].y * u[q][m].y;
              if (z > 0) sum = (whole ? mine : loop_ld1(rac, at4, m * TR * 4)) + sum;
              if (whole) mine = sum;
              if (!whole || end)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum), rac, at4, m * TR * 4, 0);
            }
          }
          if (!end) line_fft<NX, ER, false, RL, C::WAVE>(u[q], ln, tr, tw);
#pragma unroll
          for (int m = 0; m < ER; ++m)
            loop_st(rp, off, ((s * C::LR + q * C::LRP) * NX + m * TR) * 8, u[q][m]);
        }
        tm.leave(s);
      }
      tm.at += 1;
    };

    // static or per-plane propagator: FFT_y, H, IFFT_y
    auto col_phase = [&](int z, bool first) __attribute__((always_inline)) {
      float2 v[EC], hv[EC];
      const LoopCall& call = loop_args();
      const ColArgs& ca = call.ca;
      Twiddles<NY, EC> tw;
      tw.load(loop_opaque(tid0) / C::LC, ca.tw);
      tm.enter(first, sh_u);
      if (tm.dead) return;
      const __amdgpu_buffer_rsrc_t rp = loop_rsrc(ca.plane + (size_t)field * NX * NY, NX * NY * 8);
      const bool screened = call.ra.dn_kind != BPMH_DN_NONE;
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int cl = tid % C::LC, tc = tid / C::LC;
        float2* const ln = lds + cl * C::COL_LINE;
        load_cols(v, rp, s, cl, tc);
        if (whole) {
          if (screened) load_dpre(call.ra, s, z, tid / TR, tid % TR);
        }
        if (MODE == BPMH_MEAN_IGNORE && !(HKEEP && whole)) load_h(hv, ca, s, tid);
        line_fft<NY, EC, false, CL>(v, ln, tc, tw);
        if (ca.kout) record(v, call, s, z, cl, tc);
        const int x = s * C::LC + cl;
        if constexpr (MODE == BPMH_MEAN_IGNORE) {
#pragma unroll
          for (int m = 0; m < EC; ++m) v[m] = c_mul_fused(v[m], HKEEP && whole ? hk[m] : hv[m]);
        } else {
          col_h_fly<NY, EC>(kcomp2_f32(x, NX, ca.dx), n_term_f32(ca.n_eff[z], ca.k0), ca.dy, ca.dz,
                            tc, ln, hv);
#pragma unroll
          for (int m = 0; m < EC; ++m) v[m] = c_mul_fused(v[m], hv[m]);
        }
        if (ca.sw) col_scatter<NY, EC>(ca, z, field, x, tc, ln, v);
        line_fft<NY, EC, true, CL>(v, ln, tc, tw);
        store_cols(v, rp, s, cl, tc);
        tm.leave(s);
      }
      tm.at += 1;
    };

    // weighted mean: A (FFT_y, per-column sums), B (dn0, H(n0 + dn0), IFFT_y);
    // a complete team's columns stay in registers between the two
    auto weighted_phases = [&](int z, bool first) __attribute__((always_inline)) {
      const LoopCall& call = loop_args();
      const ColArgs& ca = call.ca;
      Twiddles<NY, EC> tw;
      tw.load(loop_opaque(tid0) / C::LC, ca.tw);
      tm.enter(first, sh_u);
      if (tm.dead) return;
      const __amdgpu_buffer_rsrc_t rp = loop_rsrc(ca.plane + (size_t)field * NX * NY, NX * NY * 8);
      const bool screened = call.ra.dn_kind != BPMH_DN_NONE;
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int cl = tid % C::LC, tc = tid / C::LC;
        float2* const ln = lds + cl * C::COL_LINE;
        load_cols(v, rp, s, cl, tc);
        if (whole) {
          if (screened) load_dpre(call.ra, s, z, tid / TR, tid % TR);
        }
        if (!(HKEEP && whole)) load_w(ca, s, tid);
        line_fft<NY, EC, false, CL>(v, ln, tc, tw);
        const float2 sums = col_weight_sums<NY, EC>(v, wd, tc, ln);
        if (tc == 0) ca.wpart[(size_t)field * NX + s * C::LC + cl] = sums;
        if (ca.kout) record(v, call, s, z, cl, tc);
        if (!whole) store_cols(v, rp, s, cl, tc);
        tm.leave(s);
      }
      tm.at += 1;
      tm.enter(false, sh_u);
      if (tm.dead) return;
      // dn0 in the fixed order of weighted_dn0_group
      if (tid0 < 64) {
        const __amdgpu_buffer_rsrc_t rw = loop_rsrc(ca.wpart + (size_t)field * NX, NX * 8);
        float sd = 0.f, su = 0.f;
#pragma unroll
        for (int p = 0; p < NX; p += 64) {
          const float2 w = loop_ld(rw, loop_opaque(tid0) * 8, p * 8);
          sd += w.x;
          su += w.y;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          sd += __shfl_xor(sd, o, 64);
          su += __shfl_xor(su, o, 64);
        }
        if (tid0 == 0) {
          sh_f[0] = sd / su;
          sh_f[1] = su;
        }
      }
      __syncthreads();
      const float dn0 = sh_f[0];
      const float an = n_term_f32(f_add(ca.n0, dn0), ca.k0);
      for (int s = me; s < SLOTS; s += M) {
        const int tid = loop_opaque(tid0);
        const int cl = tid % C::LC, tc = tid / C::LC;
        float2* const ln = lds + cl * C::COL_LINE;
        if (s == 0 && tid == 0) {
          ca.dn0_item[field] = dn0;
          if (ca.rec_c) {
            ca.rec_c[(size_t)(z - 1) * call.la.batch + field] = dn0;
            ca.rec_w[(size_t)(z - 1) * call.la.batch + field] = sh_f[1];
          }
        }
        if (!whole) load_cols(v, rp, s, cl, tc);
        const int x = s * C::LC + cl;
        float2 h[EC];
        col_h_fly<NY, EC>(kcomp2_f32(x, NX, ca.dx), an, ca.dy, ca.dz, tc, ln, h);
#pragma unroll
        for (int m = 0; m < EC; ++m) v[m] = c_mul_fused(v[m], h[m]);
        if (ca.sw) col_scatter<NY, EC>(ca, z, field, x, tc, ln, v);
        line_fft<NY, EC, true, CL>(v, ln, tc, tw);
        store_cols(v, rp, s, cl, tc);
        tm.leave(s);
      }
      tm.at += 1;
    };

    // plane 0 has a row phase alone (outputs of u0, FFT_x)
    const int zb = z0 == 0 ? 0 : z0 + 1;
    for (int z = zb; z <= z1 && !tm.dead; ++z) {
      if (z > 0) {
        if constexpr (MODE == BPMH_MEAN_WEIGHTED) weighted_phases(z, z == zb);
        else col_phase(z, z == zb);
      }
      if (!tm.dead) row_phase(z, z == 0);
    }
    if (tm.dead) {
      tm.give_up();
      return;
    }
  }
}

// Launch for one NX (instantiated in its own source file); false when the
// (ny, er, ec) shape is not built.
typedef bool (*loop_launch_fn)(int ny, int er, int ec, int mode, const LoopCall&, int groups, hipStream_t);
bool bpmh_loop_nx64(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_nx128(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_nx256(int, int, int, int, const LoopCall&, int, hipStream_t);
bool bpmh_loop_nx512(int, int, int, int, const LoopCall&, int, hipStream_t);

template <int NX, int NY, int ER, int EC, bool LOST>
static bool loop_launch_m(int mode, const LoopCall& c, int groups, hipStream_t s) {
  const dim3 g((unsigned)groups), b(LoopCfg<NX, NY, ER, EC>::TH);
  switch (mode) {
    case BPMH_MEAN_IGNORE:
      hipLaunchKernelGGL((k_loop<NX, NY, ER, EC, BPMH_MEAN_IGNORE, LOST>), g, b, 0, s, c);
      return true;
    case BPMH_MEAN_SIMPLE:
      hipLaunchKernelGGL((k_loop<NX, NY, ER, EC, BPMH_MEAN_SIMPLE, LOST>), g, b, 0, s, c);
      return true;
    case BPMH_MEAN_WEIGHTED:
      hipLaunchKernelGGL((k_loop<NX, NY, ER, EC, BPMH_MEAN_WEIGHTED, LOST>), g, b, 0, s, c);
      return true;
  }
  return false;
}

// the kernels whose waits give up are built for one shape
template <int NX, int NY, int ER, int EC>
constexpr bool kLoopLost = NX == 64 && NY == 64 && ER == 4 && EC == 4;

template <int NX, int NY, int ER, int EC>
static bool loop_launch_e(int mode, const LoopCall& c, int groups, hipStream_t s) {
  if (!c.la.lost) return loop_launch_m<NX, NY, ER, EC, false>(mode, c, groups, s);
  if constexpr (kLoopLost<NX, NY, ER, EC>) return loop_launch_m<NX, NY, ER, EC, true>(mode, c, groups, s);
  return false;
}

template <int NX, int NY>
static bool loop_launch_n(int er, int ec, int mode, const LoopCall& c, int groups,
                          hipStream_t s) {
  if (er == 4 && ec == 4) return loop_launch_e<NX, NY, 4, 4>(mode, c, groups, s);
  if (er == 4 && ec == 8) return loop_launch_e<NX, NY, 4, 8>(mode, c, groups, s);
  if (er == 8 && ec == 8) return loop_launch_e<NX, NY, 8, 8>(mode, c, groups, s);
  return false;
}

template <int NX>
static bool loop_launch_nx(int ny, int er, int ec, int mode, const LoopCall& c, int groups,
                           hipStream_t s) {
  switch (ny) {
    case 64: return loop_launch_n<NX, 64>(er, ec, mode, c, groups, s);
    case 128: return loop_launch_n<NX, 128>(er, ec, mode, c, groups, s);
    case 256: return loop_launch_n<NX, 256>(er, ec, mode, c, groups, s);
    case 512: return loop_launch_n<NX, 512>(er, ec, mode, c, groups, s);
  }
  return false;
}
