// All Metropolis-Hastings jumps of a step in one launch.
//
// A chain's next proposal depends on its own last accept decision alone (and,
// planar FE, on the batch acceptance of the jump before), so a workgroup keeps
// up to kJumpLanes chains in LDS and takes them through every jump:
//   1. lane k of wavefront 0 proposes for chain k and leaves its packed point
//      in LDS;
//   2. the wavefronts sum the chains' fields over the particles, the lanes
//      holding particles and the chains' points read as wavefront-wide
//      values, so a particle read once serves several chains; wavefront 0
//      first forms what the chains' targets take from the points alone;
//   3. lane k of wavefront 0 forms the field of chain k and decides.
// Only the planar FE width couples workgroups: each adds its accept and
// reject counts of a jump to a counter and, before its next proposals, waits
// for the counter to hold every workgroup's (relaxed atomics on one word: the
// counts are all that passes between workgroups, so no cache is written
// back).  Simulations, and the other emission modes' workgroups, run at their
// own pace.
//
// What bounds a jump of a few hundred chains is latency: its proposal, field
// and accept in two launches took about 16 us for 0.2 us of arithmetic.  Whole
// steps, two launches per jump -> one launch per step: planar FE mixed (600
// chains, 1000 electrons) 13.3 -> 6.0 ms, FP64 38.6 -> 4.4 ms; tip FE mixed (2200
// chains) 5.4 -> 3.9 ms; thermal-field mixed 5.5 -> 4.8 ms; 64 diodes of a pool
// mixed 14.0 -> 12.2 ms, FP64 38.7 -> 26.6 ms.
//
// Every workgroup of a simulation has to be resident for the wait to end.  A
// launch's workgroups start in order and no simulation has more than the device
// holds, so the earliest unfinished simulation always is.  The host (run_jumps)
// also sees to it that none waits long for its last workgroup's place: a launch
// fits the device, or small simulations follow large ones in the places that
// become free (uneven pools), or each jump is a launch (spin = 0), where the end of
// the launch takes the place of the wait.  Another context's work can still hold
// the CUs, so the wait is bounded: past its bound the workgroup raises `stop` and
// leaves; results go to arrays of their own (`out`), and the host repeats the
// step's jumps with a launch per jump, with the same results.  Once the first
// jump's counts are in, every workgroup is resident, so two contexts that keep each
// other's workgroups out find that out in the first wait; where the launch fits
// that is short (kFirstTicks and eight times the workgroup's own first jump: the
// workgroups of a simulation differ by one chain, and by their CU's other load).
//
// The sums' order depends on the simulation's particle count and the kind of
// context alone: with S slices, lane l of slice w takes particles
// (S r + w) 64 + l for r = 0, 1, ..., the 64 lane sums are added in a fixed tree
// and the slices' in order.  How many chains share a workgroup, and which
// wavefront takes which slice and chains, does not enter, so a simulation
// gives the same results alone and in any pool.  Forms (JumpForm): a lone
// simulation takes workgroups of four wavefronts, a slice each, over many
// CUs, or, with many particles, of sixteen wavefronts and slices, which hide
// the particles' loads; a pool workgroups of eight wavefronts that share four
// slices, two of them on a CU, so that one's decisions overlap the other's sums.
// FP64: the canonical order (partials of 256 particles, each in sequence, added in
// order): the lanes form the terms in parallel, LDS holds them, and a lane per
// (chain, chunk) adds its 256 in sequence.
#pragma once

namespace rd {

constexpr int kJumpLanes = 64;                    // most chains per workgroup
constexpr long long kSpinTicks = 25000000;        // 0.25 s of the 100 MHz wall clock
constexpr long long kFirstTicks = 200000;         // 2 ms
constexpr int kSubGroup = 32;                     // workgroups per first-level counter

// Wavefronts of a workgroup, slices of the particles, wavefronts per SIMD the
// kernel is compiled for, particles kept in LDS for all jumps of the launch
// (cathode sums; as many as leave room for that many workgroups on a CU).
template <int W, int S, int O, int H>
struct JumpForm {
  static constexpr int kWaves = W, kSlices = S, kOccupancy = O, kHeld = H, kRound = 64 * S;
};
// Measured: four-wavefront workgroups serve a lone simulation's few chains
// best, but left a pool of 64 diodes slower than a launch per jump (two
// eight-wavefront workgroups to a CU: 1.15 to 1.5 times faster); lone with
// 4000 electrons and more, each CU has few workgroups and the sixteen
// wavefronts hide the particles' loads.
using LoneForm = JumpForm<4, 4, 3, 1536>;
using LargeForm = JumpForm<16, 16, 4, 1024>;
using PoolForm = JumpForm<8, 4, 4, 2560>;
constexpr int kJumpLarge = 4096;  // particles from which a lone simulation takes LargeForm

struct JumpArgs {
  const double *X, *Y, *Z, *Q;    // FP64 sources
  const float4 *HI, *LO;          // packed sources (mixed)
  const double2* SRX;             // (x, y) nm (mixed, cathode surface)
  const float2* SRZ;              // (z, q z) nm
  const double *ru1, *ru2, *rlr;  // per jump and chain: unit normals, log-uniform ([it-1][C])
  unsigned long long* cnt;        // acceptance counters (jump_counter)
  double* width;                  // per entry: kWidthSlots values
  int* stop;                      // raised by a wait that gave up
  int C;                          // chains in all
  int it0, it1;                   // jumps it0 .. it1 - 1 of this launch
  int spin;                       // 1: all jumps in this launch; 0: a launch per jump
  long long first, later;         // bounds of the waits after jump 1 and later (ticks)
};

// Per entry: the width and rate of the jumps of either parity (a launch per
// jump), then the step's final width, rate and last counts.
constexpr int kWidthSlots = 8;

// Counter words of one jump: the total (arrivals << 48 | accepted << 24 |
// rejected; without the in-kernel wait: accepted, rejected) and, for more
// than kSubGroup workgroups, one word per kSubGroup of them, so that at most
// that many atomics meet in a word (3.9 us a round for 256 workgroups on one
// word, 1.1 us for 36).
__host__ __device__ inline int jump_words(int groups) {
  return 2 + (groups > kSubGroup ? (groups + kSubGroup - 1) / kSubGroup : 0);
}

__device__ __forceinline__ void counts_arrive(unsigned long long* w, int groups, int grp, int spin,
                                              int na, int nr) {
  if (!spin) {
    __hip_atomic_fetch_add(w, (unsigned long long)na, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(w + 1, (unsigned long long)nr, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  unsigned long long v = (1ull << 48) | ((unsigned long long)na << 24) | (unsigned long long)nr;
  if (groups > kSubGroup) {
    const int sub = grp / kSubGroup;
    const int want = min(kSubGroup, groups - sub * kSubGroup);
    v += __hip_atomic_fetch_add(w + 2 + sub, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((int)(v >> 48) != want) return;  // the last of the sub-group passes its sum on
  }
  __hip_atomic_fetch_add(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The counts of a jump once every workgroup has added its own; false: gave up.
__device__ __forceinline__ bool counts_wait(unsigned long long* w, int groups, int spin, int* stop,
                                            long long ticks, int& na, int& nr) {
  if (!spin) {
    na = (int)__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    nr = (int)__hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  const long long t0 = wall_clock64();
  unsigned long long v;
  int k = 0;
  while (((v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 48) !=
         (unsigned long long)groups) {
    // the others leave with the first workgroup that gives up
    if ((++k & 15) == 0 && __hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return false;
    if (wall_clock64() - t0 > ticks) {
      __hip_atomic_store(stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  na = (int)((v >> 24) & 0xffffff);
  nr = (int)(v & 0xffffff);
  return true;
}

// The chains of a workgroup and their proposals, in LDS: lane k of wavefront 0
// has them in registers only while it proposes or decides, so that the field
// sums have the registers.
struct ChainStore {
  double d[14][kJumpLanes];
  int i[4][kJumpLanes];
};

// One chain.
struct Chain {
  int ok = 0, acc = 0, rej = 0;
  double cx = 0, cy = 0, F = 0, sup = 0, ox = 0, oy = 0, oz = 0;
  __device__ __forceinline__ void load(const Chains& h, int c) {
    ok = h.ok[c];
    acc = h.acc[c];
    rej = h.rej[c];
    cx = h.cx[c];
    cy = h.cy[c];
    F = h.F[c];
    sup = h.sup[c];
    ox = h.ox[c];
    oy = h.oy[c];
    oz = h.oz[c];
  }
  __device__ __forceinline__ void store(const Chains& h, int c) const {
    h.acc[c] = acc;
    h.rej[c] = rej;
    h.cx[c] = cx;
    h.cy[c] = cy;
    h.F[c] = F;
    h.sup[c] = sup;
    h.ox[c] = ox;
    h.oy[c] = oy;
    h.oz[c] = oz;
  }
  __device__ __forceinline__ void put(ChainStore& m, int k) const {
    m.d[0][k] = cx;
    m.d[1][k] = cy;
    m.d[2][k] = F;
    m.d[3][k] = sup;
    m.d[4][k] = ox;
    m.d[5][k] = oy;
    m.d[6][k] = oz;
    m.i[0][k] = ok;
    m.i[1][k] = acc;
    m.i[2][k] = rej;
  }
  __device__ __forceinline__ void get(const ChainStore& m, int k) {
    cx = m.d[0][k];
    cy = m.d[1][k];
    F = m.d[2][k];
    sup = m.d[3][k];
    ox = m.d[4][k];
    oy = m.d[5][k];
    oz = m.d[6][k];
    ok = m.i[0][k];
    acc = m.i[1][k];
    rej = m.i[2][k];
  }
  // Accept/reject of jump `it` at the proposal P with field (fx, fy, fz);
  // returns 1 accepted, 2 rejected.
  __device__ __forceinline__ int decide(const SimDesc& s, int it, int first, const Proposal& P,
                                        const SiteTerms& at, double lr, double fx, double fy,
                                        double fz) {
    const bool tip = s.mode == RD_EMIT_TIP_FE;
    bool take = false;
    if (!tip || P.valid == 1) {
      const double Fn = tip ? field_normal(s.g, P.x, P.y, fx, fy, fz) : fz;
      const bool bad = (s.mode == RD_EMIT_PLANAR_GTF) ? (Fn > 0.0) : (Fn >= 0.0);
      if (!bad) {
        const double sup_new = chain_target(s.mode, s.g.ic, s.dt_q0, s.T, Fn, at.w, at.lw);
        const double alpha = sup_new - sup;
        take = sup_new >= sup || lr <= alpha;
        if (take) {
          cx = P.a;
          cy = P.b;
          sup = sup_new;
          F = Fn;
          ox = P.x;
          oy = P.y;
          oz = P.z;
        }
      }
    }
    if (s.mode == RD_EMIT_PLANAR_GTF || (tip && it > first)) {
      acc += take;
      rej += !take;
    }
    return take ? 1 : 2;
  }
};

// The proposal width of a planar FE simulation over the jumps of a launch, in
// every lane of wavefront 0 (GTF and tip: the width of the start of the step).
struct JumpWidth {
  double mh, rate;
  int na = 0, nr = 0;
  int first, fe;
  unsigned long long* w;  // counter words of jump 1
  int words, groups, grp, spin;
  long long first_wait, later_wait;
  int* stop;
  double* slot;
  long long t0 = wall_clock64();

  __device__ __forceinline__ JumpWidth(const Ent& e, const SimDesc& s, const SimState& S,
                                       const JumpArgs& a, int grp_)
      : mh(S.MH_std), rate(S.a_rate), first(nint(s.ndim * 0.25)),
        fe(s.mode == RD_EMIT_PLANAR_FE), w(a.cnt + e.part_off), words(e.pslots), groups(e.segs),
        grp(grp_), spin(a.spin), first_wait(a.first), later_wait(a.later), stop(a.stop),
        slot(a.width + (size_t)kWidthSlots * e.acc_off) {
    if (fe && !spin && a.it0 >= 2) {  // as the launch of the jump before left it
      mh = slot[(a.it0 - 1) & 1];
      rate = slot[2 + ((a.it0 - 1) & 1)];
    }
  }
  // The width after jump `it`.
  __device__ __forceinline__ bool after(int it) {
    if (groups > 1 || !spin) {
      const long long ticks = it == 1 ? first_wait + 8 * (wall_clock64() - t0) : later_wait;
      if (!counts_wait(w + (size_t)(it - 1) * words, groups, spin, stop, ticks, na, nr))
        return false;
    }
    if ((it > first) && (na + nr > 0)) {
      rate = (double)na / (double)(na + nr);
      mh = fe_width_after(mh, it, first, na, nr);
    }
    return true;
  }
  // Before the proposals of jump `it`.
  __device__ __forceinline__ bool before(int it) {
    if (!fe) return true;
    if (it >= 2 && !after(it - 1)) return false;
    if (!spin && grp == 0 && threadIdx.x == 0) {
      slot[it & 1] = mh;
      slot[2 + (it & 1)] = rate;
    }
    return true;
  }
  // Counts of jump `it` from the decisions of wavefront 0 (0: no chain).
  __device__ __forceinline__ void count(int it, int d) {
    if (!fe) return;
    na = __popcll(__ballot(d == 1));
    nr = __popcll(__ballot(d == 2));
    if ((groups > 1 || !spin) && threadIdx.x == 0)
      counts_arrive(w + (size_t)(it - 1) * words, groups, grp, spin, na, nr);
  }
  // After the last jump: the step's final width, for k_mh_finish.
  __device__ __forceinline__ void last(int ndim) {
    if (!fe || grp != 0 || !after(ndim)) return;
    if (threadIdx.x == 0) {
      slot[4] = mh;
      slot[5] = rate;
      slot[6] = na;
      slot[7] = nr;
    }
  }
};

// The proposal of lane k's chain, left in the store.
__device__ __forceinline__ Proposal jump_proposal(const SimDesc& s, double mh, int it,
                                                  ChainStore& m, int k, double u1, double u2) {
  const Proposal P = mh_proposal(s, mh, it, m.i[0][k], m.d[0][k], m.d[1][k], m.d[4][k], m.d[5][k],
                                 m.d[6][k], u1, u2);
  m.d[7][k] = P.a;
  m.d[8][k] = P.b;
  m.d[9][k] = P.x;
  m.d[10][k] = P.y;
  m.d[11][k] = P.z;
  m.i[3][k] = P.valid;
  return P;
}
__device__ __forceinline__ Proposal stored_proposal(const ChainStore& m, int k) {
  return Proposal{m.d[7][k], m.d[8][k], m.d[9][k], m.d[10][k], m.d[11][k], m.i[3][k]};
}

__device__ __forceinline__ double uniform_d(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
__device__ __forceinline__ float uniform_f(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// v.x: v of lane l ^ o for the row steps of a sum (DPP).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// a + b after exchanging the odd halves of a with the even halves of b (halves
// of 32 or 16 lanes): the even halves then hold sums of a over both halves,
// the odd ones those of b.
template <int ROW>
__device__ __forceinline__ double swap_add(double a, double b) {
  const unsigned long long ba = (unsigned long long)__double_as_longlong(a);
  const unsigned long long bb = (unsigned long long)__double_as_longlong(b);
  auto sw = [](unsigned x, unsigned y) {
    return ROW == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                     : __builtin_amdgcn_permlane16_swap(x, y, false, false);
  };
  const auto l = sw((unsigned)ba, (unsigned)bb);
  const auto h = sw((unsigned)(ba >> 32), (unsigned)(bb >> 32));
  const double p = __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0]));
  const double q = __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
  return p + q;
}

// Sums of d[0 .. T) over the wavefront's 64 lanes (T a power of two up to 8),
// the tree of every sum the same for each T: lane l ends with the sum of
// d[wave_slot<T>(l)].  While several sums remain, each step exchanges halves
// and so adds two of them at once.
template <int T>
__device__ __forceinline__ int wave_slot(int l) {
  int s = 0, w = T;
  if (w > 1) {
    w >>= 1;
    s += (l & 32) ? w : 0;
  }
  if (w > 1) {
    w >>= 1;
    s += (l & 16) ? w : 0;
  }
  if (w > 1) {
    w >>= 1;
    s += (l & 8) ? w : 0;
  }
  return s;
}
template <int T>
__device__ __forceinline__ double wave_sums(double* d, int lane) {
  int w = T;
  if (w > 1) {
    w >>= 1;
#pragma unroll
    for (int u = 0; u < T / 2; ++u) d[u] = swap_add<32>(d[u], d[u + T / 2]);
  } else {
    d[0] = swap_add<32>(d[0], d[0]);
  }
  if (w > 1) {
    w >>= 1;
#pragma unroll
    for (int u = 0; u < T / 4; ++u) d[u] = swap_add<16>(d[u], d[u + T / 4]);
  } else {
    d[0] = swap_add<16>(d[0], d[0]);
  }
  double v;
  if (w > 1) {
    const bool up = lane & 8;
    const double keep = up ? d[1] : d[0], send = up ? d[0] : d[1];
    v = keep + dpp_f64<0x128>(send);  // row_ror:8
  } else {
    v = d[0] + dpp_f64<0x128>(d[0]);
  }
  v = v + dpp_f64<0x141>(v);  // row_half_mirror: lane 7 - l of each eight
  v = v + dpp_f64<0xB1>(v);   // quad_perm 1 0 3 2
  v = v + dpp_f64<0x4E>(v);   // quad_perm 2 3 0 1
  return v;
}

// What the target of lane k's proposal takes from its point, left in the store.
// A flat cathode of one work function keeps the terms of the first jump.
__device__ __forceinline__ void store_site(const SimDesc& s, const double* wf, ChainStore& m,
                                           int k, bool again) {
  if (again && s.mode != RD_EMIT_TIP_FE && s.wf_nx == 1 && s.wf_ny == 1) return;
  const SiteTerms t = site_terms(s, wf, m.d[7][k], m.d[8][k]);
  m.d[12][k] = t.w;
  m.d[13][k] = t.lw;
}
__device__ __forceinline__ SiteTerms stored_site(const ChainStore& m, int k) {
  return SiteTerms{m.d[12][k], m.d[13][k]};
}

// First chain of a simulation's workgroup: as many for each, but for one, so that
// no workgroup waits long for the others.
__device__ __forceinline__ int jump_first(const Ent& e, int grp) {
  return (int)((long long)grp * e.nch / e.segs);
}

template <class Form>
__device__ __forceinline__ int jump_rounds(int n) {
  return (n + Form::kRound - 1) / Form::kRound;
}

// ---- mixed precision ----------------------------------------------------------

template <class Form>
struct HeldSrc {
  double2 xy[Form::kHeld];
  float2 zq[Form::kHeld];
};

// N_ic_max = 0 (planar, image charge on): sums of q z / r^3 at T chains' points
// over this lane's particles of slice w; FP32 blocks of at most kSurfBlock
// terms of one sign (see kSurfBlock), block sums in FP64.  The offsets are
// FP64 differences rounded to FP32: two instructions where the difference of
// two-part FP32 coordinates takes three, and exact before the rounding.  HELD:
// the particles are in `own`.
template <class Form, int T, bool HELD>
__device__ __forceinline__ void jump_surf0(const HeldSrc<Form>& own, const double2* srx,
                                           const float2* srz, int n, int w, int lane,
                                           const double2* tgt, double (&d)[T]) {
  double tx[T], ty[T];
  float acc[T];
#pragma unroll
  for (int u = 0; u < T; ++u) {
    tx[u] = uniform_d(tgt[u].x);
    ty[u] = uniform_d(tgt[u].y);
    acc[u] = 0.0f;
    d[u] = 0.0;
  }
  // z^2 goes into the fused sum unrounded: a product of its own would save an
  // instruction and bias all of a source's terms alike
  auto term = [&](const double2 xy, float z, float qz) {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const float dx = (float)(tx[u] - xy.x), dy = (float)(ty[u] - xy.y);
      const float ri = rsq(__builtin_fmaf(z, z, lateral2(dx, dy)));
      acc[u] = __builtin_fmaf(qz, ri * ri * ri, acc[u]);
    }
  };
  auto flush = [&]() {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      d[u] += (double)acc[u];
      acc[u] = 0.0f;
    }
  };
  const int R = jump_rounds<Form>(n);
  if (HELD) {  // padded to whole rounds
#pragma unroll 1
    for (int r = 0; r < R; ++r) {
      const int j = r * Form::kRound + w * 64 + lane;
      const float2 zq = own.zq[j];
      term(own.xy[j], zq.x, zq.y);
      if ((r & (kSurfBlock - 1)) == kSurfBlock - 1) flush();
    }
  } else {
    // rounds a batch; the next batch's loads are in flight during a batch, so
    // few chains (little arithmetic per load) take larger batches
    constexpr int B = T >= 8 ? 1 : 4;
    static_assert(kSurfBlock % B == 0, "a block is a whole number of batches");
    double2 xn[B];
    float2 zn[B];
    auto load = [&](int r) {  // (used as loaded: a select here would wait for the data)
#pragma unroll
      for (int k = 0; k < B; ++k) {
        const int j = (r + k) * Form::kRound + w * 64 + lane;
        const int i = j < n ? j : 0;
        xn[k] = srx[i];
        zn[k] = srz[i];
      }
    };
    if (R > 0) load(0);
#pragma unroll 1
    for (int r = 0; r < R; r += B) {
      double2 xc[B];
      float2 zc[B];
#pragma unroll
      for (int k = 0; k < B; ++k) {
        xc[k] = xn[k];
        zc[k] = zn[k];
      }
      if (r + B < R) load(r + B);
#pragma unroll
      for (int k = 0; k < B; ++k)
        if (r + k < R)
          term(xc[k], zc[k].x,
               (r + k) * Form::kRound + w * 64 + lane < n ? zc[k].y : 0.0f);
      if ((r & (kSurfBlock - B)) == kSurfBlock - B) flush();
    }
  }
  flush();
}

// Other planar forms, on the cathode with N_ic_max > 0 (-1/2 of the field sum,
// the series of surface_far32) or without image charges: FP32 terms, FP64 sums.  The next
// round's particle is in flight during a round, and the chains go through the
// image series side by side: they share the partners' heights, and their
// dependent operations overlap (a partner is a square root and three products in
// sequence).  Large simulations take eight chains a pass, which halves the reads
// of the particles.
template <class Form, int T, bool IC>
__device__ __forceinline__ void jump_planar(int nic, float dnm, const float4* hi,
                                            const float4* lo, int n, int w, int lane,
                                            const double2* tgt, double (&d)[T]) {
  float hx[T], hy[T], lx[T], ly[T];
#pragma unroll
  for (int u = 0; u < T; ++u) {
    split(tgt[u].x, hx[u], lx[u]);
    split(tgt[u].y, hy[u], ly[u]);
    hx[u] = uniform_f(hx[u]);
    hy[u] = uniform_f(hy[u]);
    lx[u] = uniform_f(lx[u]);
    ly[u] = uniform_f(ly[u]);
    d[u] = 0.0;
  }
  const int R = jump_rounds<Form>(n);
  float4 hn = make_float4(0, 0, 0, 0), ln = hn;
  if (w * 64 + lane < n) {
    hn = hi[w * 64 + lane];
    ln = lo[w * 64 + lane];
  }
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    const float4 h2 = hn, l2 = ln;
    const int j = (r + 1) * Form::kRound + w * 64 + lane;
    if (r + 1 < R) {  // the next round's particle
      const int i = j < n ? j : 0;
      hn = hi[i];
      ln = lo[i];
    }
    const float q = j - Form::kRound < n ? h2.w : 0.0f;  // padding has no charge
    float s[T], f[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const float dx = (hx[u] - h2.x) + (lx[u] - l2.x);
      const float dy = (hy[u] - h2.y) + (ly[u] - l2.y);
      s[u] = lateral2(dx, dy);
    }
    if (IC) {  // surface_far32 of every chain
#pragma unroll
      for (int u = 0; u < T; ++u) {
        const float ri = rsq(__builtin_fmaf(h2.z, h2.z, s[u]));
        f[u] = h2.z * (ri * ri * ri);
      }
      const float two_d = dnm + dnm;
      float up = h2.z, um = -(l2.w + dnm);
#pragma unroll 1
      for (int k = 1; k <= nic; ++k) {
        up += two_d;
#pragma unroll
        for (int u = 0; u < T; ++u) {
          float ri = rsq(__builtin_fmaf(up, up, s[u]));
          f[u] = __builtin_fmaf(up, ri * ri * ri, f[u]);
          ri = rsq(__builtin_fmaf(um, um, s[u]));
          f[u] = __builtin_fmaf(um, ri * ri * ri, f[u]);
        }
        um -= two_d;
      }
    } else {
      const float dz = -h2.z - l2.z;
#pragma unroll
      for (int u = 0; u < T; ++u) {
        const float ri = rsq(__builtin_fmaf(dz, dz, s[u]));
        f[u] = dz * (ri * ri * ri);
      }
    }
#pragma unroll
    for (int u = 0; u < T; ++u) d[u] += (double)(q * f[u]);
  }
}

// Tip: the three field sums at T chains' points (tip_pair32_target).
template <class Form, int T>
__device__ __forceinline__ void jump_tip(float kt, const float4* hi, const float4* lo, int n,
                                         int w, int lane, const float4* tgt, int tb,
                                         double (&dx)[T], double (&dy)[T], double (&dz)[T]) {
  float4 h1[T], l1[T], ih[T], il[T];
  auto uni = [](const float4 p) {
    return make_float4(uniform_f(p.x), uniform_f(p.y), uniform_f(p.z), uniform_f(p.w));
  };
#pragma unroll
  for (int u = 0; u < T; ++u) {
    h1[u] = uni(tgt[tb + u]);
    l1[u] = uni(tgt[kJumpLanes + tb + u]);
    ih[u] = uni(tgt[2 * kJumpLanes + tb + u]);
    il[u] = uni(tgt[3 * kJumpLanes + tb + u]);
    dx[u] = dy[u] = dz[u] = 0.0;
  }
  const int R = jump_rounds<Form>(n);
  float4 hn = make_float4(0, 0, 0, 0), ln = hn;
  if (w * 64 + lane < n) {
    hn = hi[w * 64 + lane];
    ln = lo[w * 64 + lane];
  }
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    float4 h2 = hn;
    const float4 l2 = ln;
    const int j = (r + 1) * Form::kRound + w * 64 + lane;
    if (r + 1 < R) {  // the next round's particle
      const int i = j < n ? j : 0;
      hn = hi[i];
      ln = lo[i];
    }
    h2.w = j - Form::kRound < n ? h2.w : 0.0f;  // padding has no charge
#pragma unroll
    for (int u = 0; u < T; ++u) {
      float cx, cy, cz;
      tip_pair32_target(h1[u], l1[u], ih[u], il[u], h2, l2, kt, cx, cy, cz);
      dx[u] += (double)cx;
      dy[u] += (double)cy;
      dz[u] += (double)cz;
    }
  }
}

// Calls pass(T, first chain) over chains [c0, c1), T at a time: TM, then fewer for
// the rest.  A rest of five or six takes TM = 8 with idle places where a term is
// cheap (its reads and set-up count), and 4 + 1 or 4 + 2 where the image series
// makes it dear (EXACT).
template <int TM, bool EXACT, class F>
__device__ __forceinline__ void jump_passes(int c0, int c1, F&& pass) {
  int tb = c0;
#pragma unroll 1
  for (; c1 - tb >= (TM == 8 ? (EXACT ? 7 : 5) : 3); tb += TM)
    pass(std::integral_constant<int, TM>{}, tb);
  if (TM == 8 && c1 - tb >= 3) {
    pass(std::integral_constant<int, 4>{}, tb);
    tb += 4;
  }
  if (c1 - tb >= 2) {
    pass(std::integral_constant<int, 2>{}, tb);
    tb += 2;
  }
  if (c1 > tb) pass(std::integral_constant<int, 1>{}, tb);
}

// SERIES: the planar forms of jump_planar, in a kernel of their own: neither's
// registers crowd the other's, and without the held particles the compute units
// hold more of its workgroups.
__host__ __device__ inline bool jump_series(const DevGeom& g) {
  return g.kind == RD_GEOM_PLANAR && !(g.ic && g.nic == 0);
}
template <int KIND, bool SERIES, class Form>
__global__ __launch_bounds__(64 * Form::kWaves, Form::kOccupancy) void k_mh_jumps32(
    const Ent* tab, int ne, const SimDesc* desc, const SimState* st, const double* wf, Chains in,
    Chains out, JumpArgs a) {
  constexpr int WAVES = Form::kWaves, kJumpSlices = Form::kSlices;
  constexpr bool kTip = KIND == RD_GEOM_TIP, kSurf0 = !kTip && !SERIES;
  __shared__ float4 tgt[kTip ? 4 : 1][kTip ? kJumpLanes : 1];
  __shared__ double2 tgt2[kTip ? 1 : kJumpLanes];  // planar: x, y (nm)
  __shared__ double red[kTip ? 3 : 1][kJumpSlices][kJumpLanes];
  __shared__ HeldSrc<Form> own[1];
  __shared__ int s_stop;
  __shared__ ChainStore store;
  const Ent e = tab[find_entry(tab, ne, blockIdx.x)];
  const SimDesc s = desc[e.slot];  // a copy: references would be read again after every barrier
  if (s.g.kind != KIND || jump_series(s.g) != SERIES) return;
  const DevGeom& g = s.g;
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int w = wv % kJumpSlices, group = wv / kJumpSlices;  // the wavefront's slice and chains
  constexpr int NG = WAVES / kJumpSlices;
  const int grp = blockIdx.x - e.wg0;
  const int k0 = jump_first(e, grp), nc = jump_first(e, grp + 1) - k0;
  const int share = (nc + NG - 1) / NG;  // chains [g0, g1) of the group
  const int g0 = min(nc, group * share), g1 = min(nc, g0 + share);
  const int c = e.cbase + k0 + lane;
  const bool mine = wv == 0 && lane < nc;  // this lane proposes and decides for a chain
  const int n = st[e.slot].n;
  const int it1 = min(a.it1, s.ndim + 1);
  if (mine) {
    Chain ch;
    ch.load(in, c);
    ch.put(store, lane);
  }
  JumpWidth width(e, s, st[e.slot], a, grp);
  if (t < kJumpLanes) {
    if (kTip)
      for (int q = 0; q < (kTip ? 4 : 1); ++q) tgt[q][kTip ? t : 0] = make_float4(0, 0, 0, 1);
    else
      tgt2[kTip ? 0 : t] = make_double2(0.0, 0.0);
  }
  if (t == 0) s_stop = 0;
  const float4* hi = a.HI + e.base;
  const float4* lo = a.LO + e.base;
  const double2* srx = a.SRX + e.base;
  const float2* srz = a.SRZ + e.base;
  const int ic = g.ic, nic = g.nic;
  const float dnm = 0.5f * (float)(2.0 * g.d * 1e9);
  const float kt = g.ic ? (float)g.ktip : 0.0f;
  // few particles stay in LDS for all jumps (padding: no charge)
  const int padded = jump_rounds<Form>(n) * Form::kRound;
  const bool held = kSurf0 && padded <= Form::kHeld;
  if (held)
    for (int j = t; j < padded; j += 64 * WAVES) {
      own[0].xy[j] = srx[j < n ? j : 0];
      const float2 zq = srz[j < n ? j : 0];
      own[0].zq[j] = make_float2(zq.x, j < n ? zq.y : 0.0f);
    }
  double u1 = 0, u2 = 0, lr = 0;
  auto draws = [&](int it) {
    const size_t o = (size_t)(it - 1) * a.C + c;
    u1 = a.ru1[o];
    u2 = a.ru2[o];
    lr = a.rlr[o];
  };
  if (mine && a.it0 < it1) draws(a.it0);
  double plr = 0;
  __syncthreads();
  for (int it = a.it0; it < it1; ++it) {
    if (wv == 0) {
      // proposals and decisions hold up every wavefront of the workgroup:
      // ahead of the field sums of other workgroups on the CU
      __builtin_amdgcn_s_setprio(3);
      if (!width.before(it)) s_stop = 1;
      if (mine) {
        const Proposal P = jump_proposal(s, width.mh, it, store, lane, u1, u2);
        if (kTip) {
          float4 h1, l1, ih1, il1;
          pack1(P.x, P.y, P.z, 0.0, g.d, h1, l1);
          pack_image(P.x, P.y, P.z, g.z0, g.R, ih1, il1);
          const int k = kTip ? lane : 0;
          tgt[0][k] = h1;
          tgt[kTip ? 1 : 0][k] = l1;
          tgt[kTip ? 2 : 0][k] = ih1;
          tgt[kTip ? 3 : 0][k] = il1;
        } else {
          tgt2[kTip ? 0 : lane] = make_double2(P.x * 1.0e9, P.y * 1.0e9);
        }
        plr = lr;
        if (it + 1 < it1) draws(it + 1);  // the next jump's, while this one's field is summed
      }
    }
    __syncthreads();
    if (s_stop) return;
    if (mine) store_site(s, wf, store, lane, it > a.it0);
    if (wv == 0) __builtin_amdgcn_s_setprio(0);
    if (kTip) {
      jump_passes<4, true>(g0, g1, [&](auto tt, int tb) {
        constexpr int T = decltype(tt)::value;
        double dx[T], dy[T], dz[T];
        jump_tip<Form, T>(kt, hi, lo, n, w, lane, &tgt[0][0], tb, dx, dy, dz);
        const double vx = wave_sums<T>(dx, lane), vy = wave_sums<T>(dy, lane),
                     vz = wave_sums<T>(dz, lane);
        const int k = tb + wave_slot<T>(lane);
        if ((lane & 7) == 0 && k < g1) {
          red[0][w][k] = vx;
          red[kTip ? 1 : 0][w][k] = vy;
          red[kTip ? 2 : 0][w][k] = vz;
        }
      });
    } else if (kSurf0) {
      jump_passes<8, SERIES>(g0, g1, [&](auto tt, int tb) {
        constexpr int T = decltype(tt)::value;
        double d[T];
        if (held)
          jump_surf0<Form, T, true>(own[0], srx, srz, n, w, lane, &tgt2[tb], d);
        else
          jump_surf0<Form, T, false>(own[0], srx, srz, n, w, lane, &tgt2[tb], d);
        const double v = wave_sums<T>(d, lane);
        const int k = tb + wave_slot<T>(lane);
        if ((lane & 7) == 0 && k < g1) red[0][w][k] = v;
      });
    } else {
      jump_passes<8, SERIES>(g0, g1, [&](auto tt, int tb) {
        constexpr int T = decltype(tt)::value;
        double d[T];
        if (ic)
          jump_planar<Form, T, true>(nic, dnm, hi, lo, n, w, lane, &tgt2[tb], d);
        else
          jump_planar<Form, T, false>(nic, dnm, hi, lo, n, w, lane, &tgt2[tb], d);
        const double v = wave_sums<T>(d, lane);
        const int k = tb + wave_slot<T>(lane);
        if ((lane & 7) == 0 && k < g1) red[0][w][k] = v;
      });
    }
    __syncthreads();
    if (wv == 0) {
      __builtin_amdgcn_s_setprio(3);
      int dec = 0;
      if (mine && store.i[0][lane] == 1) {
        const Proposal P = stored_proposal(store, lane);
        Chain ch;
        ch.get(store, lane);
        double v[kTip ? 3 : 1];
#pragma unroll
        for (int q = 0; q < (kTip ? 3 : 1); ++q) {
          v[q] = red[q][0][lane];
#pragma unroll
          for (int u = 1; u < kJumpSlices; ++u) v[q] += red[q][u][lane];
        }
        double fx = 0.0, fy = 0.0, fz = 0.0;
        const double pre = g.dfc * Consts::q_0 * 1.0e18;
        if (kTip) {
          tip_vacuum64(g, P.x, P.y, P.z, fx, fy, fz);
          fx += pre * v[0];
          fy += pre * v[kTip ? 1 : 0];
          fz += pre * v[kTip ? 2 : 0];
        } else {
          fz = g.Ez + pre * (ic ? -2.0 * v[0] : v[0]);
        }
        dec = ch.decide(s, it, width.first, P, stored_site(store, lane), plr, fx, fy, fz);
        ch.put(store, lane);
      }
      width.count(it, dec);
    }
  }
  if (mine) {
    Chain ch;
    ch.get(store, lane);
    ch.store(out, c);
  }
  // the width after the last jump (a launch per jump: in a launch of its own)
  if (wv == 0 && a.it0 <= s.ndim + 1 && (a.spin ? a.it1 > s.ndim : a.it0 == s.ndim + 1))
    width.last(s.ndim);
}

// ---- FP64 -----------------------------------------------------------------------

// Wavefront 0 proposes, sums and decides; wavefronts 1 .. 8 form terms, a lane
// per particle of a chunk, two chunks side by side (two wavefronts per SIMD:
// one alone issues an FP64 instruction every eight cycles).  The terms of one
// pass are formed while those of the pass before are summed: a sum is a serial
// chain of 256 additions (about 2000 cycles) in a few lanes, about as long as
// the wavefronts take for a pass.
constexpr int kJump64Threads = 64 + 2 * kChunk;
constexpr int kJump64T = 4;  // chains per pass

// surface_pair64's z components at T chains' points for one particle, the
// chains side by side so that their dependent operations overlap.
template <class M, int T>
__device__ __forceinline__ void surface_z64(const DevGeom& g, double pre, const double (&px)[T],
                                            const double (&py)[T], double x, double y, double zb,
                                            double (&az)[T]) {
  double dxy2[T], p0[T], iz[T];
#pragma unroll
  for (int u = 0; u < T; ++u) {
    const double dx = px[u] - x, dy = py[u] - y;
    dxy2[u] = M::lift(dx * dx + dy * dy);
    const double i0 = inv_r3_64<M>(dxy2[u] + zb * zb, g.es);
    p0[u] = pre * i0;
    iz[u] = -zb * i0;
  }
  for (int n = 1; n <= g.nic; ++n) {
    const double tnd = 2.0 * n * g.d;
    const double a = tnd - zb, b = tnd + zb;
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const double pa = a * inv_r3_64<M>(dxy2[u] + a * a, g.es);
      const double pb = b * inv_r3_64<M>(dxy2[u] + b * b, g.es);
      iz[u] = (((iz[u] + pa) - pb) - pb) + pa;
    }
  }
#pragma unroll
  for (int u = 0; u < T; ++u) az[u] = g.ic ? p0[u] * -zb + pre * iz[u] : p0[u] * (0.0 - zb);
}

template <int KIND>
__global__ __launch_bounds__(kJump64Threads, 3) void k_mh_jumps64(
    const Ent* tab, int ne, const SimDesc* desc, const SimState* st, const double* wf, Chains in,
    Chains out, JumpArgs a) {
  constexpr bool kTip = KIND == RD_GEOM_TIP;
  constexpr int K = kTip ? 3 : 1;   // field components summed
  constexpr int V = kTip ? 7 : 2;   // values of a chain's point
  constexpr int T = kJump64T;
  constexpr int NC = kTip ? 2 : 4;  // chunks of a pass
  constexpr int kSeq = K * T * NC;  // sequences of one pass: (chunk, chain, component)
  static_assert(kSeq <= 64, "a lane per sequence");
  // padded rows: the sequences' lanes read 16 bytes each without bank conflicts
  constexpr int kRow = kChunk + 2;
  __shared__ __align__(16) double term[2][kSeq][kRow];
  __shared__ double tgt[V][kJumpLanes];  // x, y (z, image distance, image)
  __shared__ double fsum[K][kJumpLanes];
  __shared__ int s_stop, s_ord;
  __shared__ ChainStore store;
  const Ent e = tab[find_entry(tab, ne, blockIdx.x)];
  const SimDesc s = desc[e.slot];
  if (s.g.kind != KIND) return;
  const DevGeom& g = s.g;
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int grp = blockIdx.x - e.wg0;
  const int k0 = jump_first(e, grp), nc = jump_first(e, grp + 1) - k0;
  const int c = e.cbase + k0 + lane;
  const bool mine = wv == 0 && lane < nc;
  const int n = st[e.slot].n;
  const int nchunks = (n + kChunk - 1) / kChunk;
  const int it1 = min(a.it1, s.ndim + 1);
  if (mine) {
    Chain ch;
    ch.load(in, c);
    ch.put(store, lane);
  }
  JumpWidth width(e, s, st[e.slot], a, grp);
  if (t < kJumpLanes)
    for (int q = 0; q < V; ++q) tgt[q][t] = 0.0;
  if (t == 0) s_stop = 0;
  const double* X = a.X + e.base;
  const double* Y = a.Y + e.base;
  const double* Z = a.Z + e.base;
  const double* Q = a.Q + e.base;
  // this lane's particle of a chunk and which half of a pass's chunks it takes
  const int p = (t - 64) & (kChunk - 1), half = wv > 4;
  // its particle of the next chunk, in flight while a chunk's terms are formed
  double xn = 0, yn = 0, zn = 0, qn = 0;
  auto load = [&](int chunk) {
    const int j = min(chunk * kChunk + p, max(n - 1, 0));
    xn = X[j];
    yn = Y[j];
    zn = Z[j];
    qn = Q[j];
  };
  // the short root and quotient sequences serve while every coordinate is
  // ordinary (rd_fp64.h); the particles do not move during the jumps
  bool ord = f64_ordinary(g.d);
  for (int j = t; j < n; j += kJump64Threads)
    ord = ord && f64_ordinary(X[j]) && f64_ordinary(Y[j]) && f64_ordinary(Z[j]);
  const bool src_ord = __syncthreads_and(ord);
  if (n > 0) load(half * (NC / 2));
  const int batches = (nchunks + NC - 1) / NC;  // passes of T chains
  double u1 = 0, u2 = 0, lr = 0;
  auto draws = [&](int it) {
    const size_t o = (size_t)(it - 1) * a.C + c;
    u1 = a.ru1[o];
    u2 = a.ru2[o];
    lr = a.rlr[o];
  };
  if (mine && a.it0 < it1) draws(a.it0);
  double plr = 0;
  __syncthreads();
  for (int it = a.it0; it < it1; ++it) {
    if (wv == 0) {
      __builtin_amdgcn_s_setprio(3);
      if (!width.before(it)) s_stop = 1;
      bool o = true;
      if (mine) {
        const Proposal P = jump_proposal(s, width.mh, it, store, lane, u1, u2);
        tgt[0][lane] = P.x;
        tgt[1][lane] = P.y;
        o = f64_ordinary(P.x) && f64_ordinary(P.y);
        if (kTip) {
          double da = 0, xi = 0, yi = 0, zi = 0;
          if (g.ic) tip_image_point64(P.x, P.y, P.z, g.z0, g.R, da, xi, yi, zi);
          tgt[kTip ? 2 : 0][lane] = P.z;
          tgt[kTip ? 3 : 0][lane] = da;
          tgt[kTip ? 4 : 0][lane] = xi;
          tgt[kTip ? 5 : 0][lane] = yi;
          tgt[kTip ? 6 : 0][lane] = zi;
          o = o && f64_ordinary(P.z) && f64_ordinary(da) && f64_ordinary(xi) &&
              f64_ordinary(yi) && f64_ordinary(zi);
        }
        plr = lr;
        if (it + 1 < it1) draws(it + 1);
      }
      const bool all = __all(o);
      if (t == 0) s_ord = all;
    }
    __syncthreads();
    if (s_stop) return;
    const bool fast = src_ord && s_ord;
    if (mine) store_site(s, wf, store, lane, it > a.it0);
    const int passes = batches * ((nc + T - 1) / T);
    double sum = 0.0;  // lane (chain, component) < T K: the chunk partials in order
    int tb = 0, bi = 0;    // chains and batch of the pass being formed
    int stb = 0, sbi = 0;  // and of the pass being summed, one behind
#pragma unroll 1
    for (int b = 0; b <= passes; ++b) {
      if (wv > 0 && b < passes) {
        const int cb = bi * NC;
        double pt[V][T];
#pragma unroll
        for (int u = 0; u < T; ++u)
#pragma unroll
          for (int v = 0; v < V; ++v) pt[v][u] = tgt[v][tb + u];  // tb + u < kJumpLanes
        auto terms = [&](auto m) {
          using M = decltype(m);
          const int ke = half ? NC : NC / 2;
#pragma unroll 1
          for (int k = half * (NC / 2); k < ke && cb + k < nchunks; ++k) {
            const bool in_n = (cb + k) * kChunk + p < n;  // beyond: terms of zero
            const double x = xn, y = yn, z = zn, q = qn * g.dfc;
            // the lane's next chunk: of this half of the pass, of the next pass
            int next = cb + k + (k + 1 < ke ? 1 : NC / 2 + 1);
            if (next >= nchunks) next = half * (NC / 2);
            load(next);
            double (*row)[kRow] = &term[b & 1][k * T * K];
            if (!kTip) {
              double az[T];
              surface_z64<M, T>(g, q, pt[0], pt[1], x, y, z, az);
#pragma unroll
              for (int u = 0; u < T; ++u) row[u][p] = in_n ? az[u] : 0.0;
            } else {
#pragma unroll
              for (int u = 0; u < T; ++u) {
                const double dx = pt[0][u] - x, dy = pt[1][u] - y, dz = pt[kTip ? 2 : 0][u] - z;
                const double r2 = M::lift(dx * dx + dy * dy) + dz * dz;
                const double rt = M::sqrt(r2);
                const double r = rt + g.es;
                const double p0 = q * M::rcp(r * r * r);
                double ax = p0 * dx, ay = p0 * dy, az = p0 * dz;
                if (g.ic) {
                  double icx, icy, icz;
                  tip_ic64<M>(dx, dy, dz, r2, rt, pt[kTip ? 4 : 0][u] - x,
                              pt[kTip ? 5 : 0][u] - y, pt[kTip ? 6 : 0][u] - z,
                              pt[kTip ? 3 : 0][u], g.R, g.ktip, icx, icy, icz);
                  ax = ax + q * icx;
                  ay = ay + q * icy;
                  az = az + q * icz;
                }
                row[u * K][p] = in_n ? ax : 0.0;
                row[u * K + (kTip ? 1 : 0)][p] = in_n ? ay : 0.0;
                row[u * K + (kTip ? 2 : 0)][p] = in_n ? az : 0.0;
              }
            }
          }
        };
        if (fast)
          terms(Fast64{});
        else
          terms(Ieee64{});
        if (++bi == batches) {
          bi = 0;
          tb += T;
        }
      }
      if (wv == 0 && b > 0) {
        // every chunk is summed to its full length: the padding's zeros do not
        // change a sum (which starts at +0, so it is never -0)
        double v = 0.0;
        if (t < kSeq) {
          const double2* row = reinterpret_cast<const double2*>(term[(b - 1) & 1][t]);
          double2 r[2][8];  // one half is read while the other is added
#pragma unroll
          for (int k = 0; k < 8; ++k) r[0][k] = row[k];
#pragma unroll
          for (int jj = 0; jj < kChunk / 16; ++jj) {
            if (jj + 1 < kChunk / 16) {
#pragma unroll
              for (int k = 0; k < 8; ++k) r[(jj + 1) & 1][k] = row[8 * (jj + 1) + k];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) v = (v + r[jj & 1][k].x) + r[jj & 1][k].y;
          }
        }
        // lane t + k T K holds chunk cb + k of lane t's sequence
        for (int k = 0; k < NC && sbi * NC + k < nchunks; ++k) {
          const double o = __shfl(v, (k * T * K + t) & 63);
          sum = sum + o;
        }
        if (++sbi == batches) {
          if (t < T * K) fsum[t % K][stb + t / K] = sum;
          sum = 0.0;
          sbi = 0;
          stb += T;
        }
      }
      __syncthreads();
    }
    if (wv == 0) {
      int dec = 0;
      if (mine && store.i[0][lane] == 1) {
        const Proposal P = stored_proposal(store, lane);
        Chain ch;
        ch.get(store, lane);
        double fx = 0.0, fy = 0.0, fz = g.Ez;
        double f[K];
#pragma unroll
        for (int k = 0; k < K; ++k) f[k] = nchunks > 0 ? fsum[k][lane] : 0.0;
        if (kTip) {
          tip_vacuum64(g, P.x, P.y, P.z, fx, fy, fz);
          fx = fx + f[0];
          fy = fy + f[kTip ? 1 : 0];
          fz = fz + f[kTip ? 2 : 0];
        } else {
          fz = fz + f[0];
        }
        dec = ch.decide(s, it, width.first, P, stored_site(store, lane), plr, fx, fy, fz);
        ch.put(store, lane);
      }
      width.count(it, dec);
    }
  }
  if (mine) {
    Chain ch;
    ch.get(store, lane);
    ch.store(out, c);
  }
  if (wv == 0 && a.it0 <= s.ndim + 1 && (a.spin ? a.it1 > s.ndim : a.it0 == s.ndim + 1))
    width.last(s.ndim);
}

}  // namespace rd
