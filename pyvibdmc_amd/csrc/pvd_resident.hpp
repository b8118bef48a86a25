// Resident discrete steps: many DMC steps in one launch, the walkers kept on chip.
//
// The launch-per-step kernels read and write every walker through HBM and pay a launch, a
// look-back and a finalisation per step.  Here workgroup b owns the walkers of a contiguous
// range of slots [base, base + cnt) for the whole launch, in LDS (a million triatomic FP32
// walkers are 36 MB; the 256 CUs hold 40 MB of LDS).  Births and deaths keep np.repeat order,
// so a workgroup's survivors stay contiguous in the global order and no walker changes
// workgroup: a step exchanges one record per workgroup (copy count, sum of c E, births) and
// every workgroup reads all records, which gives it its new base and the step's vref.  The
// per-walker arithmetic and the draws (addressed by global slot and step) are those of
// k_discrete, so populations and walkers agree bit for bit; vref agrees to the rounding of the
// summation order.
//
// Populations of the workgroups drift apart; when one outgrows its storage, or needs a round of
// NT walkers more than an even split would, all of them (every workgroup sees the same records)
// write their survivors to the global planes, meet at a barrier and load even shares again.
//
// Every workgroup waits for every other one, so all of them have to run at once.  Other kernels may
// hold some of the CUs, or wait on the rest of them themselves, so a launch first makes sure: its
// workgroups are counted, and the first of them opens the gate when the count is full, or closes it
// after a while with nothing changed and the CUs free.  (A cooperative launch gives less: it does not
// see other processes, its first one makes a queue, 3.7 ms, and those of a process run one at a time:
// two simulations of 5 000 walkers on two streams took as long together as in turn, 33 ms for 4 000
// steps each, now 19.)  A second
// launch with the same arguments, k_resident_rest, ends at once behind an open gate; behind a closed
// one the workgroups of it that do run, one or all, take the steps, with the walkers in the global
// planes.  Waits on other workgroups' records are bounded and end in ST_SPIN.  Records are single
// 64-bit words (epoch | payload) stored and read with relaxed agent-scope atomics, so a word is valid
// by itself and publishing needs no fence.
#pragma once
#include "pvd_sim.hpp"

namespace pvd {

constexpr int RES_MAXG = 256;  // workgroups of a resident launch
// least steps between redistributions that only even out the rounds: one costs 15 us at 1M walkers,
// unevenness a round of five (plain 1M: 17.0 us a step at 16, 15.9 at 32, 16.1 at 48)
constexpr int RES_REB = 32;
// Exchange area, in 64-bit words: records (4 per workgroup, by step parity), acceptance counts (by
// parity), barrier words; then two sets of RES_SET 32-bit words (the launches of a simulation use them
// in turn, each clearing the next one's), then the simulation's own words.
constexpr size_t RES_XSYNC = (size_t)RES_MAXG * (2 * 4 + 2 + 1);
// words of a set, each on a line of its own: workgroups that reported, the gate, workgroups that
// joined the second launch (RES_SHUT: no more), how many take part
enum : int { RES_ARRIVED = 0, RES_GATE = 32, RES_JOINED = 64, RES_TEAM = 96, RES_SET = 128 };
// the simulation's words, behind the sets: the last gate was closed, launches whose gate opened and
// was closed, redistributions of the walkers
enum : int { RES_CLOSED = 2 * RES_SET, RES_N_OPEN, RES_N_CLOSED, RES_N_SPREAD, RES_SYNCW };
constexpr size_t RES_XWORDS = RES_XSYNC + (RES_SYNCW + 1) / 2;
constexpr unsigned RES_OPEN = 1u, RES_SHUT = 0x80000000u;
// How long the first workgroup waits for the others, in ticks of 10 ns: at the gate 8 ms, longer than
// another launch of this kind that fills the LDS holds its CUs, and up to 10 ms more by chance (two
// processes that wait on each other's CUs should not give up together); a 64th of that where the last
// gate was closed.  In the second launch, which goes on with those that are there, 2 ms.  Nobody waits for
// the first workgroup's word longer than 60 s.
constexpr unsigned long long RES_WAIT = 800000ull, RES_WAIT_MORE = 1ull << 20, RES_TEAM_WAIT = 200000ull,
                             RES_WAIT_MAX = 6000000000ull;
constexpr unsigned RES_CLAMP = 1u << 22;  // a workgroup's published count: beyond any population bound served
constexpr long long RES_SPIN = 1ll << 24;

// PesParams / TrialParams with the parameters in the walkers' type, converted once on the host
template <typename R>
struct PesArgs {
  int kind;
  int idx[4];
  R p[12];
};
template <typename R>
struct TrialArgs {
  R balpha[PVD_MAX_TB], br0[PVD_MAX_TB], aalpha[PVD_MAX_TA], ath0[PVD_MAX_TA];
  R c0;
};

template <typename R>
struct ResArgs {
  R* buf[2];     // walker planes by step parity
  int* who[2];   // descendant tracker by step parity
  R* ext;        // per-workgroup storage of the walkers beyond the LDS
  Ctrl* ctrl;
  uint64_t* xch;
  double* tr_vref;
  double* tr_pop;
  double* tr_dteff;
  int* tr_births;
  int* tr_deaths;
  long long cap, tmax;
  double dt, alpha, n0, pop_lo, pop_hi;
  int par, branch_every, steps, capl, capb, who_on;
  int set;                                    // which set of words this launch uses
  unsigned long long gate_wait, team_wait;  // see RES_WAIT
  Rng rng;
  PesArgs<R> pes;
  TrialArgs<R> trial;
  R sigma[PVD_FUSED_MAX_COMP], inv_m[PVD_FUSED_MAX_COMP];
  float h2s[PVD_FUSED_MAX_COMP];
};

// f(0), f(1), ..., f(N - 1) with compile-time indices (arrays indexed by them stay in registers)
template <typename F, int... I>
PVD_DEV void static_for_(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
PVD_DEV void static_for(F&& f) {
  static_for_(f, std::make_integer_sequence<int, N>{});
}

// Wave scans and reductions by DPP moves (row shifts, then row broadcasts): no LDS round trips as
// in shuffles.  An inclusive scan leaves the total in lane 63; the order is fixed.
template <int CTRL, int ROWS>
PVD_DEV int dpp0(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false); }
PVD_DEV int dpp_scan(int v) {
  v += dpp0<0x111, 0xf>(v);
  v += dpp0<0x112, 0xf>(v);
  v += dpp0<0x114, 0xf>(v);
  v += dpp0<0x118, 0xf>(v);
  v += dpp0<0x142, 0xa>(v);
  v += dpp0<0x143, 0xc>(v);
  return v;
}
PVD_DEV unsigned long long first_lane(unsigned long long v) {
  return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 |
         (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}
PVD_DEV int lane_of(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
PVD_DEV int dpp_sum(int v) { return lane_of(dpp_scan(v), 63); }
PVD_DEV int dpp_max(int v) {  // of values >= 0
  v = max(v, dpp0<0x111, 0xf>(v));
  v = max(v, dpp0<0x112, 0xf>(v));
  v = max(v, dpp0<0x114, 0xf>(v));
  v = max(v, dpp0<0x118, 0xf>(v));
  v = max(v, dpp0<0x142, 0xa>(v));
  v = max(v, dpp0<0x143, 0xc>(v));
  return lane_of(v, 63);
}
template <int CTRL, int ROWS>
PVD_DEV double dpp0(double v) {
  const long long b = __double_as_longlong(v);
  const uint32_t lo = (uint32_t)dpp0<CTRL, ROWS>((int)(uint32_t)b), hi = (uint32_t)dpp0<CTRL, ROWS>((int)(b >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// sums of the first 16 lanes
PVD_DEV int dpp_sum16(int v) {
  v += dpp0<0x111, 0xf>(v);
  v += dpp0<0x112, 0xf>(v);
  v += dpp0<0x114, 0xf>(v);
  v += dpp0<0x118, 0xf>(v);
  return lane_of(v, 15);
}
PVD_DEV double lane_of(double v, int l) {
  const long long b = __double_as_longlong(v);
  const uint32_t lo = (uint32_t)lane_of((int)(uint32_t)b, l), hi = (uint32_t)lane_of((int)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
PVD_DEV double dpp_sum16(double v) {
  v += dpp0<0x111, 0xf>(v);
  v += dpp0<0x112, 0xf>(v);
  v += dpp0<0x114, 0xf>(v);
  v += dpp0<0x118, 0xf>(v);
  return lane_of(v, 15);
}
PVD_DEV double dpp_sum(double v) {
  v += dpp0<0x111, 0xf>(v);
  v += dpp0<0x112, 0xf>(v);
  v += dpp0<0x114, 0xf>(v);
  v += dpp0<0x118, 0xf>(v);
  v += dpp0<0x142, 0xa>(v);
  v += dpp0<0x143, 0xc>(v);
  return lane_of(v, 63);
}

// word p once it carries `epoch` (f: its value as first read)
PVD_DEV bool res_poll(const uint64_t* p, unsigned epoch, uint64_t& f) {
  long long spins = 0;
  while ((unsigned)(f >> 32) != epoch) {
    if (++spins > RES_SPIN) return false;
    __builtin_amdgcn_s_sleep(1);
    f = ld_relaxed(p);
  }
  return true;
}

// Rank of a lane's copies inside its wave (exclusive, in lane order), the wave's copies and its
// births, from ballots of c >= 1, c >= 2, ...: weights stay near one, so two ballots replace a
// scan.  Beyond 16 copies the scan takes over.
PVD_DEV int wave_copies(int c, int& total, int& births) {
  const unsigned long long b1 = __ballot(c > 0), b2 = __ballot(c > 1);
  auto below = [](unsigned long long b) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
  };
  int ex = below(b1) + below(b2);
  int nb = __popcll(b2);
  total = __popcll(b1) + nb;
  unsigned long long b = __ballot(c > 2);
  if (b) {
    for (int l = 3; b && l <= 16; b = __ballot(c > l), ++l) {
      ex += below(b);
      nb += __popcll(b);
      total += __popcll(b);
    }
    if (b) {
      const int inc = dpp_scan(c);
      ex = inc - c;
      total = lane_of(inc, 63);
      nb = dpp_sum(c > 1 ? c - 1 : 0);
    }
  }
  births = nb;
  return ex;
}

// Walker stride of the on-chip storage: component p of walker li at sx[li * stride + p], so the
// components share one address register; the stride is odd in banks (a 64-lane access of one
// component meets every bank once).
template <typename R, int NP>
constexpr int res_stride() {
  return sizeof(R) == 4 ? (NP | 1) : NP;
}

// W rounds of blockDim walkers per workgroup.  The first capl walkers are stored in LDS; with EXT
// later ones (a population above N0 where N0 alone fills the LDS) in a global area of the
// workgroup's own, which it alone reads and writes.
template <typename R, int NP, bool IS, int MS, int W, int NTMAX, bool EXT>
__global__ __launch_bounds__(NTMAX) void k_resident(ResArgs<R> A) {
  constexpr int NWM = NTMAX / PVD_WAVE;
  constexpr int ST = res_stride<R, NP>();
  // with few rounds the walkers stay in registers until the copies are written; more rounds are
  // moved in place, one walker's registers at a time, and read again (held, they spill)
  constexpr bool HOLD = !EXT;
  extern __shared__ __align__(16) unsigned char s_dyn[];
  __shared__ int s_wt[(W * NWM + PVD_WAVE - 1) / PVD_WAVE * PVD_WAVE];
  __shared__ double s_d[16];              // per wave: sum of c E
  __shared__ __align__(16) int4 s_t[16];  // per wave: copies, births, bad weights
  // per 64 records: copies, copies of the workgroups before this one, most copies, bad weights; sum
  // of c E; births
  __shared__ __align__(16) int4 s_res[4];
  __shared__ double s_s0[4], s_vref, s_eff, s_vref_at, s_eff_at;
  __shared__ int s_nb[4], s_acc[4], s_late;
  const int NT = blockDim.x, G = gridDim.x, blk = blockIdx.x;
  int tid = threadIdx.x;
  const int ln = lane_id(), wv = __builtin_amdgcn_readfirstlane(tid / PVD_WAVE), nwv = NT / PVD_WAVE;
  const int capl = A.capl, capb = NT * W, exts = EXT && capb > capl ? capb - capl : 0;
  // explicit address spaces: merged into generic pointers, the two storages would be read by flat
  // accesses
  typedef __attribute__((address_space(3))) R LdsR;
  typedef __attribute__((address_space(3))) int LdsI;
  typedef __attribute__((address_space(1))) R ExtR;
  typedef __attribute__((address_space(1))) int ExtI;
  LdsR* sx = (LdsR*)s_dyn;
  LdsI* sw = (LdsI*)(sx + ST * capl);
  const bool who_on = A.who_on != 0;

  // arguments that are used rarely are read again where they are used (they would fill the scalar
  // registers of the step loop)
  typedef const __attribute__((address_space(4))) ResArgs<R> Cold;
  auto cold = []() {
    Cold* p = (Cold*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
  };
  bool first = false;  // the workgroup that watches the gate (thread 0)
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  if (G > 1 && tid == 0) {
    unsigned* sync = reinterpret_cast<unsigned*>(A.xch + RES_XSYNC);
    if (blk == 0)  // nobody uses the other set: the launches before this one have ended
      for (int k = 0; k < 4; ++k) st_relaxed_u(sync + (A.set ^ 1) * RES_SET + 32 * k, 0u);
    if (A.ctrl->status == ST_OK) first = fetch_add_relaxed(sync + A.set * RES_SET + RES_ARRIVED, 1u) == 0u;
  }
  if (A.ctrl->status != ST_OK) return;
  int par = A.par;
  const int be = A.branch_every, n0i = (int)A.n0;
  const double pop_hi = A.pop_hi, pop_lo = A.pop_lo, n0 = A.n0, alpha = A.alpha;
  const long long cap = A.cap;
  // kept in registers: read again from the arguments, each use would wait for the scalar cache
  uint64_t* const xch = reinterpret_cast<uint64_t*>(first_lane((unsigned long long)A.xch));
  int n = __builtin_amdgcn_readfirstlane(A.ctrl->n[par]);
  unsigned long long step = first_lane(A.ctrl->step[par]);
  unsigned epoch = (unsigned)__builtin_amdgcn_readfirstlane((int)A.ctrl->epoch[par]);
  int base = 0, cnt = 0;

  // storage of walker li (X: it may lie beyond the LDS)
  auto ext = [&](int li) {
    ExtR* e = (ExtR*)cold()->ext + (size_t)blk * (ST + 1) * exts;
    return e + (size_t)(li - capl) * ST;
  };
  auto ext_who = [&](int li) {
    ExtR* e = (ExtR*)cold()->ext + (size_t)blk * (ST + 1) * exts + (size_t)ST * exts;
    return (ExtI*)e + (li - capl);
  };
  auto get = [&](auto X, int li, R* x) {
    if (!decltype(X)::value || li < capl) {
#pragma unroll
      for (int p = 0; p < NP; ++p) x[p] = sx[li * ST + p];
    } else {
      const ExtR* e = ext(li);
#pragma unroll
      for (int p = 0; p < NP; ++p) x[p] = e[p];
    }
  };
  auto put = [&](auto X, int li, const R* x) {
    if (!decltype(X)::value || li < capl) {
#pragma unroll
      for (int p = 0; p < NP; ++p) sx[li * ST + p] = x[p];
    } else {
      ExtR* e = ext(li);
#pragma unroll
      for (int p = 0; p < NP; ++p) e[p] = x[p];
    }
  };
  auto get_who = [&](int li) -> int {
    if (!EXT || li < capl) return sw[li];
    return *ext_who(li);
  };
  auto put_who = [&](int li, int v) {
    if (!EXT || li < capl) sw[li] = v;
    else *ext_who(li) = v;
  };
  using Any = std::integral_constant<bool, EXT>;
  using Lds = std::integral_constant<bool, false>;
  // even share of the n walkers in the planes of parity par
  auto load_share = [&]() {
    base = (int)((long long)n * blk / G);
    cnt = (int)((long long)n * (blk + 1) / G) - base;
    const R* src = cold()->buf[par] + base;
    const int* who = cold()->who[par] + base;
    for (int li = tid; li < cnt; li += NT) {
      R x[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) x[p] = src[p * cap + li];
      put(Any{}, li, x);
      if (who_on) put_who(li, who[li]);
    }
  };
  // the walkers as stored back to the planes of parity par
  auto store_share = [&]() {
    R* dst = cold()->buf[par] + base;
    int* who = cold()->who[par] + base;
    for (int li = tid; li < cnt; li += NT) {
      R x[NP];
      get(Any{}, li, x);
#pragma unroll
      for (int p = 0; p < NP; ++p) dst[p * cap + li] = x[p];
      if (who_on) who[li] = get_who(li);
    }
  };
  // all workgroups meet; `tag` is an epoch no other barrier word carries
  auto meet = [&](unsigned tag) {
    uint64_t* xbar = xch + (size_t)RES_MAXG * 10;
    store_complete();  // every wave's stores have reached its XCD's L2 ...
    __syncthreads();
    if (tid == 0) {
      fence_release();  // ... and are written back before the barrier word
      st_relaxed(xbar + blk, ((uint64_t)tag << 32) | 1u);
    }
    for (int r = tid; r < G; r += NT) {
      uint64_t f = ld_relaxed(xbar + r);
      if (!res_poll(xbar + r, tag, f)) s_late = 1;
    }
    __syncthreads();
    fence_acquire();
    return s_late == 0;
  };
  auto lost = [&]() {  // a workgroup did not answer: nothing to go on from
    if (tid == 0) {
      cold()->ctrl->status_step = (long long)step;
      cold()->ctrl->status = ST_SPIN;
    }
  };
  if (tid == 0) {
    s_late = 0;
    s_vref = s_vref_at = A.ctrl->vref[par];
    s_eff = s_eff_at = A.ctrl->eff_t;
  }
  for (int q = tid; q < (int)(sizeof(s_wt) / sizeof(int)); q += NT) s_wt[q] = 0;
  if (tid < 16) {
    s_d[tid] = 0.0;
    s_t[tid] = int4{0, 0, 0, 0};
    if (tid < 4) {
      s_res[tid] = int4{0, 0, 0, 0};
      s_s0[tid] = 0.0;
      s_nb[tid] = 0;
      s_acc[tid] = 0;
    }
  }
  load_share();
  if (G > 1) {
    if (tid == 0) {
      unsigned* sync = reinterpret_cast<unsigned*>(xch + RES_XSYNC);
      unsigned* set = sync + cold()->set * RES_SET;
      unsigned f = 0;
      if (first) {
        const unsigned long long most = cold()->gate_wait + (cold()->gate_wait ? t0 & (RES_WAIT_MORE - 1) : 0);
        const unsigned long long wait = ld_relaxed_u(sync + RES_CLOSED) ? most >> 6 : most;
        f = RES_OPEN;
        while (wait == 0 || ld_relaxed_u(set + RES_ARRIVED) != (unsigned)G) {
          if (__builtin_amdgcn_s_memrealtime() - t0 >= wait) {
            f = RES_SHUT;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
        st_relaxed_u(set + RES_GATE, f);
        st_relaxed_u(sync + RES_CLOSED, f == RES_SHUT ? 1u : 0u);
        fetch_add_relaxed(sync + (f == RES_OPEN ? RES_N_OPEN : RES_N_CLOSED), 1u);
      } else {
        while ((f = ld_relaxed_u(set + RES_GATE)) == 0u && __builtin_amdgcn_s_memrealtime() - t0 < RES_WAIT_MAX)
          __builtin_amdgcn_s_sleep(1);
      }
      s_late = f == RES_OPEN ? 0 : 1;
    }
    __syncthreads();
    if (s_late) return;
  }
  __syncthreads();

  // the last state in the planes: where a failed run is retraced from
  int n_at = n, par_at = par;
  unsigned long long step_at = step;
  const unsigned long long last_step = step + (unsigned long long)A.steps - 1;
  unsigned long long stop = ~0ull;  // retracing: the step that failed
  int fail = ST_OK, since = 0;
  for (;;) {
    // addresses are formed where they are used: hoisted out of the step loop they would take more
    // registers than there are
    asm volatile("" : "+v"(tid));
    if (!IS && step == stop) break;
    const bool branch = be <= 1 || step % (unsigned long long)be == 0;
    R x[HOLD ? W : 1][NP];
    int c[W];
    double sce = 0.0, dte = A.dt;
    const double vref = s_vref;
    int bad = 0;
    static_for<W>([&](auto K) { c[K] = 0; });
    // the rounds are a real loop (one walker's registers at a time); a value kept per round is
    // selected into its array element
    auto keep = [&](auto* arr, int k, auto v) { static_for<W>([&](auto J) { arr[J] = J == k ? v : arr[J]; }); };
    if constexpr (IS) {
      // drift move, Metropolis and local energy of every walker (k_is_move), in place; the
      // accepted moves of all workgroups give dt_eff
      R e[W];
      int acc = 0;
      static_for<W>([&](auto K) { e[K] = R(0); });
      auto moves = [&](auto X) {
#pragma unroll 1
        for (int k = 0; k * NT < cnt; ++k) {
          const int li = k * NT + tid;
          bool a = false;
          R ek = R(0);
          if (li < cnt) {
            R y[NP], disp[NP];
            double um, ub;
            get(X, li, y);
            draw_step<R, NP, false, true>(A, (long long)base + li, step, disp, um, ub, false);
            const R ke = is_move_fast<R, NP, MS>(A, disp, um, y, a);
            const R v = pes_eval_s<R, NP, MS>(A.pes, y);
            ek = v + ke;
            if (a) put(X, li, y);
          }
          keep(e, k, ek);
          acc += __popcll(__ballot(a));
        }
      };
      if (EXT && cnt > capl) moves(Any{});
      else moves(Lds{});
      if (ln == 0) s_t[wv].x = acc;
      __syncthreads();
      if (step == stop) break;
      uint64_t* xacc = xch + (size_t)RES_MAXG * (8 + (step & 1));
      if (wv == 0) {
        const int t = dpp_sum16(s_t[ln & 15].x);
        if (ln == 0) st_relaxed(xacc + blk, ((uint64_t)epoch << 32) | (unsigned)t);
      }
      // the branching uniforms while the counts travel
      float u[W];
      static_for<W>([&](auto K) {
        u[K] = 0.0f;
        if (branch && K * NT < cnt)
          u[K] = (float)draw_u<R, false>(A, (long long)base + K * NT + tid, step, RNG_BRANCH);
      });
      for (int g = wv; g * PVD_WAVE < G; g += nwv) {
        const int r = g * PVD_WAVE + ln;
        uint64_t f = 0;
        if (r < G) {
          f = ld_relaxed(xacc + r);
          if (!res_poll(xacc + r, epoch, f)) s_late = 1;
        }
        const int got = dpp_sum((int)(uint32_t)f);
        if (ln == 0) s_acc[g] = got;
      }
      __syncthreads();
      dte = dte * ((double)(unsigned)((s_acc[0] + s_acc[1]) + (s_acc[2] + s_acc[3])) / (double)n);
      static_for<W>([&](auto K) {
        if (K * NT + tid < cnt) {
          const double E = (double)e[K];
          c[K] = branch ? branch_copies<true>(E, vref, dte, (double)u[K], pop_hi, bad) : 1;
          sce += (double)c[K] * E;
        }
      });
    } else {
      auto move = [&](int li, R* y) {  // returns the copies; y: the walker, moved
        R disp[NP];
        double um, ub;
        draw_step<R, NP, false, false>(A, (long long)base + li, step, disp, um, ub, branch);
#pragma unroll
        for (int p = 0; p < NP; ++p) y[p] = y[p] + disp[p];
        const double E = (double)pes_eval_s<R, NP, MS>(A.pes, y);
        const int ck = branch ? branch_copies<sizeof(R) == 4>(E, vref, dte, ub, pop_hi, bad) : 1;
        sce += (double)ck * E;
        return ck;
      };
      if constexpr (HOLD) {
        static_for<W>([&](auto K) {
          const int li = K * NT + tid;
          if (li < cnt) {
            get(Lds{}, li, x[K]);
            c[K] = move(li, x[K]);
          }
        });
      } else {
        auto moves = [&](auto X) {
#pragma unroll 1
          for (int k = 0; k * NT < cnt; ++k) {
            const int li = k * NT + tid;
            if (li < cnt) {
              R y[NP];
              get(X, li, y);
              const int ck = move(li, y);
              put(X, li, y);
              keep(c, k, ck);
            }
          }
        };
        if (cnt > capl) moves(Any{});
        else moves(Lds{});
      }
    }
    // ranks inside the workgroup and its sums
    int births = 0, copies = 0, xc[W];
    static_for<W>([&](auto K) {
      int t = 0, nb = 0;
      xc[K] = 0;
      if (K * NT < cnt) xc[K] = wave_copies(c[K], t, nb);
      births += nb;
      copies += t;
      if (ln == 0) s_wt[K * nwv + wv] = t;
    });
    sce = dpp_sum(sce);
    const bool anybad = __any(bad != 0);
    if (ln == 0) {
      s_t[wv] = int4{(int)min((unsigned)copies, RES_CLAMP), births, anybad ? 1 : 0, 0};
      s_d[wv] = sce;
    }
    __syncthreads();
    // the workgroup's record (lane l holds wave l's sums; clamped, 16 waves' copies fit an int)
    uint64_t* rec = xch + (size_t)(step & 1) * RES_MAXG * 4;
    const int4 wt = s_t[ln & 15];
    const double wd = s_d[ln & 15];
    const int total = dpp_sum16(wt.x);
    if (wv == 0) {
      const uint64_t bits = (uint64_t)__double_as_longlong(dpp_sum16(wd));
      uint32_t word = ((uint32_t)dpp_sum16(wt.y) & 0x7FFFFFFFu) | (__any(wt.z != 0) ? 0x80000000u : 0u);
      word = ln == 2 ? (uint32_t)bits : word;
      word = ln == 1 ? (uint32_t)(bits >> 32) : word;
      word = ln == 0 ? min((unsigned)total, RES_CLAMP) : word;
      if (ln < 4) st_relaxed(rec + 4 * blk + ln, ((uint64_t)epoch << 32) | word);
    }
    // exclusive offsets of the (round, wave) pairs, by every wave: lane l holds pairs l, l + 64
    {
      const int v0 = s_wt[ln];
      const int i0 = dpp_scan(v0);
      int i1 = 0, v1 = 0;
      if constexpr (W * NWM > PVD_WAVE) {
        v1 = s_wt[PVD_WAVE + ln];
        i1 = lane_of(i0, 63) + dpp_scan(v1);
      }
      static_for<W>([&](auto K) {
        const int q = K * nwv + wv;
        int o = lane_of(i0 - v0, q & 63);
        if (W * NWM > PVD_WAVE && q >= PVD_WAVE) o = lane_of(i1 - v1, q & 63);
        xc[K] += o;
      });
    }
    if constexpr (IS && HOLD) {
      // with few rounds, the survivors' coordinates are read while the records travel
      static_for<W>([&](auto K) {
        if (K * NT < cnt && c[K] > 0) get(Lds{}, K * NT + tid, x[K]);
      });
    }
    int who_of[HOLD ? W : 1];
    if constexpr (HOLD) {
      if (who_on) static_for<W>([&](auto K) { who_of[K] = c[K] > 0 ? get_who(K * NT + tid) : 0; });
    }
    // not before the records can be there: polls that come too early slow the stores they wait for
    // (100k walkers, 256 workgroups: 6.6 us a step without, 5.3 with 24 x 64 cycles; 20k: 4.6, 4.3)
    if (G > 1) __builtin_amdgcn_s_sleep(24);
    // all records, 64 by a wave, reduced in the same fixed order in every workgroup
    for (int g = wv; g * PVD_WAVE < G; g += nwv) {
      const int r = g * PVD_WAVE + ln;
      int tot = 0, nbt = 0, flag = 0;
      double s0 = 0.0;
      if (r < G) {
        uint64_t f[4];
        static_for<4>([&](auto J) { f[J] = ld_relaxed(rec + 4 * r + J); });
        bool ok = true;
        static_for<4>([&](auto J) { ok = res_poll(rec + 4 * r + J, epoch, f[J]) && ok; });
        if (!ok) s_late = 1;
        tot = (int)(uint32_t)f[0];
        s0 = __longlong_as_double((long long)(f[1] << 32 | (uint64_t)(uint32_t)f[2]));
        nbt = (int)((uint32_t)f[3] & 0x7FFFFFFFu);
        flag = (int)((uint32_t)f[3] >> 31);
      }
      const int pre = dpp_sum(r < blk ? tot : 0), mx = dpp_max(tot);
      tot = dpp_sum(tot);
      nbt = dpp_sum(nbt);
      s0 = dpp_sum(s0);
      const bool anyflag = __any(flag != 0);
      if (ln == 0) {
        s_res[g] = int4{tot, pre, mx, anyflag ? 1 : 0};
        s_s0[g] = s0;
        s_nb[g] = nbt;
      }
    }
    __syncthreads();
    int st = ST_OK, tot, pre, mx;
    {
      const int4 p = s_res[ln & 3];
      const int late = s_late;
      tot = (lane_of(p.x, 0) + lane_of(p.x, 1)) + (lane_of(p.x, 2) + lane_of(p.x, 3));
      pre = (lane_of(p.y, 0) + lane_of(p.y, 1)) + (lane_of(p.y, 2) + lane_of(p.y, 3));
      mx = max(max(lane_of(p.z, 0), lane_of(p.z, 1)), max(lane_of(p.z, 2), lane_of(p.z, 3)));
      if (__any(late != 0)) st = ST_SPIN;
      else if (__any(p.w != 0)) st = ST_WEIGHT;
      else if ((double)tot < pop_lo || (double)tot > pop_hi) st = ST_POP;
      else if (tot > cap) st = ST_CAPACITY;
    }
    if (st != ST_OK) {
      if (st == ST_SPIN || stop != ~0ull || !meet(epoch + 1)) {
        lost();
        return;
      }
      // the walkers have moved in place: take the last state in the planes and retrace the steps
      // up to this one (the same draws and the same sums give the same walkers), under new epochs
      stop = step;
      fail = st;
      epoch += 2;
      n = n_at;
      par = par_at;
      step = step_at;
      if (tid == 0) {
        s_vref = s_vref_at;
        s_eff = s_eff_at;
      }
      since = 0;
      load_share();
      __syncthreads();
      continue;
    }
    // the step's vref and record, by the last wave (it has the fewest walkers)
    auto finish = [&]() {
      if (wv == nwv - 1) {
        const double vbar = ((s_s0[0] + s_s0[1]) + (s_s0[2] + s_s0[3])) / (double)tot;
        const double corr = (double)(tot - n0i) / n0;
        const double vnew = vbar - (alpha * corr);
        if (ln == 0) {
          s_vref = vnew;
          if (blk == 0 && (long long)step < cold()->tmax) {
            cold()->tr_vref[step] = vnew;
            cold()->tr_pop[step] = (double)tot;
            const int nbt = (s_nb[0] + s_nb[1]) + (s_nb[2] + s_nb[3]);
            cold()->tr_births[step] = nbt;
            cold()->tr_deaths[step] = n + nbt - tot;
            if (IS) {
              // advances on branching steps only (see finalize_discrete)
              s_eff = branch ? (step == 0 ? 0.0 : s_eff) + dte : 0.0;
              cold()->tr_dteff[step] = s_eff;
            }
          }
        }
      }
      n = tot;
      ++step;
      ++epoch;
    };
    par ^= 1;
    ++since;
    const bool last = step == last_step;
    const int even = (tot + G - 1) / G;
    const bool spread = mx > capb || ((mx + NT - 1) / NT > (even + NT - 1) / NT && since >= RES_REB);
    if (last || spread) {
      // survivors to their np.repeat positions in the planes
      R* dst = cold()->buf[par] + pre;
      int* who = cold()->who[par] + pre;
      static_for<W>([&](auto K) {
        if (c[K] > 0) {
          auto copy = [&](const R* y, int w) {
            for (int q = 0; q < c[K]; ++q) {
#pragma unroll
              for (int p = 0; p < NP; ++p) dst[p * cap + xc[K] + q] = y[p];
              if (who_on) who[xc[K] + q] = w;
            }
          };
          if constexpr (HOLD) {
            copy(x[K], who_of[K]);
          } else {
            R y[NP];
            get(Any{}, K * NT + tid, y);
            copy(y, who_on ? get_who(K * NT + tid) : 0);
          }
        }
      });
      finish();
      if (last) break;
      if (blk == 0 && tid == 0) fetch_add_relaxed(reinterpret_cast<unsigned*>(xch + RES_XSYNC) + RES_N_SPREAD, 1u);
      since = 0;
      if (!meet(epoch)) {
        lost();
        return;
      }
      n_at = n;
      par_at = par;
      step_at = step;
      if (tid == 0) {
        s_vref_at = s_vref;
        s_eff_at = s_eff;
      }
      load_share();
    } else {
      // compaction in place: every survivor is read before any is written
      auto write = [&](auto X, auto K, const R* y, int w) {
        if (c[K] > 0) {
          put(X, xc[K], y);
          if (who_on) put_who(xc[K], w);
        }
        for (int q = 1; __any(q < c[K]); ++q)
          if (q < c[K]) {
            put(X, xc[K] + q, y);
            if (who_on) put_who(xc[K] + q, w);
          }
      };
      auto compact = [&](auto X) {
        if constexpr (HOLD) {
          static_for<W>([&](auto K) {
            if (K * NT < cnt) write(X, K, x[K], who_of[K]);
          });
        } else {
          R y[W][NP];
          int w[W];
          static_for<W>([&](auto K) {
            if (K * NT < cnt && c[K] > 0) get(X, K * NT + tid, y[K]);
          });
          if (who_on) static_for<W>([&](auto K) { w[K] = c[K] > 0 ? get_who(K * NT + tid) : 0; });
          __syncthreads();
          static_for<W>([&](auto K) {
            if (K * NT < cnt) write(X, K, y[K], w[K]);
          });
        }
      };
      if (EXT && (cnt > capl || total > capl)) compact(Any{});
      else compact(Lds{});
      finish();
      base = pre;
      cnt = total;
    }
    __syncthreads();
  }
  // a failed step's walkers stay in the planes of its parity, as the launch-per-step kernels leave
  // them: its input (with importance sampling, moved)
  if (step == stop) store_share();
  __syncthreads();  // the last wave's vref
  if (blk == 0 && tid == 0) {
    Ctrl* C = cold()->ctrl;
    C->n[par] = n;
    C->vref[par] = s_vref;
    C->step[par] = step;
    C->epoch[par] = epoch;
    C->eff_t = s_eff;
    if (step == stop) {
      C->status_step = (long long)step;
      C->status = fail;
    }
  }
}

// The steps of a launch whose gate was closed, by those of G workgroups that run.  They take the G
// shares of k_resident in turn, with the walkers in the global planes, and follow its partition and
// its sums, so the results are the same whoever takes part.  A step is two passes over the shares (one
// more with importance sampling) and a meeting; it is bound by those and by HBM.
template <typename R, int NP, bool IS, int MS, int NTMAX>
__global__ __launch_bounds__(NTMAX) void k_resident_rest(ResArgs<R> A) {
  __shared__ double s_d[16];
  __shared__ __align__(16) int4 s_t[16];
  __shared__ int4 s_res[4];
  __shared__ double s_s0[4], s_vref;
  __shared__ int s_nb[4], s_acc[4], s_late, s_rank, s_team;
  // the shares: first slot and walkers now; copies, and those of the 64 records' earlier shares
  __shared__ int s_base[RES_MAXG], s_cnt[RES_MAXG], s_tot[RES_MAXG], s_ex[RES_MAXG];
  const int NT = blockDim.x, G = gridDim.x, tid = threadIdx.x;
  const int ln = lane_id(), wv = __builtin_amdgcn_readfirstlane(tid / PVD_WAVE), nwv = NT / PVD_WAVE;
  unsigned* sync = reinterpret_cast<unsigned*>(A.xch + RES_XSYNC);
  unsigned* set = sync + A.set * RES_SET;
  if (A.ctrl->status != ST_OK || ld_relaxed_u(set + RES_GATE) != RES_SHUT) return;
  if (tid == 0) {
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    const unsigned at = fetch_add_relaxed(set + RES_JOINED, 1u);
    unsigned team = 0;
    if (at == 0u) {
      while (ld_relaxed_u(set + RES_JOINED) < (unsigned)G && __builtin_amdgcn_s_memrealtime() - t0 < A.team_wait)
        __builtin_amdgcn_s_sleep(1);
      team = __hip_atomic_fetch_or(set + RES_JOINED, RES_SHUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      st_relaxed_u(set + RES_TEAM, team);
    } else if (!(at & RES_SHUT)) {
      while ((team = ld_relaxed_u(set + RES_TEAM)) == 0u && __builtin_amdgcn_s_memrealtime() - t0 < RES_WAIT_MAX)
        __builtin_amdgcn_s_sleep(1);
    }
    s_rank = (int)at;
    s_team = (int)team;  // 0: too late to take part
    s_late = 0;
    s_vref = A.ctrl->vref[A.par];
  }
  if (tid < 16) {
    s_d[tid] = 0.0;
    s_t[tid] = int4{0, 0, 0, 0};
    if (tid < 4) {
      s_res[tid] = int4{0, 0, 0, 0};
      s_s0[tid] = 0.0;
      s_nb[tid] = 0;
      s_acc[tid] = 0;
    }
  }
  __syncthreads();
  const int rank = s_rank, team = s_team;
  if (team == 0) return;
  int par = A.par, n = A.ctrl->n[par], since = 0;
  unsigned long long step = A.ctrl->step[par];
  unsigned epoch = A.ctrl->epoch[par];
  double eff = A.ctrl->eff_t;
  const unsigned long long end = step + (unsigned long long)A.steps;
  const int be = A.branch_every;
  // what the passes leave for each other, by slot: the copies, with importance sampling the energy
  int* cs = reinterpret_cast<int*>(A.ext);
  R* es = A.ext + A.cap;
  auto shares = [&]() {
    for (int v = tid; v < G; v += NT) {
      s_base[v] = (int)((long long)n * v / G);
      s_cnt[v] = (int)((long long)n * (v + 1) / G) - s_base[v];
    }
  };
  shares();
  __syncthreads();
  for (; step < end;) {
    const bool branch = be <= 1 || step % (unsigned long long)be == 0;
    const double vref = s_vref;
    double dte = A.dt;
    const R* src = A.buf[par];
    if constexpr (IS) {
      uint64_t* xacc = A.xch + (size_t)RES_MAXG * (8 + (step & 1));
      R* mv = A.buf[par];
      for (int v = rank; v < G; v += team) {
        const int base = s_base[v], cnt = s_cnt[v];
        int acc = 0;
        for (int k = 0; k * NT < cnt; ++k) {
          const int i = base + k * NT + tid;
          bool a = false;
          if (k * NT + tid < cnt) {
            R y[NP], disp[NP];
            double um, ub;
#pragma unroll
            for (int p = 0; p < NP; ++p) y[p] = mv[p * A.cap + i];
            draw_step<R, NP, false, true>(A, (long long)i, step, disp, um, ub, false);
            const R ke = is_move_fast<R, NP, MS>(A, disp, um, y, a);
            const R pot = pes_eval_s<R, NP, MS>(A.pes, y);
            es[i] = pot + ke;
            if (a) {
#pragma unroll
              for (int p = 0; p < NP; ++p) mv[p * A.cap + i] = y[p];
            }
          }
          acc += __popcll(__ballot(a));
        }
        if (ln == 0) s_t[wv].x = acc;
        __syncthreads();
        if (wv == 0) {
          const int t = dpp_sum16(s_t[ln & 15].x);
          if (ln == 0) st_relaxed(xacc + v, ((uint64_t)epoch << 32) | (unsigned)t);
        }
        __syncthreads();
      }
      for (int g = wv; g * PVD_WAVE < G; g += nwv) {
        const int r = g * PVD_WAVE + ln;
        uint64_t f = 0;
        if (r < G) {
          f = ld_relaxed(xacc + r);
          if (!res_poll(xacc + r, epoch, f)) s_late = 1;
        }
        const int got = dpp_sum((int)(uint32_t)f);
        if (ln == 0) s_acc[g] = got;
      }
      __syncthreads();
      dte = dte * ((double)(unsigned)((s_acc[0] + s_acc[1]) + (s_acc[2] + s_acc[3])) / (double)n);
    }
    // copies and the shares' records
    uint64_t* rec = A.xch + (size_t)(step & 1) * RES_MAXG * 4;
    for (int v = rank; v < G; v += team) {
      const int base = s_base[v], cnt = s_cnt[v];
      double sce = 0.0;
      int bad = 0, copies = 0, births = 0;
      for (int k = 0; k * NT < cnt; ++k) {
        const int i = base + k * NT + tid;
        if (k * NT + tid < cnt) {
          double E;
          int c = 1;
          if constexpr (IS) {
            E = (double)es[i];
            if (branch) {
              const float u = (float)draw_u<R, false>(A, (long long)i, step, RNG_BRANCH);
              c = branch_copies<true>(E, vref, dte, (double)u, A.pop_hi, bad);
            }
          } else {
            R y[NP], disp[NP];
            double um, ub;
            draw_step<R, NP, false, false>(A, (long long)i, step, disp, um, ub, branch);
#pragma unroll
            for (int p = 0; p < NP; ++p) y[p] = src[p * A.cap + i] + disp[p];
            E = (double)pes_eval_s<R, NP, MS>(A.pes, y);
            if (branch) c = branch_copies<sizeof(R) == 4>(E, vref, dte, ub, A.pop_hi, bad);
          }
          cs[i] = c;
          copies += c;
          births += c > 1 ? c - 1 : 0;
          sce += (double)c * E;
        }
      }
      copies = dpp_sum(copies);
      births = dpp_sum(births);
      sce = dpp_sum(sce);
      const bool anybad = __any(bad != 0);
      if (ln == 0) {
        s_t[wv] = int4{(int)min((unsigned)copies, RES_CLAMP), births, anybad ? 1 : 0, 0};
        s_d[wv] = sce;
      }
      __syncthreads();
      if (wv == 0) {
        const int4 wt = s_t[ln & 15];
        const uint64_t bits = (uint64_t)__double_as_longlong(dpp_sum16(s_d[ln & 15]));
        const int total = dpp_sum16(wt.x);
        uint32_t word = ((uint32_t)dpp_sum16(wt.y) & 0x7FFFFFFFu) | (__any(wt.z != 0) ? 0x80000000u : 0u);
        word = ln == 2 ? (uint32_t)bits : word;
        word = ln == 1 ? (uint32_t)(bits >> 32) : word;
        word = ln == 0 ? min((unsigned)total, RES_CLAMP) : word;
        if (ln < 4) st_relaxed(rec + 4 * v + ln, ((uint64_t)epoch << 32) | word);
      }
      __syncthreads();
    }
    // all records, reduced as in k_resident
    for (int g = wv; g * PVD_WAVE < G; g += nwv) {
      const int r = g * PVD_WAVE + ln;
      int tot = 0, nbt = 0, flag = 0;
      double s0 = 0.0;
      if (r < G) {
        uint64_t f[4];
        bool ok = true;
        static_for<4>([&](auto J) {
          f[J] = ld_relaxed(rec + 4 * r + J);
          ok = res_poll(rec + 4 * r + J, epoch, f[J]) && ok;
        });
        if (!ok) s_late = 1;
        tot = (int)(uint32_t)f[0];
        s0 = __longlong_as_double((long long)(f[1] << 32 | (uint64_t)(uint32_t)f[2]));
        nbt = (int)((uint32_t)f[3] & 0x7FFFFFFFu);
        flag = (int)((uint32_t)f[3] >> 31);
      }
      const int inc = dpp_scan(tot), mx = dpp_max(tot);
      if (r < G) {
        s_tot[r] = tot;
        s_ex[r] = inc - tot;
      }
      nbt = dpp_sum(nbt);
      s0 = dpp_sum(s0);
      const bool anyflag = __any(flag != 0);
      if (ln == 0) {
        s_res[g] = int4{lane_of(inc, 63), 0, mx, anyflag ? 1 : 0};
        s_s0[g] = s0;
        s_nb[g] = nbt;
      }
    }
    __syncthreads();
    const int tot = (s_res[0].x + s_res[1].x) + (s_res[2].x + s_res[3].x);
    const int mx = max(max(s_res[0].z, s_res[1].z), max(s_res[2].z, s_res[3].z));
    int st = ST_OK;
    if (s_late) st = ST_SPIN;
    else if (s_res[0].w | s_res[1].w | s_res[2].w | s_res[3].w) st = ST_WEIGHT;
    else if ((double)tot < A.pop_lo || (double)tot > A.pop_hi) st = ST_POP;
    else if (tot > A.cap) st = ST_CAPACITY;
    if (st != ST_OK) {
      // the walkers are those of the failed step, in place (with importance sampling, moved)
      if (tid == 0 && (rank == 0 || st == ST_SPIN)) {
        Ctrl* C = A.ctrl;
        C->n[par] = n;
        C->vref[par] = vref;
        C->step[par] = step;
        C->epoch[par] = epoch + 1;
        C->eff_t = eff;
        C->status_step = (long long)step;
        C->status = st;
      }
      return;
    }
    auto first_slot = [&](int v) {  // of share v's survivors
      int pre = s_ex[v];
      for (int g = 0; g < v / PVD_WAVE; ++g) pre += s_res[g].x;
      return pre;
    };
    // survivors to their np.repeat positions, share by share
    for (int v = rank; v < G; v += team) {
      const int base = s_base[v], cnt = s_cnt[v];
      int at = first_slot(v);
      R* dst = A.buf[par ^ 1];
      const int* wsrc = A.who[par];
      int* wdst = A.who[par ^ 1];
      for (int k = 0; k * NT < cnt; ++k) {
        const int i = base + k * NT + tid;
        const int c = k * NT + tid < cnt ? cs[i] : 0;
        int t, nb;
        const int o = wave_copies(c, t, nb);
        if (ln == 0) s_t[wv].x = t;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < nwv; ++w) {
          const int x = s_t[w].x;
          before += w < wv ? x : 0;
          all += x;
        }
        if (c > 0) {
          R y[NP];
#pragma unroll
          for (int p = 0; p < NP; ++p) y[p] = src[p * A.cap + i];
          if constexpr (!IS) {
            R disp[NP];
            double um, ub;
            draw_step<R, NP, false, false>(A, (long long)i, step, disp, um, ub, branch);
#pragma unroll
            for (int p = 0; p < NP; ++p) y[p] = y[p] + disp[p];
          }
          const int w = A.who_on ? wsrc[i] : 0;
          for (int q = 0; q < c; ++q) {
            const int to = at + before + o + q;
#pragma unroll
            for (int p = 0; p < NP; ++p) dst[p * A.cap + to] = y[p];
            if (A.who_on) wdst[to] = w;
          }
        }
        at += all;
        __syncthreads();
      }
    }
    const double vbar = ((s_s0[0] + s_s0[1]) + (s_s0[2] + s_s0[3])) / (double)tot;
    const double corr = (double)(tot - (int)A.n0) / A.n0;
    const double vnew = vbar - (A.alpha * corr);
    if (IS && (long long)step < A.tmax) eff = branch ? (step == 0 ? 0.0 : eff) + dte : 0.0;
    if (rank == 0 && tid == 0 && (long long)step < A.tmax) {
      A.tr_vref[step] = vnew;
      A.tr_pop[step] = (double)tot;
      const int nbt = (s_nb[0] + s_nb[1]) + (s_nb[2] + s_nb[3]);
      A.tr_births[step] = nbt;
      A.tr_deaths[step] = n + nbt - tot;
      if (IS) A.tr_dteff[step] = eff;
    }
    // the partition that k_resident would have now
    const int even = (tot + G - 1) / G;
    ++since;
    const bool spread = mx > A.capb || ((mx + NT - 1) / NT > (even + NT - 1) / NT && since >= RES_REB);
    __syncthreads();
    n = tot;
    if (spread) {
      since = 0;
      shares();
    } else {
      for (int v = tid; v < G; v += NT) {
        s_base[v] = first_slot(v);
        s_cnt[v] = s_tot[v];
      }
    }
    if (tid == 0) s_vref = vnew;
    par ^= 1;
    ++step;
    ++epoch;
    // everyone's survivors before anyone's next step
    uint64_t* xbar = A.xch + (size_t)RES_MAXG * 10;
    store_complete();
    __syncthreads();
    if (tid == 0) {
      fence_release();
      st_relaxed(xbar + rank, ((uint64_t)epoch << 32) | 1u);
    }
    for (int r = tid; r < team; r += NT) {
      uint64_t f = ld_relaxed(xbar + r);
      if (!res_poll(xbar + r, epoch, f)) s_late = 1;
    }
    __syncthreads();
    fence_acquire();
  }
  Ctrl* C = A.ctrl;
  if (rank == 0 && tid == 0) {
    C->n[par] = n;
    C->vref[par] = s_vref;
    C->step[par] = step;
    C->epoch[par] = epoch;
    C->eff_t = eff;
  }
  if (tid == 0 && s_late) {
    C->status_step = (long long)step;
    C->status = ST_SPIN;
  }
}

// The forms: FP32 and FP64 plain steps for the fused component counts, and FP32 importance sampling
// with the compiled trials.  A form is an object of its own (pvd_resident_form.hip): the first launch
// out of an object waits until all of its code is on the device, 0.35 ms and 1 ms more a megabyte
// (all forms together: 1.8 ms).
enum : int { RF_1, RF_3, RF_WATER, RF_TRIATOMIC, RF_CLUSTER, RF_WATER_IS, RF_TRIATOMIC_IS, RF_CLUSTER_IS, RF_1_F64,
             RF_3_F64, RF_WATER_F64, RF_TRIATOMIC_F64, RF_COUNT };

// W rounds of at most NTM threads in the shape for large populations
template <int F>
struct ResForm;
#define PVD_RES_FORM(F, R_, NP_, IS_, MS_, W_, NTM_)                \
  template <>                                                       \
  struct ResForm<F> {                                               \
    using R = R_;                                                   \
    static constexpr int NP = NP_, MS = MS_, W = W_, NTM = NTM_;    \
    static constexpr bool IS = IS_;                                 \
  };
PVD_RES_FORM(RF_1, float, 1, false, MS_ANY, 6, 1024)
PVD_RES_FORM(RF_3, float, 3, false, MS_ANY, 6, 1024)
PVD_RES_FORM(RF_WATER, float, 9, false, MS_PES_WATER, 6, 1024)
PVD_RES_FORM(RF_TRIATOMIC, float, 9, false, MS_ANY, 6, 1024)
PVD_RES_FORM(RF_CLUSTER, float, 18, false, MS_PES_CLUSTER, 3, 1024)
PVD_RES_FORM(RF_WATER_IS, float, 9, true, (MS_PES_WATER | MS_TRIAL_WATER), 6, 1024)
PVD_RES_FORM(RF_TRIATOMIC_IS, float, 9, true, MS_TRIAL_WATER, 6, 1024)
PVD_RES_FORM(RF_CLUSTER_IS, float, 18, true, (MS_PES_CLUSTER | MS_TRIAL_CLUSTER), 6, 512)
PVD_RES_FORM(RF_1_F64, double, 1, false, MS_ANY, 6, 1024)
PVD_RES_FORM(RF_3_F64, double, 3, false, MS_ANY, 6, 1024)
PVD_RES_FORM(RF_WATER_F64, double, 9, false, MS_PES_WATER, 6, 512)
PVD_RES_FORM(RF_TRIATOMIC_F64, double, 9, false, MS_ANY, 6, 512)
#undef PVD_RES_FORM

// a form's kernels in one of its two shapes
struct Instance {
  const void* fn;
  const void* rest;
  int W, ntmax, stride;
};
template <int F>
Instance res_instance(bool small);

}  // namespace pvd
