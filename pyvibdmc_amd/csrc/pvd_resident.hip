// Resident discrete steps (pvd_resident.hpp): the launch plan of a simulation and its launches.
#include <mutex>

#include "pvd_resident.hpp"

namespace pvd {

namespace {

// The simulations of a device that may keep walkers on chip.  A launch's workgroups hold their CUs
// while they wait for the last of them, so launches on several streams must not each get a part of
// the CUs: with three of a million walkers, two would wait for each other at their gates whenever the
// third ends (96 ms step by step, 500 to 600 so, 94 in order).  Launches that together take more than
// all CUs are therefore put in the order of their calls with events; smaller ones run beside each
// other.  With one simulation nothing is recorded: a second one's creation ends with a synchronisation
// of the device after it has joined.
struct ResDevice {
  std::mutex mu;
  std::vector<pvd_sim*> sims;
  unsigned long long turn = 0;
};
constexpr int RES_DEVICES = 64;
ResDevice& res_device(int dev) {
  static ResDevice* devices = new ResDevice[RES_DEVICES];  // not destroyed: simulations may outlive static objects
  return devices[dev];
}

// the stream waits until what is left of the others' launches fits beside `share` of the CUs
int res_wait_turn(ResDevice& D, pvd_sim* s, double share, hipStream_t st) {
  std::vector<pvd_sim*> others;
  double sum = share;
  for (pvd_sim* o : D.sims)
    if (o != s && o->res_turn) {
      others.push_back(o);
      sum += o->res_share;
    }
  std::sort(others.begin(), others.end(), [](const pvd_sim* a, const pvd_sim* b) { return a->res_turn < b->res_turn; });
  for (size_t k = 0; k < others.size() && sum > 1.0 + 1e-9; ++k) {
    HIPCHK(hipStreamWaitEvent(st, others[k]->res_done, 0));
    sum -= others[k]->res_share;
  }
  return 0;
}

// Largest dynamic LDS a workgroup of k_resident may ask for: 160 KB less its static arrays.
constexpr int RES_LDS = 160 * 1024 - 5 * 1024;

template <typename R>
Instance instance(const pvd_sim* s, bool small) {
  const int ms = s->mspec;
  if constexpr (sizeof(R) == 4) {
    if (s->is) {
      if (s->np == 9 && ms == (MS_PES_WATER | MS_TRIAL_WATER)) return res_instance<RF_WATER_IS>(small);
      if (s->np == 9 && ms == MS_TRIAL_WATER) return res_instance<RF_TRIATOMIC_IS>(small);
      if (s->np == 18 && ms == (MS_PES_CLUSTER | MS_TRIAL_CLUSTER)) return res_instance<RF_CLUSTER_IS>(small);
    } else {
      if (s->np == 1) return res_instance<RF_1>(small);
      if (s->np == 3) return res_instance<RF_3>(small);
      if (s->np == 9 && (ms & MS_PES_WATER)) return res_instance<RF_WATER>(small);
      if (s->np == 9) return res_instance<RF_TRIATOMIC>(small);
      if (s->np == 18 && (ms & MS_PES_CLUSTER)) return res_instance<RF_CLUSTER>(small);
    }
  } else if (!s->is) {
    if (s->np == 1) return res_instance<RF_1_F64>(small);
    if (s->np == 3) return res_instance<RF_3_F64>(small);
    if (s->np == 9 && (ms & MS_PES_WATER)) return res_instance<RF_WATER_F64>(small);
    if (s->np == 9) return res_instance<RF_TRIATOMIC_F64>(small);
  }
  return Instance{nullptr, nullptr, 0, 0, 0};
}

// Workgroups, threads and LDS of the resident launch, or fn = nullptr where it does not serve:
// N0 walkers must fit the LDS of the workgroups with 2 % to spare (the rest of the population's
// range lives in the per-workgroup extension), every capacity's worth of walkers the rounds, and
// the grid must be resident at once.
struct Plan {
  const void* fn;
  const void* rest;
  int grid, nt, capl, capb;
  size_t lds;
  double share;  // of the CUs
};

template <typename R>
Plan make_plan(pvd_sim* s, bool who) {
  Plan P{nullptr, nullptr, 0, 0, 0, 0, 0, 0.0};
  const long long n0 = s->cfg.num_walkers;
  const int gmax = std::min(s->cus, RES_MAXG);
  const int share = 256;
  const int g = (int)std::max(1ll, std::min<long long>(gmax, (n0 + share - 1) / share));
  const long long per = (n0 + g - 1) / g, most = (s->cap + g - 1) / g;
  const bool small = most <= 2 * 512 && per + per / 16 <= 512;
  const Instance I = instance<R>(s, small);
  if (!I.fn) return P;
  int nt = 64;
  while (nt < I.ntmax && (nt < per + per / 16 || nt * I.W < most)) nt *= 2;
  const int unit = I.stride * (int)sizeof(R) + (who ? (int)sizeof(int) : 0);
  const int capb = nt * I.W;
  const int capl = std::min(capb, RES_LDS / unit / PVD_WAVE * PVD_WAVE);
  if (per + per / 50 > (who ? capb : capl) || most > capb || (small && capl < capb)) return P;
  // the extension lives in the staging buffer (np doubles per slot)
  if ((long long)g * (capb - capl) * (I.stride + 1) * (long long)sizeof(R) > (long long)sizeof(double) * s->np * s->cap)
    return P;
  P.lds = (size_t)unit * capl;
  // the same limit from every caller: it belongs to the kernel, and another thread may be between its
  // own plan, of another size, and its launch
  if (hipFuncSetAttribute(I.fn, hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS) != hipSuccess) {
    (void)hipGetLastError();
    return P;
  }
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, I.fn, nt, P.lds) != hipSuccess ||
      (long long)per_cu * s->cus < g) {
    (void)hipGetLastError();
    return P;
  }
  P.share = (double)g / ((double)per_cu * s->cus);
  P.fn = I.fn;
  P.rest = I.rest;
  P.grid = g;
  P.nt = nt;
  P.capl = capl;
  P.capb = capb;
  return P;
}

}  // namespace

// Steps of one launch at most, a bound on how long other streams' kernels that need LDS wait: a launch
// that fills the LDS (all but the small shape do) holds the CUs for 128 steps, 2 ms for a million
// triatomics, 4 to 5 ms with importance sampling, on the Partridge-Schwenke surface and for 500 000
// clusters; 4096 steps were 60 to 180 ms (a library product on another stream beside a million
// walkers: 58 ms, now 1).  It costs nothing: even shares again make up for the launch (us a step in
// calls of 4096 and 128 steps: a million walkers 15.9, 15.6; with importance sampling 30.9, 30.9).
// RES_MIN: the fewest steps for which it is used.  A call costs about 20 us more than a step kernel's
// launch does (the second launch, walkers in and out).  us a step in calls of 16 steps, here and
// launch per step: water 1 000 walkers 4.3, 9.0; 100 000 4.8, 10.7;
// 1 000 000 15.3, 21.0; with importance sampling 31.4, 50.5; cluster with it, 500 000 36.0, 56.9.
// The first RES_REPAY steps of a simulation that asks for them a few at a time stay with the step
// kernels: the first launch of a form in a process takes 0.41 ms more (its code, see RF_1), which 5 us
// a step repay after about 80 (the first 20 steps of a million walkers: 0.46 ms, 0.75 without this rule).
constexpr int RES_STEPS = 4096, RES_STEPS_FULL = 128;
constexpr int RES_MIN = 16;
constexpr int RES_REPAY = 96;

template <typename R>
int run_resident(pvd_sim* s, int n_steps, hipStream_t st, int& done) {
  done = 0;
  s->steps_asked += n_steps;
  if (s->cont || !s->xch || s->htrial || s->cfg.pes.kind == PES_EXTERNAL || n_steps < RES_MIN ||
      s->steps_asked < RES_REPAY || s->res_dev < 0 || s->res_dev >= RES_DEVICES)
    return 0;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return 0;
  }
  const Plan P = make_plan<R>(s, s->who_on);
  if (!P.fn) return 0;
  ResArgs<R> A;
  std::memset(&A, 0, sizeof(A));
  for (int b = 0; b < 2; ++b) {
    A.buf[b] = (R*)s->coords[b];
    A.who[b] = s->who[b];
  }
  A.ext = (R*)s->stage;
  A.ctrl = s->ctrl;
  A.xch = s->xch;
  A.tr_vref = s->tr_vref;
  A.tr_pop = s->tr_pop;
  A.tr_dteff = s->tr_dteff;
  A.tr_births = s->tr_births;
  A.tr_deaths = s->tr_deaths;
  A.cap = s->cap;
  A.tmax = s->tmax;
  const StepArgs<R> S = make_args<R>(s);
  A.dt = S.dt;
  A.alpha = S.alpha;
  A.n0 = S.n0;
  A.pop_lo = S.pop_lo;
  A.pop_hi = S.pop_hi;
  A.branch_every = s->cfg.branch_every > 0 ? s->cfg.branch_every : 1;
  A.capl = P.capl;
  A.capb = P.capb;
  A.gate_wait = s->res_gate_wait;
  A.team_wait = s->res_team_wait;
  A.who_on = s->who_on ? 1 : 0;
  A.rng = S.rng;
  A.pes.kind = S.pes.kind;
  std::memcpy(A.pes.idx, S.pes.idx, sizeof(A.pes.idx));
  for (int k = 0; k < 12; ++k) A.pes.p[k] = (R)S.pes.p[k];
  for (int k = 0; k < PVD_MAX_TB; ++k) {
    A.trial.balpha[k] = (R)S.trial.balpha[k];
    A.trial.br0[k] = (R)S.trial.br0[k];
  }
  for (int k = 0; k < PVD_MAX_TA; ++k) {
    A.trial.aalpha[k] = (R)S.trial.aalpha[k];
    A.trial.ath0[k] = (R)S.trial.ath0[k];
  }
  A.trial.c0 = (R)S.trial.c0;
  for (int p = 0; p < s->np; ++p) {
    A.sigma[p] = (R)S.sigma[p];
    A.inv_m[p] = (R)S.inv_m[p];
    A.h2s[p] = S.h2s[p];
  }
  ResDevice& D = res_device(s->res_dev);
  std::lock_guard<std::mutex> lock(D.mu);
  const bool shared = D.sims.size() > 1;
  if (shared) {
    if (!s->res_done) HIPCHK(hipEventCreateWithFlags(&s->res_done, hipEventDisableTiming));
    const int rc = res_wait_turn(D, s, P.share, st);
    if (rc) return rc;
  }
  while (done < n_steps) {
    A.steps = std::min(P.lds > RES_LDS / 2 ? RES_STEPS_FULL : RES_STEPS, n_steps - done);
    A.par = (int)(s->next_step & 1);
    void* args[] = {&A};
    A.set = (int)(s->res_launches & 1);
    HIPCHK(hipLaunchKernel(P.fn, dim3(P.grid), dim3(P.nt), args, P.lds, st));
    if (P.grid == 1) {
      ++s->res_alone;
    } else {
      ++s->res_launches;
      HIPCHK(hipLaunchKernel(P.rest, dim3(P.grid), dim3(P.nt), args, 0, st));
    }
    s->next_step += A.steps;
    s->epoch_next += 2 * (unsigned)A.steps + 2;  // a failed launch retraces its steps under new epochs
    done += A.steps;
  }
  if (shared) {
    HIPCHK(hipEventRecord(s->res_done, st));
    s->res_share = P.share;
    s->res_stream = st;
    s->res_turn = ++D.turn;
  }
  return 0;
}

void resident_join(pvd_sim* s) {
  if (!s->xch || s->res_dev < 0 || s->res_dev >= RES_DEVICES) return;
  ResDevice& D = res_device(s->res_dev);
  std::lock_guard<std::mutex> lock(D.mu);
  D.sims.push_back(s);
}

void resident_leave(pvd_sim* s) {
  if (!s->xch || s->res_dev < 0 || s->res_dev >= RES_DEVICES) return;
  ResDevice& D = res_device(s->res_dev);
  std::lock_guard<std::mutex> lock(D.mu);
  D.sims.erase(std::remove(D.sims.begin(), D.sims.end(), s), D.sims.end());
  if (s->res_done) (void)hipEventDestroy(s->res_done);
  s->res_done = nullptr;
}

void resident_idle(pvd_sim* s, hipStream_t st) {
  if (!s->res_turn || s->res_stream != st) return;
  std::lock_guard<std::mutex> lock(res_device(s->res_dev).mu);
  s->res_turn = 0;
}

template int run_resident<float>(pvd_sim*, int, hipStream_t, int&);
template int run_resident<double>(pvd_sim*, int, hipStream_t, int&);

}  // namespace pvd
