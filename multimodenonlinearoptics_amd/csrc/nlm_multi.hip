// nlm_multi.hip -- heterogeneous batches: many independent propagations of
// different media (model, nFreqs, nZSteps, dispersion, pump) in one graph launch.
//
// Each instance is one batchSignalSimulation row of its own medium
// (src/_NonlinearMedium.cpp:378-444; the FNLM overload
// src/_FullyNonlinearMedium.hpp:8-11).  Instances are grouped into classes by
// (model, log2 N); every class runs as one persistent kernel whose workgroups
// take instances from a device work queue (one atomic counter per class) in
// order of decreasing nZ, so long propagations start first and short ones fill
// the tail.  What a medium's pump contributes is formed before the propagations, for
// all steps at once (nlm_multi_stage.hip): the step tables of one-mode media, the
// pump rows of multi-mode media with a linear pump; media whose tables or rows do not
// fit in memory generate their rows inside the kernel (InlinePump).  Chi3 (nonlinear
// pump) and Chi2SFGOPA (two pumps) start from their plan's device pump grids.  Every
// solver has a kernel (Chi3GNLSE with its transforms inside the RK stages).
// Everything is captured into one hipGraph (staging, then the classes on four
// chains); nlm_multi_launch replays it.
//
// The number of persistent workgroups of a class is chosen by a small
// autotuner at creation: each class is timed alone for a few grid sizes and
// the fastest kept (per process, keyed by model, log2 N and instance count).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <tuple>
#include <vector>

#include "nlm_internal.hpp"
#include "nlm_multi.hpp"

__global__ void k_zero_ints(int* p, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0;
}

// Kernel of a class: models sharing a right-hand side share kernels (Chi2AFC
// runs Chi2SFG's, Chi2ASHG Chi2SHG's).
static int class_model(int model) {
  return model == NLM_CHI2AFC ? NLM_CHI2SFG : model == NLM_CHI2ASHG ? NLM_CHI2SHG : model;
}

static multi_fn pick_multi(int model, int L, int form) {
  switch (class_model(model)) {
    case NLM_CHI3: return nlm_pick_multi_0(L, form);
    case NLM_CHI2PDC: return nlm_pick_multi_1(L, form);
    case NLM_CHI2SFG: return nlm_pick_multi_2(L, form);
    case NLM_CHI2SFGPDC: return nlm_pick_multi_4(L, form);
    case NLM_CHI2SFGII: return nlm_pick_multi_5(L, form);
    case NLM_CHI2PDCII: return nlm_pick_multi_6(L, form);
    case NLM_CHI2SFGOPA: return nlm_pick_multi_7(L, form);
    case NLM_CHI2SFGXPM: return nlm_pick_multi_8(L, form);
    case NLM_CHI2SHG: return nlm_pick_multi_9(L, form);
    case NLM_CHI2SHGOPA: return nlm_pick_multi_10(L, form);
    case NLM_CHI2DSFG: return nlm_pick_multi_11(L, form);
    case NLM_CHI2SHGXPM: return nlm_pick_multi_12(L, form);
    case NLM_CHI3GNLSE: return nlm_pick_multi_14(L, form);
  }
  return nullptr;
}

struct MultiClass {
  int model, L, count, grid;
  int form;         // MULTI_FIELD, MULTI_INLINE, MULTI_MODES or MULTI_TAB
  int stage;        // STAGE_*: what is formed before the propagation kernel
  size_t staged;    // its bytes
  int chunkOff = 0, nChunks = 0;
  multi_fn fn;
  size_t orderOff;  // offset of this class's instance order in the order array
  hipStream_t stream = nullptr;
  hipEvent_t done = nullptr;
};

struct nlm_multi_s {
  int n = 0;
  std::vector<int> N, nOut;
  std::vector<size_t> outOff;
  DevBuf<cplx> inBuf, outBuf, envBuf;
  DevBuf<double> realBuf;
  DevBuf<MultiInst> inst;
  DevBuf<int> order, counters;
  DevBuf<cplx> stageBuf;  // step tables and pump rows of the staged classes
  DevBuf<int> chunks;     // their chunks (instance, first step)
  std::vector<MultiClass> classes;
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, t0 = nullptr, t1 = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // host copy of the last launch's outputs, made by the first nlm_multi_output after it
  std::mutex outMu;
  std::vector<cplx> hostOut;
  bool hostOutOf = false;
  float lastMs = 0.f;
};

static std::mutex g_tune_mu;
static std::map<std::tuple<int, int, int, int>, int> g_tuned;  // (model, L, form, count) -> grid

static void launch_stage(nlm_multi_s* m, const MultiClass& c, const cplx* tw, hipStream_t s) {
  nlm_multi_stage(c.stage, c.model, c.L, m->inst.p, m->chunks.p + 2 * (size_t)c.chunkOff, c.nChunks, tw, s);
}

static int run_class(nlm_multi_s* m, const MultiClass& c, int grid, const cplx* tw, hipStream_t s) {
  launch_stage(m, c, tw, s);
  hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, m->counters.p + (&c - m->classes.data()), 1);
  c.fn(m->inst.p, m->order.p + c.orderOff, c.count, m->counters.p + (&c - m->classes.data()), tw, grid, s);
  HIP_TRY(hipGetLastError());
  return NLM_OK;
}

extern "C" int nlm_multi_destroy(nlm_multi* m) {
  if (!m) return NLM_OK;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  if (m->exec) (void)hipGraphExecDestroy(m->exec);
  if (m->graph) (void)hipGraphDestroy(m->graph);
  for (auto& c : m->classes) {
    if (c.stream) (void)hipStreamDestroy(c.stream);
    if (c.done) (void)hipEventDestroy(c.done);
  }
  if (m->fork) (void)hipEventDestroy(m->fork);
  if (m->t0) (void)hipEventDestroy(m->t0);
  if (m->t1) (void)hipEventDestroy(m->t1);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return NLM_OK;
}

extern "C" int nlm_multi_create(int n, const nlm_multi_item* items, int autotune, nlm_multi** out) {
  return nlm_multi_create_staged(n, items, autotune, -1, out);
}

extern "C" int nlm_multi_create_staged(int n, const nlm_multi_item* items, int autotune, int64_t stage_bytes,
                                       nlm_multi** out) {
  if (!out || n < 0 || (n > 0 && !items)) return set_err(NLM_INVALID_ARGUMENT, "invalid arguments");
  *out = nullptr;
  autotune &= 1;  // bit 1 (stage the pump rows) is accepted; staging is the rule below
  nlm_multi_s* m = new nlm_multi_s();
  auto fail = [&](int code) {
    nlm_multi_destroy(m);
    return code;
  };
  m->n = n;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&m->fork) != hipSuccess || hipEventCreate(&m->t0) != hipSuccess ||
      hipEventCreate(&m->t1) != hipSuccess)
    return fail(set_err(NLM_DEVICE_ERROR, "stream/event creation failed"));

  // sizes of the packed per-instance buffers
  size_t inTot = 0, outTot = 0, envTot = 0, realTot = 0;
  std::map<std::tuple<int, int, int>, std::vector<int>> byClass;  // (class model, L, generated pump)
  m->N.resize(n);
  m->nOut.resize(n);
  m->outOff.resize(n);
  for (int i = 0; i < n; i++) {
    const nlm_multi_item& it = items[i];
    nlm_plan* p = it.plan;
    if (!p) return fail(set_err(NLM_INVALID_ARGUMENT, "null plan in item"));
    const bool pumped = p->nP > 0;
    const bool inl = pumped && it.envelope != nullptr;
    if (inl && (p->nP != 1 || p->model == NLM_CHI3))
      return fail(set_err(NLM_INVALID_ARGUMENT,
                          "a pump generated in the batch needs a single linear pump; pass no envelope and run the "
                          "medium's pump simulation instead"));
    if (!pick_multi(p->model, p->L, inl ? MULTI_INLINE : MULTI_FIELD) && !pick_multi(p->model, p->L, MULTI_MODES))
      return fail(set_err(NLM_INVALID_ARGUMENT, "heterogeneous batches take nFreqs a power of two, 32..4096"));
    if (!it.input || it.cols <= 0 || it.cols % p->N != 0 || it.cols / p->N > p->nS)
      return fail(set_err(NLM_INVALID_ARGUMENT, "Signals not of correct length!"));
    if (it.input_mode < 0 || it.input_mode >= p->nS)
      return fail(set_err(NLM_INVALID_ARGUMENT, "inputModes does not match any mode in the system"));
    if (it.n_out < 1 || it.n_out > p->nS) return fail(set_err(NLM_INVALID_ARGUMENT, "Requested no outputs!"));
    for (int q = 0; q < it.n_out; q++)
      if (it.outputs[q] < 0 || it.outputs[q] >= p->nS)
        return fail(set_err(NLM_INVALID_ARGUMENT, "output mode out of range"));
    if (inl && !it.disp_pump)
      return fail(set_err(NLM_INVALID_ARGUMENT, "a generated pump needs the pump dispersion"));
    if (pumped && !inl)
      if (int e = check_pumps_ready(p)) return fail(e);
    m->N[i] = p->N;
    m->nOut[i] = it.n_out;
    m->outOff[i] = outTot;
    inTot += it.cols;
    outTot += (size_t)it.n_out * p->N;
    if (inl) {
      envTot += p->N;
      realTot += p->N + (it.strength ? 2 * (size_t)p->nZ - 1 : 0);
    }
    byClass[std::make_tuple(class_model(p->model), p->L, inl ? 1 : 0)].push_back(i);
  }
  int e;
  if ((e = m->inBuf.ensure(inTot)) || (e = m->outBuf.ensure(outTot)) || (e = m->envBuf.ensure(envTot)) ||
      (e = m->realBuf.ensure(realTot)) || (e = m->inst.ensure(n)) || (e = m->order.ensure(n)))
    return fail(e);

  // descriptors and packed uploads
  std::vector<MultiInst> hi(n);
  std::vector<cplx> hin(inTot), henv(envTot);
  std::vector<double> hreal(realTot);
  size_t io = 0, eo = 0, ro = 0;
  for (int i = 0; i < n; i++) {
    const nlm_multi_item& it = items[i];
    nlm_plan* p = it.plan;
    MultiInst& d = hi[i];
    memset(&d, 0, sizeof d);
    d.dstep = p->dstep.p;
    d.halfIn = p->halfIn.p;
    d.halfOut = p->halfOut.p;
    d.coef = p->coef.p;
    d.cconst = p->cconst.p;
    std::memcpy(hin.data() + io, it.input, sizeof(cplx) * it.cols);
    d.in = m->inBuf.p + io;
    io += it.cols;
    d.out = m->outBuf.p + m->outOff[i];
    d.nZ = p->nZ;
    d.inTime = it.in_time_domain ? 1 : 0;
    d.inCols = it.cols;
    d.nOut = it.n_out;
    for (int q = 0; q < 4; q++) d.inPos[q] = d.outPos[q] = -1;
    input_channels(p->nS, it.cols / p->N, it.input_mode, d.inPos);
    for (int q = 0; q < it.n_out; q++) d.outPos[it.outputs[q]] = q;
    d.raman = p->raman.p;
    d.filt = p->filt.p;
    if (p->nP > 0 && !it.envelope) {
      d.pump0 = p->pumpT[0].p;
      d.pump1 = p->nP > 1 ? p->pumpT[1].p : nullptr;
    }
    if (p->nP > 0 && it.envelope) {
      std::memcpy(henv.data() + eo, it.envelope, sizeof(cplx) * p->N);
      d.env = m->envBuf.p + eo;
      eo += p->N;
      std::memcpy(hreal.data() + ro, it.disp_pump, sizeof(double) * p->N);
      d.Dp = m->realBuf.p + ro;
      ro += p->N;
      if (it.strength) {
        std::memcpy(hreal.data() + ro, it.strength, sizeof(double) * (2 * (size_t)p->nZ - 1));
        d.strength = m->realBuf.p + ro;
        ro += 2 * (size_t)p->nZ - 1;
      }
      d.dzp = it.dzp;
    }
  }
  // What each class stages, the largest fields first (they are the longest chains and
  // gain most) while everything staged fits the caller's limit, by default a quarter of the
  // device memory and half of what is free: the step table of one-mode media (32 bytes per point and step), or
  // the pump rows of multi-mode media with a generated pump (as many bytes).  A class
  // that does not fit generates its rows in the kernel, or reads its grids.
  // SHG / PDC media of nFreqs 256..4096, nZSteps 200..4000, launch ms with every class
  // generating its rows and the modes sharing lanes -> now: 2000 media 156 -> 132 (the
  // N = 4096 tables take 54 GB of the budget, the other classes generate theirs), 500
  // media 149 -> 68 (all staged, 27 GB).
  // Where the buffer cannot be had after all (memory taken since by another thread or process),
  // half of it is tried, and in the end none.
  std::vector<MultiClass> cls;
  std::vector<std::vector<int>> members;
  for (auto& kv : byClass) {
    MultiClass c;
    c.model = std::get<0>(kv.first);
    c.L = std::get<1>(kv.first);
    cls.push_back(c);
    members.push_back(kv.second);
  }
  std::vector<int> bySize(cls.size());
  for (size_t k = 0; k < cls.size(); k++) bySize[k] = (int)k;
  std::stable_sort(bySize.begin(), bySize.end(), [&](int a, int b) { return cls[a].L > cls[b].L; });
  // the forms for a budget in bytes; returns the elements that they stage
  const auto choose = [&](size_t budget) {
    size_t total = 0;
    for (int k : bySize) {
      MultiClass& c = cls[k];
      const nlm_multi_item& it = items[members[k][0]];
      const bool inl = it.plan->nP > 0 && it.envelope != nullptr;
      const bool groups = pick_multi(c.model, c.L, MULTI_MODES) != nullptr;
      const bool table = pick_multi(c.model, c.L, MULTI_TAB) != nullptr;
      c.stage = STAGE_NONE;
      c.staged = 0;
      c.form = inl ? MULTI_INLINE : groups ? MULTI_MODES : MULTI_FIELD;
      if (!table && !(inl && groups)) continue;
      size_t need = 0;
      for (int i : members[k]) need += (size_t)2 * hi[i].nZ * m->N[i];
      if (need * sizeof(cplx) > budget) continue;
      budget -= need * sizeof(cplx);
      total += need;
      c.staged = need * sizeof(cplx);
      c.stage = !table ? STAGE_ROWS : inl ? STAGE_TAB : STAGE_TAB_GRID;
      c.form = table ? MULTI_TAB : MULTI_MODES;
    }
    return total;
  };
  size_t freeB = 0, totalB = 0;
  if (hipMemGetInfo(&freeB, &totalB) != hipSuccess) freeB = totalB = 0;
  size_t stageTot = choose(stage_bytes < 0 ? std::min(totalB / 4, freeB / 2) : (size_t)stage_bytes);
  while (m->stageBuf.ensure(stageTot)) {
    (void)hipGetLastError();
    stageTot = choose(stageTot * sizeof(cplx) / 2);
  }
  for (auto& c : cls) {
    c.fn = pick_multi(c.model, c.L, c.form);
    if (!c.fn) return fail(set_err(NLM_INVALID_ARGUMENT, "heterogeneous batches take nFreqs a power of two, 32..4096"));
  }
  if ((e = m->counters.ensure(cls.size() + 1))) return fail(e);
  std::vector<int> hchunks;
  size_t stageOff = 0;
  // the classes' longest-first orders
  std::vector<int> hord;
  hord.reserve(n);
  for (size_t k = 0; k < cls.size(); k++) {
    MultiClass c = cls[k];
    if (c.stage != STAGE_NONE) {
      c.chunkOff = (int)(hchunks.size() / 2);
      for (int i : members[k]) {
        if (c.stage == STAGE_ROWS) hi[i].pump0 = m->stageBuf.p + stageOff;
        else hi[i].tab = m->stageBuf.p + stageOff;
        stageOff += (size_t)2 * hi[i].nZ * m->N[i];
        for (int s = 1; s < hi[i].nZ || s == 1; s += MULTI_CHUNK) {
          hchunks.push_back(i);
          hchunks.push_back(s);
        }
      }
      c.nChunks = (int)(hchunks.size() / 2) - c.chunkOff;
    }
    std::vector<int> idx = members[k];
    std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) { return hi[a].nZ > hi[b].nZ; });
    c.orderOff = hord.size();
    hord.insert(hord.end(), idx.begin(), idx.end());
    c.count = (int)idx.size();
    c.grid = 1;
    m->classes.push_back(c);
  }
  if (!hchunks.empty()) {
    if ((e = m->chunks.ensure(hchunks.size()))) return fail(e);
    HIP_TRY(hipMemcpy(m->chunks.p, hchunks.data(), sizeof(int) * hchunks.size(), hipMemcpyHostToDevice));
  }
  if (n > 0) {
    HIP_TRY(hipMemcpy(m->inst.p, hi.data(), sizeof(MultiInst) * n, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(m->order.p, hord.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(m->inBuf.p, hin.data(), sizeof(cplx) * inTot, hipMemcpyHostToDevice));
    if (envTot) HIP_TRY(hipMemcpy(m->envBuf.p, henv.data(), sizeof(cplx) * envTot, hipMemcpyHostToDevice));
    if (realTot) HIP_TRY(hipMemcpy(m->realBuf.p, hreal.data(), sizeof(double) * realTot, hipMemcpyHostToDevice));
  }

  // grid sizes: autotuned per class (timed alone) or the default of four
  // workgroups per CU, never more workgroups than instances
  const int cus = device_cus();
  for (auto& c : m->classes) {
    const cplx* tw = nullptr;
    if ((e = get_twiddles(1 << c.L, &tw))) return fail(e);
    const int cand[4] = {cus, 2 * cus, 4 * cus, 8 * cus};
    int best = std::min(c.count, 4 * cus);
    const auto key = std::make_tuple(c.model, c.L, c.form, c.count);
    bool cached = false;
    {
      std::lock_guard<std::mutex> lk(g_tune_mu);
      auto f = g_tuned.find(key);
      if (f != g_tuned.end()) {
        best = f->second;
        cached = true;
      }
    }
    if (autotune && !cached && c.count > cus) {
      float bestMs = 1e30f;
      for (int g : cand) {
        const int grid = std::min(c.count, g);
        if ((e = run_class(m, c, grid, tw, m->stream))) return fail(e);  // warm
        HIP_TRY(hipEventRecord(m->t0, m->stream));
        if ((e = run_class(m, c, grid, tw, m->stream))) return fail(e);
        HIP_TRY(hipEventRecord(m->t1, m->stream));
        HIP_TRY(hipEventSynchronize(m->t1));
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, m->t0, m->t1));
        if (ms < bestMs) {
          bestMs = ms;
          best = grid;
        }
        if (grid == c.count) break;
      }
      std::lock_guard<std::mutex> lk(g_tune_mu);
      g_tuned[key] = best;
    }
    c.grid = std::max(1, best);
    if (hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c.done, hipEventDisableTiming) != hipSuccess)
      return fail(set_err(NLM_DEVICE_ERROR, "stream/event creation failed"));
  }

  // Capture on at most four chains, one per hardware queue (a process has four, and
  // work of streams that share one runs in order anyway): the classes by decreasing
  // estimated time, each appended, its staging first, to the chain that is free first,
  // so that the longest propagations start at once.  No chain waits for another: with
  // the staging in a chain of its own and the staged classes waiting for it, the
  // graph's branches were put on the queues in another order and the longest class
  // started last (500 SHG / PDC media 127 ms).
  if (!m->classes.empty()) {
    constexpr int CHAINS = 4;
    const int nc = (int)m->classes.size(), chains = std::min(CHAINS, nc);
    std::vector<int> byCost(nc);
    std::vector<double> cost(nc);
    for (int k = 0; k < nc; k++) {
      const MultiClass& c = m->classes[k];
      byCost[k] = k;
      // microseconds per step of one propagation beside others: step-table classes, and
      // the others (several modes or transforms per step); staging writes 32 bytes per
      // point and step at ~2 TB/s
      static const double tabUs[8] = {1.6, 1.6, 1.6, 1.6, 2.0, 2.4, 4.6, 7.4};
      static const double otherUs[8] = {3.2, 3.2, 3.2, 3.2, 3.2, 6.0, 8.0, 14.0};
      cost[k] = (c.form == MULTI_TAB ? tabUs : otherUs)[c.L - 5] * hi[hord[c.orderOff]].nZ;
      if (c.stage != STAGE_NONE)
        for (int j = 0; j < c.count; j++) cost[k] += hi[hord[c.orderOff + j]].nZ * (double)(1 << c.L) * 1.6e-5;
    }
    std::stable_sort(byCost.begin(), byCost.end(), [&](int a, int b) { return cost[a] > cost[b]; });
    double load[CHAINS] = {0, 0, 0, 0};
    HIP_TRY(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
    hipLaunchKernelGGL(k_zero_ints, dim3((nc + 255) / 256), dim3(256), 0, m->stream, m->counters.p, nc);
    hipError_t ce = hipGetLastError();
    if (ce == hipSuccess) ce = hipEventRecord(m->fork, m->stream);
    for (int q = 0; q < chains && ce == hipSuccess; q++) ce = hipStreamWaitEvent(m->classes[q].stream, m->fork, 0);
    for (int k : byCost) {
      if (ce != hipSuccess) break;
      const MultiClass& c = m->classes[k];
      int q = 0;
      for (int j = 1; j < chains; j++)
        if (load[j] < load[q]) q = j;
      load[q] += cost[k];
      hipStream_t s = m->classes[q].stream;
      const cplx* tw = nullptr;
      (void)get_twiddles(1 << c.L, &tw);
      launch_stage(m, c, tw, s);
      c.fn(m->inst.p, m->order.p + c.orderOff, c.count, m->counters.p + k, tw, c.grid, s);
      ce = hipGetLastError();
    }
    for (int q = 0; q < chains && ce == hipSuccess; q++) {
      ce = hipEventRecord(m->classes[q].done, m->classes[q].stream);
      if (ce == hipSuccess) ce = hipStreamWaitEvent(m->stream, m->classes[q].done, 0);
    }
    hipGraph_t g = nullptr;
    hipError_t ee = hipStreamEndCapture(m->stream, &g);
    if (ce != hipSuccess || ee != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return fail(set_err(NLM_DEVICE_ERROR, std::string("graph capture failed: ") +
                                                hipGetErrorString(ce != hipSuccess ? ce : ee)));
    }
    m->graph = g;
    HIP_TRY(hipGraphInstantiate(&m->exec, m->graph, nullptr, nullptr, 0));
  }
  *out = m;
  return NLM_OK;
}

extern "C" int nlm_multi_launch(nlm_multi* m) {
  if (!m) return set_err(NLM_INVALID_ARGUMENT, "null batch");
  if (!m->exec) return NLM_OK;
  // held until the graph is queued: an output in between would keep the launch before's
  // results as this one's
  std::lock_guard<std::mutex> lk(m->outMu);
  m->hostOutOf = false;
  HIP_TRY(hipEventRecord(m->t0, m->stream));
  HIP_TRY(hipGraphLaunch(m->exec, m->stream));
  HIP_TRY(hipEventRecord(m->t1, m->stream));
  return NLM_OK;
}

extern "C" int nlm_multi_sync(nlm_multi* m, double* ms) {
  if (!m) return set_err(NLM_INVALID_ARGUMENT, "null batch");
  HIP_TRY(hipStreamSynchronize(m->stream));
  if (ms) {
    float f = 0.f;
    if (m->exec) HIP_TRY(hipEventElapsedTime(&f, m->t0, m->t1));
    *ms = f;
  }
  return NLM_OK;
}

extern "C" int nlm_multi_output(nlm_multi* m, int i, double* out) {
  if (!m || !out) return set_err(NLM_INVALID_ARGUMENT, "null argument");
  if (i < 0 || i >= m->n) return set_err(NLM_INVALID_ARGUMENT, "instance index out of range");
  // all outputs in one copy: one at a time they cost ~13 us each
  std::lock_guard<std::mutex> lk(m->outMu);
  if (!m->hostOutOf) {
    const size_t total = m->outOff[m->n - 1] + (size_t)m->nOut[m->n - 1] * m->N[m->n - 1];
    try {
      m->hostOut.resize(total);
    } catch (const std::bad_alloc&) {  // no room on the host for all of them: this one alone
      const HostCopy c = {out, m->outBuf.p + m->outOff[i], sizeof(cplx) * m->nOut[i] * m->N[i]};
      return nlm_to_host(&c, 1, m->stream);
    }
    const HostCopy c = {m->hostOut.data(), m->outBuf.p, total * sizeof(cplx)};
    if (int e = nlm_to_host(&c, 1, m->stream)) return e;
    m->hostOutOf = true;
  }
  memcpy(out, m->hostOut.data() + m->outOff[i], sizeof(cplx) * m->nOut[i] * m->N[i]);
  return NLM_OK;
}

extern "C" int nlm_multi_grid(nlm_multi* m, int c, int32_t* model, int32_t* log2n, int32_t* count, int32_t* grid) {
  if (!m) return set_err(NLM_INVALID_ARGUMENT, "null batch");
  if (c < 0 || c >= (int)m->classes.size()) return set_err(NLM_INVALID_ARGUMENT, "class index out of range");
  if (model) *model = m->classes[c].model;
  if (log2n) *log2n = m->classes[c].L;
  if (count) *count = m->classes[c].count;
  if (grid) *grid = m->classes[c].grid;
  return NLM_OK;
}

extern "C" int nlm_multi_form(nlm_multi* m, int c, int32_t* form, int64_t* staged_bytes) {
  if (!m) return set_err(NLM_INVALID_ARGUMENT, "null batch");
  if (c < 0 || c >= (int)m->classes.size()) return set_err(NLM_INVALID_ARGUMENT, "class index out of range");
  if (form) *form = m->classes[c].form;
  if (staged_bytes) *staged_bytes = (int64_t)m->classes[c].staged;
  return NLM_OK;
}

extern "C" int nlm_multi_classes(nlm_multi* m) { return m ? (int)m->classes.size() : 0; }
