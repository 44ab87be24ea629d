// nlm_internal.hpp -- plan state and host helpers shared by the engine's
// translation units (not part of the C-ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/nlm.h"
#include "nlm_copy.hpp"
#include "nlm_prop.hpp"

#define HIP_TRY(expr)                                                                              \
  do {                                                                                             \
    hipError_t e_ = (expr);                                                                        \
    if (e_ != hipSuccess)                                                                          \
      return set_err(NLM_DEVICE_ERROR, std::string("HIP error in ") + #expr + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  int ensure(size_t count) {
    if (count <= n && p) return NLM_OK;
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    if (count == 0) return NLM_OK;
    hipError_t e = hipMalloc((void**)&p, count * sizeof(T));
    if (e != hipSuccess) return set_err(NLM_DEVICE_ERROR, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    n = count;
    return NLM_OK;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

// whether ptr is memory of `device` that this process's HIP runtime knows
bool nlm_on_device(const void* ptr, int device);

// What a replay of the staged z loop reads from device memory (nlm_big.hip): its first step
// and the caller's output.
struct BigArgs {
  int step;
  cplx* out;
};

struct nlm_plan_s {
  int model = 0, N = 0, L = 0, nZ = 0, nS = 0, nP = 0, NC = 0, NCC = 0;
  int device = 0;
  hipStream_t own = nullptr, stream = nullptr;
  const cplx* tw = nullptr;
  DevBuf<cplx> dstep, halfIn, halfOut, coef, cconst, raman, filt;
  DevBuf<cplx> pumpT[2], pumpF[2];
  DevBuf<cplx> gridF, gridT;
  DevBuf<cplx> G, C, S, in, out, env, F0, dsp, relI;
  DevBuf<double> Dp, strength;
  int greensRows = 0, greensCols = 0;
  bool timing = false;
  hipEvent_t ev[6] = {};
  double last_ms[3] = {0, 0, 0};
  // Green's forward kept for the adjoint
  bool pumpLinear = false, hasStrength = false;
  double dzp = 0;
  DevBuf<cplx> ckpt, gG, gC, gS, gcoefPart, gcoef, gpumpPart, gpump, gF0Part, gF0, gtmp, gslice;
  DevBuf<cplx> scale;
  DevBuf<cplx> cascade[2][2];  // products of nlm_greens_cascade whose last plan this is
  // staged transform for Chi3GNLSE batches with nFreqs >= 8192 and the gradient (nlm_big.hip)
  DevBuf<cplx> bigState, bigH;
  int ramanReal = 0;  // the Raman response is the spectrum of a real one
  DevBuf<BigArgs> bigArgs;
  hipGraphExec_t bigExec = nullptr;
  int bigKey[6] = {0, 0, 0, 0, 0, 0};
  const void* bigStatePtr = nullptr;
  // Last asynchronous call that used the plan's scratch (bigState, the any-length path's table
  // and workspaces): the next call on them may be on another stream (nlm_plan_set_stream).
  hipEvent_t scratchDone = nullptr;
  bool scratchBusy = false, scratchUsed = false;
  DevBuf<cplx> anyScratch;  // workspaces of the any-length path (nlm_any.hip) when they exceed LDS
  DevBuf<cplx> stepTab;  // RK4 step propagators of one-mode undepleted media [nZ][N][2]
  int stepTable = 1;      // use them (nlm_plan_set_step_table)
  int ckptEvery = 0, nSeg = 0, gNIn = 0, gNOut = 0, gInTime = 0, gHasScale = 0;
  // differentiable Chi3GNLSE batch (nlm_batch_forward / nlm_batch_adjoint)
  int bRows = 0;
  DevBuf<cplx> adjWork, adjSeg;
  // state generation: bumped by every change the adjoints depend on (coefficients,
  // pump grids, the Green's rows in G); adjGen is the generation a differentiable
  // forward left, which its adjoint requires unchanged
  unsigned long long gen = 0, adjGen = 0;
};

inline void plan_touch(nlm_plan_s* p) { ++p->gen; }

void fill_common(nlm_plan_s* p, KParams& kp);
int check_pumps_ready(nlm_plan_s* p);
int launch_prop_kernel(nlm_plan_s* p, const KParams& kp);
// the same with the step-propagator table [nZ][N][2] in a caller's buffer (used when
// uses_step_table(p)); allocates nothing
int launch_prop_kernel_tab(nlm_plan_s* p, const KParams& kp, cplx* tab, bool may_tune = false);
bool uses_step_table(const nlm_plan_s* p);
// Before work on the plan's scratch: the stream waits for the asynchronous call that used it
// last.  A capturing stream is left alone; the order of its replays is the caller's.
bool stream_capturing(hipStream_t s);
int scratch_wait(nlm_plan_s* p);
// After an asynchronous call: records it if it used the scratch.
int scratch_mark(nlm_plan_s* p);
int get_twiddles(int n, const cplx** out);
// input channel feeding each mode (-1: none), src/_NonlinearMedium.hpp:164-198
void input_channels(int nS, int nCh, int inputMode, int* inPos);
// Chi3GNLSE batches staged through memory (nlm_big.hip): nFreqs 16384 / 32768, which no
// workgroup can hold
bool nlm_big_supported(int model, int L);
// and 8192 up to a row per CU, although one workgroup could hold a field
bool nlm_big_better(nlm_plan_s* p, int rows);
int nlm_big_batch(nlm_plan_s* p, const cplx* in, int rows, int cols, int inTime, int inPos, int nOut, int outPos,
                  cplx* out);
// Any even nFreqs outside the power-of-two kernels (nlm_any.hip): not a power of
// two, 2 and 4, or above 8192.  Plans of these lengths have L = 0.
bool nlm_any_size(int n);
// may_alloc = false: fail instead of allocating the device workspace that
// lengths above the LDS workspace need.  tab: a step table [nZ][N][2] of the caller's
// for the media that use one, or nullptr
int nlm_any_prop(nlm_plan_s* p, const KParams& kp, cplx* tab = nullptr, bool may_alloc = true);
// whether that many fields run with a step table where there is room for one
bool nlm_any_uses_table(const nlm_plan_s* p, int fields);
int nlm_any_pump_linear(nlm_plan_s* p, const double* strength_dev, double dzp);
int nlm_any_pump_chi3(nlm_plan_s* p, double dzp);
int nlm_any_pump_import(nlm_plan_s* p, int q, const cplx* sigF, int nzs, double dzs, const double* Ds,
                        const double* Dp, const double* omega, double dzp, double bd, double z, double zs);
int nlm_any_fft(const cplx* in, cplx* out, int n, int count, bool inverse, hipStream_t s, DevBuf<cplx>* scratch);
void tic(nlm_plan_s* p, int slot);
void collect_timing(nlm_plan_s* p, int a0, int a1, int slot);
void launch_greens_assemble(const cplx* G, cplx* C, cplx* S, int N, int nIn, int nOut, int nb, const cplx* scale,
                            hipStream_t s);
