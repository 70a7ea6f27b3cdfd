// sLSTM forward / decode engine for MI355X (gfx950, CDNA4): kernels + C ABI.
//
// One persistent launch runs all T timesteps.  A head's recurrent matrix R
// [dh x 4dh] is split by OUTPUT UNIT over G = ceil(dh/16) workgroups ("head
// group"); each workgroup keeps its 64 columns of R (4 gates x 16 units) in
// VGPRs for the whole sequence, computes R.h with MFMA (K split over the 4
// waves, partial sums reduced through LDS), and runs the exponential-gating
// pointwise update with c, n, m in fp32 registers.  The only thing exchanged
// per step is h_t: every workgroup stores its 16 units of h_t into a ring of
// 8 step slots in the workspace (laid out [row tile][member][16 rows][16 units],
// so that polls and stores move whole cache lines) and the other members of the
// group poll those very words until none of them carries the "not written yet"
// pattern the ring was pre-filled with.  One memory round trip per step, no
// flags, no atomics-with-return, no grid barrier.  A decode step (T = 1) is a
// different kernel: a tiled GEMM + gating with no waits between workgroups.
//
// Equations follow xlstm/blocks/slstm/src/vanilla/slstm.py:19-37 with the
// per-element n == 0 rule of xlstm/blocks/slstm/src/cuda/slstm_pointwise.cu:79.
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <mutex>

#include "xlstm_amd.h"

#include "slstm_device_common.h"
#include "slstm_seq_kernel.h"
#include "slstm_seq_roles_kernel.h"
#include "slstm_seq_pair_kernel.h"
#include "slstm_step_kernel.h"
#include "slstm_step_pipe_kernel.h"
#include "slstm_step_small_kernel.h"
#include "slstm_layer_step_kernel.h"
#include "slstm_backward_rules.h"
#include "slstm_backward_kernels.h"
#include "slstm_layer_kernels.h"
#include "slstm_layer_f32_kernels.h"
#include "slstm_local_kernel.h"
#include "slstm_backward_unit_kernel.h"
#include "slstm_backward_quad_kernel.h"
#include "slstm_backward_step_kernel.h"
#include "slstm_step_feed_kernel.h"
#include "slstm_backward_params_kernel.h"
#include "slstm_backward_params_slab_kernel.h"
#include "slstm_serial_bound.h"

// ---------------------------------------------------------------------------
// Scratch of the entry point that allocates nothing (xs_slstm_forward_static): status block, placement words and
// exchange ring in an array that every GPU the library runs on holds until the process ends.  In host code the
// array's name is only a stand-in: the device address comes from hipGetSymbolAddress, once per device.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[XS_STATIC_SCRATCH_BYTES];

namespace {

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

constexpr size_t kStatusBytes = 256;
constexpr int kMaxWg = 4096;
constexpr size_t kHeaderBytes = kStatusBytes + (size_t)kMaxWg * 4;  // status block + placement words (multiple of 256)

// upper bound on the elements of the exchange ring [8 slots][head groups][G][rows][16]:
// the head groups of one launch never cover more than B rounded up to 64 rows per head
inline size_t xbuf_elems(int B, int NH, int dh) {
  // (with row tiles of 4 or 8 rows a block still spans 16 rows, hence the factor 4)
  return (size_t)8 * NH * ((dh + 15) / 16) * ((size_t)(B + 63) / 64 * 64) * 16 * 4;
}

typedef void (*SeqKernel)(SeqParams);

template <bool BF16, int NCH, bool FULL>
SeqKernel pick_mt(int MT, bool burst) {
  switch (MT) {
    case 1: return (burst && NCH <= 4) ? slstm_seq_kernel<BF16, NCH, 1, FULL, NCH <= 4> : slstm_seq_kernel<BF16, NCH, 1, FULL, false>;
    case 2: return slstm_seq_kernel<BF16, NCH, 2, FULL, NCH <= 4>;
    default: return nullptr;
  }
}

// (chunk counts below those here have head dims that stay in one compute unit: slstm_local_kernel.h)
template <bool BF16, bool FULL>
SeqKernel pick_quad(int nch) {
  if (nch == 2) return slstm_seq_kernel<BF16, 2, 1, FULL, false, false, true>;
  if (nch == 4) return slstm_seq_kernel<BF16, 4, 1, FULL, false, false, true>;
  if constexpr (!BF16) {
    if (nch == 8) return slstm_seq_kernel<BF16, 8, 1, FULL, false, false, true>;
  }
  return nullptr;
}

// the kernels of a training forward beyond the head dims that stay in one compute unit
template <bool BF16, int NCH, bool FULL>
SeqKernel pick_train_n(bool quad, bool burst) {
  if (quad) return slstm_seq_kernel<BF16, NCH, 1, FULL, false, false, NCH <= (BF16 ? 4 : 8), 2>;
  return (burst && NCH <= 4) ? slstm_seq_kernel<BF16, NCH, 1, FULL, NCH <= 4, false, false, 2> : slstm_seq_kernel<BF16, NCH, 1, FULL, false, false, false, 2>;
}
template <bool BF16, bool FULL>
SeqKernel pick_train(int nch, bool quad, bool burst) {
  switch (nch) {
    case 2: return pick_train_n<BF16, 2, FULL>(quad, burst);
    case 4: return pick_train_n<BF16, 4, FULL>(quad, burst);
    case 8: return pick_train_n<BF16, 8, FULL>(quad, burst);
    default: return nullptr;
  }
}

template <bool BF16, bool FULL>
SeqKernel pick_roles_kernel(int nch) {
  switch (nch) {
    case 1: return slstm_seq_roles_kernel<BF16, 1, FULL>;
    case 2: return slstm_seq_roles_kernel<BF16, 2, FULL>;
    case 4: return slstm_seq_roles_kernel<BF16, 4, FULL>;
    case 8: return slstm_seq_roles_kernel<BF16, 8, FULL>;
    default: return nullptr;
  }
}

template <bool BF16, bool FULL>
SeqKernel pick_kernel(int nch, int MT, bool burst) {
  switch (nch) {
    case 2: return pick_mt<BF16, 2, FULL>(MT, burst);
    case 4: return pick_mt<BF16, 4, FULL>(MT, burst);
    case 8: return pick_mt<BF16, 8, FULL>(MT, burst);
    default: return nullptr;
  }
}

int validate(const xs_slstm_args *a, bool step, bool own_scratch = false) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (step && a->T != 1) return fail(XS_ERR_SHAPE, "xs_slstm_step needs T == 1, got %d", a->T);
  if (step && a->r_dtype != a->wx_dtype) return fail(XS_ERR_DTYPE, "xs_slstm_step needs the recurrent matrix in the dtype of wx");
  if (a->wx_dtype != XS_F32 && a->wx_dtype != XS_BF16) return fail(XS_ERR_DTYPE, "wx_dtype %d not supported", a->wx_dtype);
  if (a->r_dtype != XS_F32 && a->r_dtype != XS_BF16) return fail(XS_ERR_DTYPE, "r_dtype %d not supported", a->r_dtype);
  if (a->wx_dtype == XS_F32 && a->r_dtype != XS_F32) return fail(XS_ERR_DTYPE, "float32 wx needs a float32 recurrent matrix");
  if (!a->r || !a->bias || !a->s_out) return fail(XS_ERR_NULL, "r, bias and s_out are required");
  if (a->s0) {  // other workgroups still read s0 while the first ones write s_out
    const uintptr_t lo0 = (uintptr_t)a->s0, lo1 = (uintptr_t)a->s_out;
    const uintptr_t bytes = (uintptr_t)16 * (uintptr_t)a->B * (uintptr_t)a->NH * (uintptr_t)a->dh;
    if (lo0 < lo1 + bytes && lo1 < lo0 + bytes && bytes) return fail(XS_ERR_SHAPE, "s_out must not overlap s0");
  }
  if (a->B > 0 && a->T > 0 && (!a->wx || !a->h_out)) return fail(XS_ERR_NULL, "wx and h_out are required");
  if (a->dh % 8 != 0) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not a multiple of 8", a->dh);
  const long long H = (long long)a->NH * a->dh;
  if (a->B > 0 && a->T > 0) {
    if (a->wx_stride_t < 4 * H || (a->B > 1 && a->wx_stride_b < 4 * H))
      return fail(XS_ERR_SHAPE, "wx strides (%lld, %lld) overlap the innermost 4*H = %lld elements", (long long)a->wx_stride_b, (long long)a->wx_stride_t, 4 * H);
    if (a->reset && a->reset_stride_b < a->T) return fail(XS_ERR_SHAPE, "reset row stride %lld < T", (long long)a->reset_stride_b);
  }
  const uintptr_t al = 16;
  const long long esz = a->wx_dtype == XS_BF16 ? 2 : 4;
  if (a->B > 0 && a->T > 0 &&
      (((uintptr_t)a->wx % al) || ((a->wx_stride_b * esz) % 16) || ((a->wx_stride_t * esz) % 16)))
    return fail(XS_ERR_ALIGN, "wx and its row/step strides must be 16-byte aligned");
  if (((uintptr_t)a->r % al) || ((uintptr_t)a->h_out % al) || ((uintptr_t)a->s0 % al) || ((uintptr_t)a->s_out % al) ||
      ((uintptr_t)a->h_prev % al))
    return fail(XS_ERR_ALIGN, "r, h_out, s0, s_out and h_prev must be 16-byte aligned");
  if (a->h_prev && !a->s0) return fail(XS_ERR_NULL, "h_prev is a copy of the y plane of s0: s0 is required with it");
  if (!own_scratch) {  // (the entry point with a scratch array of its own checks what the launches really need)
    if (!a->workspace || a->workspace_bytes < xs_slstm_workspace_bytes(a->B, a->T, a->NH, a->dh))
      return fail(XS_ERR_WORKSPACE, "workspace missing or smaller than xs_slstm_workspace_bytes()");
    if ((uintptr_t)a->workspace % 256) return fail(XS_ERR_ALIGN, "workspace must be 256-byte aligned");
  }
  return XS_OK;
}

// compute units of the current device (asked for once: a decoded token looks at it several times)
int device_cus() {
  static std::atomic<int> known[64];  // (0: not asked yet)
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  if (dev >= 0 && dev < 64 && (cus = known[dev].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
  if (dev >= 0 && dev < 64) known[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// Raises a kernel's dynamic-LDS limit once per (kernel, device); the attribute call is not free and
// a decode loop would otherwise pay it every token.
int ensure_dynamic_lds(const void *kernel, size_t bytes) {
  struct Done { const void *kernel; int device; size_t bytes; };
  static std::mutex mu;
  static Done done[256];  // (a fixed table: nothing on the launch path allocates, host memory included)
  static int ndone = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return fail(XS_ERR_DEVICE, "cannot query the current device");
  std::lock_guard<std::mutex> lock(mu);
  for (int i = 0; i < ndone; ++i)
    if (done[i].kernel == kernel && done[i].device == dev && done[i].bytes >= bytes) return XS_OK;
  const hipError_t ea = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (ea != hipSuccess) return fail(XS_ERR_LAUNCH, "cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(ea));
  if (ndone < 256) done[ndone++] = Done{kernel, dev, bytes};  // (a full table only means the attribute is set again next time)
  return XS_OK;
}

StepParams step_params(const xs_slstm_args *a) {
  StepParams p;
  p.wx = a->wx; p.wx_sb = a->wx_stride_b;
  p.r = a->r; p.r_bf16 = a->r_dtype == XS_BF16;
  p.bias = a->bias; p.s0 = a->s0;
  p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  p.h_out = a->h_out; p.s_out = a->s_out;
  p.status = (xs_slstm_status *)a->workspace;
  p.B = a->B; p.NH = a->NH; p.dh = a->dh;
  p.n_unit_tiles = (a->dh + 31) / 32;
  p.n_row_tiles = (a->B + 63) / 64;
  p.h_prev = nullptr;
  p.spin_limit = a->spin_limit > 0 ? (a->spin_limit < (1ll << 30) ? (int)a->spin_limit : (1 << 30)) : (1 << 22);
  return p;
}

int run_step(const xs_slstm_args *a) {
  hipStream_t stream = (hipStream_t)a->stream;
  const int B = a->B, NH = a->NH, dh = a->dh;
  const bool bf16 = a->wx_dtype == XS_BF16;
  if (B == 0) return XS_OK;
  const int epc = bf16 ? 8 : 4;
  int nch = 1;
  while (nch * 16 * epc < dh) nch *= 2;  // the sequence kernel's K quarters are nch slabs wide
  if (nch > 8) return fail(XS_ERR_UNSUPPORTED, "head dim %d too large for %s operands (max %d)", dh, bf16 ? "bf16" : "fp32", 8 * 16 * epc);
  if ((long long)B * 4 * NH * dh * (bf16 ? 2 : 4) < 32) return fail(XS_ERR_SHAPE, "wx too small");
  StepParams p = step_params(a);
  const long long nwg = (long long)NH * p.n_unit_tiles * p.n_row_tiles;
  if (nwg > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tiles for one step launch");
  // Small batches: workgroups of 16 rows x 16 units (slstm_step_small_kernel.h), as long as there are at most so many of
  // them per compute unit; beyond, what every row tile reads of R costs more than the other kernels' longer way.  us a step
  // replayed from a graph, this kernel / the others, on either side of the line: bf16 4 heads of 512, 64 rows (2 per compute unit) 8.3 / 10.5,
  // 80 rows 10.7 / 10.5; 8 heads of 256, 64 rows (2) 5.0 / 5.5, 128 rows 8.0 / 6.0; 4 heads of 1024, 16 rows (1) 7.8 / 9.9, 32 rows
  // 12.6 / 11.0; float32 4 heads of 256, 256 rows (4) 14.7 / 16.6, 512 rows 24.0 / 17.4.
  const int small_rows = (B + 15) / 16, small_units = (dh + 15) / 16;
  if ((long long)NH * small_units * small_rows <= (long long)device_cus() * (bf16 ? (nch == 8 ? 1 : 2) : 4)) {
    p.n_unit_tiles = small_units;
    p.n_row_tiles = small_rows;
    p.h_prev = bf16 && a->s0 && !a->reset ? a->h_prev : nullptr;
    void (*k)(StepParams) = bf16 ? (p.h_prev ? pick_step_small<true, true>(nch) : pick_step_small<true, false>(nch)) : pick_step_small<false, false>(nch);
    hipLaunchKernelGGL(k, dim3((unsigned)(NH * p.n_unit_tiles * p.n_row_tiles)), dim3(256), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "step kernel launch failed: %s", hipGetErrorString(e));
    return XS_OK;
  }
  const dim3 grid((unsigned)nwg);
  int nch_log2 = 0;
  while ((1 << nch_log2) < nch) ++nch_log2;
  // steady-state decode: whole tiles, a state, no mask -> the variant without clamping
  const bool full = a->s0 && !a->reset && B % 64 == 0 && dh % 32 == 0 && dh == nch * 16 * epc;
  // slab width in MFMA k-steps: the whole K range when it fits LDS (dh <= 256 bf16 / 128 fp32)
  const int slabch = nch == 1 ? 4 : (nch == 2 ? 8 : 2);
  const int nbuf = slabch >= 4 ? 1 : 2;
  // one slab: eight waves in two roles (operands + MFMA / pointwise operands + gating), the sums of one row tile cross in 16 KiB of LDS
  const bool split = slabch >= 4;
  const size_t lds = (size_t)nbuf * (64 + 128) * (slabch * 64 + 16) + (split ? 4 * 256 * 16 : 0);
  typedef void (*StepKernel)(StepParams, int);
  StepKernel kern;
  const bool hint = full && bf16 && a->h_prev != nullptr;  // operand already in bf16 (h_out of the previous step)
  p.h_prev = hint ? a->h_prev : nullptr;
  // the steady state of bf16 decoding with the previous h at hand, head dim 256: the pipelined kernel (row tiles move
  // through fetch, MFMA, gating and store one behind the other); its buffer offsets are 31-bit
  if (hint && dh == 256 && 63ll * a->wx_stride_b * 2 + 4ll * NH * dh * 2 < (1ll << 31) && 4ll * B * NH * dh * 4 < (1ll << 31)) {
    const size_t plds = (size_t)2 * 64 * 256 + 3 * 64 * 128 + 4 * 64 * 64 + 2 * 128 * 256 + 64;  // h, c/n/m, W.x, R (later the sums), counters
    void (*pk)(StepParams) = slstm_step_pipe_kernel<8>;
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(pk), plds);
    if (rc != XS_OK) return rc;
    hipLaunchKernelGGL(pk, grid, dim3(kStepPipeThreads), plds, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "step kernel launch failed: %s", hipGetErrorString(e));
    return XS_OK;
  }
  // R prepared in slabs (xs_slstm_tile_r_for_steps) and the recurrent operand in the type of the operands: the kernel
  // whose feeder waves bring the slabs to LDS, for the head dims whose K range is walked in slabs
  if (a->r_tiled && slabch == 2 && dh % 64 == 0 && (!bf16 || a->h_prev || !a->s0) && (long long)B * NH * dh * (bf16 ? 2 : 4) < (1ll << 31)) {
    StepFeedParams q;
    q.B = B; q.NH = NH; q.dh = dh; q.nch = nch;
    q.wx = a->wx; q.wx_sb = a->wx_stride_b;
    q.r_tiled = a->r_tiled;
    q.h_prev = a->s0 ? (bf16 ? a->h_prev : (const void *)a->s0) : nullptr;
    q.bias = a->bias; q.s0 = a->s0; q.reset = a->reset; q.reset_sb = a->reset_stride_b;
    q.h_out = a->h_out; q.s_out = a->s_out; q.status = (xs_slstm_status *)a->workspace;
    if (((uintptr_t)a->r_tiled % 16) || ((uintptr_t)q.h_prev % 16)) return fail(XS_ERR_ALIGN, "r_tiled and h_prev must be 16-byte aligned");
    void (*fk)(StepFeedParams) = bf16 ? slstm_step_feed_kernel<true> : slstm_step_feed_kernel<false>;
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(fk), (size_t)step_feed_lds_bytes());
    if (rc != XS_OK) return rc;
    const long long fwg = (long long)NH * (dh / 32) * ((B + 63) / 64);
    hipLaunchKernelGGL(fk, dim3((unsigned)fwg), dim3(512), step_feed_lds_bytes(), stream, q);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "step kernel launch failed: %s", hipGetErrorString(e));
    return XS_OK;
  }
#define XS_PICK(BF, SC, SP) (full ? slstm_step_tile_kernel<BF, SC, true, false, SP> : slstm_step_tile_kernel<BF, SC, false, false, SP>)
#define XS_PICK_HINT(SC, SP) (hint ? slstm_step_tile_kernel<true, SC, true, true, SP> : XS_PICK(true, SC, SP))
  if (bf16) kern = slabch == 4 ? XS_PICK_HINT(4, true) : (slabch == 8 ? XS_PICK_HINT(8, true) : XS_PICK_HINT(2, false));
  else kern = slabch == 4 ? XS_PICK(false, 4, true) : (slabch == 8 ? XS_PICK(false, 8, true) : XS_PICK(false, 2, false));
#undef XS_PICK_HINT
#undef XS_PICK
  if (lds > 64 * 1024) {  // the single-slab variant at dh = 256 needs 99 KiB of the 160 KiB of LDS
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
    if (rc != XS_OK) return rc;
  }
  hipLaunchKernelGGL(kern, grid, dim3(split ? 512 : 256), lds, stream, p, nch_log2);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "step kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// the type of d_wx that a backward call asks for
int d_wx_type(const xs_slstm_bwd_args *a, int *is_bf16) {
  *is_bf16 = 0;
  if (a->d_wx_dtype == XS_F32) return XS_OK;
  if (a->d_wx_dtype != XS_BF16 || a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "d_wx_dtype must be XS_F32, or XS_BF16 with dtype XS_BF16");
  if (a->d_wx && (((uintptr_t)a->d_wx % 16) || (a->d_wx_stride_b % 8) || (a->d_wx_stride_t % 8)))
    return fail(XS_ERR_ALIGN, "d_wx in bf16 must be 16-byte aligned and its strides multiples of 8 elements");
  *is_bf16 = 1;
  return XS_OK;
}

// ---- small heads: the kernels that keep a head in one compute unit (slstm_local_kernel.h)
// (float32 beyond head dim 64 multiplies faster over several: 0.79 against 1.57 us a step at head dim 128)
inline bool local_head(int dh, bool bf16) { return dh <= (bf16 ? kLocalMaxHeadDim : 64); }
// the head dims that xs_slstm_train_forward / _backward cover
inline bool trains(int dh, bool bf16) { return dh >= 8 && dh % 8 == 0 && dh <= (bf16 ? 1024 : 512); }
inline int local_waves(int dh) { return (dh + 15) / 16; }

template <bool BF16, bool COEF>
void (*pick_local(int w))(LocalParams) {
  if constexpr (BF16) {
    switch (w) {
      case 5: return slstm_local_kernel<BF16, 5, COEF>;
      case 6: return slstm_local_kernel<BF16, 6, COEF>;
      case 7: return slstm_local_kernel<BF16, 7, COEF>;
      case 8: return slstm_local_kernel<BF16, 8, COEF>;
    }
  }
  switch (w) {
    case 1: return slstm_local_kernel<BF16, 1, COEF>;
    case 2: return slstm_local_kernel<BF16, 2, COEF>;
    case 3: return slstm_local_kernel<BF16, 3, COEF>;
    default: return slstm_local_kernel<BF16, 4, COEF>;
  }
}
template <bool BF16, bool DWX16>
void (*pick_local_bwd(int w))(LocalBwdParams) {
  if constexpr (BF16) {
    switch (w) {
      case 5: return slstm_local_bwd_kernel<BF16, 5, DWX16>;
      case 6: return slstm_local_bwd_kernel<BF16, 6, DWX16>;
      case 7: return slstm_local_bwd_kernel<BF16, 7, DWX16>;
      case 8: return slstm_local_bwd_kernel<BF16, 8, DWX16>;
    }
  }
  switch (w) {
    case 1: return slstm_local_bwd_kernel<BF16, 1, DWX16>;
    case 2: return slstm_local_bwd_kernel<BF16, 2, DWX16>;
    case 3: return slstm_local_bwd_kernel<BF16, 3, DWX16>;
    default: return slstm_local_bwd_kernel<BF16, 4, DWX16>;
  }
}
// workgroups of a launch over (row tile of 4 rows, head) pairs: a multiple of 8 (one range per XCD)
inline long long local_grid(int B, int NH) { return ((long long)((B + 3) / 4) * NH + 7) / 8 * 8; }

// heads head0 .. NH - 1 (head0 > 0: behind launches of other kernels for the heads in front)
int run_local(const xs_slstm_args *a, float *coef, int head0 = 0) {
  const bool bf16 = a->wx_dtype == XS_BF16;
  const int w = local_waves(a->dh);
  const long long grid = local_grid(a->B, a->NH - head0);
  if (grid > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many row tiles for one launch");
  LocalParams p;
  const size_t esz = bf16 ? 2 : 4, units = (size_t)head0 * a->dh;  // (an offset of the pointers: the kernel has no head of its own to add)
  p.wx = (const char *)a->wx + units * esz; p.wx_sb = a->wx_stride_b; p.wx_st = a->wx_stride_t;
  p.r_bf16 = a->r_dtype == XS_BF16;
  p.r = (const char *)a->r + units * 4 * a->dh * (p.r_bf16 ? 2 : 4);
  p.bias = a->bias + 4 * units; p.s0 = a->s0 ? a->s0 + units : nullptr; p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  p.h_out = (char *)a->h_out + units * esz; p.s_out = a->s_out + units; p.status = (xs_slstm_status *)a->workspace; p.coef = coef;
  p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh; p.heads = a->NH - head0;
  void (*k)(LocalParams);
  if (coef) k = bf16 ? pick_local<true, true>(w) : pick_local<false, true>(w);
  else k = bf16 ? pick_local<true, false>(w) : pick_local<false, false>(w);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(64 * w), 0, (hipStream_t)a->stream, p);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "sequence kernel launch failed: %s", hipGetErrorString(e));
}

// ---- the unit-split reverse kernel (slstm_backward_unit_kernel.h): how a call is cut into launches
struct UnitPlan { int G, W, CT, RT, heads, groups; };  // members of 16 CT units; row tile; heads of a launch; row tiles per head of a launch
// The first form of the list with which all of a head slice's row tiles fit at once; tiles of 16 rows in several launches
// where none does.  us a step (bf16): head dim 256, 64 rows 1.77 with {2, 8} and 2.91 with two launches of {2, 4}; head
// dim 512, 32 rows 2.16 with {2, 8} and 3.31 with {2, 16}; head dim 1024, 16 rows 3.81 and 6.11.  A group of up to 32
// members sits on one XCD, which members of 32 units give every head dim of bf16.
int unit_plan(int B, int NH, int dh, bool bf16, UnitPlan &u) {
  const int cus = device_cus();
  if (cus <= 0) return fail(XS_ERR_DEVICE, "cannot query the device");
  u.W = (dh + 15) / 16;
  const int per_xcd = cus / 8;
  static const int forms[2][4][2] = {{{1, 4}, {1, 16}}, {{1, 4}, {2, 4}, {2, 8}, {2, 16}}};  // {CT, RT}: float32, bf16
  bool found = false;
  for (int i = 0; i < (bf16 ? 4 : 2); ++i) {
    const int ct = forms[bf16][i][0], rt = forms[bf16][i][1], members = (u.W + ct - 1) / ct, capacity = members > 32 ? 0 : 8 * (per_xcd / members);
    if (capacity < 1) continue;
    const int heads = NH < capacity ? NH : capacity, groups = capacity / heads, tiles = (B + rt - 1) / rt;
    u.G = members; u.CT = ct; u.RT = rt; u.heads = heads; u.groups = groups < tiles ? groups : tiles;
    found = true;
    if (tiles <= groups) break;
  }
  if (!found) return fail(XS_ERR_DEVICE, "a head of %d units does not fit the compute units of this device's XCDs", dh);
  return XS_OK;
}
inline size_t unit_slot_bytes(const UnitPlan &u, int esz) { return (size_t)unit_bwd_slot_members(u.G, u.RT, u.CT, esz == 2) * u.RT * 64 * u.CT * esz; }
inline size_t unit_ring_bytes(const UnitPlan &u, int esz) { return kBwdRing * u.heads * u.groups * unit_slot_bytes(u, esz); }

template <int UW>
void (*pick_bwd_quad(int dh, bool dwx_bf16))(BwdSplitParams) {
  if (dwx_bf16) return dh == 64 ? slstm_bwd_quad_kernel<1, UW, true> : (dh == 128 ? slstm_bwd_quad_kernel<2, UW, true> : slstm_bwd_quad_kernel<4, UW, true>);
  return dh == 64 ? slstm_bwd_quad_kernel<1, UW> : (dh == 128 ? slstm_bwd_quad_kernel<2, UW> : slstm_bwd_quad_kernel<4, UW>);
}

template <bool BF16, int RT, int CT, bool DWX16>
void (*pick_unit_bwd(int gq))(UnitBwdParams) {
  if constexpr (!BF16) {
    if (gq <= 2) return slstm_bwd_unit_kernel<BF16, 2, RT, CT, DWX16>;
  }
  if constexpr (CT == 2) {
    if (gq <= 2) return slstm_bwd_unit_kernel<BF16, 2, RT, CT, DWX16>;
    if (gq <= 4) return slstm_bwd_unit_kernel<BF16, 4, RT, CT, DWX16>;
    return nullptr;
  } else {
    if (gq <= 4) return slstm_bwd_unit_kernel<BF16, 4, RT, CT, DWX16>;
    if (gq <= 8) return slstm_bwd_unit_kernel<BF16, 8, RT, CT, DWX16>;
    return nullptr;
  }
}
template <bool DWX16>
void (*pick_unit_bwd_bf16(int rt, int ct, int gq))(UnitBwdParams) {
  if (ct == 1) return pick_unit_bwd<true, 4, 1, DWX16>(gq);
  return rt == 4 ? pick_unit_bwd<true, 4, 2, DWX16>(gq) : (rt == 8 ? pick_unit_bwd<true, 8, 2, DWX16>(gq) : pick_unit_bwd<true, 16, 2, DWX16>(gq));
}

int run_unit_backward(const xs_slstm_bwd_args *a, int64_t d_h_sb, int64_t d_h_st, int r_dtype, int dwx_bf16, float clip, uint32_t *abort_host) {
  const bool bf16 = a->dtype == XS_BF16;
  const int esz = bf16 ? 2 : 4;
  UnitPlan u;
  int rc = unit_plan(a->B, a->NH, a->dh, bf16, u);
  if (rc != XS_OK) return rc;
  if (!a->exchange || !a->counters) return fail(XS_ERR_NULL, "exchange and counters are required at this head dim");
  if (((uintptr_t)a->exchange % 16) || ((uintptr_t)a->d_h % 16) || (d_h_sb * esz) % 16 || (d_h_st * esz) % 16)
    return fail(XS_ERR_ALIGN, "exchange, d_h and its strides must be 16-byte aligned");
  if (16 * d_h_sb * esz >= (1ll << 31) || (a->reset && 16 * a->reset_stride_b + a->T >= (1ll << 31)))
    return fail(XS_ERR_UNSUPPORTED, "rows of d_h or of the reset mask lie too far apart");
  UnitBwdParams p;
  p.coef = a->coef; p.d_h = a->d_h; p.d_h_sb = d_h_sb; p.d_h_st = d_h_st; p.d_s_final = a->d_s_final;
  p.r = a->r; p.r_bf16 = r_dtype == XS_BF16; p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  p.d_wx = a->d_wx; p.d_wx_sb = a->d_wx_stride_b; p.d_wx_st = a->d_wx_stride_t; p.d_s0 = a->d_s0;
  p.xch = (char *)a->exchange; p.abort_word = a->counters; p.placement = a->counters + 1; p.abort_host = abort_host;
  p.spin_limit = a->spin_limit != 0 ? a->spin_limit : kDefaultSpinLimit;
  p.cut = a->recurrent_cut != 0; p.clip = clip;
  p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh; p.G = u.G; p.W = u.W;
  const int gq = (u.G + 4 * u.CT - 1) / (4 * u.CT);  // members of a wave's share of K
  void (*k)(UnitBwdParams);
  if (bf16) k = dwx_bf16 ? pick_unit_bwd_bf16<true>(u.RT, u.CT, gq) : pick_unit_bwd_bf16<false>(u.RT, u.CT, gq);
  else k = u.RT == 4 ? pick_unit_bwd<false, 4, 1, false>(gq) : pick_unit_bwd<false, 16, 1, false>(gq);
  if (!k) return fail(XS_ERR_UNSUPPORTED, "no reverse kernel for head dim %d", a->dh);
  const int lds = unit_bwd_lds_bytes(u.RT, u.CT, bf16);
  rc = ensure_dynamic_lds((const void *)k, (size_t)lds);
  if (rc != XS_OK) return rc;
  hipStream_t stream = (hipStream_t)a->stream;
  bool first = true;
  for (int h0 = 0; h0 < a->NH; h0 += u.heads)
    for (int b0 = 0; b0 < a->B; b0 += u.RT * u.groups) {
      p.head0 = h0; p.NHL = h0 + u.heads <= a->NH ? u.heads : a->NH - h0;
      p.b0 = b0; p.bend = b0 + u.RT * u.groups < a->B ? b0 + u.RT * u.groups : a->B;
      p.NBT = (p.bend - b0 + u.RT - 1) / u.RT;
      const int ng = p.NHL * p.NBT;
      const long long n16 = (long long)kBwdRing * ng * (long long)unit_slot_bytes(u, esz) / 16;
      hipLaunchKernelGGL(slstm_bwd_arm_kernel, dim3((unsigned)((n16 + 255) / 256 < 1024 ? (n16 + 255) / 256 : 1024)), dim3(256), 0, stream,
                         (uint4 *)p.xch, n16, first ? p.abort_word : p.placement, ng + (first ? 1 : 0));
      first = false;
      hipLaunchKernelGGL(k, dim3(8u * u.G * ((ng + 7) / 8)), dim3(unit_bwd_threads(u.CT)), lds, stream, p);
    }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "backward kernel launch failed: %s", hipGetErrorString(e));
}

int run_train_backward(const xs_slstm_bwd_args *a, int64_t d_h_sb, int64_t d_h_st, int r_dtype, uint32_t *abort_host) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (a->dtype != XS_F32 && a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "dtype must be XS_F32 or XS_BF16");
  const bool bf16 = a->dtype == XS_BF16;
  if (r_dtype != XS_F32 && !(r_dtype == XS_BF16 && bf16)) return fail(XS_ERR_DTYPE, "r_dtype must be XS_F32, or XS_BF16 with dtype XS_BF16");
  if (!trains(a->dh, bf16)) return fail(XS_ERR_UNSUPPORTED, "head dim %d: a multiple of 8 up to %d", a->dh, bf16 ? 1024 : 512);
  if (a->B == 0 || a->T == 0) return XS_OK;
  int dwx_bf16 = 0;
  const int rc = d_wx_type(a, &dwx_bf16);
  if (rc != XS_OK) return rc;
  if (!a->coef || !a->d_h || !a->r || !a->d_wx || !a->d_s0) return fail(XS_ERR_NULL, "coef, d_h, r, d_wx and d_s0 are required");
  if ((uintptr_t)a->coef % 16) return fail(XS_ERR_ALIGN, "coef must be 16-byte aligned");
  const long long H = (long long)a->NH * a->dh;
  if (a->d_wx_stride_t < 4 * H || (a->B > 1 && a->d_wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "d_wx strides overlap the innermost 4*H elements");
  if (a->reset && a->reset_stride_b < a->T) return fail(XS_ERR_SHAPE, "reset row stride %lld < T", (long long)a->reset_stride_b);
  const float clip = (a->recurrent_clipval > 0.0f && a->recurrent_clipval < __builtin_inff()) ? a->recurrent_clipval : 0.0f;
  if (!local_head(a->dh, bf16)) return run_unit_backward(a, d_h_sb, d_h_st, r_dtype, dwx_bf16, clip, abort_host);
  const long long grid = local_grid(a->B, a->NH);
  if (grid > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many row tiles for one launch");
  const int w = local_waves(a->dh);
  LocalBwdParams p;
  p.coef = a->coef; p.d_h = a->d_h; p.d_h_sb = d_h_sb; p.d_h_st = d_h_st; p.d_s_final = a->d_s_final;
  p.r = a->r; p.r_bf16 = r_dtype == XS_BF16; p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  p.d_wx = a->d_wx; p.d_wx_sb = a->d_wx_stride_b; p.d_wx_st = a->d_wx_stride_t; p.d_s0 = a->d_s0;
  p.cut = a->recurrent_cut != 0; p.clip = clip;
  p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
  void (*k)(LocalBwdParams) = bf16 ? (dwx_bf16 ? pick_local_bwd<true, true>(w) : pick_local_bwd<true, false>(w)) : pick_local_bwd<false, false>(w);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(64 * w), 0, (hipStream_t)a->stream, p);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "backward kernel launch failed: %s", hipGetErrorString(e));
}

// Calls of several host threads that share a workspace and a stream run one after the other on the device, but only if the
// launches of one call - the workspace is cleared, then used - are not interleaved with another's: a call holds the lock of
// its workspace while it launches.
std::mutex &launches_into(const void *workspace) {
  static std::mutex mu[64];
  return mu[((uintptr_t)workspace >> 8) % 64];
}

template <int NCH>
SeqKernel pick_pair_n(int MT, int rows, bool coef) {
  if (MT == 2) return coef ? slstm_seq_pair_kernel<NCH, 2, 16, 2> : slstm_seq_pair_kernel<NCH, 2, 16, 0>;
  if constexpr (NCH == 8) {  // (smaller heads come here with full tiles only)
    if (rows == 4) return coef ? slstm_seq_pair_kernel<NCH, 1, 4, 2> : slstm_seq_pair_kernel<NCH, 1, 4, 0>;
    if (rows == 8) return coef ? slstm_seq_pair_kernel<NCH, 1, 8, 2> : slstm_seq_pair_kernel<NCH, 1, 8, 0>;
  }
  return coef ? slstm_seq_pair_kernel<NCH, 1, 16, 2> : slstm_seq_pair_kernel<NCH, 1, 16, 0>;
}
SeqKernel pick_pair(int nch, int MT, int rows, bool coef) {
  switch (nch) {
    case 2: return pick_pair_n<2>(MT, rows, coef);
    case 4: return pick_pair_n<4>(MT, rows, coef);
    case 8: return pick_pair_n<8>(MT, rows, coef);
    default: return nullptr;
  }
}

// Do two workgroups of every form of slstm_seq_pair_kernel share a compute unit, as its placement needs?
bool pair_resident() {
  static const bool resident = [] {
    for (int nch = 2; nch <= 8; nch *= 2)
      for (int form = 0; form < 8; ++form) {
        const SeqKernel k = pick_pair(nch, form >> 1 == 3 ? 2 : 1, 4 << (form >> 1), form & 1);
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(k), kPairThreads, 0) != hipSuccess || n < 2) return false;
      }
    return true;
  }();
  return resident;
}

// need != nullptr: launch nothing, only say whether a kernel takes every launch of this call and how many bytes of
// workspace they touch
int run_forward(const xs_slstm_args *a, size_t *need = nullptr, uint32_t *abort_host = nullptr, float *train_coef = nullptr) {
  hipStream_t stream = (hipStream_t)a->stream;
  const int B = a->B, T = a->T, NH = a->NH, dh = a->dh;
  const long long H = (long long)NH * dh;
  const bool bf16 = a->wx_dtype == XS_BF16;
  const bool dry = need != nullptr;
  if (dry) *need = kHeaderBytes;

  // status block + per-workgroup placement words start clean: with the exchange ring in front of the first launch, here
  // where there is none
  if (!dry && (B == 0 || T == 0))
    hipLaunchKernelGGL(fill_u32_kernel, dim3(4), dim3(256), 0, stream, (uint32_t *)a->workspace, kHeaderBytes / 4, 0u);
  if (B == 0) return XS_OK;
  if (T == 0) {
    if (dry) return XS_OK;
    const size_t n = (size_t)4 * B * H;
    hipLaunchKernelGGL(copy_state_kernel, dim3(256), dim3(256), 0, stream, a->s0, a->s_out, n);
    return hipGetLastError() == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "state copy launch failed");
  }

  // kernel shape
  const int epc = bf16 ? 8 : 4;
  int nch = 1;
  while (nch * 16 * epc < dh) nch *= 2;  // four waves cover nch * 16 * epc input units
  if (nch > 8) return fail(XS_ERR_UNSUPPORTED, "head dim %d too large for %s operands (max %d)", dh, bf16 ? "bf16" : "fp32", 8 * 16 * epc);
  const int G = (dh + 15) / 16;
  const int cus = device_cus();
  if (cus <= 0) return fail(XS_ERR_DEVICE, "cannot query the device");
  if (G > cus) return fail(XS_ERR_UNSUPPORTED, "ceil(dh/16) = %d workgroups of one head exceed the %d compute units; they must all be resident", G, cus);

  // Every workgroup of a head group waits for the others, so all groups of a launch must be resident at once, and
  // the placement deals groups out per XCD: a group of up to 32 workgroups sits on ONE XCD, a larger even one on
  // an XCD pair, anything else is spread over the device.  What a launch may hold is therefore counted per XCD
  // (one workgroup per compute unit), not per device: with 24 workgroups per group an XCD of 32 compute units
  // holds one group, not 32 * 8 / 24 of the device's.
  const int cus_per_xcd = cus / 8 > 0 ? cus / 8 : 1;
  // The gating waves of the kernel of four row tiles, and the kernel with two workgroups per compute unit, address W.x, the
  // mask and h_out as a scalar base plus a 32-bit offset per lane inside four rows / one row tile.
  const long long esz = bf16 ? 2 : 4;
  const bool offsets_fit = 4ll * a->wx_stride_b * esz + 4ll * NH * dh * esz < 0xFFFFFF00ll &&
                           (!a->reset || 4ll * a->reset_stride_b < 0xFFFFFF00ll) && 16ll * NH * dh * esz < (1ll << 31);
  // Heads of more workgroups than an XCD has compute units, sequences that are not short: two workgroups per compute unit and a head on
  // one XCD (slstm_seq_pair_kernel).  R is then read once for every 32 rows instead of 64 before the first step, and 64 peers shake
  // hands: 4 heads of 1024, us a call, on XCD pairs / on one XCD: B 64 T 40 143 / 151, T 100 361 / 346, T 300 1016 / 937; B 16 T 17 68 / 76, T 40
  // 119 / 114, T 300 700 / 514; B 2 T 9 49 / 47; 4 x 768 B 64 T 40 161 / 137.  (A training forward takes one row tile per workgroup on XCD
  // pairs, four times the launches.)
  // Smaller heads, batches that fill the device with more than one row tile per workgroup at one workgroup per compute unit: two of them
  // where that makes one row tile per workgroup of two, or fewer launches (T 300, us a call, one / two workgroups per compute unit: B 64 4 x 512
  // 697 / 538, B 128 4 x 256 631 / 453, B 200 3 x 320 1291 / 749; but B 128 4 x 512, two row tiles of 16 in place of four, 671 / 761, B 256 8 x 256
  // 1160 / 1390; T 20 the same, T 64 B 64 4 x 512 165 / 125), and in training, where a workgroup has one row tile otherwise (B 112 T 100 12 x 144
  // 1222 / 1038 with the backward pass, B 64 T 100 4 x 512 845 / 802).
  const int pair_groups = 8 * (2 * cus_per_xcd / G), row_tiles = (B + 15) / 16;
  const int per_pair = pair_groups > 0 ? pair_groups / (NH < pair_groups ? NH : pair_groups) : 0;  // row tiles of a head at once
  bool pair = bf16 && nch >= 2 && per_pair > 0 && offsets_fit && !a->coef_out && T >= (train_coef || row_tiles <= per_pair ? 32 : 64);
  if (pair && G <= 32) {
    const int groups = 8 * (cus_per_xcd / G), per_one = groups > 0 ? groups / (NH < groups ? NH : groups) : 0;
    pair = per_one > 0 && row_tiles > per_one && (train_coef || row_tiles <= per_pair ||
                                   (row_tiles + 2 * per_pair - 1) / (2 * per_pair) < (row_tiles + 4 * per_one - 1) / (4 * per_one));
  }
  pair = pair && pair_resident();
  const int span = pair ? 64 : 32;
  int capacity;  // head groups per launch
  if (pair) capacity = pair_groups;
  else if (G <= 32) capacity = 8 * (cus_per_xcd / G);
  else if (G <= 64 && G % 2 == 0) capacity = 4 * ((2 * cus_per_xcd) / G);
  else capacity = cus / G;
  if (capacity < 1) return fail(XS_ERR_DEVICE, "a head group of %d workgroups does not fit the %d compute units of this device's XCDs", G, cus);
  // Heads are independent (block-diagonal R): when the groups of all heads do not fit at once, the heads go in
  // several launches, as many per launch as fit.
  const int heads_per_launch = NH < capacity ? NH : capacity;
  if (!dry && heads_per_launch < NH) {  // a call is refused as a whole: no slice of heads after another has been launched
    size_t bytes = 0;
    const int rc = run_forward(a, &bytes, nullptr, train_coef);
    if (rc != XS_OK) return rc;
  }
  std::unique_lock<std::mutex> launches;
  if (!dry) launches = std::unique_lock<std::mutex>(launches_into(a->workspace));
  int launch_no = 0;
  for (int head0 = 0; head0 < NH; head0 += heads_per_launch) {
  const int NHL = head0 + heads_per_launch <= NH ? heads_per_launch : NH - head0;

  // batch tiling: the fewest rows per workgroup such that all groups of one launch are co-resident
  const int tiles = (B + 15) / 16;
  const int max_groups_per_head = capacity / NHL;  // >= 1
  int MT = 1;
  // (a training forward that leaves its coefficients: one row tile per workgroup, more launches)
  while ((pair || !train_coef) && MT < (pair ? 2 : 4) && (tiles + MT - 1) / MT > max_groups_per_head) MT *= 2;
  // (where four rows span more than 32-bit offsets reach - sequences of a gigabyte per row -, the batch goes through the kernel of
  // two row tiles in more launches instead)
  if (MT == 4 && !offsets_fit) MT = 2;
  // small heads stay in one compute unit, all heads that are left in one launch (nothing waits, so nothing has to be
  // resident at once), unless the batch is one for the kernel of four row tiles.  (The slices of heads but the last are of
  // one size: where the first goes to that kernel, a last one of fewer heads may still come here.)
  if (MT < 4 && !a->coef_out && !train_coef && local_head(dh, bf16)) return dry ? XS_OK : run_local(a, nullptr, head0);
  int rows_per_wg = 16 * MT;
  if (MT == 1 && (!pair || nch == 8)) {  // spare compute units: smaller row tiles, smaller exchanges
    for (int r = 4; r < 16; r *= 2)
      if ((B + r - 1) / r <= max_groups_per_head) { rows_per_wg = r; break; }
  }
  const int rows_per_launch = rows_per_wg * max_groups_per_head;

  for (int b0 = 0; b0 < B; b0 += rows_per_launch) {
    const int bend = b0 + rows_per_launch < B ? b0 + rows_per_launch : B;
    // the variant without per-chunk masks: no K tail and, with several row tiles, no missing rows in this launch
    const bool full = dh == nch * 16 * epc && (MT == 1 || (bend - b0) % rows_per_wg == 0);
    // the feeder fetches W.x in bursts where the prefetch waves cannot cover it: row tiles of 8 rows or more
    const bool burst = rows_per_wg >= 8;
    // four row tiles per workgroup: the kernel with MFMA waves and gating waves; one or two: the kernel in which
    // every compute wave does both
    const bool roles = MT == 4;
    SeqKernel kern;
    if (roles)
      kern = bf16 ? (full ? pick_roles_kernel<true, true>(nch) : pick_roles_kernel<true, false>(nch))
                  : (full ? pick_roles_kernel<false, true>(nch) : pick_roles_kernel<false, false>(nch));
    else
      kern = bf16 ? (full ? pick_kernel<true, true>(nch, MT, burst) : pick_kernel<true, false>(nch, MT, burst))
                  : (full ? pick_kernel<false, true>(nch, MT, burst) : pick_kernel<false, false>(nch, MT, burst));
    // row tiles of at most 4 rows: the compute waves split the columns by unit, not K (head groups on one XCD)
    const bool quad = MT == 1 && rows_per_wg == 4 && G <= 32;
    if (quad) kern = bf16 ? (full ? pick_quad<true, true>(nch) : pick_quad<true, false>(nch)) : (full ? pick_quad<false, true>(nch) : pick_quad<false, false>(nch));
    if (pair) kern = pick_pair(nch, MT, rows_per_wg, train_coef != nullptr);
    else if (train_coef) kern = bf16 ? (full ? pick_train<true, true>(nch, quad, burst) : pick_train<true, false>(nch, quad, burst))
                                : (full ? pick_train<false, true>(nch, quad, burst) : pick_train<false, false>(nch, quad, burst));
    if (a->coef_out) {  // a training forward: the same kernel, leaving the backward pass its coefficients
      if (!quad || !bf16 || (dh != 128 && dh != 256) || rows_per_launch < B)
        return fail(XS_ERR_UNSUPPORTED, "coef_out: the call does not run in row tiles of 4 rows of one kernel (bf16, head dim 128 or 256, "
                                        "ceil(B/4) * NH * dh/16 workgroups on the device at once)");
      if (((uintptr_t)a->coef_out % 4)) return fail(XS_ERR_ALIGN, "coef_out must be 4-byte aligned");
      kern = nch == 1 ? slstm_seq_kernel<true, 1, 1, true, false, false, true, 1> : slstm_seq_kernel<true, 2, 1, true, false, false, true, 1>;
    }
#ifdef XS_SMALL_BATCH_FMA
    // the measured alternative for small batches (see the kernel): only in a library built for that measurement
    if (MT == 1 && rows_per_wg == 4 && nch <= 2 && full) {
      if (bf16) kern = nch == 1 ? slstm_seq_kernel<true, 1, 1, true, false, true> : slstm_seq_kernel<true, 2, 1, true, false, true>;
      else kern = nch == 1 ? slstm_seq_kernel<false, 1, 1, true, false, true> : slstm_seq_kernel<false, 2, 1, true, false, true>;
    }
#endif
    if (!kern) return fail(XS_ERR_UNSUPPORTED, "no kernel for nch=%d MT=%d", nch, MT);
    const int NBT = (bend - b0 + rows_per_wg - 1) / rows_per_wg;
    const int ngroups = NHL * NBT;
    // grid shapes of the three placements the kernel knows: one XCD per group, two XCDs per group, spread
    const int grid = G <= span ? 8 * G * ((ngroups + 7) / 8)
                             : ((G <= 64 && G % 2 == 0) ? 8 * (G / 2) * ((ngroups + 3) / 4) : ngroups * G);
    if (grid > kMaxWg) return fail(XS_ERR_UNSUPPORTED, "grid %d too large", grid);
    if (dry) {
      const size_t ring = (size_t)kRing * ngroups * G * 16 * MT * 16 * (bf16 ? 2 : 4);
      if (kHeaderBytes + ring > *need) *need = kHeaderBytes + ring;
      continue;
    }
    {  // every word of the exchange ring starts as "not written yet"; the status block and the placement words are clear
       // (a later launch of the call: the placement words alone, what the earlier ones said in the status block stays)
      const size_t words = (size_t)kRing * ngroups * G * 16 * MT * 16 * (bf16 ? 2 : 4) / 4;
      const int blocks = (int)((words / 4 + 255) / 256);
      const size_t skip = launch_no++ > 0 ? kStatusBytes : 0;
      hipLaunchKernelGGL(clear_workspace_kernel, dim3(blocks < 16 ? 16 : (blocks > 1024 ? 1024 : blocks)), dim3(256), 0, stream,
                         (uint32_t *)((char *)a->workspace + skip), (kHeaderBytes - skip) / 4,
                         (uint32_t *)((char *)a->workspace + kHeaderBytes), words);
    }
    SeqParams p;
    p.wx = a->wx; p.wx_sb = a->wx_stride_b; p.wx_st = a->wx_stride_t;
    p.r = a->r; p.r_bf16 = a->r_dtype == XS_BF16;
    p.bias = a->bias; p.s0 = a->s0;
    p.reset = a->reset; p.reset_sb = a->reset_stride_b;
    p.h_out = a->h_out; p.s_out = a->s_out;
    p.status = (xs_slstm_status *)a->workspace;
    p.wg_xcc = (uint32_t *)((char *)a->workspace + kStatusBytes);
    p.xbuf = (char *)a->workspace + kHeaderBytes;
    p.B = B; p.T = T; p.NH = NH; p.dh = dh;
    p.b0 = b0; p.bend = bend; p.G = G; p.span = span; p.NBT = NBT; p.rows_per_wg = rows_per_wg;
    p.head0 = head0; p.NHL = NHL;
    p.spin_limit = a->spin_limit;
    p.coef_out = train_coef ? train_coef : a->coef_out;
    p.abort_host = abort_host;
    // a prefetch wave issues 2 (bf16) or 4 (fp32) scalar loads per batch row of a tile; 8 per wave and iteration
    // and 16 in all are what the scalar cache sustains, a tile that needs more goes without (prefetch waves that
    // fall behind hold up the barriers: measured 2x slower)
    {
      const int rows_in_tile = rows_per_wg < 16 ? rows_per_wg : 16;
      const int want = (rows_in_tile * (bf16 ? 2 : 4) + 7) / 8;
      p.prefetch = want <= max_prefetch_waves(nch) ? want : 0;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(pair ? kPairThreads : (roles ? kRolesThreads : kThreads + 64 * p.prefetch)), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "sequence kernel launch failed: %s", hipGetErrorString(e));
  }
  }  // heads of one launch
  return XS_OK;
}

// ---- backward pass with one launch per step (split == 3): slstm_fwd_walk_kernel and slstm_bwd_step_kernel.  Both keep
// what a launch hands to the next in the caller's `exchange` buffer: the forward walk (a launch per kFwdWalkSteps
// steps) a state [4,B,H] float32 (its y plane holds the y of the initial state in the type of the operands) and R in
// the walk's slabs; the reverse pass two
// sets of gate deltas in the type of the operands, in tiles of 64 rows.
int run_backward_stepwise(const xs_slstm_bwd_args *a, bool prepare) {
  const bool bf16 = a->dtype == XS_BF16;
  const int esz = bf16 ? 2 : 4;
  const int B = a->B, T = a->T, NH = a->NH, dh = a->dh;
  const long long H = (long long)NH * dh, BH = (long long)B * H;
  hipStream_t stream = (hipStream_t)a->stream;
  int dwx_bf16 = 0;
  {
    const int rc = d_wx_type(a, &dwx_bf16);
    if (rc != XS_OK) return rc;
  }
  if (!a->exchange) return fail(XS_ERR_NULL, "exchange is required with one launch per step");
  if (((uintptr_t)a->exchange % 16) || ((uintptr_t)a->coef % 16)) return fail(XS_ERR_ALIGN, "exchange and coef must be 16-byte aligned");
  const long long nwg = (long long)NH * (dh / 32) * ((B + 63) / 64);
  if (nwg > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tiles for one step launch");
  if (prepare) {
    if (!a->wx || !a->r || !a->bias || !a->h_out) return fail(XS_ERR_NULL, "wx, r, bias and h_out are required");
    if (a->wx_stride_t < 4 * H || (B > 1 && a->wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "wx strides overlap the innermost 4*H elements");
    if (((uintptr_t)a->wx % 16) || ((a->wx_stride_b * esz) % 16) || ((a->wx_stride_t * esz) % 16))
      return fail(XS_ERR_ALIGN, "wx and its row/step strides must be 16-byte aligned");
    if (((uintptr_t)a->r % 16) || ((uintptr_t)a->s0 % 16) || ((uintptr_t)a->bias % 16) || ((uintptr_t)a->h_out % 16))
      return fail(XS_ERR_ALIGN, "r, s0, bias and h_out must be 16-byte aligned");
    if (BH * esz >= (1ll << 31)) return fail(XS_ERR_UNSUPPORTED, "a step's outputs of 2 GiB or more");
    char *const ws = (char *)a->exchange;
    float *const state = (float *)ws;              // [4,B,H]; the y plane: the y of the initial state in the type of the operands
    char *const r_tiled = ws + 16 * BH;
    void (*init)(const void *, void *, const float *, void *, int, int, int) = bf16 ? slstm_fwd_walk_init_kernel<true> : slstm_fwd_walk_init_kernel<false>;
    hipLaunchKernelGGL(init, dim3(1024), dim3(256), 0, stream, a->r, (void *)r_tiled, a->s0, (void *)state, B, NH, dh);
    FwdWalkParams p;
    p.B = B; p.T = T; p.NH = NH; p.dh = dh;
    p.wx = a->wx; p.wx_sb = a->wx_stride_b; p.wx_st = a->wx_stride_t;
    p.r_tiled = r_tiled; p.bias = a->bias; p.state = state;
    p.h_out = a->h_out; p.h_init = a->s0 ? (const void *)state : nullptr;
    p.reset = a->reset; p.reset_sb = a->reset_stride_b; p.coef = a->coef;
    void (*kern)(FwdWalkParams) = bf16 ? slstm_fwd_walk_kernel<true> : slstm_fwd_walk_kernel<false>;
    {
      const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), (size_t)fwd_walk_lds_bytes());
      if (rc != XS_OK) return rc;
    }
    for (int t = 0; t < T; t += kFwdWalkSteps) {  // (a launch covers kFwdWalkSteps steps: one pass over R for all of them)
      p.t = t;
      p.nsteps = T - t < kFwdWalkSteps ? T - t : kFwdWalkSteps;
      p.state_in = t == 0 ? a->s0 : state;
      hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(kBwdStepThreads), fwd_walk_lds_bytes(), stream, p);
    }
  } else {
    if (!a->d_h || !a->r_t || !a->d_wx || !a->d_s0) return fail(XS_ERR_NULL, "d_h, r_t, d_wx and d_s0 are required");
    if (((uintptr_t)a->r_t % 16) || ((uintptr_t)a->d_h % 16) || ((uintptr_t)a->d_s0 % 16) || ((uintptr_t)a->d_s_final % 16))
      return fail(XS_ERR_ALIGN, "r_t, d_h, d_s0 and d_s_final must be 16-byte aligned");
    if (((uintptr_t)a->d_wx % 16) || (a->d_wx_stride_b % 4) || (a->d_wx_stride_t % 4))
      return fail(XS_ERR_ALIGN, "d_wx and its row/step strides must be 16-byte aligned");
    if (a->d_wx_stride_t < 4 * H || (B > 1 && a->d_wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "d_wx strides overlap the innermost 4*H elements");
    BwdStepParams q;
    q.B = B; q.T = T; q.NH = NH; q.dh = dh;
    q.coef = a->coef; q.d_h = a->d_h; q.d_s_final = a->d_s_final; q.r_t = a->r_t;
    q.reset = a->reset; q.reset_sb = a->reset_stride_b;
    q.d_wx = (float *)a->d_wx; q.d_wx_sb = a->d_wx_stride_b; q.d_wx_st = a->d_wx_stride_t; q.d_wx_bf16 = dwx_bf16; q.d_s0 = a->d_s0;
    q.cut = a->recurrent_cut != 0;
    q.clip = (a->recurrent_clipval > 0.0f && a->recurrent_clipval < __builtin_inff()) ? a->recurrent_clipval : 0.0f;
    char *const deltas[2] = {(char *)a->exchange, (char *)a->exchange + 4ll * ((B + 63) / 64 * 64) * H * esz};  // (tiles of 64 rows)
    void (*kern)(BwdStepParams) = bf16 ? slstm_bwd_step_kernel<true> : slstm_bwd_step_kernel<false>;
    {
      const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), (size_t)bwd_step_lds_bytes());
      if (rc != XS_OK) return rc;
    }
    for (int t = T - 1; t >= -1; --t) {
      q.t = t; q.first = t == T - 1;
      q.delta_out = deltas[(t + 1) & 1];
      q.delta_in = deltas[t & 1];  // (what the launch of step t + 1 wrote)
      hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(kBwdStepThreads), bwd_step_lds_bytes(), stream, q);
    }
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "backward step kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// ---- backward pass: the forward walk that leaves the coefficients, and the reverse-time kernel
int run_backward(const xs_slstm_bwd_args *a, bool prepare) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (a->dtype != XS_F32 && a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "dtype must be XS_F32 or XS_BF16");
  if (a->split == 3) {
    // one launch per step: the head dims the forward covers beyond those of the persistent kernels, and those next below
    const int lo = a->dtype == XS_BF16 ? 512 : 256;
    if (a->dh % 64 != 0 || a->dh < lo || a->dh > 2 * lo)
      return fail(XS_ERR_UNSUPPORTED, "backward pass with one launch per step: head dim %d not supported (%d to %d in steps of 64)", a->dh, lo, 2 * lo);
  } else if (a->dh != 64 && a->dh != 128 && a->dh != 256 && !(a->dh == 512 && a->dtype == XS_BF16 && (prepare || a->split)))
    return fail(XS_ERR_UNSUPPORTED, "backward pass: head dim %d not supported (64, 128, 256; 512 in bf16 over several compute units; "
                "up to 1024 in bf16 and 512 in float32 with one launch per step, split = 3)", a->dh);
  if (a->B == 0 || a->T == 0) return XS_OK;
  const bool bf16 = a->dtype == XS_BF16;
  const long long H = (long long)a->NH * a->dh;
  int dwx_bf16 = 0;
  if (!prepare) {
    const int rc = d_wx_type(a, &dwx_bf16);
    if (rc != XS_OK) return rc;
  }
  if (!a->coef) return fail(XS_ERR_NULL, "coef is required");
  if (a->reset && a->reset_stride_b < a->T) return fail(XS_ERR_SHAPE, "reset row stride %lld < T", (long long)a->reset_stride_b);
  hipStream_t stream = (hipStream_t)a->stream;
  if (a->split == 3) return run_backward_stepwise(a, prepare);
  if (prepare) {
    if (!a->wx || !a->r || !a->h_out || !a->bias) return fail(XS_ERR_NULL, "wx, r, h_out and bias are required");
    if (a->wx_stride_t < 4 * H || (a->B > 1 && a->wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "wx strides overlap the innermost 4*H elements");
    {  // (W.x and the outputs go straight into LDS in pieces of 16 bytes, R is read in such pieces)
      const long long esz = bf16 ? 2 : 4;
      if (((uintptr_t)a->wx % 16) || ((a->wx_stride_b * esz) % 16) || ((a->wx_stride_t * esz) % 16))
        return fail(XS_ERR_ALIGN, "wx and its row/step strides must be 16-byte aligned");
      if (((uintptr_t)a->r % 16) || ((uintptr_t)a->h_out % 16) || ((uintptr_t)a->s0 % 16) || ((uintptr_t)a->coef % 16))
        return fail(XS_ERR_ALIGN, "r, h_out, s0 and coef must be 16-byte aligned");
    }
    BwdPrepParams p;
    p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
    p.wx = a->wx; p.wx_sb = a->wx_stride_b; p.wx_st = a->wx_stride_t;
    p.r = a->r; p.h_out = a->h_out; p.bias = a->bias; p.s0 = a->s0; p.reset = a->reset; p.reset_sb = a->reset_stride_b; p.coef = a->coef;
    p.tiled = a->split == 2 ? 4 : (a->split ? 16 : 0);
    // (batch row, head) pairs dealt out over the XCDs, the dh / 64 slices of a pair on one of them
    const long long blocks = ((long long)a->B * a->NH + 7) / 8 * 8 * (a->dh / 64);
    if (blocks > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many elements for one launch");
    void (*kp)(BwdPrepParams) = nullptr;
    switch (a->dh) {
      case 64: kp = bf16 ? slstm_bwd_prepare_kernel<true, 64> : slstm_bwd_prepare_kernel<false, 64>; break;
      case 128: kp = bf16 ? slstm_bwd_prepare_kernel<true, 128> : slstm_bwd_prepare_kernel<false, 128>; break;
      case 256: kp = bf16 ? slstm_bwd_prepare_kernel<true, 256> : slstm_bwd_prepare_kernel<false, 256>; break;
      default: kp = slstm_bwd_prepare_kernel<true, 512>; break;  // (512 with bf16: checked above)
    }
    const int plds = bwd_prepare_lds_bytes(bf16, a->dh);
    const int rc = ensure_dynamic_lds((const void *)kp, (size_t)plds);
    if (rc != XS_OK) return rc;
    hipLaunchKernelGGL(kp, dim3((unsigned)blocks), dim3(kPrepThreads), plds, stream, p);
  } else {
    if (!a->d_h || !a->r_t || !a->d_wx || !a->d_s0) return fail(XS_ERR_NULL, "d_h, r_t, d_wx and d_s0 are required");
    if (((uintptr_t)a->r_t % 16)) return fail(XS_ERR_ALIGN, "r_t must be 16-byte aligned");
    // (d_h and the coefficients are fetched in pieces of 16 bytes, d_wx is written in pairs of floats)
    if (((uintptr_t)a->d_h % 16) || ((uintptr_t)a->coef % 16)) return fail(XS_ERR_ALIGN, "d_h and coef must be 16-byte aligned");
    if (((uintptr_t)a->d_wx % 8) || (a->d_wx_stride_b % 2) || (a->d_wx_stride_t % 2))
      return fail(XS_ERR_ALIGN, "d_wx must be 8-byte aligned and its strides even");
    if (a->d_wx_stride_t < 4 * H || (a->B > 1 && a->d_wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "d_wx strides overlap the innermost 4*H elements");
    // (0, negative, NaN or infinite: no clipping)
    const float clip = (a->recurrent_clipval > 0.0f && a->recurrent_clipval < __builtin_inff()) ? a->recurrent_clipval : 0.0f;
    if (a->split == 2) {
      // row tiles of 4 rows (bf16, head dims up to 256): four times the workgroups of the 16-row kernel, a shorter step
      if (!bf16 || (a->dh != 64 && a->dh != 128 && a->dh != 256))
        return fail(XS_ERR_UNSUPPORTED, "backward pass with row tiles of 4 rows: bf16 and head dim 64, 128 or 256 (got %d)", a->dh);
      if (!a->exchange || !a->counters) return fail(XS_ERR_NULL, "exchange and counters are required with split");
      if (((uintptr_t)a->exchange % 16)) return fail(XS_ERR_ALIGN, "exchange must be 16-byte aligned");
      if (a->reset && 3 * a->reset_stride_b + a->T >= 0x7FFFFF00ll) return fail(XS_ERR_UNSUPPORTED, "reset rows too far apart for row tiles of 4 rows");
      if (3 * H * 2 + 1024 >= 0x7FFFFF00ll) return fail(XS_ERR_UNSUPPORTED, "rows too long for row tiles of 4 rows");
      const int S = a->dh / 64;
      const long long ngroups = (long long)a->NH * ((a->B + 3) / 4);
      const long long groups_per_xcd = (ngroups + 7) / 8;
      // prefetching workgroups per XCD: one per 40 KB that the XCD's groups read per step (a compute unit draws some
      // 65 GB/s from memory, a step takes about a microsecond; one per 20 or 10 KB gains nothing), as far as there are compute units left
      const long long step_bytes = groups_per_xcd * S * (4 * 9 * 64 * 4 + 4 * 64 * 2);
      const long long want = step_bytes > 280000 ? 8 : (step_bytes + 39999) / 40000;
      // 32 units a workgroup where twice the workgroups leave these their room, else 64 (figures at the kernel)
      const int uw = 8 * (groups_per_xcd * (a->dh / 32) + want) <= device_cus() ? 32 : 64;
      const long long grid = groups_per_xcd * 8 * (a->dh / uw);
      if (grid > device_cus()) return fail(XS_ERR_DEVICE, "%lld workgroups of the backward pass with row tiles of 4 rows do not fit %d compute units at once", grid, device_cus());
      BwdSplitParams q;
      q.B = a->B; q.T = a->T; q.NH = a->NH; q.dh = a->dh;
      q.coef = a->coef; q.d_h = a->d_h; q.d_s_final = a->d_s_final; q.r_ts = a->r_t;
      q.reset = a->reset; q.reset_sb = a->reset_stride_b;
      q.d_wx = (float *)a->d_wx; q.d_wx_sb = a->d_wx_stride_b; q.d_wx_st = a->d_wx_stride_t; q.d_s0 = a->d_s0;
      q.xch = a->exchange; q.abort_word = a->counters; q.progress = a->counters + 1; q.placement = a->counters + 1 + ngroups;
      q.main_locals = (int)(grid / 8);
      const long long room = (device_cus() - grid) / 8;
      const int prefetchers = (int)(want < room ? want : room);
      q.spin_limit = a->spin_limit != 0 ? a->spin_limit : kDefaultSpinLimit;
      q.cut = a->recurrent_cut != 0; q.clip = clip;
      const long long n16 = (long long)kBwdRing * ngroups * 4 * 4 * a->dh * 2 / 16;
      hipLaunchKernelGGL(slstm_bwd_arm_kernel, dim3((unsigned)((n16 + 255) / 256 < 1024 ? (n16 + 255) / 256 : 1024)), dim3(256), 0, stream,
                         (uint4 *)a->exchange, n16, a->counters, (int)(1 + 2 * ngroups));
      void (*kq)(BwdSplitParams) = uw == 32 ? pick_bwd_quad<32>(a->dh, dwx_bf16) : pick_bwd_quad<64>(a->dh, dwx_bf16);
      const int lds = bwd_quad_lds_bytes(uw);
      {
        const int rc = ensure_dynamic_lds((const void *)kq, (size_t)lds);
        if (rc != XS_OK) return rc;
      }
      hipLaunchKernelGGL(kq, dim3((unsigned)(grid + 8 * prefetchers)), dim3(bwd_quad_threads(uw)), lds, stream, q);
      const hipError_t es = hipGetLastError();
      if (es != hipSuccess) return fail(XS_ERR_LAUNCH, "backward kernel launch failed: %s", hipGetErrorString(es));
      return XS_OK;
    }
    if (a->split) {
      if (a->dh != 64 && a->dh != 128 && a->dh != 256 && !(a->dh == 512 && bf16))
        return fail(XS_ERR_UNSUPPORTED, "backward pass over several compute units per head: head dim %d not supported", a->dh);
      if (!a->exchange || !a->counters) return fail(XS_ERR_NULL, "exchange and counters are required with split");
      const int S = a->dh / 64;
      const long long ngroups = (long long)a->NH * ((a->B + 15) / 16);
      const long long grid = (ngroups + 7) / 8 * 8 * S;
      if (grid > device_cus()) return fail(XS_ERR_DEVICE, "%lld workgroups of the split backward pass do not fit %d compute units at once", grid, device_cus());
      BwdSplitParams q;
      q.B = a->B; q.T = a->T; q.NH = a->NH; q.dh = a->dh;
      q.coef = a->coef; q.d_h = a->d_h; q.d_s_final = a->d_s_final; q.r_ts = a->r_t;
      q.reset = a->reset; q.reset_sb = a->reset_stride_b;
      q.d_wx = (float *)a->d_wx; q.d_wx_sb = a->d_wx_stride_b; q.d_wx_st = a->d_wx_stride_t; q.d_s0 = a->d_s0;
      if (((uintptr_t)a->exchange % 16)) return fail(XS_ERR_ALIGN, "exchange must be 16-byte aligned");
      q.xch = a->exchange; q.abort_word = a->counters; q.progress = a->counters + 1; q.placement = a->counters + 1 + ngroups;
      q.main_locals = (int)(grid / 8);
      // prefetching workgroups per XCD, as for the row tiles of 4 rows below: one per 40 KB that the XCD's groups read
      // per step, as far as there are compute units left
      int prefetchers = 0;
      {
        const long long groups_per_xcd = (ngroups + 7) / 8;
        const long long step_bytes = groups_per_xcd * S * (kBwdCoefBytes + 16 * 64 * (bf16 ? 2 : 4));
        long long want = (step_bytes + 39999) / 40000;
        const long long room = (device_cus() - grid) / 8;
        if (want > room) want = room;
        if (want > 8) want = 8;
        prefetchers = (int)(want < 0 ? 0 : want);
      }
      q.spin_limit = a->spin_limit != 0 ? a->spin_limit : kDefaultSpinLimit;  // (negative: every wait gives up at once)
      q.cut = a->recurrent_cut != 0; q.clip = clip;
      const long long n16 = (long long)kBwdRing * ngroups * 16 * 4 * a->dh * (bf16 ? 2 : 4) / 16;
      hipLaunchKernelGGL(slstm_bwd_arm_kernel, dim3((unsigned)((n16 + 255) / 256 < 1024 ? (n16 + 255) / 256 : 1024)), dim3(256), 0, stream,
                         (uint4 *)a->exchange, n16, a->counters, (int)(1 + 2 * ngroups));
      void (*ks)(BwdSplitParams) = nullptr;
      bool feed = true;  // (feeder waves where the registers allow twelve waves)
      if (a->dh == 64) ks = bf16 ? slstm_bwd_split_kernel<true, 1, true> : slstm_bwd_split_kernel<false, 1, true>;
      else if (a->dh == 128) ks = bf16 ? slstm_bwd_split_kernel<true, 2, true> : slstm_bwd_split_kernel<false, 2, true>;
      else if (a->dh == 256 && bf16) ks = slstm_bwd_split_kernel<true, 4, true>;
      else if (a->dh == 256) { ks = slstm_bwd_split_kernel<false, 4, false>; feed = false; }
      else { ks = slstm_bwd_split_kernel<true, 8, false>; feed = false; }
      if (dwx_bf16) {
        if (a->dh == 64) ks = slstm_bwd_split_kernel<true, 1, true, true>;
        else if (a->dh == 128) ks = slstm_bwd_split_kernel<true, 2, true, true>;
        else if (a->dh == 256) ks = slstm_bwd_split_kernel<true, 4, true, true>;
        else ks = slstm_bwd_split_kernel<true, 8, false, true>;
      }
      const int lds = bwd_split_lds_bytes(feed, bf16);
      {
        const int rc = ensure_dynamic_lds((const void *)ks, (size_t)lds);
        if (rc != XS_OK) return rc;
      }
      hipLaunchKernelGGL(ks, dim3((unsigned)(grid + 8 * prefetchers)), dim3(feed ? 768 : 512), lds, stream, q);
      const hipError_t es = hipGetLastError();
      if (es != hipSuccess) return fail(XS_ERR_LAUNCH, "backward kernel launch failed: %s", hipGetErrorString(es));
      return XS_OK;
    }
    BwdParams p;
    p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
    p.coef = a->coef; p.d_h = a->d_h; p.d_s_final = a->d_s_final; p.r_t = a->r_t;
    p.reset = a->reset; p.reset_sb = a->reset_stride_b;
    p.d_wx = (float *)a->d_wx; p.d_wx_sb = a->d_wx_stride_b; p.d_wx_st = a->d_wx_stride_t; p.d_wx_bf16 = dwx_bf16; p.d_s0 = a->d_s0;
    p.cut = a->recurrent_cut != 0; p.clip = clip;
    void (*kern)(BwdParams) = nullptr;
    int waves = 0;
#ifndef XS_BWD_NB256
#define XS_BWD_NB256 2
#endif
    if (a->dh == 64) { kern = bf16 ? slstm_bwd_kernel<true, 1, 4> : slstm_bwd_kernel<false, 1, 4>; waves = 4; }
    else if (a->dh == 128) { kern = bf16 ? slstm_bwd_kernel<true, 1, 8> : slstm_bwd_kernel<false, 1, 8>; waves = 8; }
    else { kern = bf16 ? slstm_bwd_kernel<true, XS_BWD_NB256, 16 / XS_BWD_NB256> : slstm_bwd_kernel<false, XS_BWD_NB256, 16 / XS_BWD_NB256>; waves = 16 / XS_BWD_NB256; }
    const int esz = bf16 ? 2 : 4;
    const size_t lds = (size_t)16 * (4 * a->dh + 16 / esz) * esz;  // the delta tile
    if (lds > 64 * 1024) {
      const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
      if (rc != XS_OK) return rc;
    }
    const long long blocks = (long long)a->NH * ((a->B + 15) / 16);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(waves * 64), lds, stream, p);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "backward kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// ---- backward pass: R in the operand order of the reverse kernels (xs_slstm_bwd_args::r_t), one thread per element of
// the result: its place says which (gate unit k = g dh + a, input unit d) it holds, and R[h][k][d] is read from the
// forward's layout.  mode = xs_slstm_bwd_args::split.
template <typename T>
__global__ __launch_bounds__(256) void slstm_bwd_tile_r_kernel(const T *r, T *r_t, int NH, int dh, int mode, int epc) {
  const long long per_head = 4ll * dh * dh, n = (long long)NH * per_head;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x; o < n; o += stride) {
    const int h = (int)(o / per_head);
    long long v = o - (long long)h * per_head;
    int k, d;
    if (mode == 0) {         // [d / 16][k / KC][(k % KC) / EPC][d % 16][k % EPC], KC = 4 EPC
      const int e = (int)(v % epc); v /= epc;
      const int r16 = (int)(v & 15); v >>= 4;
      const int c = (int)(v & 3); v >>= 2;
      const int nkc = 4 * dh / (4 * epc);
      const int kc = (int)(v % nkc); v /= nkc;
      k = (kc * 4 + c) * epc + e;
      d = (int)v * 16 + r16;
    } else if (mode == 3) {  // [d / 32][k / KS][d % 32][k % KS], KS = 32 EPC / 2 (256 bytes)
      const int ks = 16 * epc;
      const int e = (int)(v % ks); v /= ks;
      const int r32 = (int)(v & 31); v >>= 5;
      const int nsl = 4 * dh / ks;
      const int sl = (int)(v % nsl); v /= nsl;
      k = sl * ks + e;
      d = (int)v * 32 + r32;
    } else {                 // [dh / 64][8 waves][k-steps of a wave][4 column blocks][4][16 columns][EPC], K reordered
      const int ksteps = 4 * dh / 8 / (4 * epc);
      const int e = (int)(v % epc); v /= epc;
      const int r16 = (int)(v & 15); v >>= 4;
      const int c = (int)(v & 3); v >>= 2;
      const int cb = (int)(v & 3); v >>= 2;
      const int kst = (int)(v % ksteps); v /= ksteps;
      const int w = (int)(v & 7); v >>= 3;
      const int kk = ((w * ksteps + kst) * 4 + c) * epc + e;  // the kernel's K index
      d = ((int)v * 4 + cb) * 16 + r16;
      if (mode == 1) k = ((kk & 255) >> 6) * dh + (kk >> 8) * 64 + (kk & 63);  // kk = 256 (a / 64) + 64 g + a % 64
      else k = (kk & 3) * dh + (kk >> 2);                                     // kk = 4 a + g
    }
    r_t[o] = r[((long long)h * 4 * dh + k) * dh + d];
  }
}

int run_backward_tile_r(const xs_slstm_bwd_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims NH=%d dh=%d", a->NH, a->dh);
  if (a->dtype != XS_F32 && a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "dtype must be XS_F32 or XS_BF16");
  if (a->split < 0 || a->split > 3) return fail(XS_ERR_UNSUPPORTED, "split = %d", a->split);
  if (!a->r || !a->r_t) return fail(XS_ERR_NULL, "r and r_t are required");
  const bool bf16 = a->dtype == XS_BF16;
  const int epc = bf16 ? 8 : 4;
  if (a->split == 2 && !bf16) return fail(XS_ERR_UNSUPPORTED, "row tiles of 4 rows go with XS_BF16");
  if (a->dh % 64 != 0) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not one of the backward kernels'", a->dh);
  hipStream_t stream = (hipStream_t)a->stream;
  const long long n = 4ll * a->NH * a->dh * a->dh;
  const unsigned blocks = (unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
  if (bf16) hipLaunchKernelGGL(slstm_bwd_tile_r_kernel<uint16_t>, dim3(blocks), dim3(256), 0, stream, (const uint16_t *)a->r, (uint16_t *)a->r_t, a->NH, a->dh, a->split, epc);
  else hipLaunchKernelGGL(slstm_bwd_tile_r_kernel<uint32_t>, dim3(blocks), dim3(256), 0, stream, (const uint32_t *)a->r, (uint32_t *)a->r_t, a->NH, a->dh, a->split, epc);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "tiling kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// ---- backward pass: the gradients of R and the bias from the gate deltas and the forward's outputs
int run_backward_params(const xs_slstm_bwd_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (a->dtype != XS_F32 && a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "dtype must be XS_F32 or XS_BF16");
  if (a->dh % 8 != 0) return fail(XS_ERR_UNSUPPORTED, "backward pass: head dim %d is not a multiple of 8", a->dh);
  if (!a->d_r || !a->d_bias) return fail(XS_ERR_NULL, "d_r and d_bias are required");
  const bool bf16 = a->dtype == XS_BF16;
  const long long H = (long long)a->NH * a->dh;
  int dwx_bf16 = 0;
  {
    const int rc = d_wx_type(a, &dwx_bf16);
    if (rc != XS_OK) return rc;
  }
  hipStream_t stream = (hipStream_t)a->stream;
  const size_t nr = (size_t)a->NH * 4 * a->dh * a->dh, nb = (size_t)4 * H;
  if (((uintptr_t)a->d_r % 4) || ((uintptr_t)a->d_bias % 4)) return fail(XS_ERR_ALIGN, "d_r and d_bias must be 4-byte aligned");
  const bool empty = a->B == 0 || a->T == 0;
  if (!empty) {
    if (!a->d_wx || !a->h_out) return fail(XS_ERR_NULL, "d_wx and h_out are required");
    if (a->d_wx_stride_t < 4 * H || (a->B > 1 && a->d_wx_stride_b < 4 * H)) return fail(XS_ERR_SHAPE, "d_wx strides overlap the innermost 4*H elements");
    if (((uintptr_t)a->d_wx % 16) || (a->d_wx_stride_b % 4) || (a->d_wx_stride_t % 4))
      return fail(XS_ERR_ALIGN, "d_wx and its row/step strides must be 16-byte aligned");
    if (((uintptr_t)a->h_out % 16) || ((uintptr_t)a->s0 % 16)) return fail(XS_ERR_ALIGN, "h_out and s0 must be 16-byte aligned");
    if (a->reset && a->reset_stride_b < a->T) return fail(XS_ERR_SHAPE, "reset row stride %lld < T", (long long)a->reset_stride_b);
    // (a chunk of 32 steps is read through one buffer descriptor: its offsets are 31-bit)
    if (32ll * a->d_wx_stride_t * (dwx_bf16 ? 2 : 4) >= (1ll << 31) || 32ll * a->B * H * (bf16 ? 2 : 4) >= (1ll << 31))
      return fail(XS_ERR_UNSUPPORTED, "32 steps of d_wx or of the outputs span 2 GiB or more: run the batch in slices of rows");
  }
  // (the slices of K are added into the results: they start at zero)
  hipLaunchKernelGGL(clear_two_kernel, dim3(256), dim3(256), 0, stream, (uint32_t *)a->d_r, nr, (uint32_t *)a->d_bias, nb);
  if (!empty) {
    BwdParamParams p;
    p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
    p.dhp = (a->dh + 63) / 64 * 64;
    p.d_wx = (const float *)a->d_wx; p.d_wx_sb = a->d_wx_stride_b; p.d_wx_st = a->d_wx_stride_t;
    p.h_out = a->h_out; p.s0 = a->s0; p.reset = a->reset; p.reset_sb = a->reset_stride_b;
    p.d_r = a->d_r; p.d_bias = a->d_bias;
    p.tchunks = (a->T + kParamKC - 1) / kParamKC;
    const int nt = p.dhp % 256 == 0 ? 256 : (p.dhp % 128 == 0 ? 128 : 64);
    const bool slab = dwx_bf16 != 0;  // deltas in bf16: the kernel whose operands go straight to LDS
    const int tiles = (4 * p.dhp / (slab ? kSlabMT : kParamMT)) * (p.dhp / nt);
    const long long nchunks = (long long)a->B * p.tchunks;
    if (nchunks > 0x7FFFFFFF - 8) return fail(XS_ERR_UNSUPPORTED, "too many chunks of 32 steps for one launch");
    // slices of K: enough workgroups for two per compute unit (slab: its LDS takes a compute unit to itself), no slice
    // shorter than four chunks
    const int cus = device_cus() > 0 ? device_cus() : 256;
    const long long base = (long long)a->NH * tiles;
    // (4 or 8 per compute unit: 10 to 30 % slower.)
    // (head, slice) groups are dealt out over the XCDs, group i on XCD i % 8: a multiple of 8 of them keeps every XCD
    // busy (4 heads of 1024 are 512 tiles and one slice each by the rule above: four XCDs idle, twice the time)
    auto whole_xcds = [&](long long k) {
      if (k < 1) k = 1;
      while ((a->NH * k) % 8 != 0 && a->NH * k < 64) ++k;
      return k;
    };
    long long ks = whole_xcds(slab ? cus / base : (2ll * cus + base - 1) / base);
    // float32, one per compute unit, half the atomics: with 256 columns a tile wherever the tiles alone are no more than that; with fewer columns
    // where it fills the device exactly and a slice is short.  us, two -> one per compute unit: 4 x 256 B 32 T 256 206 -> 181, 6 x 256 373 -> 328,
    // 8 x 512 1177 -> 1170; 8 x 128 B 6 T 250 (6 chunks a slice) 45.8 -> 38.5, 4 x 128 B 32 T 256 (16) 72.2 -> 69.0, B 100 T 128 (25) 80 -> 86, 16 x 128
    // B 32 T 256 (64) 176 -> 183; not filled, or with a last round that is nearly empty: 8 x 192 283 -> 429, 4 x 384 452 -> 588
    if (!slab && !bf16 && base <= cus) {
      const long long one = whole_xcds(cus / base);
      if (nt == 256 || (base * one == cus && nchunks < 20 * one)) ks = one;
    }
    if (ks > nchunks / 4) ks = nchunks / 4;
    if (ks < 1) ks = 1;
    p.ksplit = (int)ks;
    const long long groups = (long long)a->NH * ks;
    const long long grid = (groups + 7) / 8 * 8 * tiles;
    if (grid > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tiles for one launch");
    void (*kern)(BwdParamParams);
    if (bf16) kern = nt == 256 ? slstm_bwd_param_kernel<true, 256> : (nt == 128 ? slstm_bwd_param_kernel<true, 128> : slstm_bwd_param_kernel<true, 64>);
    else kern = nt == 256 ? slstm_bwd_param_kernel<false, 256> : (nt == 128 ? slstm_bwd_param_kernel<false, 128> : slstm_bwd_param_kernel<false, 64>);
    size_t lds = (size_t)bwd_param_lds_bytes(bf16, nt);
    if (slab) {
      kern = nt == 256 ? slstm_bwd_param_slab_kernel<256> : (nt == 128 ? slstm_bwd_param_slab_kernel<128> : slstm_bwd_param_slab_kernel<64>);
      lds = (size_t)param_slab_lds_bytes(nt);
    }
    if (lds > 64 * 1024) {
      const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
      if (rc != XS_OK) return rc;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), lds, stream, p);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "parameter gradient kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

int check_conv(const xs_conv_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->D <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d D=%d", a->B, a->T, a->D);
  if (a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "xs_causal_conv_silu computes on bf16 tensors only");
  if (a->K < 2 || a->K > 4) return fail(XS_ERR_UNSUPPORTED, "convolution of %d taps not supported (2..4)", a->K);
  if (a->D % 8 != 0) return fail(XS_ERR_UNSUPPORTED, "D = %d is not a multiple of 8", a->D);
  if (a->ring_out && (a->T != 1 || a->reset)) return fail(XS_ERR_SHAPE, "ring_out goes with a single unmasked token (T == 1, no reset mask)");
  if (a->B == 0 || a->T == 0) return XS_OK;
  if (!a->x || !a->weight || !a->out) return fail(XS_ERR_NULL, "x, weight and out are required");
  if ((uintptr_t)a->ring_out % 16) return fail(XS_ERR_ALIGN, "ring_out must be 16-byte aligned");
  if (a->ring_out && a->conv_state) {  // other threads still read the old ring while the first ones write the new one
    const uintptr_t lo0 = (uintptr_t)a->conv_state, lo1 = (uintptr_t)a->ring_out;
    const uintptr_t sb = (uintptr_t)(a->conv_state_stride_b ? a->conv_state_stride_b : (long long)(a->K - 1) * a->D) * 2;
    const uintptr_t n0 = sb * (uintptr_t)(a->B - 1) + (uintptr_t)(a->K - 1) * a->D * 2, n1 = (uintptr_t)a->B * a->K * a->D * 2;
    if (lo0 < lo1 + n1 && lo1 < lo0 + n0) return fail(XS_ERR_SHAPE, "ring_out must not overlap conv_state");
  }
  if (a->x_stride_t < a->D || (a->B > 1 && a->x_stride_b < a->D)) return fail(XS_ERR_SHAPE, "x strides overlap the innermost D elements");
  if (a->reset && a->reset_stride_b < a->T) return fail(XS_ERR_SHAPE, "reset row stride %lld < T", (long long)a->reset_stride_b);
  if (a->conv_state && a->conv_state_stride_b && (a->conv_state_stride_b < (long long)(a->K - 1) * a->D || a->conv_state_stride_b % 8))
    return fail(XS_ERR_SHAPE, "conv_state row stride %lld too small or not 16-byte aligned", (long long)a->conv_state_stride_b);
  if (((uintptr_t)a->x % 16) || ((a->x_stride_b * 2) % 16) || ((a->x_stride_t * 2) % 16) || ((uintptr_t)a->conv_state % 16) ||
      ((uintptr_t)a->weight % 16) || ((uintptr_t)a->bias % 16) || ((uintptr_t)a->out % 16))
    return fail(XS_ERR_ALIGN, "x and its strides, conv_state, weight, bias and out must be 16-byte aligned");
  return XS_OK;
}

int run_conv(const xs_conv_args *a, void *x_out = nullptr) {
  const int rc = check_conv(a);
  if (rc != XS_OK || a->B == 0 || a->T == 0) return rc;
  if (x_out) {
    if (!a->ring_out) return fail(XS_ERR_NULL, "x_out goes with ring_out");
    if ((uintptr_t)x_out % 16) return fail(XS_ERR_ALIGN, "x_out must be 16-byte aligned");
    const long long row = 2ll * a->D, x_sb = a->B > 1 ? 2 * a->x_stride_b : 0, taps = (a->K - 1) * row, taps_sb = a->conv_state_stride_b ? 2 * a->conv_state_stride_b : taps;
    const struct { const char *name; const void *p; long long bytes; } others[4] = {
        {"x", a->x, (a->B - 1) * x_sb + row}, {"conv_state", a->conv_state, a->conv_state ? (a->B - 1) * taps_sb + taps : 0}, {"out", a->out, a->B * row}, {"ring_out", a->ring_out, a->B * a->K * row}};
    for (const auto &o : others)
      if ((uintptr_t)x_out < (uintptr_t)o.p + o.bytes && (uintptr_t)o.p < (uintptr_t)x_out + a->B * row) return fail(XS_ERR_SHAPE, "x_out must not overlap %s", o.name);
  }
  const long long threads = (long long)a->B * a->T * (a->D / 8);
  const long long blocks = ((threads + 255) / 256 + 7) / 8 * 8;  // a multiple of 8: the kernel deals them out by XCD
  if (blocks > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one launch");
  ConvParams p;
  p.x = (const uint16_t *)a->x; p.x_sb = a->x_stride_b; p.x_st = a->x_stride_t;
  p.state = (const uint16_t *)a->conv_state;
  p.state_sb = a->conv_state_stride_b ? a->conv_state_stride_b : (long long)(a->K - 1) * a->D;
  p.w = (const uint16_t *)a->weight; p.bias = (const uint16_t *)a->bias;
  p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  p.out = (uint16_t *)a->out;
  p.ring_out = (uint16_t *)a->ring_out; p.x_out = (uint16_t *)x_out;
  p.B = a->B; p.T = a->T; p.D = a->D;
  hipStream_t stream = (hipStream_t)a->stream;
  void (*kern)(ConvParams) = a->K == 2 ? causal_conv_silu_kernel<2> : (a->K == 3 ? causal_conv_silu_kernel<3> : causal_conv_silu_kernel<4>);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "convolution kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

template <int BM, int BN, int D>
int launch_gates(const xs_gates_args *a, GatesParams p, hipStream_t stream) {
  p.n_tiles = 4 * a->NH * (a->dh / BN);
  p.m_tiles = (a->M + BM - 1) / BM;
  const int w_major = p.m_tiles <= 8;
  const long long grid = w_major ? (long long)8 * ((p.n_tiles + 7) / 8) * p.m_tiles : (long long)8 * ((p.m_tiles + 7) / 8) * p.n_tiles;
  if (grid > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tiles for one launch");
  if ((long long)BM * a->x_stride_row * 2 >= (1ll << 31) || (long long)BM * a->x_conv_stride_row * 2 >= (1ll << 31))
    return fail(XS_ERR_UNSUPPORTED, "%d rows of x span 2 GiB or more", BM);
  void (*kern)(GatesParams, int) = headwise_gates_kernel<BM, BN, D>;
  const size_t lds = (size_t)D * (BM + BN) * 128;
  if (lds > 64 * 1024) {
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
    if (rc != XS_OK) return rc;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, stream, p, w_major);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "gate projection kernel launch failed: %s", hipGetErrorString(e));
}

// Tiles of the general kernel, by the number of tokens (us at 4 heads of 1024; the kernel before it in brackets):
// up to 32 token tiles of 16 (M 1: 7.3 [101], M 30: 8.1 [103]); 128 x 128 tiles where the head dim allows them and they
// fill the compute units (M 1024: 43 [215], M 16384: 786 [2828]); 64 x 64 in between and for the other head dims (M 64:
// 9.3 [106]; 4 heads of 192, M 4096: 17.3 [40.7]).  A ring of few slots lets several workgroups share a compute unit,
// which is worth more than slabs asked for further ahead.
int launch_gates_tiles(const xs_gates_args *a, const GatesParams &p, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) return fail(XS_ERR_DEVICE, "cannot query the device");
  if (a->M <= 32) return launch_gates<16, 64, 4>(a, p, stream);
  if (a->dh % 128 == 0 && (long long)((a->M + 127) / 128) * 4 * a->NH * (a->dh / 128) >= cus) return launch_gates<128, 128, 2>(a, p, stream);
  return launch_gates<64, 64, 3>(a, p, stream);
}

int check_gates(const xs_gates_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->M < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims M=%d NH=%d dh=%d", a->M, a->NH, a->dh);
  if (a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "xs_headwise_gates computes on bf16 tensors only");
  if (a->dh % 64 != 0) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not a multiple of 64", a->dh);
  if (a->M == 0) return XS_OK;
  const long long H = (long long)a->NH * a->dh;
  if (!a->x || !a->x_conv || !a->out || !a->w[0] || !a->w[1] || !a->w[2] || !a->w[3])
    return fail(XS_ERR_NULL, "x, x_conv, the four weights and out are required");
  if (a->x_stride_row < H || a->x_conv_stride_row < H || a->out_stride_row < 4 * H)
    return fail(XS_ERR_SHAPE, "a row stride is smaller than the row");
  if (((uintptr_t)a->x % 16) || ((uintptr_t)a->x_conv % 16) || ((uintptr_t)a->out % 16) || ((a->x_stride_row * 2) % 16) ||
      ((a->x_conv_stride_row * 2) % 16) || ((a->out_stride_row * 2) % 16) || ((uintptr_t)a->w[0] % 16) ||
      ((uintptr_t)a->w[1] % 16) || ((uintptr_t)a->w[2] % 16) || ((uintptr_t)a->w[3] % 16))
    return fail(XS_ERR_ALIGN, "x, x_conv, out, their row strides and the weights must be 16-byte aligned");
  return XS_OK;
}

int run_gates(const xs_gates_args *a) {
  const int rc = check_gates(a);
  if (rc != XS_OK || a->M == 0) return rc;
  GatesParams p;
  p.x = (const uint16_t *)a->x; p.xc = (const uint16_t *)a->x_conv;
  p.x_sr = a->x_stride_row; p.xc_sr = a->x_conv_stride_row;
  for (int g = 0; g < 4; ++g) p.w[g] = (const uint16_t *)a->w[g];
  p.out = (uint16_t *)a->out; p.out_sr = a->out_stride_row;
  p.M = a->M; p.NH = a->NH; p.dh = a->dh;
  hipStream_t stream = (hipStream_t)a->stream;
  const int combos = 2 * a->NH;               // (head, operand)
  const int bm = a->dh == 256 ? 64 : 32;      // the resident kernel's tokens per tile: threads / 8
  const int cus = device_cus();
  if (cus <= 0) return fail(XS_ERR_DEVICE, "cannot query the device");
  const int parts = cus / combos > 1 ? cus / combos : 1;
  if ((a->dh == 128 || a->dh == 256) && (a->M + bm - 1) / bm >= 4 * parts) {
    // weights resident in registers, workgroups walk over token tiles: pays from four tiles per workgroup on (8 heads of
    // 256, M 4096: 34 us against 49 with the general kernel; M 1024, one tile each: 16.7 against 13.6)
    p.m_tiles = (a->M + bm - 1) / bm;
    p.n_tiles = combos;
    if (a->dh == 256) hipLaunchKernelGGL(headwise_gates_resident_kernel<4>, dim3((unsigned)(combos * parts)), dim3(512), 0, stream, p, combos, parts);
    else hipLaunchKernelGGL(headwise_gates_resident_kernel<2>, dim3((unsigned)(combos * parts)), dim3(256), 0, stream, p, combos, parts);
  } else if ((a->dh == 128 || a->dh == 256) && a->M <= 256) {
    // a decode step: every compute unit fetches its share of the weights once, the whole K range at once (8 heads of 128,
    // M 256: 3.4 us against 3.8)
    p.m_tiles = (a->M + 63) / 64;
    p.n_tiles = 4 * a->NH * (a->dh / 64);
    const size_t lds = (size_t)128 * (a->dh * 2 + 16);
    void (*kern)(GatesParams) = a->dh == 256 ? headwise_gates_slab_kernel<4> : headwise_gates_slab_kernel<2>;
    if (lds > 64 * 1024) {
      const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
      if (rc != XS_OK) return rc;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.m_tiles * p.n_tiles)), dim3(256), lds, stream, p);
  } else {
    return launch_gates_tiles(a, p, stream);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "gate projection kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

int run_group_norm(const xs_norm_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (a->dtype != XS_BF16) return fail(XS_ERR_DTYPE, "xs_headwise_group_norm computes on bf16 tensors only");
  if (a->dh % 4 != 0 || a->dh > 1024) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not a multiple of 4 up to 1024", a->dh);
  if (a->B == 0 || a->T == 0) return XS_OK;
  if (!a->x || !a->out) return fail(XS_ERR_NULL, "x and out are required");
  if (((uintptr_t)a->x % 8) || ((uintptr_t)a->out % 8) || ((uintptr_t)a->weight % 8) || (a->x_stride_b % 4) || (a->x_stride_t % 4) || (a->x_stride_h % 4))
    return fail(XS_ERR_ALIGN, "x, weight, out and the strides of x must be 8-byte aligned");
  const long long groups = (long long)a->B * a->T * a->NH;
  const long long blocks = (groups + 3) / 4;
  if (blocks > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one launch");
  NormParams p;
  p.x = (const uint16_t *)a->x; p.x_sb = a->x_stride_b; p.x_st = a->x_stride_t; p.x_sh = a->x_stride_h;
  p.weight = (const uint16_t *)a->weight; p.out = (uint16_t *)a->out; p.eps = a->eps;
  p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
  const int pieces = (a->dh + 255) / 256;
  void (*kern)(NormParams) = pieces == 1 ? headwise_group_norm_kernel<1> : (pieces == 2 ? headwise_group_norm_kernel<2> : headwise_group_norm_kernel<4>);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)a->stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "group norm kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// ---- one decoded token of a layer up to its hidden state (slstm_layer_step_kernel.h)
// How its kernel splits it; ut 0: not at all, the kernels of its parts are the faster way.
// us a token with the group norm behind it, replayed from a graph, the parts' kernels -> this one.  One workgroup of 16 units
// a compute unit: 4 heads of 64, 7 rows 11.9 -> 6.7, 4 of 256, 64 rows 14.5 -> 9.6, 4 of 512, 7 rows 16.0 -> 12.6.  Up to two, as one of
// 32 units: 8 of 256, 64 rows 15.6 -> 11.0 (as two 13.0), 4 of 512, 64 rows 22.2 -> 17.4 (24.8).  Beyond, several row tiles
// a workgroup of 32 units: 8 of 256, 128 rows 18.5 -> 14.3, 256 rows 23.0 -> 20.8, 16 of 256, 256 rows (16 a compute unit, each
// as many again 5.6 us against 4.2) 34.4 -> 32.0.  Head dims beyond 256 have no registers for several row tiles, 1024 (its
// whole head in a convolution, 32 products in one chain) gains nothing: 1 row 24.0 -> 24.0, 16 rows 26.0 -> 27.3.
struct LayerStepSplit { int nch, ut, row_groups; bool loop; };
LayerStepSplit layer_step_split(int B, int NH, int dh, int K) {
  LayerStepSplit s{1, 0, (B + 15) / 16, false};
  while (s.nch * 128 < dh) s.nch *= 2;
  const long long cus = device_cus(), wgs = (long long)NH * (dh / 16) * s.row_groups;  // workgroups of 16 rows x 16 units
  if (K != 4 || s.nch > 4 || cus <= 0 || wgs > (s.nch <= 2 ? 16 : 2) * cus) return s;
  s.ut = wgs <= cus ? 1 : 2;
  if (wgs > 2 * cus) {
    s.loop = true;
    s.row_groups = (int)std::min<long long>(s.row_groups, std::max(1ll, cus / ((long long)NH * (dh / 32))));
  }
  return s;
}
int run_layer_step(const xs_layer_step_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  xs_slstm_args cell = a->cell;
  const int B = cell.B, NH = cell.NH, dh = cell.dh;
  const long long D = (long long)NH * dh;
  if (cell.wx_dtype != XS_BF16) return fail(XS_ERR_DTYPE, "xs_layer_step computes on bf16 tensors only");
  if (NH <= 0 || dh <= 0 || dh % 64) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not a multiple of 64", dh);
  if (!cell.s0 || cell.reset) return fail(XS_ERR_UNSUPPORTED, "a layer's step goes with a state and without a mask");
  if (B > 0 && (!a->x || !a->ring_out)) return fail(XS_ERR_NULL, "x and ring_out are required");
  cell.wx = a->x; cell.wx_stride_b = cell.wx_stride_t = 4 * D;  // (not read)
  int rc = validate(&cell, true);
  if (rc != XS_OK || B == 0) return rc;
  const LayerStepSplit split = layer_step_split(B, NH, dh, a->K);
  if (!split.ut) return fail(XS_ERR_UNSUPPORTED, "xs_layer_step does not take %d rows of %d heads of %d with %d taps", B, NH, dh, a->K);
  xs_conv_args conv{};
  conv.B = B; conv.T = 1; conv.D = (int32_t)D; conv.K = a->K; conv.dtype = XS_BF16;
  conv.x = a->x; conv.x_stride_b = conv.x_stride_t = D;
  conv.conv_state = a->conv_state; conv.conv_state_stride_b = a->conv_state_stride_b;
  conv.weight = a->conv_w; conv.bias = a->conv_b; conv.out = conv.ring_out = a->ring_out;
  xs_gates_args gates{};
  gates.M = B; gates.NH = NH; gates.dh = dh; gates.dtype = XS_BF16;
  gates.x = gates.x_conv = a->x; gates.x_stride_row = gates.x_conv_stride_row = D;
  for (int g = 0; g < 4; ++g) gates.w[g] = a->gate_w[g];
  gates.out = a->ring_out; gates.out_stride_row = 4 * D;
  if ((rc = check_conv(&conv)) != XS_OK || (rc = check_gates(&gates)) != XS_OK) return rc;
  if ((uintptr_t)a->x_out % 16) return fail(XS_ERR_ALIGN, "x_out must be 16-byte aligned");
  // other workgroups of a head still read its x and its taps while the first ones write
  const long long row = D * 2, taps_sb = a->conv_state_stride_b ? a->conv_state_stride_b * 2 : 3 * row;
  const struct { const char *name; const void *p; long long bytes; } in[2] = {{"x", a->x, B * row}, {"conv_state", a->conv_state, a->conv_state ? (B - 1) * taps_sb + 3 * row : 0}},
      out[4] = {{"ring_out", a->ring_out, 4 * B * row}, {"h_out", cell.h_out, B * row}, {"s_out", cell.s_out, 8 * B * row}, {"x_out", a->x_out, a->x_out ? B * row : 0}};
  for (const auto &i : in)
    for (const auto &o : out)
      if ((uintptr_t)i.p < (uintptr_t)o.p + o.bytes && (uintptr_t)o.p < (uintptr_t)i.p + i.bytes) return fail(XS_ERR_SHAPE, "%s must not overlap %s", o.name, i.name);
  LayerStepParams p;
  p.step = step_params(&cell);
  p.step.n_unit_tiles = dh / (16 * split.ut);
  p.step.n_row_tiles = split.row_groups;
  p.step.h_prev = cell.h_prev;
  p.row_tiles = (B + 15) / 16;
  p.x = (const uint16_t *)a->x;
  p.state = (const uint16_t *)a->conv_state;
  p.state_sb = a->conv_state_stride_b ? a->conv_state_stride_b : 3 * D;
  p.conv_w = (const uint16_t *)a->conv_w; p.conv_b = (const uint16_t *)a->conv_b;
  for (int g = 0; g < 4; ++g) p.gate_w[g] = (const uint16_t *)a->gate_w[g];
  p.ring_out = (uint16_t *)a->ring_out; p.x_out = (uint16_t *)a->x_out;
  const LayerStepKernel kern = cell.h_prev ? pick_layer_step<true>(split.nch, split.ut, split.loop) : pick_layer_step<false>(split.nch, split.ut, split.loop);
  const size_t lds = (size_t)layer_step_lds_bytes(split.nch);
  if (lds + 25600 * split.ut > 64 * 1024 && (rc = ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds)) != XS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(NH * p.step.n_unit_tiles * p.step.n_row_tiles)), dim3(256 * split.ut), lds, (hipStream_t)cell.stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "layer step kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// ---- the float32 layer around the cell (slstm_layer_f32_kernels.h)
int layer_launched(const char *what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? XS_OK : fail(XS_ERR_LAUNCH, "%s launch failed: %s", what, hipGetErrorString(e));
}
bool layer_misaligned(std::initializer_list<const void *> ptrs) {
  for (const void *q : ptrs)
    if ((uintptr_t)q % 16) return true;
  return false;
}
int layer_check(const xs_layer_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->B < 0 || a->T < 0 || a->NH <= 0 || a->dh <= 0) return fail(XS_ERR_SHAPE, "bad dims B=%d T=%d NH=%d dh=%d", a->B, a->T, a->NH, a->dh);
  if (a->dh % 4 || a->dh > 512) return fail(XS_ERR_UNSUPPORTED, "head dim %d is not a multiple of 4 up to 512", a->dh);
  if ((long long)a->B * a->T > (1ll << 29)) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one call");
  return XS_OK;
}
// how a backward pass splits its sums over tokens
struct LayerSplit { int conv_blocks, slices, slice_tokens; size_t gate_floats, conv_floats; };
LayerSplit layer_split(int B, int T, int NH, int dh, int K) {
  LayerSplit s;
  const long long M = (long long)B * T, D = (long long)NH * dh, up = (dh + 63) / 64;
  s.conv_blocks = (int)(((long long)B * ((T + kConvBackRun - 1) / kConvBackRun) + 7) / 8);
  // 1024 workgroups, four a compute unit, but slices of 256 tokens and more (us at 4096 tokens x 4 heads of 128 in 8, 16, 32
  // slices 31.0, 28.5, 29.5; 6732 x 8 of 256 in 1, 2, 4: 346, 303, 295)
  const long long tiles = 4 * NH * up * up, want = std::max(1ll, std::min(1024 / tiles, (M + 255) / 256));
  s.slice_tokens = (int)(((M + want - 1) / want + kProductK - 1) / kProductK * kProductK);
  s.slices = (int)((M + s.slice_tokens - 1) / s.slice_tokens);
  s.gate_floats = s.slices > 1 ? (size_t)s.slices * 4 * D * dh : 0;
  s.conv_floats = (size_t)s.conv_blocks * D * (K + 1);
  return s;
}
LayerConvParams layer_conv_params(const xs_layer_args *a) {
  LayerConvParams p{};
  p.B = a->B; p.T = a->T; p.D = a->NH * a->dh;
  p.x = a->x; p.x_sb = a->x_stride_b; p.x_st = a->x_stride_t;
  p.state = a->conv_state; p.state_sb = a->conv_state_stride_b ? a->conv_state_stride_b : (long long)(a->K - 1) * p.D;
  p.w = a->conv_w; p.bias = a->conv_b;
  p.reset = a->reset; p.reset_sb = a->reset_stride_b;
  return p;
}
LayerProductParams layer_product_params(const xs_layer_args *a) {
  LayerProductParams p{};
  const long long D = (long long)a->NH * a->dh;
  p.a[0] = a->x_conv; p.a_sb[0] = a->T * D; p.a_st[0] = D;
  p.a[1] = a->x; p.a_sb[1] = a->x_stride_b; p.a_st[1] = a->x_stride_t;
  for (int g = 0; g < 4; ++g) { p.w[g] = a->gate_w[g]; p.d_w[g] = a->d_gate_w[g]; }
  p.wx = a->wx; p.d_wx = a->d_wx; p.d_a[0] = a->d_x_conv; p.d_a[1] = a->d_x;
  p.M = a->B * a->T; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
  p.m_tiles = (p.M + 63) / 64; p.slices = 1; p.slice_tokens = p.M;
  return p;
}
template <LayerProduct MODE>
int launch_layer_product(LayerProductParams p, hipStream_t stream) {
  const int up = (p.dh + 63) / 64;
  // (INPUTS: the operand x behind x_conv, and not at all where its gradient is not wanted)
  p.tiles = MODE == LayerProduct::WEIGHTS ? 4 * up * up : (MODE == LayerProduct::INPUTS ? (p.d_a[1] ? 2 : 1) : 4) * up;
  const long long pairs = (long long)p.NH * (MODE == LayerProduct::WEIGHTS ? p.slices : p.m_tiles);
  const long long grid = 8 * ((pairs + 7) / 8) * p.tiles;
  if (grid > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tiles for one launch");
  p.pairs = (int)pairs; p.pairs_per_xcd = (int)((pairs + 7) / 8);
  hipLaunchKernelGGL(layer_product_f32_kernel<MODE>, dim3((unsigned)grid), dim3(256), 0, stream, p);
  return layer_launched("projection kernel");
}

int layer_front_check(const xs_layer_args *a) {
  const long long D = (long long)a->NH * a->dh;
  if (a->K < 2 || a->K > 4) return fail(XS_ERR_UNSUPPORTED, "convolution of %d taps not supported (2..4)", a->K);
  if (!a->x || !a->conv_w || !a->gate_w[0] || !a->gate_w[1] || !a->gate_w[2] || !a->gate_w[3] || !a->x_conv)
    return fail(XS_ERR_NULL, "x, the weights and x_conv are required");
  if (a->x_stride_t < D || (a->B > 1 && a->x_stride_b < D)) return fail(XS_ERR_SHAPE, "x strides overlap the innermost D elements");
  if (a->x_stride_b % 4 || a->x_stride_t % 4 || layer_misaligned({a->x, a->conv_w, a->conv_b, a->gate_w[0], a->gate_w[1], a->gate_w[2], a->gate_w[3], a->x_conv}))
    return fail(XS_ERR_ALIGN, "x, its strides, the weights and x_conv must be 16-byte aligned");
  return XS_OK;
}

int run_layer_front(const xs_layer_args *a) {
  int rc = layer_check(a);
  if (rc != XS_OK || a->B == 0 || a->T == 0) return rc;
  if ((rc = layer_front_check(a)) != XS_OK) return rc;
  const long long D = (long long)a->NH * a->dh;
  if (!a->wx) return fail(XS_ERR_NULL, "wx is required");
  if (a->conv_state && a->conv_state_stride_b && (a->conv_state_stride_b < (a->K - 1) * D || a->conv_state_stride_b % 4))
    return fail(XS_ERR_SHAPE, "conv_state row stride %lld too small or not 16-byte aligned", (long long)a->conv_state_stride_b);
  if (layer_misaligned({a->conv_state, a->wx})) return fail(XS_ERR_ALIGN, "conv_state and wx must be 16-byte aligned");
  LayerConvParams c = layer_conv_params(a);
  c.out = a->x_conv;
  const long long threads = (long long)a->B * ((a->T + kConvRun - 1) / kConvRun) * (D / 4), blocks = (threads + 255) / 256;
  if (blocks > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one launch");
  void (*kern)(LayerConvParams) = a->K == 2 ? layer_conv_f32_kernel<2> : (a->K == 3 ? layer_conv_f32_kernel<3> : layer_conv_f32_kernel<4>);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)a->stream, c);
  if ((rc = layer_launched("convolution kernel")) != XS_OK) return rc;
  return launch_layer_product<LayerProduct::PROJECT>(layer_product_params(a), (hipStream_t)a->stream);
}

template <int L, int P>
void launch_layer_norm(const LayerNormParams &p, hipStream_t stream) {
  const long long groups = (long long)p.B * p.T * p.NH;
  hipLaunchKernelGGL((layer_norm_f32_kernel<L, P>), dim3((unsigned)((groups + 256 / L - 1) / (256 / L))), dim3(256), 0, stream, p);
}
int run_layer_norm(const xs_layer_args *a) {
  const int rc = layer_check(a);
  if (rc != XS_OK || a->B == 0 || a->T == 0) return rc;
  if (!a->h || !a->out) return fail(XS_ERR_NULL, "h and out are required");
  if (layer_misaligned({a->h, a->norm_w, a->out})) return fail(XS_ERR_ALIGN, "h, norm_w and out must be 16-byte aligned");
  if ((long long)a->B * a->T * a->NH > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one launch");
  LayerNormParams p{};
  p.y = a->h; p.weight = a->norm_w; p.out = a->out; p.eps = a->eps;
  p.B = a->B; p.T = a->T; p.NH = a->NH; p.dh = a->dh;
  hipStream_t stream = (hipStream_t)a->stream;
  if (a->dh <= 64) launch_layer_norm<16, 1>(p, stream);
  else if (a->dh <= 128) launch_layer_norm<32, 1>(p, stream);
  else if (a->dh <= 256) launch_layer_norm<64, 1>(p, stream);
  else launch_layer_norm<64, 2>(p, stream);
  return layer_launched("group norm kernel");
}

int run_layer_front_backward(const xs_layer_args *a) {
  int rc = layer_check(a);
  if (rc != XS_OK || a->B == 0 || a->T == 0) return rc;
  if ((rc = layer_front_check(a)) != XS_OK) return rc;
  const bool gates = a->d_gate_w[0] || a->d_gate_w[1] || a->d_gate_w[2] || a->d_gate_w[3], conv = a->d_conv_w || a->d_conv_b, inputs = a->d_x || conv;
  if (!a->d_wx || !a->scratch || (inputs && !a->d_x_conv)) return fail(XS_ERR_NULL, "d_wx, scratch and, for d_x and the convolution's gradients, d_x_conv are required");
  if (a->conv_state) return fail(XS_ERR_UNSUPPORTED, "no gradient through a convolution that continues from a state");
  if (layer_misaligned({a->d_wx, a->d_x_conv, a->d_x, a->scratch, a->d_gate_w[0], a->d_gate_w[1], a->d_gate_w[2], a->d_gate_w[3]}))
    return fail(XS_ERR_ALIGN, "d_wx, d_x_conv, d_x, scratch and d_gate_w must be 16-byte aligned");
  const LayerSplit split = layer_split(a->B, a->T, a->NH, a->dh, a->K);
  hipStream_t stream = (hipStream_t)a->stream;
  const long long D = (long long)a->NH * a->dh;
  LayerProductParams g = layer_product_params(a);
  if (inputs && (rc = launch_layer_product<LayerProduct::INPUTS>(g, stream)) != XS_OK) return rc;
  g.slices = split.slices; g.slice_tokens = split.slice_tokens; g.partial = a->scratch;
  if (gates && (rc = launch_layer_product<LayerProduct::WEIGHTS>(g, stream)) != XS_OK) return rc;
  float *const conv_partial = a->scratch + split.gate_floats;
  if (inputs) {
    LayerConvParams c = layer_conv_params(a);
    c.state = nullptr;
    c.d_out = a->d_x_conv; c.d_x = a->d_x; c.partial = conv ? conv_partial : nullptr;
    const int piece_blocks = (int)((D / 4 + 31) / 32);
    if ((long long)piece_blocks * split.conv_blocks > 0x7FFFFFFF) return fail(XS_ERR_UNSUPPORTED, "too many tokens for one launch");
    void (*kern)(LayerConvParams, int) = a->K == 2 ? layer_conv_backward_f32_kernel<2> : (a->K == 3 ? layer_conv_backward_f32_kernel<3> : layer_conv_backward_f32_kernel<4>);
    hipLaunchKernelGGL(kern, dim3((unsigned)(piece_blocks * split.conv_blocks)), dim3(256), 0, stream, c, piece_blocks);
    if ((rc = layer_launched("convolution gradient kernel")) != XS_OK) return rc;
  }
  LayerReduceParams r{};
  auto region = [](const float *partial, long long n, int parts) { return LayerReduceParams::Region{partial, n, parts, (int)((n + 63) / 64)}; };
  r.region[0] = region(a->scratch, gates && split.slices > 1 ? 4 * D * a->dh : 0, split.slices);
  r.region[1] = region(conv_partial, conv ? D * (a->K + 1) : 0, split.conv_blocks);
  if (!r.region[0].blocks && !r.region[1].blocks) return XS_OK;
  for (int i = 0; i < 4; ++i) r.d_w[i] = a->d_gate_w[i];
  r.d_conv_w = a->d_conv_w; r.d_conv_b = a->conv_b ? a->d_conv_b : nullptr;
  r.per_gate = D * a->dh; r.taps = a->K;
  hipLaunchKernelGGL(layer_reduce_kernel, dim3((unsigned)(r.region[0].blocks + r.region[1].blocks)), dim3(256), 0, stream, r);
  return layer_launched("sum kernel");
}

// ---- measurement: one stage of the dependency chain of a timestep, alone (slstm_serial_bound.h)
int run_stage(const xs_measure_args *a) {
  if (!a) return fail(XS_ERR_NULL, "args is NULL");
  if (a->steps <= 0) return fail(XS_ERR_SHAPE, "steps must be positive");
  hipStream_t stream = (hipStream_t)a->stream;
  StageParams p{};
  p.steps = a->steps;
  p.words = nullptr;
  if (a->stage == XS_STAGE_LAUNCH) {
    for (int i = 0; i < a->steps; ++i) hipLaunchKernelGGL(stage_empty_kernel, dim3(1), dim3(64), 0, stream);
  } else {
    if (!a->workspace || ((uintptr_t)a->workspace % 256)) return fail(XS_ERR_WORKSPACE, "a 256-byte aligned workspace is required");
    p.words = (unsigned int *)a->workspace;
    if (a->stage == XS_STAGE_EXCHANGE) {
      const int G = a->members;
      if (G != 8 && G != 16 && G != 32 && G != 64) return fail(XS_ERR_SHAPE, "members must be 8, 16, 32 or 64");
      if (a->rows < 1 || a->rows > 16) return fail(XS_ERR_SHAPE, "rows must be 1..16");
      const int cus = device_cus();
      const int per_xcd = a->two_xcds ? G / 2 : G;
      if (cus <= 0 || per_xcd > cus / 8) return fail(XS_ERR_DEVICE, "%d workgroups do not fit one XCD of this device at once", per_xcd);
      const size_t ring = (size_t)kRing * G * 512;
      if (a->workspace_bytes < 256 + ring) return fail(XS_ERR_WORKSPACE, "the exchange stage needs %zu bytes of workspace", 256 + ring);
      p.members = G; p.two_xcds = a->two_xcds ? 1 : 0; p.rows = a->rows;
      p.ring = (char *)a->workspace + 256;
      p.spin_limit = kDefaultSpinLimit;
      hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, stream, (uint32_t *)a->workspace, (size_t)64, 0u);
      hipLaunchKernelGGL(fill_u32_kernel, dim3(64), dim3(256), 0, stream, (uint32_t *)p.ring, ring / 4, kSentinel32);
      void (*k)(StageParams) = G == 8 ? stage_exchange_kernel<1> : (G == 16 ? stage_exchange_kernel<2> : (G == 32 ? stage_exchange_kernel<4> : stage_exchange_kernel<8>));
      // tiles of at most 4 rows inside one XCD: the layout and the polls of the kernel for such tiles
      if (a->rows <= 4 && !a->two_xcds && G <= 32)
        k = G == 8 ? stage_exchange_quad_kernel<4> : (G == 16 ? stage_exchange_quad_kernel<8> : stage_exchange_quad_kernel<16>);
      hipLaunchKernelGGL(k, dim3(8 * per_xcd), dim3(256), 0, stream, p);
    } else if (a->stage == XS_STAGE_CHAIN) {
      const int G = 16;  // (head dim 256)
      const int cus = device_cus();
      const int per_xcd = cus > 0 ? (cus / 8) / G : 0;  // head groups per XCD, as many as fit: the product's launch at config 2
      if (per_xcd < 1) return fail(XS_ERR_DEVICE, "a head group of %d workgroups does not fit one XCD of this device", G);
      if (a->rows < 1 || a->rows > 16) return fail(XS_ERR_SHAPE, "rows must be 1..16");
      const size_t ring = (size_t)8 * per_xcd * kRing * G * 512;
      if (a->workspace_bytes < 256 + ring) return fail(XS_ERR_WORKSPACE, "the chain stage needs %zu bytes of workspace", 256 + ring);
      p.members = G; p.two_xcds = 0; p.rows = a->rows;
      p.ring = (char *)a->workspace + 256;
      p.spin_limit = kDefaultSpinLimit;
      hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, stream, (uint32_t *)a->workspace, (size_t)64, 0u);
      hipLaunchKernelGGL(fill_u32_kernel, dim3(64), dim3(256), 0, stream, (uint32_t *)p.ring, ring / 4, kSentinel32);
      hipLaunchKernelGGL(stage_chain_kernel, dim3(8 * per_xcd * G), dim3(256), 0, stream, p);
    } else if (a->stage == XS_STAGE_CONTRACTION) {
      if (a->workspace_bytes < 256) return fail(XS_ERR_WORKSPACE, "256 bytes of workspace are required");
      hipLaunchKernelGGL(stage_contraction_kernel<2>, dim3(1), dim3(256), 0, stream, p);
    } else if (a->stage == XS_STAGE_GATING) {
      if (a->workspace_bytes < 256) return fail(XS_ERR_WORKSPACE, "256 bytes of workspace are required");
      hipLaunchKernelGGL(stage_gating_kernel, dim3(1), dim3(256), 0, stream, p);
    } else {
      return fail(XS_ERR_SHAPE, "unknown stage %d", a->stage);
    }
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "measurement kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

// host side of the static scratch array: its device address, per device
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

int static_scratch(void **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return fail(XS_ERR_DEVICE, "cannot query the current device");
  if (dev < 0 || dev >= kMaxDevices) return fail(XS_ERR_DEVICE, "device %d beyond the %d this entry point keeps scratch for", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));  // this device's copy of the array
    if (e != hipSuccess || !ptr) return fail(XS_ERR_DEVICE, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return XS_OK;
}

}  // namespace

extern "C" {

int xs_abi_version(void) { return XS_ABI_VERSION; }

const char *xs_last_error(void) { return g_err; }

size_t xs_slstm_workspace_bytes(int32_t B, int32_t T, int32_t NH, int32_t dh) {
  if (B < 0 || T < 0 || NH <= 0 || dh <= 0) return 0;
  return kHeaderBytes + xbuf_elems(B, NH, dh) * 4;
}

int xs_slstm_forward_watched(const xs_slstm_args *args, uint32_t *abort_host) {
  g_err[0] = 0;
  const int rc = validate(args, false);
  if (rc != XS_OK) return rc;
  if (args->coef_out) {  // a training forward: is this one of the calls that can leave the coefficients? (launches nothing)
    if (args->T < 1 || args->B < 1) return fail(XS_ERR_UNSUPPORTED, "coef_out: nothing to do for an empty call");
    size_t need = 0;
    const int rd = run_forward(args, &need);
    if (rd != XS_OK) return rd;
    return run_forward(args, nullptr, abort_host);  // (also for one token: the step kernels keep no gate values)
  }
  // one token: the tiled step kernel (no waits between compute units, bit-identical to the sequence kernel)
  if (args->T == 1 && args->B > 0 && args->r_dtype == args->wx_dtype) return run_step(args);
  return run_forward(args, nullptr, abort_host);
}

int xs_slstm_forward(const xs_slstm_args *args) { return xs_slstm_forward_watched(args, nullptr); }

int xs_slstm_forward_static(const xs_slstm_args *args) {
  g_err[0] = 0;
  int rc = validate(args, false, true);
  if (rc != XS_OK) return rc;
  if (args->coef_out) return fail(XS_ERR_UNSUPPORTED, "coef_out goes with xs_slstm_forward");
  xs_slstm_args a = *args;
  rc = static_scratch(&a.workspace);
  if (rc != XS_OK) return rc;
  a.workspace_bytes = XS_STATIC_SCRATCH_BYTES;
  if (a.T == 1 && a.B > 0 && a.r_dtype == a.wx_dtype) return run_step(&a);  // (touches the status block only)
  size_t need = 0;
  rc = run_forward(&a, &need);  // what the launches of this call would touch; launches nothing
  if (rc != XS_OK) return rc;
  if (need > (size_t)XS_STATIC_SCRATCH_BYTES)
    return fail(XS_ERR_WORKSPACE, "this call needs %zu bytes of scratch, the static array holds %zu: use xs_slstm_forward with a workspace",
                need, (size_t)XS_STATIC_SCRATCH_BYTES);
  return run_forward(&a);
}

size_t xs_slstm_train_coef_floats(int32_t B, int32_t T, int32_t NH, int32_t dh, int32_t dtype) {
  if (B < 1 || T < 1 || NH < 1 || (dtype != XS_F32 && dtype != XS_BF16) || !trains(dh, dtype == XS_BF16)) return 0;
  return (size_t)T * ((B + 3) / 4) * NH * ((dh + 15) / 16) * 576;
}

size_t xs_slstm_train_exchange_bytes(int32_t B, int32_t NH, int32_t dh, int32_t dtype) {
  if (B < 1 || NH < 1 || (dtype != XS_F32 && dtype != XS_BF16) || !trains(dh, dtype == XS_BF16) || local_head(dh, dtype == XS_BF16)) return 0;
  UnitPlan u;
  return unit_plan(B, NH, dh, dtype == XS_BF16, u) == XS_OK ? unit_ring_bytes(u, dtype == XS_BF16 ? 2 : 4) : 0;
}

int xs_slstm_train_forward(const xs_slstm_args *args, float *coef, uint32_t *abort_host) {
  g_err[0] = 0;
  const int rc = validate(args, false);
  if (rc != XS_OK) return rc;
  if (!coef || ((uintptr_t)coef % 16)) return fail(coef ? XS_ERR_ALIGN : XS_ERR_NULL, "coef is required, 16-byte aligned");
  if (args->coef_out) return fail(XS_ERR_UNSUPPORTED, "coef_out goes with xs_slstm_forward");
  if (!xs_slstm_train_coef_floats(args->B, args->T, args->NH, args->dh, args->wx_dtype))
    return fail(XS_ERR_UNSUPPORTED, "a training forward: at least one row and step, head dims up to 1024 (bf16) and 512 (float32)");
  if (local_head(args->dh, args->wx_dtype == XS_BF16)) return run_local(args, coef);
  return run_forward(args, nullptr, abort_host, coef);
}

int xs_slstm_train_backward(const xs_slstm_bwd_args *args, int64_t d_h_stride_b, int64_t d_h_stride_t, int32_t r_dtype, uint32_t *abort_host) {
  g_err[0] = 0;
  return run_train_backward(args, d_h_stride_b, d_h_stride_t, r_dtype, abort_host);
}

int xs_slstm_step(const xs_slstm_args *args) {
  g_err[0] = 0;
  const int rc = validate(args, true);
  if (rc != XS_OK) return rc;
  if (args->coef_out) return fail(XS_ERR_UNSUPPORTED, "coef_out goes with xs_slstm_forward");
  return run_step(args);
}

int xs_slstm_backward_prepare(const xs_slstm_bwd_args *args) {
  g_err[0] = 0;
  return run_backward(args, true);
}

int xs_slstm_backward(const xs_slstm_bwd_args *args) {
  g_err[0] = 0;
  return run_backward(args, false);
}

int xs_measure_stage(const xs_measure_args *args) {
  g_err[0] = 0;
  return run_stage(args);
}

int xs_slstm_backward_params(const xs_slstm_bwd_args *args) {
  g_err[0] = 0;
  return run_backward_params(args);
}

int xs_slstm_tile_r_for_steps(const void *r, void *r_tiled, int32_t NH, int32_t dh, int32_t dtype, void *stream) {
  g_err[0] = 0;
  if (!r || !r_tiled) return fail(XS_ERR_NULL, "r and r_tiled are required");
  if (NH <= 0 || dh <= 0 || dh % 64 != 0) return fail(XS_ERR_SHAPE, "bad dims NH=%d dh=%d (a multiple of 64)", NH, dh);
  if (dtype != XS_F32 && dtype != XS_BF16) return fail(XS_ERR_DTYPE, "dtype must be XS_F32 or XS_BF16");
  if (((uintptr_t)r % 16) || ((uintptr_t)r_tiled % 16)) return fail(XS_ERR_ALIGN, "r and r_tiled must be 16-byte aligned");
  void (*init)(const void *, void *, const float *, void *, int, int, int) = dtype == XS_BF16 ? slstm_fwd_walk_init_kernel<true> : slstm_fwd_walk_init_kernel<false>;
  hipLaunchKernelGGL(init, dim3(1024), dim3(256), 0, (hipStream_t)stream, r, r_tiled, (const float *)nullptr, (void *)nullptr, 0, NH, dh);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(XS_ERR_LAUNCH, "tiling kernel launch failed: %s", hipGetErrorString(e));
  return XS_OK;
}

int xs_slstm_backward_tile_r(const xs_slstm_bwd_args *args) {
  g_err[0] = 0;
  return run_backward_tile_r(args);
}

int xs_causal_conv_silu(const xs_conv_args *args) {
  g_err[0] = 0;
  return run_conv(args);
}

int xs_causal_conv_silu_token(const xs_conv_args *args, void *x_out) {
  g_err[0] = 0;
  if (!x_out) return fail(XS_ERR_NULL, "x_out is required");
  return run_conv(args, x_out);
}

int xs_headwise_gates(const xs_gates_args *args) {
  g_err[0] = 0;
  return run_gates(args);
}

int xs_headwise_group_norm(const xs_norm_args *args) {
  g_err[0] = 0;
  return run_group_norm(args);
}

int xs_layer_front(const xs_layer_args *args) {
  g_err[0] = 0;
  return run_layer_front(args);
}

int xs_layer_norm(const xs_layer_args *args) {
  g_err[0] = 0;
  return run_layer_norm(args);
}

int xs_layer_step_fits(int32_t B, int32_t NH, int32_t dh, int32_t K) {
  return B > 0 && NH > 0 && dh > 0 && dh % 64 == 0 && layer_step_split(B, NH, dh, K).ut > 0;
}

int xs_layer_step(const xs_layer_step_args *args) {
  g_err[0] = 0;
  return run_layer_step(args);
}

size_t xs_layer_scratch_floats(int32_t B, int32_t T, int32_t NH, int32_t dh, int32_t K) {
  if (B <= 0 || T <= 0 || NH <= 0 || dh <= 0 || K <= 0) return 0;
  const LayerSplit s = layer_split(B, T, NH, dh, K);
  return s.gate_floats + s.conv_floats;
}

int xs_layer_front_backward(const xs_layer_args *args) {
  g_err[0] = 0;
  return run_layer_front_backward(args);
}

}  // extern "C"
