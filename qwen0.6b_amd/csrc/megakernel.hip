// Qwen3-0.6B batch-1 decode engine for MI355X (gfx950): one
// persistent kernel runs whole token steps (embedding, 28 layers, final norm,
// tied lm_head, argmax) and, in generate mode, feeds each argmax back as the
// next step's input without returning to the host.
//
// Design (from measurements on MI355X):
//  * one 512-thread workgroup per CU; workgroup w runs on XCD w % 8, and the
//    work partition (qwen_layout.h) keeps each kv head's QKV rows, attention
//    splits, softmax combine, o_proj and a 384-row slice of the MLP inside one
//    XCD. Per layer only two steps cross XCDs: the sums of the 8 per-XCD
//    o_proj and down partials into the residual stream (each workgroup reads
//    its 32 rows from the 8 XCDs);
//  * no grid barrier: every hand-off is an exchange buffer of 8-byte slots
//    carrying payload + step tag, written with device-scope stores and polled
//    with device-scope loads (one-way latency 0.3-0.5 us; a fence-based flag
//    costs 1-2 us more);
//  * waves 0-3 compute: each polls a quarter of a stage's input, the quarters
//    meet in LDS, and each wave computes a quarter of the stage's rows and
//    stores its own results. They hold no outstanding weight loads, so a poll
//    never waits behind a prefetch;
//  * waves 4-7 stream every stage's weights and K/V rows with LDS-DMA
//    (global_load_lds_dwordx4) into a 128 KB ring of 1 KB lines, up to 128
//    lines ahead of the compute waves; a compute wave reads its lines into
//    registers (and frees them) while it waits for its input, so only the
//    arithmetic follows the input's arrival. In the lm_head the loader waves
//    compute rows alongside the compute waves, and the last fifth of the
//    vocabulary is claimed at run time by groups of 8 workgroups (one per XCD);
//  * the residual stream stays fp32 inside the workgroup that owns its rows;
//    only the all-gathered copies are fp16;
//  * every wait is bounded by a wall-clock deadline; a missed deadline sets a
//    status word and all waves leave, so a broken exchange cannot hang the GPU.
//
// Reference behaviour followed: Tools/megakernel/megakernel.cu:763-920 (op
// order), 242-291 (QKV), 308-553 (q/k norm, RoPE, KV write, attention),
// 558-709 (o_proj, post-norm, SiLU*up, down), 893-919 (final norm),
// 1001-1144 (lm_head + argmax), 1150-1314 (launchers).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_ext.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include <type_traits>
#include <cstring>
#include <mutex>

#include "qwen_layout.h"
#include "qwen_megakernel.h"

using namespace ql;

typedef unsigned int u32;
typedef unsigned long long u64;
typedef u32 v4u __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

constexpr float RMS_EPS = 1e-6f;
constexpr u32 ST_TIMEOUT = 1u;
constexpr u32 ST_BAD_TOKEN = 2u;
// XCC id of the executing wave: s_getreg of hardware register 20 (XCC_ID), bits [3:0]
__device__ __forceinline__ u32 xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | 20); }
constexpr int DMA_DEPTH = 16;  // LDS-DMA lines a loader wave keeps in flight
// optional device timestamps (wall clock) per workgroup and stage of one token
constexpr int TRACE_EVENTS = 6;
enum TraceEvent : int {
  TR_POLL = 0,   // compute wave 0 starts waiting for the stage input
  TR_INPUT = 1,  // compute wave 0 has the stage input
  TR_SYNC = 2,   // attention: the wave's partial is in LDS (before the merge barrier);
                 // lm_head stage: compute wave 0 finished its lm_head rows
  TR_STORE = 3,  // compute wave 0 stored its results (and they were acknowledged)
  TR_LINES = 4,  // layer stages: compute wave 0 has the stage's ring lines;
                 // lm_head stage: compute wave 0 has the argmax partials of all workgroups
  TR_MERGE = 5,  // attention: compute wave 0 passed the barrier before the split merge;
                 // lm_head stage: loader wave 0 finished its lm_head rows
};
QL_HD int trace_stages(int L) { return NSTAGE * L + 1; }

struct KParams {
  const _Float16* embed;
  const LDGLayerWeight* layers;
  const _Float16* final_norm;
  const _Float16* lm_head;
  const _Float16* cos_t;
  const _Float16* sin_t;
  _Float16* k_cache;
  _Float16* v_cache;
  _Float16* hidden_out;    // [1024] fp16
  float* norm_out;         // [1024] fp32
  int* out_tokens;         // [num_steps]
  const int* forced;       // nullable [num_steps]
  float* logits_out;       // nullable [num_steps][VOCAB]
  float* hidden_steps;     // nullable [num_steps][HIDDEN]
  const _Float16* in_vec;  // MODE_LMHEAD / MODE_MLP input [1024]
  float* out_vec;          // MODE_MLP output [1024]
  u64* ws;                 // exchange slots
  u32* status;             // status word (device scope)
  u64 deadline;            // wall-clock ticks a single wait may take
  u64* trace;              // nullable [NWG][trace_stages(L)][TRACE_EVENTS]
  int trace_token;         // token index whose stages are traced
  int* out_count;          // nullable: steps run (the generation stops after eos)
  int eos;                 // stop after the first step whose argmax is this id (-1: never)
  int mode, num_layers, first_token, start_pos, num_steps, max_seq;
  float attn_scale;
  u32 epoch0;
  // the sampling build of the kernel: every next token is the argmax of logit / temperature +
  // Gumbel noise (seed, position) instead of the logit's (temperature sampling, on the device)
  float temperature;
  u64 seed;
  int sample;              // host side: launch the sampling build
  // the sampling builds with top_k >= 1: the token is drawn from the top-k (then top-p, when
  // top_p < 1) tokens of the step's logits instead of from all of them; top_k = VOCAB: top-p
  // alone. 1 <= top_k <= TOPK_MAX: the `sampled` build (draw_topk); larger: `dsampled`
  // (draw_dist); top_k = 0: `tsampled` (temperature alone)
  int top_k;
  float top_p;
  LDGLayerWeight own_layer;  // MODE_MLP: the block's weights
};
constexpr int TOPK_MAX = 128;  // largest top_k of the `sampled` build

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): 10 rounds of two 32x32 -> 64 multiplies
// with the published multipliers and key increments; returns the first output word
__device__ __forceinline__ u32 philox_x0(u32 c0, u32 c1, u32 c2, u32 c3, u32 k0, u32 k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const u64 p0 = (u64)0xD2511F53u * c0, p1 = (u64)0xCD9E8D57u * c2;
    const u32 n0 = (u32)(p1 >> 32) ^ c1 ^ k0, n2 = (u32)(p0 >> 32) ^ c3 ^ k1;
    c0 = n0;
    c1 = (u32)p1;
    c2 = n2;
    c3 = (u32)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c0;
}

// Gumbel(0, 1) noise of token j at `step` (the position of the step's input token) under `seed`:
// g = -log(-log(u)) with u = (top 23 bits of Philox of counter (j, step, 0, 0), key (seed low,
// seed high), + 0.5) / 2^23, every step exact in fp32, so u lies in [2^-24, 1 - 2^-24] (24 bits
// would round the largest value up to 1.0 and give g = +inf)
__device__ __forceinline__ float gumbel(u64 seed, u32 step, u32 j) {
  const u32 x = philox_x0(j, step, 0u, 0u, (u32)seed, (u32)(seed >> 32));
  const float u = ((float)(x >> 9) + 0.5f) * (1.0f / 8388608.0f);
  return -logf(-logf(u));
}

// order-preserving key: larger floats give larger keys; NaN gives 0 (below -inf)
__device__ __forceinline__ u32 fkey(float v) {
  if (v != v) return 0u;
  const u32 b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(u32 k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// unnormalised probability exp((l - M) / T) in units of 2^-40; 0 for NaN (M is the largest
// logit, so the value is at most 2^40 and a vocabulary's sum fits 64 bits)
__device__ __forceinline__ u64 mass(float l, float M, float T) {
  if (l != l) return 0;
  return (u64)(expf((l - M) / T) * 1099511627776.0f);
}

// (key << 32 | ~index): the larger of two is the larger key, then the lower index
__device__ __forceinline__ u64 pack_best(u32 key, int idx) { return ((u64)key << 32) | (u64)(0xffffffffu - (u32)idx); }
__device__ __forceinline__ int best_index(u64 b) { return (int)(0xffffffffu - (u32)b); }

// ------------------------------------------------------------------------------------
// device code: the production kernel, and a copy that records per-stage timestamps

namespace fast {
constexpr bool kTrace = false;
constexpr bool kSample = false;
constexpr bool kTopK = false;
constexpr bool kDist = false;
constexpr bool kMlp = false;
#include "decode_body.inc"
}  // namespace fast

namespace traced {
constexpr bool kTrace = true;
constexpr bool kSample = false;
constexpr bool kTopK = false;
constexpr bool kDist = false;
constexpr bool kMlp = false;
#include "decode_body.inc"
}  // namespace traced

namespace sampled {
constexpr bool kTrace = false;
constexpr bool kSample = true;
constexpr bool kTopK = true;
constexpr bool kDist = false;
constexpr bool kMlp = false;
#include "decode_body.inc"
}  // namespace sampled

// top_k > TOPK_MAX and top-p alone: the sampling build whose draw splits the selections over
// every workgroup's slice when the published entries cannot decide them (draw_dist)
namespace dsampled {
constexpr bool kTrace = false;
constexpr bool kSample = true;
constexpr bool kTopK = true;
constexpr bool kDist = true;
constexpr bool kMlp = false;
#include "decode_body.inc"
}  // namespace dsampled

// temperature alone: the sampling build without the top-k draw, whose code would otherwise
// share (and reshape) this kernel's register allocation
namespace tsampled {
constexpr bool kTrace = false;
constexpr bool kSample = true;
constexpr bool kTopK = false;
constexpr bool kDist = false;
constexpr bool kMlp = false;
#include "decode_body.inc"
}  // namespace tsampled

// the isolated MLP block alone, with the one layer's pointers in the arguments (a table in memory took a
// copy that the host waited for, or a kernel of its own: 15.9 -> 11.1 us per call; the same choice at run
// time in the greedy build made its tokens 1% slower, by its scalar registers)
namespace isolated {
constexpr bool kTrace = false;
constexpr bool kSample = false;
constexpr bool kTopK = false;
constexpr bool kDist = false;
constexpr bool kMlp = true;
#include "decode_body.inc"
}  // namespace isolated

// the batched prefill kernel (namespace pf)
#include "prefill_body.inc"

// the token sampler (namespace smp)
#include "sample_body.inc"

// one workgroup per CU, as the decode kernel: each records the XCC it runs on
__global__ void __launch_bounds__(BLOCK, 1) qwen_placement_probe(u32* out) {
  if (threadIdx.x == 0) out[blockIdx.x] = xcc_id();
}

// the prefill kernel's geometry (two 256-thread workgroups per CU): each records its XCC
__global__ void __launch_bounds__(pf::NT, pf::WG_PER_CU) qwen_placement_probe_pf(u32* out) {
  if (threadIdx.x == 0) out[blockIdx.x] = xcc_id();
}

// zeroes n 8-byte words (a kernel, not hipMemsetAsync: callers may capture the stream)
__global__ void qwen_zero_words(u64* p, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0;
}

// Exchange workspace of qwen_generate_nosync_noalloc: the same layout as the workspace the
// other entry points allocate (slots, status line, lm_head pool counters), as module memory,
// one copy per device. Host code never uses this name as an address: it uses the pointer
// hipGetSymbolAddress returns for the current device (DeviceState::fixed).
static_assert(WORKSPACE_BYTES % 256 == 0, "whole 256-byte lines");
static __device__ __align__(256) unsigned char scratch[WORKSPACE_BYTES];

// ------------------------------------------------------------------------------------
// host side

namespace {

constexpr int MAX_DEVICES = 16;
constexpr u64 DEFAULT_WAIT_US = 500000;

// one exchange workspace (WORKSPACE_BYTES) and the token epoch its tags continue from
struct Workspace {
  u64* ws = nullptr;
  u32* status = nullptr;
  u32 epoch = 1;
};

struct DeviceState {
  bool init = false;
  int err = QWEN_OK;
  Workspace heap;                 // hipMalloc'd on first use by the allocating entry points
  Workspace fixed;                // the `scratch` array of this device (no allocation)
  char* pf = nullptr;             // prefill activations (PF_BYTES), on first use
  char* smp = nullptr;            // the sampler's work area (SMP_BYTES), allocated on first use
  u32 smp_parity = 0;             // sampler launches so far (selects the work area copy)
  hipEvent_t order = nullptr;     // end of the last launch (see launch_resident)
  u64 clk_khz = 100000;
  u64 deadline = 0;
  u64* trace = nullptr;
  long long trace_elems = 0;
  int trace_token = -1;
};

std::mutex g_mu;
DeviceState g_dev[MAX_DEVICES];
// What the library allocates (workspaces, the prefill and sampler buffers) is held until the process ends and released with it; no exit handler
// calls into the HIP runtime.

int zero_words(void* p, long bytes, hipStream_t s) {
  hipLaunchKernelGGL(qwen_zero_words, dim3(NWG), dim3(256), 0, s, (u64*)p, bytes / 8);
  return hipGetLastError() == hipSuccess ? QWEN_OK : QWEN_ERR_LAUNCH;
}

// The prefill builds: one-workgroup-per-CU kernels with tiles for at most 16, 64, .. 1024 positions, then
// the two-workgroups-per-CU kernel for longer prompts. The last line lies where 128-position tiles stop
// giving one tile per CU (1025 positions are 288 QKV tiles for 256 workgroups): at 999 positions the
// short build takes 2.41 ms against 2.86, at 1919 a one-workgroup-per-CU build 3.83 against 3.72.
constexpr int PF_CLASS_MAX[] = {16, 64, 128, 256, 512, 1024};
constexpr int PF_CLASSES = sizeof(PF_CLASS_MAX) / sizeof(int);
static_assert(PF_CLASS_MAX[PF_CLASSES - 1] == PF_MID_MAX, "class limits");
int prefill_class(int n) {
  int k = 0;
  while (k < PF_CLASSES && n > PF_CLASS_MAX[k]) ++k;
  return k;
}

// Every kernel whose workgroups wait for each other, with the grid it is launched with: one round of the
// chip's CUs, which all of it must fit at once (device_state checks each; nothing else is launched by
// launch_resident).
struct Build {
  const void* kernel;
  int grid, threads;
};
enum BuildId : int { DEC_GREEDY, DEC_TRACED, DEC_TOPK, DEC_DIST, DEC_TEMP, DEC_MLP, SAMPLER, PREFILL };  // + prefill_class
const Build BUILDS[] = {
    {(const void*)fast::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)traced::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)sampled::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)dsampled::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)tsampled::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)isolated::qwen_decode_kernel, NWG, BLOCK},
    {(const void*)smp::qwen_sample_kernel, smp::NB, smp::NT},
    {(const void*)pf::qwen_prefill_mid_kernel<16>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_mid_kernel<64>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_mid_kernel<128>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_mid_kernel<256>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_mid_kernel<512>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_mid_kernel<1024>, NWG, pf::MNT},
    {(const void*)pf::qwen_prefill_kernel, pf::NWG_PF, pf::NT},
};
static_assert(sizeof(BUILDS) / sizeof(Build) == PREFILL + PF_CLASSES + 1, "a build per prefill class, then the long one");

// The engine's kernels wait for their own workgroups, so all of a launch's must be resident at once:
// its grid is one round of the chip (one or two workgroups per CU, checked against the occupancy), and
// no two of these launches may share the chip, nor the device's workspaces. Each launch therefore
// follows the one before it, on whatever stream: `order` is the event of the last one's end, set by
// the launch itself (hipExtLaunchKernel), and every call's stream waits for it before its first
// operation. The runtime's cooperative launch gives the same guarantee by passing through a queue of
// its own, 18-20 us per call (a sampler launch with nothing to select 27 -> 7 us, the lm_head 78 ->
// 63); an event recorded after a plain launch costs 3 us more than one that belongs to it.
// A captured call puts the same wait and the same record into the graph, as event nodes, so that each
// replay waits for the launch before it and later ones wait for the replay: the order is that of the
// host's calls, hipGraphLaunch among them, which the program makes one after the other. (Its launch stays
// a cooperative one: grids of replays that threads launch at once, out of any order, do not meet.)

// Whether the stream is being captured. Where the runtime cannot say (or the capture has failed) nothing
// may be sent to the stream: a launch taken for a captured one would be in no order.
int capture_state(hipStream_t stream, bool* captured) {
  hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &c) != hipSuccess || c == hipStreamCaptureStatusInvalidated) return QWEN_ERR_LAUNCH;
  *captured = c == hipStreamCaptureStatusActive;
  return QWEN_OK;
}
// adds a node to the stream's capture that waits for the event, or records it, at every replay
int capture_event(hipStream_t stream, hipEvent_t event, bool record) {
  hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  hipGraph_t graph = nullptr;
  const hipGraphNode_t* last = nullptr;
  size_t n = 0;
  if (hipStreamGetCaptureInfo_v2(stream, &c, &id, &graph, &last, &n) != hipSuccess || c != hipStreamCaptureStatusActive)
    return QWEN_ERR_LAUNCH;
  hipGraphNode_t node = nullptr;
  const hipError_t e = record ? hipGraphAddEventRecordNode(&node, graph, last, n, event)
                              : hipGraphAddEventWaitNode(&node, graph, last, n, event);
  return e == hipSuccess &&
                 hipStreamUpdateCaptureDependencies(stream, &node, 1, hipStreamSetCaptureDependencies) == hipSuccess
             ? QWEN_OK
             : QWEN_ERR_LAUNCH;
}
// makes the stream wait for the device's last launch; caller holds g_mu
int order_after(DeviceState* st, hipStream_t stream, bool captured) {
  if (captured) return capture_event(stream, st->order, /*record=*/false);
  return hipStreamWaitEvent(stream, st->order, 0) == hipSuccess ? QWEN_OK : QWEN_ERR_LAUNCH;
}
// false for a stream whose queue is restricted to some of the CUs (hipExtStreamCreateWithCUMask): a grid
// that needs all of them never gets resident there. The cooperative queue, which such a stream's
// launches then pass through, is not restricted (the question costs 0.2 us per call).
bool whole_chip(hipStream_t stream) {
  u32 mask[NWG / 32] = {};
  if (hipExtStreamGetCUMask(stream, NWG / 32, mask) != hipSuccess) return false;
  for (u32 m : mask)
    if (m != 0xffffffffu) return false;
  return true;
}
// launches one of BUILDS; caller holds g_mu, and the stream has waited for the last launch (order_after)
int launch_resident(DeviceState* st, int build, void** args, hipStream_t stream, bool captured) {
  const Build& b = BUILDS[build];
  if (captured || !whole_chip(stream)) {
    if (hipLaunchCooperativeKernel(b.kernel, dim3(b.grid), dim3(b.threads), args, 0, stream) != hipSuccess)
      return QWEN_ERR_LAUNCH;
    if (captured) return capture_event(stream, st->order, /*record=*/true);
    return hipEventRecord(st->order, stream) == hipSuccess ? QWEN_OK : QWEN_ERR_LAUNCH;
  }
  return hipExtLaunchKernel(b.kernel, dim3(b.grid), dim3(b.threads), args, 0, stream, nullptr, st->order, 0) == hipSuccess
             ? QWEN_OK
             : QWEN_ERR_LAUNCH;
}

// The workgroups w of the decode launch (256 x 512) and of the prefill launches with equal w % 8 must
// run on one XCD: the decode's work partition and XCD-local exchange stores, and the prefill's per-XCD
// barrier (one L2 write-back and invalidate per XCD) rely on it ("XCD w % 8" in their comments: which
// of the chip's XCDs that is does not matter). The dispatcher deals workgroups out in turn, from an XCD
// that differs from queue to queue and changes when a queue is mapped anew (2400 launches of both
// geometries, cooperative and plain, between other kernels: always w -> (w + r) % 8, r = 0, 6 or 7).
// Checked once per device and geometry with a probe launch that writes into `buf` (n words).
int check_placement(const void* probe, int n, int threads, u32* buf, hipStream_t s) {
  void* args[] = {&buf};
  if (hipLaunchCooperativeKernel(probe, dim3(n), dim3(threads), args, 0, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return QWEN_ERR_LAUNCH;
  static u32 xcc[2 * NWG];
  if (n > 2 * NWG || hipMemcpy(xcc, buf, sizeof(u32) * n, hipMemcpyDeviceToHost) != hipSuccess)
    return QWEN_ERR_LAUNCH;
  for (int w = 0; w < n; ++w)
    if ((xcc[w] & 15) != ((xcc[0] & 15) + xcd_of(w)) % NXCD) {
      fprintf(stderr, "qwen_megakernel: workgroup %d of %d runs on XCC %u, workgroup 0 on %u: not one XCD per w %% 8\n", w, n,
              xcc[w] & 15, xcc[0] & 15);
      return QWEN_ERR_DEVICE;
    }
  return QWEN_OK;
}

// Device checks and the fixed workspace, once per device; allocates nothing. (Caller holds g_mu.)
int device_state(DeviceState** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return QWEN_ERR_DEVICE;
  DeviceState& st = g_dev[dev];
  if (!st.init) {
    st.init = true;
    st.err = QWEN_ERR_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return st.err;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0 || prop.multiProcessorCount != NWG || !prop.cooperativeLaunch) {
      fprintf(stderr, "qwen_megakernel: needs a 256-CU gfx950 device with cooperative launch (got %s, %d CUs)\n",
              prop.gcnArchName, prop.multiProcessorCount);
      return st.err;
    }
    for (const Build& b : BUILDS) {
      int occ = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, b.kernel, b.threads, 0) != hipSuccess || occ * NWG < b.grid)
        return st.err;
    }
    int clk_khz = 0;
    if (hipDeviceGetAttribute(&clk_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || clk_khz <= 0)
      clk_khz = 100000;
    st.clk_khz = (u64)clk_khz;
    st.deadline = st.clk_khz * DEFAULT_WAIT_US / 1000;  // 0.5 s per single wait
    // this device's copy of `scratch`: its address, never the host-side name
    void* fixed = nullptr;
    if (hipGetSymbolAddress(&fixed, HIP_SYMBOL(scratch)) != hipSuccess || fixed == nullptr) {
      st.err = QWEN_ERR_LAUNCH;
      return st.err;
    }
    st.err = check_placement((const void*)qwen_placement_probe, NWG, BLOCK, (u32*)fixed, nullptr);
    if (st.err != QWEN_OK) return st.err;
    if (zero_words(fixed, WORKSPACE_BYTES, nullptr) != QWEN_OK ||
        hipEventCreateWithFlags(&st.order, hipEventDisableTiming) != hipSuccess ||
        hipEventRecord(st.order, nullptr) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
      st.err = QWEN_ERR_LAUNCH;
      return st.err;
    }
    st.fixed.ws = (u64*)fixed;
    st.fixed.status = (u32*)((char*)fixed + TOTAL_SLOTS * 8);
    st.err = QWEN_OK;
  }
  if (st.err != QWEN_OK) return st.err;
  *out = &st;
  return QWEN_OK;
}

// The allocating entry points' workspace, on first use. (Caller holds g_mu.)
int heap_workspace(DeviceState* st) {
  if (st->heap.ws) return QWEN_OK;
  void* p = nullptr;
  if (hipMalloc(&p, WORKSPACE_BYTES) != hipSuccess) return QWEN_ERR_LAUNCH;
  if (hipMemset(p, 0, WORKSPACE_BYTES) != hipSuccess) {
    (void)hipFree(p);
    return QWEN_ERR_LAUNCH;
  }
  st->heap.ws = (u64*)p;
  st->heap.status = (u32*)((char*)p + TOTAL_SLOTS * 8);
  return QWEN_OK;
}

// launches the decode kernel on the heap workspace, or (fixed = true) on the device's
// `scratch` array, in which case nothing is allocated
int launch(KParams& P, hipStream_t stream, bool fixed = false) {
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK) return rc;
  if (!fixed && (rc = heap_workspace(st)) != QWEN_OK) return rc;
  Workspace& w = fixed ? st->fixed : st->heap;
  // a trace buffer must hold every stage of every workgroup of this launch's layers
  if (st->trace && (long long)NWG * trace_stages(P.num_layers) * TRACE_EVENTS > st->trace_elems) return QWEN_ERR_ARG;
  // the traced build is the greedy kernel: a sampled launch while tracing would return argmax ids
  if (st->trace && P.sample) return QWEN_ERR_ARG;
  bool captured = false;
  if ((rc = capture_state(stream, &captured)) != QWEN_OK) return rc;
  if (P.mode == MODE_MLP && captured) return QWEN_ERR_LAUNCH;  // (the MLP block never was capturable)
  if ((rc = order_after(st, stream, captured)) != QWEN_OK) return rc;
  P.ws = w.ws;
  P.status = w.status;
  P.deadline = st->deadline;
  P.trace = st->trace;
  P.trace_token = st->trace_token;
  P.epoch0 = w.epoch;
  // epochs are 24-bit in the tag; wrap back to 1 (never 0: a zeroed slot is never "ready")
  u64 next = (u64)w.epoch + (u64)P.num_steps + 1;
  if (next >= (1u << 24)) {
    if (zero_words(w.ws, TOTAL_SLOTS * 8, stream) != QWEN_OK) return QWEN_ERR_LAUNCH;
    P.epoch0 = 1;
    next = 1 + (u64)P.num_steps + 1;
  }
  w.epoch = (u32)next;
  void* args[] = {&P};
  const int build = P.trace              ? DEC_TRACED
                    : P.mode == MODE_MLP ? DEC_MLP
                    : P.sample           ? (P.top_k > TOPK_MAX ? DEC_DIST : P.top_k > 0 ? DEC_TOPK : DEC_TEMP)
                                         : DEC_GREEDY;
  return launch_resident(st, build, args, stream, captured);
}

// prefill activations for up to MAX_SEQ_LIMIT positions: residual X fp32 [n, 1024], q and the
// attention output fp16 [n, 2048] each, SiLU * up fp16 [n, 3072], the next RMSNorm's gained input
// fp16 [n, 1024] and its block sums of squares fp32 [n, 64], then the barrier counters and
// the split attention items' arrival counters (zeroed before every launch), the timestamps and
// the split items' partial results
constexpr long PF_X = 0;
constexpr long PF_Q = PF_X + (long)MAX_SEQ_LIMIT * HIDDEN * 4;
constexpr long PF_AO = PF_Q + (long)MAX_SEQ_LIMIT * QSZ * 2;
constexpr long PF_IM = PF_AO + (long)MAX_SEQ_LIMIT * QSZ * 2;
constexpr long PF_XN = PF_IM + (long)MAX_SEQ_LIMIT * INTER * 2;
constexpr long PF_SSQ = PF_XN + (long)MAX_SEQ_LIMIT * HIDDEN * 2;
constexpr long PF_BAR = PF_SSQ + (long)MAX_SEQ_LIMIT * pf::SSB * 4;
constexpr int PF_NTS = 1 + 1 + 5 * MAX_LAYERS;  // launch start, then every grid barrier
constexpr long PF_BAR_LINES = 4096;              // barrier words: 8 XCDs x 64 arrivals, 8 copies of 8 leaders
constexpr long PF_ACNT = PF_BAR + PF_BAR_LINES;
constexpr long PF_BAR_BYTES = PF_BAR_LINES + 4L * pf::MAX_QB * NKV;
constexpr long PF_TS = PF_BAR + PF_BAR_BYTES;
constexpr long PF_PART = (PF_TS + 8L * ((PF_NTS + 31) / 32 * 32) + 255) / 256 * 256;
constexpr long PF_BYTES = PF_PART + 4L * pf::MAX_PSLOTS * NKV * pf::PART_FLOATS;
static_assert(PF_BAR_BYTES % 4 == 0 && PF_PART % 256 == 0, "prefill workspace alignment");
static_assert(4L * (64 + 32) * NXCD <= PF_BAR_LINES, "the barrier words fit their lines");

// sampler buffer: the sampler's work area (two copies, chosen by launch parity)
constexpr long SMP_WORK = 0;
constexpr long SMP_BYTES = (smp::WORK_BYTES + 255) / 256 * 256;

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// temperature, top_k and top_p as the sampler reads them (NaN refused)
bool sample_args_ok(float temperature, int top_k, float top_p) {
  return temperature == temperature && top_k >= 0 && top_p == top_p;
}

// the decode kernel's top_k for a draw with these arguments (checked by sample_args_ok):
// temperature <= 0 is the argmax (1); no top-k (0 or >= VOCAB) is VOCAB with top_p < 1 (top-p
// alone) and 0 without (temperature alone)
int device_top_k(float temperature, int top_k, float top_p) {
  if (!(temperature > 0.f)) return 1;
  if (top_k == 0 || top_k >= VOCAB) return top_p < 1.f ? VOCAB : 0;
  return top_k;
}

// the device's sampler buffer (allocated and cleared on first use); caller holds g_mu
int sampler_buffer(DeviceState* st, hipStream_t stream) {
  if (st->smp) return QWEN_OK;
  int rc = heap_workspace(st);  // the status word the sampler reports to
  if (rc != QWEN_OK) return rc;
  void* p = nullptr;
  if (hipMalloc(&p, SMP_BYTES) != hipSuccess) return QWEN_ERR_LAUNCH;
  if (zero_words(p, SMP_BYTES, stream) != QWEN_OK) {
    (void)hipFree(p);
    return QWEN_ERR_LAUNCH;
  }
  st->smp = (char*)p;
  return QWEN_OK;
}

// one sampler launch on the device's work area; caller holds g_mu
int launch_sampler(DeviceState* st, smp::SParams& S, hipStream_t stream) {
  bool captured = false;
  int rc = capture_state(stream, &captured);
  if (rc != QWEN_OK || (rc = order_after(st, stream, captured)) != QWEN_OK) return rc;
  S.work = (u64*)(st->smp + SMP_WORK);
  S.parity = st->smp_parity++;
  S.status = st->heap.status;
  S.deadline = st->deadline;
  void* args[] = {&S};
  return launch_resident(st, SAMPLER, args, stream, captured);
}

int fill_decode(KParams& P, const void* embed, const LDGLayerWeight* lw, const void* fnorm, const void* lm_head,
                const void* cos_t, const void* sin_t, void* kc, void* vc, void* hidden, void* norm_out,
                int num_layers, int start, int steps, int max_seq, float scale) {
  if (!embed || !lw || !fnorm || !lm_head || !cos_t || !sin_t || !kc || !vc || !hidden || !norm_out) return QWEN_ERR_ARG;
  if (!aligned16(lw) || !aligned16(embed) || !aligned16(lm_head) || !aligned16(kc) || !aligned16(vc) ||
      !aligned16(cos_t) || !aligned16(sin_t) || !aligned16(hidden) || !aligned16(norm_out) || !aligned16(fnorm))
    return QWEN_ERR_ARG;
  // max_seq must keep every ring line of 4 positions inside the cache
  if (num_layers < 1 || num_layers > MAX_LAYERS || steps < 1 || start < 0 || max_seq < 4 || (max_seq & 3) != 0 ||
      (long)start + steps > (long)max_seq || max_seq > MAX_SEQ_LIMIT)
    return QWEN_ERR_ARG;
  memset(&P, 0, sizeof(P));
  P.eos = -1;
  P.embed = (const _Float16*)embed;
  P.layers = lw;
  P.final_norm = (const _Float16*)fnorm;
  P.lm_head = (const _Float16*)lm_head;
  P.cos_t = (const _Float16*)cos_t;
  P.sin_t = (const _Float16*)sin_t;
  P.k_cache = (_Float16*)kc;
  P.v_cache = (_Float16*)vc;
  P.hidden_out = (_Float16*)hidden;
  P.norm_out = (float*)norm_out;
  P.mode = MODE_DECODE;
  P.num_layers = num_layers;
  P.start_pos = start;
  P.num_steps = steps;
  P.max_seq = max_seq;
  P.attn_scale = scale;
  return QWEN_OK;
}

}  // namespace

extern "C" int launch_ldg_decode_direct(int input_token_id, int* output_token_id, const void* embed_weight,
                                        const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                        const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                        void* k_cache, void* v_cache, void* hidden_buffer, void*, void*, void*,
                                        void*, void*, void*, void*, void* g_normalized, void*, void*,
                                        int num_layers, int position, int max_seq_len, float attn_scale,
                                        hipStream_t stream) {
  KParams P;
  int rc = fill_decode(P, embed_weight, layer_weights, final_norm_weight, lm_head_weight, cos_table, sin_table,
                       k_cache, v_cache, hidden_buffer, g_normalized, num_layers, position, 1, max_seq_len,
                       attn_scale);
  if (rc != QWEN_OK) return rc;
  if (!output_token_id || input_token_id < 0 || input_token_id >= VOCAB) return QWEN_ERR_ARG;
  P.first_token = input_token_id;
  P.out_tokens = output_token_id;
  return launch(P, stream);
}

extern "C" int launch_ldg_decode_persistent(int input_token_id, int* output_token_id, const void* embed_weight,
                                            const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                            const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                            void* k_cache, void* v_cache, void* hidden_buffer, void* a, void* b,
                                            void* c, void* d, void* e, void* f, void* g, void* g_normalized, void* h,
                                            void* i, int num_layers, int position, int cache_len, int max_seq_len,
                                            float attn_scale, hipStream_t stream) {
  (void)cache_len;  // unused by the reference too: its kernel reads the position (megakernel.cu:1211-1230)
  return launch_ldg_decode_direct(input_token_id, output_token_id, embed_weight, layer_weights, final_norm_weight,
                                  lm_head_weight, cos_table, sin_table, k_cache, v_cache, hidden_buffer, a, b, c, d,
                                  e, f, g, g_normalized, h, i, num_layers, position, max_seq_len, attn_scale, stream);
}

extern "C" int qwen_generate_ex(int first_token_id, int num_steps, const int* forced_tokens, const void* embed_weight,
                                const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                void* k_cache, void* v_cache, void* hidden_buffer, void* g_normalized,
                                int* output_log, float* logits_out, float* hidden_steps, int num_layers,
                                int start_position, int max_seq_len, float attn_scale, hipStream_t stream) {
  KParams P;
  int rc = fill_decode(P, embed_weight, layer_weights, final_norm_weight, lm_head_weight, cos_table, sin_table,
                       k_cache, v_cache, hidden_buffer, g_normalized, num_layers, start_position, num_steps,
                       max_seq_len, attn_scale);
  if (rc != QWEN_OK) return rc;
  if (!output_log || first_token_id < 0 || first_token_id >= VOCAB) return QWEN_ERR_ARG;
  if ((logits_out && !aligned16(logits_out)) || (hidden_steps && !aligned16(hidden_steps))) return QWEN_ERR_ARG;
  P.first_token = first_token_id;
  P.out_tokens = output_log;
  P.forced = forced_tokens;
  P.logits_out = logits_out;
  P.hidden_steps = hidden_steps;
  return launch(P, stream);
}

extern "C" int qwen_generate_until(int first_token_id, int num_steps, int eos_token_id, const void* embed_weight,
                                   const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                   const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                   void* k_cache, void* v_cache, void* hidden_buffer, void* g_normalized,
                                   int* output_log, int* out_count, int num_layers, int start_position,
                                   int max_seq_len, float attn_scale, hipStream_t stream) {
  KParams P;
  int rc = fill_decode(P, embed_weight, layer_weights, final_norm_weight, lm_head_weight, cos_table, sin_table,
                       k_cache, v_cache, hidden_buffer, g_normalized, num_layers, start_position, num_steps,
                       max_seq_len, attn_scale);
  if (rc != QWEN_OK) return rc;
  if (!output_log || !out_count || first_token_id < 0 || first_token_id >= VOCAB || eos_token_id < 0 ||
      eos_token_id >= VOCAB)
    return QWEN_ERR_ARG;
  P.first_token = first_token_id;
  P.out_tokens = output_log;
  P.out_count = out_count;
  P.eos = eos_token_id;
  return launch(P, stream);
}

extern "C" int launch_ldg_generate_nosync(int first_token_id, int num_steps, const void* embed_weight,
                                          const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                          const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                          void* k_cache, void* v_cache, void* hidden_buffer, void*, void*, void*,
                                          void*, void*, void*, void*, void* g_normalized, void*, void*,
                                          int* output_log, int num_layers, int start_position, int max_seq_len,
                                          float attn_scale, hipStream_t stream) {
  return qwen_generate_ex(first_token_id, num_steps, nullptr, embed_weight, layer_weights, final_norm_weight,
                          lm_head_weight, cos_table, sin_table, k_cache, v_cache, hidden_buffer, g_normalized,
                          output_log, nullptr, nullptr, num_layers, start_position, max_seq_len, attn_scale, stream);
}

// launch_ldg_generate_nosync on the device's fixed `scratch` workspace: no allocation in this
// call or in its first-use set-up on a device. The workspace need does not depend on the
// arguments; their limits are those of launch_ldg_generate_nosync (QWEN_ERR_ARG beyond them,
// and on a stream that is being captured).
extern "C" int qwen_generate_nosync_noalloc(int first_token_id, int num_steps, const void* embed_weight,
                                            const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                            const void* lm_head_weight, const void* cos_table,
                                            const void* sin_table, void* k_cache, void* v_cache,
                                            void* hidden_buffer, void*, void*, void*, void*, void*, void*, void*,
                                            void* g_normalized, void*, void*, int* output_log, int num_layers,
                                            int start_position, int max_seq_len, float attn_scale,
                                            hipStream_t stream) {
  KParams P;
  int rc = fill_decode(P, embed_weight, layer_weights, final_norm_weight, lm_head_weight, cos_table, sin_table,
                       k_cache, v_cache, hidden_buffer, g_normalized, num_layers, start_position, num_steps,
                       max_seq_len, attn_scale);
  if (rc != QWEN_OK) return rc;
  if (!output_log || first_token_id < 0 || first_token_id >= VOCAB) return QWEN_ERR_ARG;
  // Not for stream capture: the tags' token epochs are kernel arguments, so a replayed graph
  // would reuse them against slots that already carry them, and a device's first call
  // synchronises with the host (placement probe).
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return QWEN_ERR_ARG;
  P.first_token = first_token_id;
  P.out_tokens = output_log;
  return launch(P, stream, /*fixed=*/true);
}

extern "C" int qwen_prefill(const int* ids, int n, const void* embed_weight, const LDGLayerWeight* layer_weights,
                            const void* cos_table, const void* sin_table, void* k_cache, void* v_cache,
                            void* hidden_buffer, int num_layers, int start_position, int max_seq_len,
                            float attn_scale, hipStream_t stream) {
  if (!ids || !embed_weight || !layer_weights || !cos_table || !sin_table || !k_cache || !v_cache || !hidden_buffer)
    return QWEN_ERR_ARG;
  if (!aligned16(embed_weight) || !aligned16(layer_weights) || !aligned16(cos_table) || !aligned16(sin_table) ||
      !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(hidden_buffer))
    return QWEN_ERR_ARG;
  if (n < 1 || num_layers < 1 || num_layers > MAX_LAYERS || start_position < 0 || max_seq_len < 4 ||
      (max_seq_len & 3) != 0 || max_seq_len > MAX_SEQ_LIMIT || (long)start_position + n > (long)max_seq_len)
    return QWEN_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK) return rc;
  if ((rc = heap_workspace(st)) != QWEN_OK) return rc;
  if (!st->pf) {
    void* p = nullptr;
    if (hipMalloc(&p, PF_BYTES) != hipSuccess) return QWEN_ERR_LAUNCH;
    if ((rc = check_placement((const void*)qwen_placement_probe_pf, pf::NWG_PF, pf::NT, (u32*)p, stream)) != QWEN_OK) {
      (void)hipFree(p);
      return rc;
    }
    st->pf = (char*)p;
  }
  pf::PParams P;
  memset(&P, 0, sizeof(P));
  P.ids = ids;
  P.embed = (const _Float16*)embed_weight;
  P.layers = layer_weights;
  P.cos_t = (const _Float16*)cos_table;
  P.sin_t = (const _Float16*)sin_table;
  P.kc = (_Float16*)k_cache;
  P.vc = (_Float16*)v_cache;
  P.hidden_out = (_Float16*)hidden_buffer;
  P.X = (float*)(st->pf + PF_X);
  P.Q = (_Float16*)(st->pf + PF_Q);
  P.AO = (_Float16*)(st->pf + PF_AO);
  P.IM = (_Float16*)(st->pf + PF_IM);
  P.XN = (_Float16*)(st->pf + PF_XN);
  P.SSQ = (float*)(st->pf + PF_SSQ);
  P.bar = (u32*)(st->pf + PF_BAR);
  P.acnt = (u32*)(st->pf + PF_ACNT);
  P.ts = (u64*)(st->pf + PF_TS);
  P.part = (float*)(st->pf + PF_PART);
  P.status = st->heap.status;
  P.deadline = st->deadline;
  P.n = n;
  P.start = start_position;
  P.num_layers = num_layers;
  P.max_seq = max_seq_len;
  P.attn_scale = attn_scale;
  const int cls = prefill_class(n);
  if (!pf_plan(n, start_position, P.plan)) return QWEN_ERR_ARG;
  bool captured = false;
  if ((rc = capture_state(stream, &captured)) != QWEN_OK || (rc = order_after(st, stream, captured)) != QWEN_OK) return rc;
  if (zero_words(P.bar, PF_BAR_BYTES, stream) != QWEN_OK) return QWEN_ERR_LAUNCH;
  void* args[] = {&P};
  return launch_resident(st, PREFILL + cls, args, stream, captured);
}

extern "C" int qwen_prefill_timestamps(unsigned long long* out, int max_entries) {
  if (!out || max_entries < 1) return QWEN_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK) return rc;
  const int n = max_entries < PF_NTS ? max_entries : PF_NTS;
  if (!st->pf) {
    memset(out, 0, sizeof(unsigned long long) * n);
    return QWEN_OK;
  }
  if (hipDeviceSynchronize() != hipSuccess) return QWEN_ERR_LAUNCH;
  if (hipMemcpy(out, st->pf + PF_TS, sizeof(unsigned long long) * n, hipMemcpyDeviceToHost) != hipSuccess)
    return QWEN_ERR_LAUNCH;
  return QWEN_OK;
}

extern "C" int qwen_sample(const float* logits, int n, float temperature, int top_k, float top_p,
                           unsigned long long seed, unsigned int step, int* out_token, hipStream_t stream) {
  if (!logits || !out_token || n < 1 || n > smp::MAX_N || !sample_args_ok(temperature, top_k, top_p))
    return QWEN_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK || (rc = sampler_buffer(st, stream)) != QWEN_OK) return rc;
  smp::SParams S;
  memset(&S, 0, sizeof(S));
  S.logits = logits;
  S.n = n;
  S.temperature = temperature;
  S.top_k = top_k;
  S.top_p = top_p;
  S.seed = seed;
  S.step = step;
  S.out_token = out_token;
  return launch_sampler(st, S, stream);
}

extern "C" int qwen_generate_sampled(int first_token_id, int num_steps, int eos_token_id, const void* embed_weight,
                                     const LDGLayerWeight* layer_weights, const void* final_norm_weight,
                                     const void* lm_head_weight, const void* cos_table, const void* sin_table,
                                     void* k_cache, void* v_cache, void* hidden_buffer, void* g_normalized,
                                     int* output_log, int* out_count, int num_layers, int start_position,
                                     int max_seq_len, float attn_scale, float temperature, int top_k, float top_p,
                                     unsigned long long seed, hipStream_t stream) {
  KParams P;
  // the whole range is checked before anything is launched
  int rc = fill_decode(P, embed_weight, layer_weights, final_norm_weight, lm_head_weight, cos_table, sin_table,
                       k_cache, v_cache, hidden_buffer, g_normalized, num_layers, start_position, num_steps,
                       max_seq_len, attn_scale);
  if (rc != QWEN_OK) return rc;
  if (!output_log || first_token_id < 0 || first_token_id >= VOCAB || eos_token_id < -1 || eos_token_id >= VOCAB ||
      !sample_args_ok(temperature, top_k, top_p))
    return QWEN_ERR_ARG;
  // one launch of num_steps steps, every token drawn inside the decode kernel (eos checked on the
  // device as in qwen_generate_until): temperature <= 0 is the argmax (top_k 1); temperature
  // alone runs the `tsampled` build, top-k (then top-p) and top-p alone the `sampled` /
  // `dsampled` builds
  P.first_token = first_token_id;
  P.out_tokens = output_log;
  P.out_count = out_count;
  P.eos = eos_token_id;
  P.temperature = temperature;
  P.seed = seed;
  P.sample = 1;
  P.top_k = device_top_k(temperature, top_k, top_p);
  P.top_p = top_p;
  return launch(P, stream);
}

extern "C" int qwen_lm_head_argmax(const void* hidden_f16, const void* weight, int* out_token, float* logits_out,
                                   hipStream_t stream) {
  if (!hidden_f16 || !weight || !out_token || !aligned16(hidden_f16) || !aligned16(weight)) return QWEN_ERR_ARG;
  if (logits_out && !aligned16(logits_out)) return QWEN_ERR_ARG;
  KParams P;
  memset(&P, 0, sizeof(P));
  P.eos = -1;
  P.lm_head = (const _Float16*)weight;
  P.in_vec = (const _Float16*)hidden_f16;
  P.out_tokens = out_token;
  P.logits_out = logits_out;
  P.mode = MODE_LMHEAD;
  P.num_layers = 1;
  P.num_steps = 1;
  P.max_seq = MAX_SEQ_LIMIT;
  return launch(P, stream);
}

extern "C" int qwen_lm_head_sample(const void* hidden_f16, const void* weight, float temperature, int top_k,
                                   float top_p, unsigned long long seed, int position, int* out_token,
                                   float* logits_out, hipStream_t stream) {
  if (!hidden_f16 || !weight || !out_token || !aligned16(hidden_f16) || !aligned16(weight)) return QWEN_ERR_ARG;
  if (logits_out && !aligned16(logits_out)) return QWEN_ERR_ARG;
  if (!(temperature > 0.f) || !sample_args_ok(temperature, top_k, top_p) || position < 0) return QWEN_ERR_ARG;
  KParams P;
  memset(&P, 0, sizeof(P));
  P.eos = -1;
  P.lm_head = (const _Float16*)weight;
  P.in_vec = (const _Float16*)hidden_f16;
  P.out_tokens = out_token;
  P.logits_out = logits_out;
  P.mode = MODE_LMHEAD;
  P.num_layers = 1;
  P.num_steps = 1;
  P.start_pos = position;
  P.max_seq = MAX_SEQ_LIMIT;
  P.temperature = temperature;
  P.seed = seed;
  P.sample = 1;
  P.top_k = device_top_k(temperature, top_k, top_p);
  P.top_p = top_p;
  return launch(P, stream);
}

extern "C" int qwen_mlp_block(const void* x_f16, const void* post_norm_weight, const void* gate_weight,
                              const void* up_weight, const void* down_weight, float* y_out, hipStream_t stream) {
  if (!x_f16 || !post_norm_weight || !gate_weight || !up_weight || !down_weight || !y_out) return QWEN_ERR_ARG;
  if (!aligned16(x_f16) || !aligned16(post_norm_weight) || !aligned16(gate_weight) || !aligned16(up_weight) ||
      !aligned16(down_weight) || !aligned16(y_out))
    return QWEN_ERR_ARG;
  KParams P;
  memset(&P, 0, sizeof(P));
  P.eos = -1;
  P.own_layer.post_attn_layernorm_weight = post_norm_weight;
  P.own_layer.gate_proj_weight = gate_weight;
  P.own_layer.up_proj_weight = up_weight;
  P.own_layer.down_proj_weight = down_weight;
  P.in_vec = (const _Float16*)x_f16;
  P.out_vec = y_out;
  P.mode = MODE_MLP;
  P.num_layers = 1;
  P.num_steps = 1;
  P.max_seq = MAX_SEQ_LIMIT;
  return launch(P, stream);
}

namespace {

// status word of one workspace: 0, or the error it reports (the workspace is then cleared
// and its epochs restart)
int take_status(Workspace& w) {
  if (!w.ws) return QWEN_OK;
  u32 s = 0;
  if (hipMemcpy(&s, w.status, sizeof(s), hipMemcpyDeviceToHost) != hipSuccess) return QWEN_ERR_LAUNCH;
  if (s == 0) return QWEN_OK;
  // a failed launch leaves slots in an unknown state: start clean
  if (zero_words(w.ws, WORKSPACE_BYTES, nullptr) != QWEN_OK || hipDeviceSynchronize() != hipSuccess)
    return QWEN_ERR_LAUNCH;
  w.epoch = 1;
  return (s & ST_BAD_TOKEN) ? QWEN_ERR_BAD_TOKEN : QWEN_ERR_TIMEOUT;
}

}  // namespace

extern "C" int qwen_last_error(void) {
  std::lock_guard<std::mutex> lock(g_mu);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return QWEN_ERR_DEVICE;
  DeviceState& st = g_dev[dev];
  if (!st.init) return QWEN_OK;
  if (st.err != QWEN_OK) return st.err;
  if (hipDeviceSynchronize() != hipSuccess) return QWEN_ERR_LAUNCH;
  const int a = take_status(st.heap);
  const int b = take_status(st.fixed);
  // a failed sampler launch can leave its work area (histograms, barrier words) dirty
  if (a != QWEN_OK && st.smp &&
      (zero_words(st.smp + SMP_WORK, smp::WORK_BYTES / 8 * 8, nullptr) != QWEN_OK || hipDeviceSynchronize() != hipSuccess))
    return QWEN_ERR_LAUNCH;
  return a != QWEN_OK ? a : b;
}

extern "C" int qwen_set_wait_deadline_us(long long us) {
  if (us < 0) return QWEN_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK) return rc;
  st->deadline = st->clk_khz * (us == 0 ? DEFAULT_WAIT_US : (u64)us) / 1000;
  if (st->deadline == 0) st->deadline = 1;
  return QWEN_OK;
}

extern "C" int qwen_abi_version(void) { return QWEN_ABI_VERSION; }

extern "C" int qwen_set_trace(unsigned long long* buf, long long elems, int token) {
  if (buf && elems <= 0) return QWEN_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState* st = nullptr;
  int rc = device_state(&st);
  if (rc != QWEN_OK) return rc;
  st->trace = buf;
  st->trace_elems = buf ? elems : 0;
  st->trace_token = buf ? token : -1;
  return QWEN_OK;
}

extern "C" int qwen_trace_events(void) { return TRACE_EVENTS; }
