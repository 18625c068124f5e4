// C-ABI shim over the prebuilt gfx950 code object (q8gemv_kernels.hip).
//
// Host side only: hipModuleLoad / hipModuleGetFunction at init, then argument
// validation and hipModuleLaunchKernel per call.  The ABI is declared in
// include/q8gemv.h.
#include "q8gemv.h"
#include "qwen3_decode.h"
#include "prefill_split.h"
#include "shim_internal.h"
#include "step_roles.h"

#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

// hipExtModuleLaunchKernel lives in hip/hip_ext.h, which pulls in the device
// headers; its C declaration is all the shim needs.
extern "C" hipError_t hipExtModuleLaunchKernel(hipFunction_t f, uint32_t globalWorkSizeX,
                                               uint32_t globalWorkSizeY, uint32_t globalWorkSizeZ,
                                               uint32_t localWorkSizeX, uint32_t localWorkSizeY,
                                               uint32_t localWorkSizeZ, size_t sharedMemBytes,
                                               hipStream_t hStream, void** kernelParams,
                                               void** extra, hipEvent_t startEvent,
                                               hipEvent_t stopEvent, uint32_t flags);

namespace {

struct KindInfo {
  const char* name;
  int64_t n, k;
};

// create_q8_irpa.py:185-224 (shapes), qwen3_full.mlir:772-777 (stacked params)
constexpr KindInfo kKinds[5] = {
    {"attn_q", 2048, 1024},
    {"attn_kv", 1024, 1024},
    {"attn_o", 1024, 2048},
    {"gate_up", 6144, 1024},
    {"ffn_dn", 1024, 3072},
};

constexpr int kVocabMaxWorkgroups = 8192;
constexpr uint32_t kDefaultSpinLimit = 1u << 20;  // dec_step: poll rounds before a wait gives up
constexpr int kQ8MaxWorkgroups = 65536;
constexpr int64_t kBatchWavesPerCu = 10;  // q8gemv_batch default
constexpr size_t kVocabWorkspaceBytes = 256;
constexpr int kBatchMaxCount = 1 << 20;
constexpr size_t kBatchHeaderBytes = 16;
constexpr size_t kBatchEntryBytes = 40;

// Device layout of one batch table entry (q8gemv_kernels.hip, Q8BatchEntry).
struct BatchEntry {
  const void* w;
  const void* x;
  void* y;
  int32_t n_rows;
  int32_t p;
  int32_t unit_begin;
  int32_t reserved;
};
static_assert(sizeof(BatchEntry) == kBatchEntryBytes, "batch entry layout");

// The six reference executables (kernels/cuda/dispatch_*.mlir:5-9): ordinal,
// export name, push-constant count, workgroup size and count of this build's
// substitution stubs.
struct HalDispatch {
  int ordinal;
  const char* name;
  int constants;
  uint32_t block;
  uint32_t grid;
};
constexpr HalDispatch kHalDispatches[6] = {
    {3, "decode_dispatch_3_matmul_2048x1x1024_f16", 2, 64, 512},
    {4, "decode_dispatch_4_matmul_1024x1x1024_f16", 3, 64, 256},
    {12, "decode_dispatch_12_matmul_1024x1x2048_f16", 2, 64, 256},
    {18, "decode_dispatch_18_matmul_6144x1x1024_f16", 2, 64, 1536},
    {20, "decode_dispatch_20_matmul_1024x1x3072_f16", 2, 64, 256},
    {24, "decode_dispatch_24_matmul_151936x1x1024_f16", 1, 256, 1024},
};

struct State {
  std::mutex mu;
  bool ready = false;
  int device = -1;
  int compute_units = 0;
  hipModule_t module = nullptr;
  hipFunction_t q8[3] = {};  // K = 1024, 2048, 3072
  hipFunction_t q8batch = nullptr;
  int batch_threads = 64;  // q8gemv_batch_k's declared workgroup size
  hipFunction_t q8qkv = nullptr;
  hipFunction_t hal[6] = {};  // IREE HAL-ABI kernels, in kHalDispatches order
  hipFunction_t vocab = nullptr;
  hipFunction_t vocab_finalize = nullptr;
  hipFunction_t argmax = nullptr;  // argmax_f16_k
  hipFunction_t ws_reset = nullptr;
  hipFunction_t copy = nullptr;
  hipFunction_t calib_empty = nullptr, calib_handoff = nullptr, calib_chase = nullptr,
                read = nullptr;
  // Tuning knobs: process-wide, set under mu, read without it (atomics), so a
  // setter never races a launch on another thread; each call reads a knob
  // once.
  std::atomic<int> batch_wgs{0};  // 0 = default
  hipModule_t dec_module = nullptr;  // decode_gfx950.hsaco (optional)
  hipFunction_t dec_embed = nullptr, dec_qkv = nullptr, dec_attn = nullptr,
                dec_o = nullptr, dec_gu = nullptr, dec_dn = nullptr, dec_vocab = nullptr,
                dec_final = nullptr, dec_adv = nullptr, dec_clear = nullptr, dec_step = nullptr;
  hipModule_t pf_module = nullptr;  // prefill_gfx950.hsaco (optional)
  hipFunction_t pf_embed = nullptr, pf_norm = nullptr, pf_gemm_qkv = nullptr, pf_gemm_res = nullptr,
                pf_gemm_qkv_m32 = nullptr, pf_gemm_res_m32 = nullptr, pf_gemm_swiglu = nullptr,
                pf_gemm_part = nullptr, pf_gemm_part_m32 = nullptr, pf_res_reduce = nullptr,
                pf_res_reduce_norm = nullptr, pf_rope = nullptr,
                pf_attn = nullptr, pf_attn_merge = nullptr, pf_set_pos = nullptr;
  // the f16 GEMMs (pf_gemm_f16*: over the f16 layer matrices) and their
  // expansion from Q8_0 (pf_expand_q8)
  hipFunction_t pf_f16_qkv_44 = nullptr, pf_f16_qkv_24 = nullptr,
                pf_f16_qkv_22p = nullptr,
                pf_f16_sw_46w = nullptr, pf_f16_sw_44 = nullptr, pf_f16_sw_24 = nullptr,
                pf_f16_sw_22 = nullptr,
                pf_f16_res_22 = nullptr, pf_f16_res_12k = nullptr,
                pf_f16_part_22 = nullptr, pf_f16_part_22k = nullptr, pf_f16_part_12k = nullptr,
                pf_f16_part_44k = nullptr, pf_expand = nullptr;
  // [64 x 64, 128 x 64 tiles][attn_o, ffn_down][K ranges - 1]
  hipFunction_t pf_f16_res_pipe[2][2][2] = {};
  // the row products (prefill_rows.h): [instance, fewest tokens first][0: f16
  // weights, 1: Q8_0]
  hipFunction_t pf_rows_qkv_rope[2] = {}, pf_rows_qkv[2][2] = {}, pf_rows_gu[4][2] = {},
                pf_rows_o[2][2] = {}, pf_rows_dn[2][2] = {};
  std::atomic<int> pf_tile_rows{0};   // prefill GEMM token tile: 0 = by shape, 32, 64 or 128
  std::atomic<int> pf_attn_split{0};  // prefill attention positions per split in blocks of 32
  std::atomic<int> step_single{-1};   // single-launch decode step: -1 unknown, 0 off, 1 on
  int64_t step_slots = 0;  // dec_step workgroups the device holds at once
  // poll rounds before a dec_step wait gives up
  std::atomic<uint32_t> step_spin_limit{kDefaultSpinLimit};
  // Single-launch steps of different streams run one after another: each
  // needs all its workgroups resident at once, and two at a time do not fit.
  // step_ev is recorded after every such launch (outside graph capture) and a
  // launch on another stream first waits for it.
  std::mutex step_mu;
  hipEvent_t step_ev = nullptr;
  hipStream_t step_last = nullptr;
  // steps re-run with the per-phase launches after a single launch gave up
  std::atomic<uint64_t> step_fallbacks{0};
  // test hook: the single launch this many launches from now is forced to
  // give up at its start (-1: none)
  std::atomic<int64_t> force_abort_in{-1};
  int noalloc_rc = Q8_ERR_NOT_INITIALIZED;  // set-up status of the allocation-free entry point
  std::string noalloc_err;
  std::atomic<int> vocab_wgs{0};  // 0 = default
};

State g;

thread_local std::string t_err;
thread_local hipEvent_t t_start = nullptr;
thread_local hipEvent_t t_stop = nullptr;

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  t_err = buf;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(Q8_ERR_HIP, "%s failed: %s (%d)", what, hipGetErrorString(e), (int)e);
}

#define HIP_TRY(expr)                                 \
  do {                                                \
    hipError_t _e = (expr);                           \
    if (_e != hipSuccess) return hip_fail(_e, #expr); \
  } while (0)

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

std::string default_code_object() {
  Dl_info info;
  if (dladdr(reinterpret_cast<void*>(&q8gemv_init), &info) && info.dli_fname) {
    std::string p(info.dli_fname);
    size_t slash = p.rfind('/');
    std::string dir = slash == std::string::npos ? std::string(".") : p.substr(0, slash);
    return dir + "/q8gemv_gfx950.hsaco";
  }
  return "q8gemv_gfx950.hsaco";
}

int launch(hipFunction_t fn, uint32_t grid, uint32_t block, void** args, hipStream_t stream) {
  hipError_t e;
  if (t_start != nullptr || t_stop != nullptr) {
    hipEvent_t s = t_start, p = t_stop;
    t_start = t_stop = nullptr;
    e = hipExtModuleLaunchKernel(fn, grid * block, 1, 1, block, 1, 1, 0, stream, args, nullptr,
                                 s, p, 0);
  } else {
    e = hipModuleLaunchKernel(fn, grid, 1, 1, block, 1, 1, 0, stream, args, nullptr);
  }
  if (e != hipSuccess) return hip_fail(e, "kernel launch");
  return Q8_OK;
}

int launch2(hipFunction_t fn, uint32_t gx, uint32_t gy, uint32_t block, void** args,
            hipStream_t stream) {
  hipError_t e = hipModuleLaunchKernel(fn, gx, gy, 1, block, 1, 1, 0, stream, args, nullptr);
  if (e != hipSuccess) return hip_fail(e, "kernel launch");
  return Q8_OK;
}

int check_ready() {
  if (!g.ready) return fail(Q8_ERR_NOT_INITIALIZED, "q8gemv_init() has not succeeded");
  return Q8_OK;
}

int cu_count() { return g.compute_units > 0 ? g.compute_units : 256; }

int q8_launch(const void* w_layer, int64_t n_rows, int64_t k, const void* x, void* y,
              void* stream) {
  const int64_t quads = (n_rows + 3) / 4;  // one wave per row quad
  const void* w_arg = w_layer;
  const void* x_arg = x;
  void* y_arg = y;
  int n_arg = (int)n_rows;
  void* args[] = {&w_arg, &x_arg, &y_arg, &n_arg};
  return launch(g.q8[k / 1024 - 1], (uint32_t)quads, 64, args, static_cast<hipStream_t>(stream));
}

int validate_gemv(const void* w_layer, int64_t n_rows, int64_t k, const void* x_f16,
                  const void* y_f16) {
  if (!w_layer || !x_f16 || !y_f16) return fail(Q8_ERR_NULL_POINTER, "null w, x or y");
  if (k != 1024 && k != 2048 && k != 3072)
    return fail(Q8_ERR_BAD_SHAPE, "K=%lld not in {1024, 2048, 3072}", (long long)k);
  if (n_rows < 1 || n_rows > (1LL << 24))
    return fail(Q8_ERR_BAD_SHAPE, "n_rows=%lld outside [1, 2^24]", (long long)n_rows);
  if (!aligned(w_layer, 16)) return fail(Q8_ERR_MISALIGNED, "weights not 16-byte aligned");
  if (!aligned(x_f16, 16)) return fail(Q8_ERR_MISALIGNED, "x not 16-byte aligned");
  if (!aligned(y_f16, 2)) return fail(Q8_ERR_MISALIGNED, "y not 2-byte aligned");
  return Q8_OK;
}

int vocab_grid() {
  const int set = g.vocab_wgs.load(std::memory_order_relaxed);
  if (set > 0) return set;
  // One workgroup (four waves) per CU: with the matrix read from HBM (three
  // copies taken in turn) 1 / 2 / 4 per CU measured 49.7 / 50.7 / 52.6 us.
  int wgs = cu_count();
  return wgs > kVocabMaxWorkgroups ? kVocabMaxWorkgroups : wgs;
}

}  // namespace

extern "C" {

int q8gemv_init(const char* code_object_path) {
  std::lock_guard<std::mutex> lock(g.mu);
  if (g.ready) return Q8_OK;
  std::string path = code_object_path ? std::string(code_object_path) : default_code_object();
  FILE* f = std::fopen(path.c_str(), "rb");
  if (!f) return fail(Q8_ERR_CODE_OBJECT, "cannot open code object %s", path.c_str());
  std::fclose(f);
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  hipModule_t mod = nullptr;
  hipError_t e = hipModuleLoad(&mod, path.c_str());
  if (e != hipSuccess)
    return fail(Q8_ERR_CODE_OBJECT, "hipModuleLoad(%s): %s", path.c_str(), hipGetErrorString(e));
  e = hipModuleGetFunction(&g.q8[0], mod, "q8gemv_p1");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.q8[1], mod, "q8gemv_p2");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.q8[2], mod, "q8gemv_p3");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.q8batch, mod, "q8gemv_batch_k");
  g.batch_threads = 64;
  if (e == hipSuccess) {
    int threads = 0;
    if (hipFuncGetAttribute(&threads, HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK, g.q8batch) ==
            hipSuccess &&
        threads >= 64 && threads % 64 == 0)
      g.batch_threads = threads;
  }
  if (e == hipSuccess) e = hipModuleGetFunction(&g.q8qkv, mod, "q8gemv_qkv_k");
  for (int i = 0; i < 6 && e == hipSuccess; ++i)
    e = hipModuleGetFunction(&g.hal[i], mod, kHalDispatches[i].name);
  if (e != hipSuccess) {
    (void)hipModuleUnload(mod);
    return fail(Q8_ERR_CODE_OBJECT, "Q8_0 GEMV kernels missing from %s", path.c_str());
  }
  e = hipModuleGetFunction(&g.vocab, mod, "vocab_gemv_argmax_k1024");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.vocab_finalize, mod, "vocab_argmax_finalize");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.argmax, mod, "argmax_f16_k");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.ws_reset, mod, "vocab_workspace_reset");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.copy, mod, "stream_copy_b128");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.read, mod, "stream_read_b128");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.calib_empty, mod, "calib_empty");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.calib_handoff, mod, "calib_handoff");
  if (e == hipSuccess) e = hipModuleGetFunction(&g.calib_chase, mod, "calib_chase");
  if (e != hipSuccess) {
    (void)hipModuleUnload(mod);
    return fail(Q8_ERR_CODE_OBJECT, "vocab / copy kernels missing from %s", path.c_str());
  }
  // The decode-step kernels live in a second code object next to the first
  // (or next to this library); without it the qwen3_decode_* calls report
  // Q8_ERR_CODE_OBJECT.
  {
    const size_t slash = path.rfind('/');
    std::string dir = slash == std::string::npos ? std::string(".") : path.substr(0, slash);
    std::string dpath = dir + "/decode_gfx950.hsaco";
    FILE* df = std::fopen(dpath.c_str(), "rb");
    if (!df) {
      std::string lib = default_code_object();
      dpath = lib.substr(0, lib.rfind('/')) + "/decode_gfx950.hsaco";
      df = std::fopen(dpath.c_str(), "rb");
    }
    if (df) {
      std::fclose(df);
      hipModule_t dm = nullptr;
      if (hipModuleLoad(&dm, dpath.c_str()) == hipSuccess) {
        struct {
          hipFunction_t* fn;
          const char* name;
        } names[] = {{&g.dec_embed, "dec_embed"},     {&g.dec_qkv, "dec_qkv"},
                     {&g.dec_attn, "dec_attention"},
                     {&g.dec_o, "dec_o_res"},         {&g.dec_gu, "dec_gu_swiglu"},
                     {&g.dec_dn, "dec_down_res"},     {&g.dec_vocab, "dec_vocab_argmax"},
                     {&g.dec_final, "dec_finalize"},  {&g.dec_adv, "dec_advance"},
                     {&g.dec_clear, "dec_scratch_clear"}, {&g.dec_step, "dec_step"}};
        bool ok = true;
        for (auto& n : names) ok = ok && hipModuleGetFunction(n.fn, dm, n.name) == hipSuccess;
        if (ok) {
          g.dec_module = dm;
        } else {
          (void)hipModuleUnload(dm);
          for (auto& n : names) *n.fn = nullptr;
        }
      }
    }
  }
  // The batched prompt kernels live in a third code object beside the decode
  // one; without it qwen3_prefill_batched reports Q8_ERR_CODE_OBJECT.
  if (g.dec_module) {
    const size_t slash = path.rfind('/');
    std::string dir = slash == std::string::npos ? std::string(".") : path.substr(0, slash);
    std::string ppath = dir + "/prefill_gfx950.hsaco";
    FILE* pf = std::fopen(ppath.c_str(), "rb");
    if (!pf) {
      std::string lib = default_code_object();
      ppath = lib.substr(0, lib.rfind('/')) + "/prefill_gfx950.hsaco";
      pf = std::fopen(ppath.c_str(), "rb");
    }
    if (pf) {
      std::fclose(pf);
      hipModule_t pm = nullptr;
      if (hipModuleLoad(&pm, ppath.c_str()) == hipSuccess) {
        struct {
          hipFunction_t* fn;
          const char* name;
        } names[] = {{&g.pf_embed, "pf_embed"},
                     {&g.pf_norm, "pf_rmsnorm"},
                     {&g.pf_gemm_qkv, "pf_gemm_q8"},
                     {&g.pf_gemm_res, "pf_gemm_q8_res"},
                     {&g.pf_gemm_qkv_m32, "pf_gemm_q8_m32"},
                     {&g.pf_gemm_res_m32, "pf_gemm_q8_res_m32"},
                     {&g.pf_gemm_swiglu, "pf_gemm_q8_swiglu"},
                     {&g.pf_rope, "pf_qk_rope_cache"},
                     {&g.pf_attn, "pf_attention"},
                     {&g.pf_attn_merge, "pf_attn_merge"},
                     {&g.pf_gemm_part, "pf_gemm_q8_part"},
                     {&g.pf_gemm_part_m32, "pf_gemm_q8_part_m32"},
                     {&g.pf_res_reduce, "pf_res_reduce"},
                     {&g.pf_res_reduce_norm, "pf_res_reduce_norm"},
                     {&g.pf_set_pos, "pf_set_pos"},
                     {&g.pf_f16_qkv_44, "pf_gemm_f16_qkv_44"},
                     {&g.pf_f16_qkv_24, "pf_gemm_f16_qkv_24"},
                     {&g.pf_f16_qkv_22p, "pf_gemm_f16_qkv_22p"},
                     {&g.pf_f16_sw_46w, "pf_gemm_f16_swiglu_46w"},
                     {&g.pf_f16_sw_44, "pf_gemm_f16_swiglu_44"},
                     {&g.pf_f16_sw_24, "pf_gemm_f16_swiglu_24"},
                     {&g.pf_f16_sw_22, "pf_gemm_f16_swiglu_22"},
                     {&g.pf_f16_res_22, "pf_gemm_f16_res_22"},
                     {&g.pf_f16_res_12k, "pf_gemm_f16_res_12k"},
                     {&g.pf_f16_res_pipe[0][0][0], "pf_gemm_f16_res_o_p1"},
                     {&g.pf_f16_res_pipe[0][0][1], "pf_gemm_f16_res_o_p2"},
                     {&g.pf_f16_res_pipe[0][1][0], "pf_gemm_f16_res_dn_p1"},
                     {&g.pf_f16_res_pipe[0][1][1], "pf_gemm_f16_res_dn_p2"},
                     {&g.pf_f16_res_pipe[1][0][0], "pf_gemm_f16_res_o_w1"},
                     {&g.pf_f16_res_pipe[1][0][1], "pf_gemm_f16_res_o_w2"},
                     {&g.pf_f16_res_pipe[1][1][0], "pf_gemm_f16_res_dn_w1"},
                     {&g.pf_f16_res_pipe[1][1][1], "pf_gemm_f16_res_dn_w2"},
                     {&g.pf_f16_part_22, "pf_gemm_f16_part_22"},
                     {&g.pf_f16_part_22k, "pf_gemm_f16_part_22k"},
                     {&g.pf_f16_part_12k, "pf_gemm_f16_part_12k"},
                     {&g.pf_f16_part_44k, "pf_gemm_f16_part_44k"},
                     {&g.pf_rows_qkv_rope[0], "pf_rows_qkv_rope"},
                     {&g.pf_rows_qkv_rope[1], "pf_rows_qkv_rope_q8"},
                     {&g.pf_rows_qkv[0][0], "pf_rows_qkv_11"},
                     {&g.pf_rows_qkv[0][1], "pf_rows_qkv_q8_11"},
                     {&g.pf_rows_qkv[1][0], "pf_rows_qkv_12"},
                     {&g.pf_rows_qkv[1][1], "pf_rows_qkv_q8_12"},
                     {&g.pf_rows_gu[0][0], "pf_rows_gu_12"},
                     {&g.pf_rows_gu[0][1], "pf_rows_gu_q8_12"},
                     {&g.pf_rows_gu[1][0], "pf_rows_gu_22"},
                     {&g.pf_rows_gu[1][1], "pf_rows_gu_q8_22"},
                     {&g.pf_rows_gu[2][0], "pf_rows_gu_24"},
                     {&g.pf_rows_gu[2][1], "pf_rows_gu_q8_24"},
                     {&g.pf_rows_gu[3][0], "pf_rows_gu_26"},
                     {&g.pf_rows_gu[3][1], "pf_rows_gu_q8_26"},
                     {&g.pf_rows_o[0][0], "pf_rows_o_1"},
                     {&g.pf_rows_o[0][1], "pf_rows_o_q8_1"},
                     {&g.pf_rows_o[1][0], "pf_rows_o_2"},
                     {&g.pf_rows_o[1][1], "pf_rows_o_q8_2"},
                     {&g.pf_rows_dn[0][0], "pf_rows_dn_1"},
                     {&g.pf_rows_dn[0][1], "pf_rows_dn_q8_1"},
                     {&g.pf_rows_dn[1][0], "pf_rows_dn_2"},
                     {&g.pf_rows_dn[1][1], "pf_rows_dn_q8_2"},
                     {&g.pf_expand, "pf_expand_q8"}};
        bool ok = true;
        for (auto& n : names) ok = ok && hipModuleGetFunction(n.fn, pm, n.name) == hipSuccess;
        if (ok) {
          g.pf_module = pm;
        } else {
          (void)hipModuleUnload(pm);
          for (auto& n : names) *n.fn = nullptr;
        }
      }
    }
  }
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 256;
  // The single-launch step needs its workgroups resident together (they
  // wait on each other's tagged words; there is no grid barrier): a device
  // whose CUs hold them all at once (two per CU), checked from the kernel's
  // occupancy.  It is launched as an ordinary kernel: a cooperative launch
  // of the same grid measured 19.6 us of launch cost against 2.1 (empty
  // kernel, back to back), 559.8 -> 541.8 us per step.  Should a concurrent
  // kernel on another stream keep some of the workgroups from starting, the
  // bounded waits of the resident ones give up and the step reports status
  // bit 1 (every workgroup then exits) instead of hanging.
  g.step_slots = 0;
  if (g.dec_step) {
    int per_cu = 0;
    if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, g.dec_step, 256, 0) ==
        hipSuccess)
      g.step_slots = (int64_t)per_cu * cus;
  }
  // The single launch is the default where it can run: no kernel boundaries,
  // and every workgroup requests its next weights before it waits.
  if (g.step_single.load() < 0) g.step_single = g.step_slots >= kStepWgs ? 1 : 0;
  g.module = mod;
  g.device = dev;
  g.compute_units = cus;
  g.batch_wgs = 0;
  g.vocab_wgs = 0;
  g.ready = true;
  // the allocation-free entry point's scratch on this device (address and a
  // zero fill; an error here leaves that one entry point unavailable)
  g.noalloc_rc = q8_shim::noalloc_setup(dev);
  if (g.noalloc_rc != Q8_OK) g.noalloc_err = t_err;
  return Q8_OK;
}

void q8gemv_shutdown(void) {
  std::lock_guard<std::mutex> lock(g.mu);
  if (!g.ready) return;
  (void)hipModuleUnload(g.module);
  g.module = nullptr;
  g.q8[0] = g.q8[1] = g.q8[2] = g.q8batch = g.q8qkv = nullptr;
  std::memset(g.hal, 0, sizeof(g.hal));
  if (g.dec_module) (void)hipModuleUnload(g.dec_module);
  g.dec_module = nullptr;
  g.dec_embed = g.dec_qkv = g.dec_attn = g.dec_o = g.dec_gu = g.dec_dn =
      g.dec_vocab = g.dec_final = g.dec_adv = g.dec_clear = g.dec_step = nullptr;
  g.step_slots = 0;
  {
    std::lock_guard<std::mutex> step_lock(g.step_mu);
    if (g.step_ev) (void)hipEventDestroy(g.step_ev);
    g.step_ev = nullptr;
    g.step_last = nullptr;
  }
  if (g.pf_module) (void)hipModuleUnload(g.pf_module);
  g.pf_module = nullptr;
  g.pf_embed = g.pf_norm = g.pf_gemm_qkv = g.pf_gemm_res = g.pf_gemm_qkv_m32 = g.pf_gemm_res_m32 =
      g.pf_gemm_swiglu = g.pf_rope = g.pf_attn = g.pf_attn_merge = g.pf_set_pos = nullptr;
  g.pf_gemm_part = g.pf_gemm_part_m32 = g.pf_res_reduce = g.pf_res_reduce_norm = nullptr;
  g.pf_f16_qkv_44 = g.pf_f16_qkv_24 = g.pf_f16_qkv_22p = g.pf_f16_sw_46w =
      g.pf_f16_sw_44 = g.pf_f16_sw_24 = g.pf_f16_sw_22 = nullptr;
  std::memset(g.pf_f16_res_pipe, 0, sizeof(g.pf_f16_res_pipe));
  std::memset(g.pf_rows_qkv_rope, 0, sizeof(g.pf_rows_qkv_rope));
  std::memset(g.pf_rows_qkv, 0, sizeof(g.pf_rows_qkv));
  std::memset(g.pf_rows_gu, 0, sizeof(g.pf_rows_gu));
  std::memset(g.pf_rows_o, 0, sizeof(g.pf_rows_o));
  std::memset(g.pf_rows_dn, 0, sizeof(g.pf_rows_dn));
  g.pf_f16_res_22 = g.pf_f16_res_12k = g.pf_f16_part_22 = g.pf_f16_part_22k =
      g.pf_f16_part_12k = g.pf_f16_part_44k = g.pf_expand = nullptr;
  g.vocab = g.vocab_finalize = g.argmax = g.ws_reset = g.copy = nullptr;
  g.calib_empty = g.calib_handoff = g.calib_chase = g.read = nullptr;
  g.ready = false;
}

const char* q8gemv_last_error(void) { return t_err.c_str(); }

int q8gemv_kind_shape(int kind, int64_t* n, int64_t* k, int64_t* bytes_per_layer) {
  if (kind < 0 || kind > 4) return fail(Q8_ERR_INVALID_KIND, "invalid kind %d", kind);
  const KindInfo& ki = kKinds[kind];
  if (n) *n = ki.n;
  if (k) *k = ki.k;
  if (bytes_per_layer) *bytes_per_layer = ki.n * ki.k / Q8_BLOCK_ELEMS * Q8_BLOCK_BYTES;
  return Q8_OK;
}

int q8gemv_rows(const void* w_layer, int64_t n_rows, int64_t k, const void* x_f16, void* y_f16,
                void* stream) {
  int rc = validate_gemv(w_layer, n_rows, k, x_f16, y_f16);
  if (rc) return rc;
  rc = check_ready();
  if (rc) return rc;
  return q8_launch(w_layer, n_rows, k, x_f16, y_f16, stream);
}

int q8gemv(int kind, const void* w_stacked, int64_t layer, const void* x_f16, void* y_f16,
           void* stream) {
  if (kind < 0 || kind > 4) return fail(Q8_ERR_INVALID_KIND, "invalid kind %d", kind);
  if (!w_stacked || !x_f16 || !y_f16) return fail(Q8_ERR_NULL_POINTER, "null w, x or y");
  if (layer < 0 || layer >= Q8_NUM_LAYERS)
    return fail(Q8_ERR_LAYER_RANGE, "layer %lld outside [0, %d)", (long long)layer,
                Q8_NUM_LAYERS);
  const KindInfo& ki = kKinds[kind];
  const int64_t bpl = ki.n * ki.k / Q8_BLOCK_ELEMS * Q8_BLOCK_BYTES;
  const void* w_layer = static_cast<const uint8_t*>(w_stacked) + layer * bpl;
  return q8gemv_rows(w_layer, ki.n, ki.k, x_f16, y_f16, stream);
}

int decode_dispatch_3_matmul_2048x1x1024_f16(const void* q8_stacked, int64_t layer,
                                             const void* x_f16, void* y_f16, void* stream) {
  return q8gemv(Q8_ATTN_Q, q8_stacked, layer, x_f16, y_f16, stream);
}
int decode_dispatch_4_matmul_1024x1x1024_f16(const void* q8_stacked, int64_t layer,
                                             const void* x_f16, void* y_f16, void* stream) {
  return q8gemv(Q8_ATTN_KV, q8_stacked, layer, x_f16, y_f16, stream);
}
int decode_dispatch_12_matmul_1024x1x2048_f16(const void* q8_stacked, int64_t layer,
                                              const void* x_f16, void* y_f16, void* stream) {
  return q8gemv(Q8_ATTN_O, q8_stacked, layer, x_f16, y_f16, stream);
}
int decode_dispatch_18_matmul_6144x1x1024_f16(const void* q8_stacked, int64_t layer,
                                              const void* x_f16, void* y_f16, void* stream) {
  return q8gemv(Q8_GATE_UP, q8_stacked, layer, x_f16, y_f16, stream);
}
int decode_dispatch_20_matmul_1024x1x3072_f16(const void* q8_stacked, int64_t layer,
                                              const void* x_f16, void* y_f16, void* stream) {
  return q8gemv(Q8_FFN_DN, q8_stacked, layer, x_f16, y_f16, stream);
}

int q8gemv_desc_for_kind(int kind, const void* w_stacked, int64_t layer, const void* x_f16,
                         void* y_f16, q8gemv_desc* out) {
  if (kind < 0 || kind > 4) return fail(Q8_ERR_INVALID_KIND, "invalid kind %d", kind);
  if (!w_stacked || !out) return fail(Q8_ERR_NULL_POINTER, "null w_stacked or out");
  if (layer < 0 || layer >= Q8_NUM_LAYERS)
    return fail(Q8_ERR_LAYER_RANGE, "layer %lld outside [0, %d)", (long long)layer,
                Q8_NUM_LAYERS);
  const KindInfo& ki = kKinds[kind];
  const int64_t bpl = ki.n * ki.k / Q8_BLOCK_ELEMS * Q8_BLOCK_BYTES;
  out->w_layer = static_cast<const uint8_t*>(w_stacked) + layer * bpl;
  out->x_f16 = x_f16;
  out->y_f16 = y_f16;
  out->n_rows = ki.n;
  out->k = ki.k;
  return Q8_OK;
}

int q8gemv_qkv(const void* wq_stacked, const void* wk_stacked, const void* wv_stacked,
               int64_t layer, const void* x_f16, void* yq_f16, void* yk_f16, void* yv_f16,
               void* stream) {
  if (!wq_stacked || !wk_stacked || !wv_stacked || !x_f16 || !yq_f16 || !yk_f16 || !yv_f16)
    return fail(Q8_ERR_NULL_POINTER, "null weight, x or y pointer");
  if (layer < 0 || layer >= Q8_NUM_LAYERS)
    return fail(Q8_ERR_LAYER_RANGE, "layer %lld outside [0, %d)", (long long)layer,
                Q8_NUM_LAYERS);
  if (!aligned(wq_stacked, 16) || !aligned(wk_stacked, 16) || !aligned(wv_stacked, 16))
    return fail(Q8_ERR_MISALIGNED, "weights not 16-byte aligned");
  if (!aligned(x_f16, 16)) return fail(Q8_ERR_MISALIGNED, "x not 16-byte aligned");
  if (!aligned(yq_f16, 2) || !aligned(yk_f16, 2) || !aligned(yv_f16, 2))
    return fail(Q8_ERR_MISALIGNED, "y not 2-byte aligned");
  int rc = check_ready();
  if (rc) return rc;
  const int64_t bpl_q = 2048LL * 1024 / Q8_BLOCK_ELEMS * Q8_BLOCK_BYTES;
  const int64_t bpl_kv = 1024LL * 1024 / Q8_BLOCK_ELEMS * Q8_BLOCK_BYTES;
  const void* wq = static_cast<const uint8_t*>(wq_stacked) + layer * bpl_q;
  const void* wk = static_cast<const uint8_t*>(wk_stacked) + layer * bpl_kv;
  const void* wv = static_cast<const uint8_t*>(wv_stacked) + layer * bpl_kv;
  const void* x = x_f16;
  void* yq = yq_f16;
  void* yk = yk_f16;
  void* yv = yv_f16;
  void* args[] = {&wq, &wk, &wv, &x, &yq, &yk, &yv};
  return launch(g.q8qkv, 1024, 64, args, static_cast<hipStream_t>(stream));
}

int q8gemv_hal_dispatch(int ordinal, const void* binding0, const void* binding1, void* binding2,
                        const uint32_t* push_constants, int n_constants, void* stream) {
  return q8gemv_hal_dispatch_grid(ordinal, binding0, binding1, binding2, push_constants,
                                  n_constants, 0, 0, stream);
}

int q8gemv_hal_dispatch_grid(int ordinal, const void* binding0, const void* binding1,
                             void* binding2, const uint32_t* push_constants, int n_constants,
                             uint32_t workgroups, uint32_t workgroup_size, void* stream) {
  int idx = -1;
  for (int i = 0; i < 6; ++i)
    if (kHalDispatches[i].ordinal == ordinal) idx = i;
  if (idx < 0) return fail(Q8_ERR_INVALID_KIND, "no substituted dispatch with ordinal %d", ordinal);
  const HalDispatch& hd = kHalDispatches[idx];
  if (!binding0 || !binding1 || !binding2 || !push_constants)
    return fail(Q8_ERR_NULL_POINTER, "null binding or push-constant pointer");
  if (n_constants != hd.constants)
    return fail(Q8_ERR_BAD_ARGUMENT, "%s takes %d push constants, got %d", hd.name, hd.constants,
                n_constants);
  if (!aligned(binding0, 16) || !aligned(binding1, 16) || !aligned(binding2, 2))
    return fail(Q8_ERR_MISALIGNED, "bindings 0/1 need 16-byte, binding 2 2-byte alignment");
  if (ordinal != 24) {
    const int lo = ordinal == 4 ? 1 : 0;
    const uint64_t layer = (uint64_t)push_constants[lo] | ((uint64_t)push_constants[lo + 1] << 32);
    if (layer >= (uint64_t)Q8_NUM_LAYERS)
      return fail(Q8_ERR_LAYER_RANGE, "layer %llu outside [0, %d)", (unsigned long long)layer,
                  Q8_NUM_LAYERS);
  }
  if ((ordinal == 4 || ordinal == 24) && (push_constants[0] & 1u))
    return fail(Q8_ERR_MISALIGNED, "output byte offset %u is odd", push_constants[0]);
  const uint32_t block = workgroup_size ? workgroup_size : hd.block;
  const uint32_t grid = workgroups ? workgroups : hd.grid;
  if (block % 64 != 0 || block > 256)
    return fail(Q8_ERR_BAD_ARGUMENT, "workgroup size %u is not 64, 128, 192 or 256", block);
  if (grid > 0x7fffffffu)
    return fail(Q8_ERR_BAD_ARGUMENT, "%u workgroups is too many", grid);
  int rc = check_ready();
  if (rc) return rc;
  const void* b0 = binding0;
  const void* b1 = binding1;
  void* b2 = binding2;
  uint32_t c[3] = {push_constants[0], hd.constants > 1 ? push_constants[1] : 0u,
                   hd.constants > 2 ? push_constants[2] : 0u};
  void* args3[] = {&b0, &b1, &b2, &c[0]};
  void* args5[] = {&b0, &b1, &b2, &c[0], &c[1]};
  void* args6[] = {&b0, &b1, &b2, &c[0], &c[1], &c[2]};
  void** args = hd.constants == 1 ? args3 : hd.constants == 2 ? args5 : args6;
  return launch(g.hal[idx], grid, block, args, static_cast<hipStream_t>(stream));
}

size_t q8gemv_batch_table_bytes(int count) {
  if (count < 1 || count > kBatchMaxCount) return 0;
  return kBatchHeaderBytes + kBatchEntryBytes * (size_t)count;
}

int q8gemv_batch_encode(const q8gemv_desc* descs, int count, void* host_table,
                        size_t table_bytes, int32_t* total_units) {
  if (!descs || !host_table || !total_units) return fail(Q8_ERR_NULL_POINTER, "null argument");
  if (count < 1 || count > kBatchMaxCount)
    return fail(Q8_ERR_BAD_ARGUMENT, "count %d outside [1, %d]", count, kBatchMaxCount);
  if (table_bytes < q8gemv_batch_table_bytes(count))
    return fail(Q8_ERR_BAD_ARGUMENT, "table needs %zu bytes, got %zu",
                q8gemv_batch_table_bytes(count), table_bytes);
  uint8_t* t = static_cast<uint8_t*>(host_table);
  int64_t units = 0;
  for (int i = 0; i < count; ++i) {
    const q8gemv_desc& d = descs[i];
    int rc = validate_gemv(d.w_layer, d.n_rows, d.k, d.x_f16, d.y_f16);
    if (rc) {
      std::string msg = t_err;
      return fail(rc, "descriptor %d: %s", i, msg.c_str());
    }
    BatchEntry be;
    be.w = d.w_layer;
    be.x = d.x_f16;
    be.y = d.y_f16;
    be.n_rows = (int32_t)d.n_rows;
    be.p = (int32_t)(d.k / 1024);
    be.unit_begin = (int32_t)units;
    be.reserved = 0;
    std::memcpy(t + kBatchHeaderBytes + kBatchEntryBytes * (size_t)i, &be, sizeof(be));
    units += (d.n_rows + 3) / 4 * (d.k / 1024);
    if (units >= (1LL << 31)) return fail(Q8_ERR_BAD_SHAPE, "batch too large");
  }
  int32_t header[4] = {count, (int32_t)units, 0, 0};
  std::memcpy(t, header, sizeof(header));
  *total_units = (int32_t)units;
  return Q8_OK;
}

int q8gemv_batch(const void* device_table, int count, int32_t total_units, void* stream) {
  if (!device_table) return fail(Q8_ERR_NULL_POINTER, "null table");
  if (!aligned(device_table, 16)) return fail(Q8_ERR_MISALIGNED, "table not 16-byte aligned");
  if (count < 1 || count > kBatchMaxCount)
    return fail(Q8_ERR_BAD_ARGUMENT, "count %d outside [1, %d]", count, kBatchMaxCount);
  if (total_units < count) return fail(Q8_ERR_BAD_ARGUMENT, "total_units %d < count", total_units);
  int rc = check_ready();
  if (rc) return rc;
  // default: 10 waves per CU (the 28-layer sweep from HBM, three weight
  // copies taken in turn: 8 / 9 / 10 / 10.5 / 11 / 12 per CU measured 74.1 /
  // 72.1 / 71.6 / 75.5 / 72.3 / 72.3 us)
  const int set_wgs = g.batch_wgs.load(std::memory_order_relaxed);
  const int64_t cap = set_wgs > 0 ? set_wgs : kBatchWavesPerCu * 64 / g.batch_threads * cu_count();
  const int64_t grid = total_units < cap ? total_units : cap;
  const void* t_arg = device_table;
  int c_arg = count;
  int u_arg = total_units;
  void* args[] = {&t_arg, &c_arg, &u_arg};
  return launch(g.q8batch, (uint32_t)grid, (uint32_t)g.batch_threads, args,
                static_cast<hipStream_t>(stream));
}

size_t vocab_argmax_workspace_bytes(void) { return kVocabWorkspaceBytes; }

int vocab_argmax_workspace_reset(void* workspace, void* stream) {
  if (!workspace) return fail(Q8_ERR_NULL_POINTER, "null workspace");
  if (!aligned(workspace, 16)) return fail(Q8_ERR_MISALIGNED, "workspace not 16-byte aligned");
  int rc = check_ready();
  if (rc) return rc;
  void* ws = workspace;
  void* args[] = {&ws};
  return launch(g.ws_reset, 1, 64, args, static_cast<hipStream_t>(stream));
}

int f16_gemv_argmax_rows(const void* w_f16, int64_t n_rows, const void* x_f16, void* logits_f16,
                         int32_t* token, void* workspace, void* stream) {
  if (!workspace) return fail(Q8_ERR_NULL_POINTER, "null workspace");
  if (!aligned(workspace, 16)) return fail(Q8_ERR_MISALIGNED, "workspace not 16-byte aligned");
  int rc = q8_shim::validate_f16_argmax(w_f16, n_rows, x_f16, logits_f16, token);
  if (rc) return rc;
  return q8_shim::launch_f16_argmax(w_f16, n_rows, x_f16, logits_f16, token, workspace,
                                    static_cast<hipStream_t>(stream));
}

}  // extern "C"

namespace q8_shim {

int error(int code, const char* msg) { return fail(code, "%s", msg); }

int hip_error(hipError_t e, const char* what) { return hip_fail(e, what); }

int noalloc_ready() {
  int rc = check_ready();
  if (rc) return rc;
  if (g.noalloc_rc != Q8_OK)
    return fail(g.noalloc_rc, "allocation-free scratch unavailable: %s", g.noalloc_err.c_str());
  return Q8_OK;
}

int validate_f16_argmax(const void* w_f16, int64_t n_rows, const void* x_f16,
                        const void* logits_f16, const int32_t* token) {
  if (!w_f16 || !x_f16 || !token) return fail(Q8_ERR_NULL_POINTER, "null w, x or token");
  if (n_rows < 1 || n_rows >= (1LL << 31))
    return fail(Q8_ERR_BAD_SHAPE, "n_rows=%lld outside [1, 2^31)", (long long)n_rows);
  if (!aligned(w_f16, 16)) return fail(Q8_ERR_MISALIGNED, "weights not 16-byte aligned");
  if (!aligned(x_f16, 16)) return fail(Q8_ERR_MISALIGNED, "x not 16-byte aligned");
  if (logits_f16 && !aligned(logits_f16, 2))
    return fail(Q8_ERR_MISALIGNED, "logits not 2-byte aligned");
  if (!aligned(token, 4)) return fail(Q8_ERR_MISALIGNED, "token not 4-byte aligned");
  return check_ready();
}

int launch_f16_argmax(const void* w_f16, int64_t n_rows, const void* x_f16, void* logits_f16,
                      int32_t* token, void* workspace, hipStream_t s) {
  int rc;
  const void* w_arg = w_f16;
  const void* x_arg = x_f16;
  void* l_arg = logits_f16;
  int n_arg = (int)n_rows;
  int32_t* t_arg = token;
  void* ws_arg = workspace;
  void* args[] = {&w_arg, &x_arg, &l_arg, &n_arg, &ws_arg};
  rc = launch(g.vocab, (uint32_t)vocab_grid(), 256, args, s);
  if (rc) return rc;
  void* fargs[] = {&ws_arg, &t_arg};
  return launch(g.vocab_finalize, 1, 64, fargs, s);
}

}  // namespace q8_shim

extern "C" {

int vocab_gemv_argmax(const void* w_f16, const void* x_f16, void* logits_f16, int32_t* token,
                      void* workspace, void* stream) {
  return f16_gemv_argmax_rows(w_f16, Q8_VOCAB_ROWS, x_f16, logits_f16, token, workspace, stream);
}

int decode_dispatch_24_matmul_151936x1x1024_f16(const void* w_f16, const void* x_f16,
                                                void* logits_f16, int32_t* token,
                                                void* workspace, void* stream) {
  return vocab_gemv_argmax(w_f16, x_f16, logits_f16, token, workspace, stream);
}

int f16_argmax(const void* values_f16, int64_t n, int32_t* token, void* workspace,
               void* stream) {
  if (!values_f16 || !token || !workspace)
    return fail(Q8_ERR_NULL_POINTER, "null values, token or workspace");
  if (n < 1 || n >= (1LL << 31)) return fail(Q8_ERR_BAD_SHAPE, "n=%lld outside [1, 2^31)", (long long)n);
  if (!aligned(values_f16, 16)) return fail(Q8_ERR_MISALIGNED, "values not 16-byte aligned");
  if (!aligned(token, 4)) return fail(Q8_ERR_MISALIGNED, "token not 4-byte aligned");
  if (!aligned(workspace, 16)) return fail(Q8_ERR_MISALIGNED, "workspace not 16-byte aligned");
  int rc = check_ready();
  if (rc) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const void* v_arg = values_f16;
  int n_arg = (int)n;
  void* ws_arg = workspace;
  int32_t* t_arg = token;
  // one workgroup per 2048 values (8 per thread), at most one per compute unit
  const int64_t want = (n + 2047) / 2048;
  const uint32_t grid = (uint32_t)(want < cu_count() ? want : cu_count());
  void* args[] = {&v_arg, &n_arg, &ws_arg};
  rc = launch(g.argmax, grid, 256, args, s);
  if (rc) return rc;
  void* fargs[] = {&ws_arg, &t_arg};
  return launch(g.vocab_finalize, 1, 64, fargs, s);
}

int q8gemv_batch_set_workgroups(int workgroups) {
  if (workgroups < 0 || workgroups > kQ8MaxWorkgroups)
    return fail(Q8_ERR_BAD_ARGUMENT, "workgroups %d outside [0, %d]", workgroups, kQ8MaxWorkgroups);
  std::lock_guard<std::mutex> lock(g.mu);
  g.batch_wgs = workgroups;
  return Q8_OK;
}

int vocab_set_workgroups(int workgroups) {
  if (workgroups < 0 || workgroups > kVocabMaxWorkgroups)
    return fail(Q8_ERR_BAD_ARGUMENT, "workgroups %d outside [0, %d]", workgroups,
                kVocabMaxWorkgroups);
  std::lock_guard<std::mutex> lock(g.mu);
  g.vocab_wgs = workgroups;
  return Q8_OK;
}

int vocab_get_workgroups(int* workgroups) {
  if (!workgroups) return fail(Q8_ERR_NULL_POINTER, "null output");
  *workgroups = vocab_grid();
  return Q8_OK;
}

// ---------------------------------------------------------------- runtime

int q8rt_device_count(int* count) {
  if (!count) return fail(Q8_ERR_NULL_POINTER, "null count");
  HIP_TRY(hipGetDeviceCount(count));
  return Q8_OK;
}

int q8rt_set_device(int device) {
  HIP_TRY(hipSetDevice(device));
  return Q8_OK;
}

int q8rt_device_info(char* name, int name_len, int* compute_units, int64_t* total_mem) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, dev));
  if (name && name_len > 0) {
    std::snprintf(name, (size_t)name_len, "%s (%s)", prop.name, prop.gcnArchName);
  }
  if (compute_units) *compute_units = prop.multiProcessorCount;
  if (total_mem) *total_mem = (int64_t)prop.totalGlobalMem;
  return Q8_OK;
}

int q8rt_malloc(void** ptr, size_t bytes) {
  if (!ptr) return fail(Q8_ERR_NULL_POINTER, "null ptr");
  HIP_TRY(hipMalloc(ptr, bytes));
  return Q8_OK;
}

int q8rt_free(void* ptr) {
  HIP_TRY(hipFree(ptr));
  return Q8_OK;
}

int q8rt_memcpy_htod(void* dst, const void* src, size_t bytes) {
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  HIP_TRY(hipDeviceSynchronize());
  return Q8_OK;
}

int q8rt_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return Q8_OK;
}

int q8rt_memcpy_dtod(void* dst, const void* src, size_t bytes) {
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
  HIP_TRY(hipDeviceSynchronize());
  return Q8_OK;
}

int q8rt_memset(void* ptr, int value, size_t bytes) {
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemset(ptr, value, bytes));
  HIP_TRY(hipDeviceSynchronize());
  return Q8_OK;
}

int q8rt_device_synchronize(void) {
  HIP_TRY(hipDeviceSynchronize());
  return Q8_OK;
}

int q8rt_stream_create(void** stream) {
  if (!stream) return fail(Q8_ERR_NULL_POINTER, "null stream");
  hipStream_t s = nullptr;
  HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  *stream = s;
  return Q8_OK;
}

int q8rt_stream_destroy(void* stream) {
  HIP_TRY(hipStreamDestroy(static_cast<hipStream_t>(stream)));
  return Q8_OK;
}

int q8rt_stream_synchronize(void* stream) {
  HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return Q8_OK;
}

int q8rt_event_create(void** event) {
  if (!event) return fail(Q8_ERR_NULL_POINTER, "null event");
  hipEvent_t e = nullptr;
  HIP_TRY(hipEventCreate(&e));
  *event = e;
  return Q8_OK;
}

int q8rt_event_destroy(void* event) {
  HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)));
  return Q8_OK;
}

int q8rt_event_record(void* event, void* stream) {
  HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), static_cast<hipStream_t>(stream)));
  return Q8_OK;
}

int q8rt_event_synchronize(void* event) {
  HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(event)));
  return Q8_OK;
}

int q8rt_event_elapsed_ms(float* ms, void* start, void* stop) {
  if (!ms) return fail(Q8_ERR_NULL_POINTER, "null ms");
  HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
  return Q8_OK;
}

int q8rt_graph_begin_capture(void* stream) {
  HIP_TRY(hipStreamBeginCapture(static_cast<hipStream_t>(stream), hipStreamCaptureModeThreadLocal));
  return Q8_OK;
}

int q8rt_graph_end_capture(void* stream, void** graph_exec) {
  if (!graph_exec) return fail(Q8_ERR_NULL_POINTER, "null graph_exec");
  hipGraph_t graph = nullptr;
  HIP_TRY(hipStreamEndCapture(static_cast<hipStream_t>(stream), &graph));
  hipGraphExec_t exec = nullptr;
  hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
  *graph_exec = exec;
  return Q8_OK;
}

int q8rt_graph_launch(void* graph_exec, void* stream) {
  HIP_TRY(hipGraphLaunch(static_cast<hipGraphExec_t>(graph_exec), static_cast<hipStream_t>(stream)));
  return Q8_OK;
}

int q8rt_graph_destroy(void* graph_exec) {
  HIP_TRY(hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph_exec)));
  return Q8_OK;
}

int q8rt_stream_copy(void* dst, const void* src, size_t bytes, void* stream) {
  if ((!dst || !src) && bytes) return fail(Q8_ERR_NULL_POINTER, "null dst or src");
  if (bytes % 16 || !aligned(dst, 16) || !aligned(src, 16))
    return fail(Q8_ERR_MISALIGNED, "copy needs 16-byte aligned pointers and sizes");
  int rc = check_ready();
  if (rc) return rc;
  int64_t n16 = (int64_t)(bytes / 16);
  int64_t grid = (n16 + 255) / 256;
  if (grid > 8192) grid = 8192;
  if (grid < 1) grid = 1;
  const void* s_arg = src;
  void* d_arg = dst;
  void* args[] = {&s_arg, &d_arg, &n16};
  return launch(g.copy, (uint32_t)grid, 256, args, static_cast<hipStream_t>(stream));
}

int q8rt_stream_read(const void* src, size_t bytes, void* stream) {
  if (!src && bytes) return fail(Q8_ERR_NULL_POINTER, "null src");
  if (bytes % 16 || !aligned(src, 16))
    return fail(Q8_ERR_MISALIGNED, "read needs a 16-byte aligned pointer and size");
  int rc = check_ready();
  if (rc) return rc;
  int64_t n16 = (int64_t)(bytes / 16);
  int64_t grid = (n16 + 255) / 256;
  if (grid > 8192) grid = 8192;
  if (grid < 1) grid = 1;
  const void* s_arg = src;
  void* sink = const_cast<void*>(src);  // written only if a thread's XOR equals `never`
  uint32_t never = 0x9e3779b9u;
  void* args[] = {&s_arg, &sink, &n16, &never};
  return launch(g.read, (uint32_t)grid, 256, args, static_cast<hipStream_t>(stream));
}

int q8rt_time_next_launch(void* start_event, void* stop_event) {
  t_start = static_cast<hipEvent_t>(start_event);
  t_stop = static_cast<hipEvent_t>(stop_event);
  return Q8_OK;
}

}  // extern "C"

namespace {

// A stream, two events and device buffers for a measurement, released on
// every return path (after the stream has drained).
struct CalibScope {
  hipStream_t st = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  void* buf[3] = {nullptr, nullptr, nullptr};
  ~CalibScope() {
    if (st) (void)hipStreamSynchronize(st);
    for (void* b : buf)
      if (b) (void)hipFree(b);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
  }
};

}  // namespace

extern "C" {

int q8rt_launch_cost(int cooperative, int workgroups, int threads, size_t lds_bytes,
                     int launches, float* us_per_launch) {
  if (!us_per_launch) return fail(Q8_ERR_NULL_POINTER, "null output");
  if (workgroups < 1 || workgroups > 65536 || threads < 1 || threads > 1024 ||
      lds_bytes > 160 * 1024 || launches < 1 || launches > 100000)
    return fail(Q8_ERR_BAD_ARGUMENT, "launch shape %d x %d, %zu LDS bytes, %d launches",
                workgroups, threads, lds_bytes, launches);
  int rc = check_ready();
  if (rc) return rc;
  CalibScope c;
  HIP_TRY(hipStreamCreate(&c.st));
  HIP_TRY(hipEventCreate(&c.e0));
  HIP_TRY(hipEventCreate(&c.e1));
  auto one = [&]() -> hipError_t {
    if (cooperative)
      return hipModuleLaunchCooperativeKernel(g.calib_empty, workgroups, 1, 1, threads, 1, 1,
                                              (unsigned)lds_bytes, c.st, nullptr);
    return hipModuleLaunchKernel(g.calib_empty, workgroups, 1, 1, threads, 1, 1,
                                 (unsigned)lds_bytes, c.st, nullptr, nullptr);
  };
  for (int i = 0; i < 16; ++i) HIP_TRY(one());  // warm-up
  HIP_TRY(hipEventRecord(c.e0, c.st));
  for (int i = 0; i < launches; ++i) HIP_TRY(one());
  HIP_TRY(hipEventRecord(c.e1, c.st));
  HIP_TRY(hipEventSynchronize(c.e1));
  float ms = 0.0f;
  HIP_TRY(hipEventElapsedTime(&ms, c.e0, c.e1));
  *us_per_launch = ms * 1e3f / (float)launches;
  return Q8_OK;
}

// Mirrors HandoffArgs in q8gemv_kernels.hip.
struct HandoffArgsHost {
  void* words;
  void* pub;
  void* recv;
  int32_t producers, consumers, n_words, replicas, rounds;
  uint32_t seq, period, spin_limit;
};

int q8rt_handoff_latency(int producers, int consumers, int n_words, int replicas, int rounds,
                         float* latency_us, int* failed) {
  if (!latency_us || !failed) return fail(Q8_ERR_NULL_POINTER, "null output");
  if (producers < 1 || consumers < 1 || producers + consumers > 512 || n_words < 1 ||
      n_words > 4096 || n_words % producers != 0 || replicas < 1 || replicas > 16 ||
      rounds < 1 || rounds > 255)
    return fail(Q8_ERR_BAD_ARGUMENT,
                "hand-off of %d words (%d replicas) from %d to %d workgroups over %d rounds",
                n_words, replicas, producers, consumers, rounds);
  int rc = check_ready();
  if (rc) return rc;
  static std::atomic<uint32_t> calls{0};
  CalibScope c;
  HIP_TRY(hipStreamCreate(&c.st));
  const size_t wbytes = ((size_t)replicas * n_words + 1) * 8;
  HIP_TRY(hipMalloc(&c.buf[0], wbytes));
  HIP_TRY(hipMalloc(&c.buf[1], (size_t)rounds * producers * 4));
  HIP_TRY(hipMalloc(&c.buf[2], (size_t)rounds * consumers * 4));
  HIP_TRY(hipMemsetAsync(c.buf[0], 0, wbytes, c.st));
  HIP_TRY(hipMemsetAsync(c.buf[1], 0, (size_t)rounds * producers * 4, c.st));
  HIP_TRY(hipMemsetAsync(c.buf[2], 0, (size_t)rounds * consumers * 4, c.st));
  HandoffArgsHost a{c.buf[0], c.buf[1], c.buf[2], producers, consumers, n_words, replicas, rounds,
                    1u + (calls.fetch_add(1) & 0xffffu), 2000u /* 20 us */, 1u << 16};
  void* args[] = {&a};
  HIP_TRY(hipModuleLaunchKernel(g.calib_handoff, producers + consumers, 1, 1, 256, 1, 1, 0, c.st,
                                args, nullptr));
  std::vector<uint32_t> pub((size_t)rounds * producers), recv((size_t)rounds * consumers);
  HIP_TRY(hipMemcpyAsync(pub.data(), c.buf[1], pub.size() * 4, hipMemcpyDeviceToHost, c.st));
  HIP_TRY(hipMemcpyAsync(recv.data(), c.buf[2], recv.size() * 4, hipMemcpyDeviceToHost, c.st));
  HIP_TRY(hipStreamSynchronize(c.st));
  int bad = 0;
  for (int r = 0; r < rounds; ++r) {
    uint32_t last = 0;
    bool have = true;
    for (int p = 0; p < producers; ++p) {
      const uint32_t v = pub[(size_t)r * producers + p];
      if (v == 0) have = false;
      if (p == 0 || (int32_t)(v - last) > 0) last = v;
    }
    for (int q = 0; q < consumers; ++q) {
      const uint32_t v = recv[(size_t)r * consumers + q];
      float& out = latency_us[(size_t)r * consumers + q];
      if (!have || v == 0) {
        out = std::numeric_limits<float>::quiet_NaN();
        ++bad;
      } else {
        out = (float)(int32_t)(v - last) * 0.01f;  // 10 ns ticks
      }
    }
  }
  *failed = bad;
  return Q8_OK;
}

int q8rt_memory_latency(int hops, float* ns_per_load, int* xcds) {
  if (!ns_per_load || !xcds) return fail(Q8_ERR_NULL_POINTER, "null output");
  if (hops < 16 || hops > 65536)
    return fail(Q8_ERR_BAD_ARGUMENT, "%d hops outside [16, 65536]", hops);
  int rc = check_ready();
  if (rc) return rc;
  // A cycle through `hops` distinct 128-byte lines of a 64 MiB region, in a
  // fixed pseudo-random order starting (and ending) at line 0.
  constexpr uint32_t kWords = 16u << 20;  // 64 MiB of u32
  constexpr uint32_t kLines = kWords / 32;
  constexpr size_t kScrub = (size_t)1 << 30;
  std::vector<uint32_t> line(kLines);
  for (uint32_t i = 0; i < kLines; ++i) line[i] = i;
  uint64_t st = 0x9e3779b97f4a7c15ull;
  for (uint32_t i = kLines - 1; i > 1; --i) {  // shuffle lines 1.. (line 0 starts the cycle)
    st = st * 6364136223846793005ull + 1442695040888963407ull;
    const uint32_t j = 1 + (uint32_t)((st >> 33) % i);
    std::swap(line[i], line[j]);
  }
  std::vector<uint32_t> next(kWords, 0u);
  for (int h = 0; h < hops; ++h) next[(size_t)line[h] * 32] = line[(h + 1) % hops] * 32;
  CalibScope c;
  HIP_TRY(hipStreamCreate(&c.st));
  HIP_TRY(hipMalloc(&c.buf[0], (size_t)kWords * 4));
  HIP_TRY(hipMalloc(&c.buf[1], kScrub));
  HIP_TRY(hipMalloc(&c.buf[2], 64 * 4));  // ticks [0, 8), XCD ids [16, 24)
  HIP_TRY(hipMemcpyAsync(c.buf[0], next.data(), (size_t)kWords * 4, hipMemcpyHostToDevice, c.st));
  HIP_TRY(hipMemsetAsync(c.buf[1], 0, kScrub, c.st));
  uint32_t* ticks = static_cast<uint32_t*>(c.buf[2]);
  uint32_t host[24];
  auto chase = [&](int passes, int xcd) -> int {
    HIP_TRY(hipMemsetAsync(c.buf[2], 0xff, 64 * 4, c.st));
    const void* n_arg = c.buf[0];
    uint32_t mask = kWords - 1;
    int h_arg = hops, p_arg = passes, x_arg = xcd;
    uint32_t* t_arg = ticks;
    uint32_t* x_out = ticks + 16;
    void* args[] = {&n_arg, &mask, &h_arg, &p_arg, &x_arg, &t_arg, &x_out};
    // one workgroup per XCD (workgroups go to the XCDs in turn)
    HIP_TRY(hipModuleLaunchKernel(g.calib_chase, 8, 1, 1, 64, 1, 1, 0, c.st, args, nullptr));
    HIP_TRY(hipMemcpyAsync(host, c.buf[2], sizeof(host), hipMemcpyDeviceToHost, c.st));
    HIP_TRY(hipStreamSynchronize(c.st));
    return Q8_OK;
  };
  const float nan = std::numeric_limits<float>::quiet_NaN();
  auto per_load = [&](uint32_t t) { return t == 0xffffffffu ? nan : (float)t * 10.0f / hops; };
  // 1 GiB read (4x the memory-side cache): neither L2 nor the MALL holds a
  // line of the cycle; then pass 1 from HBM, pass 2 from this XCD's L2
  if ((rc = q8rt_stream_read(c.buf[1], kScrub, c.st))) return rc;
  if ((rc = chase(2, -1))) return rc;
  ns_per_load[0] = per_load(host[0]);
  ns_per_load[2] = per_load(host[1]);
  const int x0 = host[2] == 0xffffffffu ? -1 : (int)host[2];
  xcds[0] = x0;
  // the same lines from another XCD, whose L2 never saw them: the MALL
  ns_per_load[1] = nan;
  xcds[1] = -1;
  if (x0 >= 0) {
    if ((rc = chase(1, (x0 + 1) % 8))) return rc;
    ns_per_load[1] = per_load(host[0]);
    xcds[1] = host[1] == 0xffffffffu ? -1 : (int)host[1];
  }
  return Q8_OK;
}

}  // extern "C"

// ------------------------------------------------------------ decode step

namespace {

constexpr int kLayers = 28;
constexpr int kVocabRows = 151936;
constexpr int64_t kKvRow = 8 * 128;  // f16 elements per cache slot
constexpr int kKvHeads = 8;
// attention workgroups (partials) per kv head at most: 16 above kAttnShortCtx positions, else 8
constexpr int kAttnGroupsHost = 16;
constexpr int32_t kGenerateBatch = 4;  // tokens between EOS checks (qwen3_full.mlir:1412)


// Scratch layout (bytes).  Key + status first; every region 256-byte aligned.
constexpr size_t kScrKey = 0;        // u64 argmax key
constexpr size_t kScrStatus = 8;     // u32 status
constexpr size_t kScrHA = 256;       // f16[1024]
constexpr size_t kScrHB = kScrHA + 2048;
constexpr size_t kScrRes = kScrHB + 2048;
constexpr size_t kScrQ = kScrRes + 2048;     // f16[2048]
constexpr size_t kScrK = kScrQ + 4096;       // f16[1024]
constexpr size_t kScrV = kScrK + 2048;       // f16[1024]
constexpr size_t kScrAttn = kScrV + 2048;    // f16[2048]
constexpr size_t kScrAct = kScrAttn + 4096;  // f16[3072]
constexpr size_t kScrXn = kScrAct + 6144;    // f16[1024] rms_norm(h, attn_norm)
constexpr size_t kScrQr = kScrXn + 2048;     // f16[2048] q after head norm + RoPE
constexpr size_t kScrFn = kScrQr + 4096;     // f16[1024] rms_norm(res, ffn_norm)
constexpr size_t kScrOn = kScrFn + 2048;     // f16[1024] rms_norm(h, output_norm)
constexpr size_t kScrPart = kScrOn + 2048;   // f32[16][16][132] attention partials
constexpr size_t kScrSeq = 16;       // u32 step sequence number (single-launch step)
constexpr size_t kScrStarted = 128;  // u32 the last launch whose grid was resident
// tagged words of the single-launch step (u64; map in decode_kernels.hip)
// the single-launch step's tagged words per layer parity: h, attention output,
// attn_o + residual output and SwiGLU output in 4 replicas each, q/k/v and
// the attention partials once (layout in decode_kernels.hip)
constexpr size_t kStepWordsParity = 4 * 512 + 1024 + 512 + 512 + 16 * 16 * 130 + 4 * 1024 +
                                    4 * 512 + 4 * 1536;
constexpr size_t kStepWords = 2 * kStepWordsParity + 2 * kStepWgs + kStepExtra;
constexpr size_t kScrWords = (kScrPart + 16 * kAttnGroupsHost * 132 * 4 + 255) / 256 * 256;
constexpr size_t kScrBytes = kScrWords + kStepWords * 8;


const uint8_t* cb(const void* p) { return static_cast<const uint8_t*>(p); }
uint8_t* mb(void* p) { return static_cast<uint8_t*>(p); }

// Kernel argument of dec_step (decode_kernels.hip, same member order).
struct StepParams {
  const void* token_embd;
  const void* attn_norm;
  const void* ffn_norm;
  const void* q_norm;
  const void* k_norm;
  const void* wq;
  const void* wk;
  const void* wv;
  const void* wo;
  const void* wgu;
  const void* wdn;
  const void* output_norm;
  const void* output_w;
  void* k_cache;
  void* v_cache;
  const int32_t* token_in;
  int32_t* token_out;
  int32_t* pos;
  void* logits;
  int32_t* out;
  void* words;
  void* seq;
  void* last_started;
  void* status;
  void* on_out;
  void* stamps;
  int32_t max_seq;
  int32_t advance;
  int32_t head;
  uint32_t spin_limit;
};

// One single-launch decode step (dec_step), ordered after the last one
// launched on any other stream (see State::step_ev; not under graph capture,
// where the caller orders its graphs).
int launch_step(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                const int32_t* token_in, int32_t* token_out, int32_t* pos, void* logits,
                int32_t* out, int advance, int head, void* scratch, hipStream_t st) {
  StepParams p;
  p.token_embd = w->token_embd;
  p.attn_norm = w->attn_norm;
  p.ffn_norm = w->ffn_norm;
  p.q_norm = w->q_norm;
  p.k_norm = w->k_norm;
  p.wq = w->wq;
  p.wk = w->wk;
  p.wv = w->wv;
  p.wo = w->wo;
  p.wgu = w->wgu;
  p.wdn = w->wdn;
  p.output_norm = w->output_norm;
  p.output_w = w->output_w;
  p.k_cache = k_cache;
  p.v_cache = v_cache;
  p.token_in = token_in;
  p.token_out = token_out;
  p.pos = pos;
  p.logits = logits;
  p.out = out;
  p.words = mb(scratch) + kScrWords;
  p.seq = mb(scratch) + kScrSeq;
  p.last_started = mb(scratch) + kScrStarted;
  p.status = mb(scratch) + kScrStatus;
  p.on_out = mb(scratch) + kScrOn;
  p.stamps = mb(scratch) + kScrPart;  // unused by this step unless built with timestamps
  p.max_seq = (int32_t)max_seq;
  p.advance = advance ? 1 : 0;
  p.head = head ? 1 : 0;
  p.spin_limit = g.step_spin_limit.load(std::memory_order_relaxed);
  if (g.force_abort_in.load(std::memory_order_relaxed) >= 0 && g.force_abort_in.fetch_sub(1) == 0)
    p.spin_limit = 0;  // the test hook: workgroup 0 gives up at its start
  void* args[] = {&p};
  const uint32_t grid = (uint32_t)step_grid(max_seq);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  HIP_TRY(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone) {
    hipError_t e = hipModuleLaunchKernel(g.dec_step, grid, 1, 1, 256, 1, 1, 0, st, args,
                                         nullptr);
    if (e != hipSuccess) return hip_fail(e, "launch of dec_step");
    return Q8_OK;
  }
  std::lock_guard<std::mutex> lock(g.step_mu);
  // The event only orders launches on this device, so it records without a
  // system-scope fence (the default fence, an L2 writeback, measured 3 us
  // per step; without it 1 us).
  if (g.step_ev == nullptr)
    HIP_TRY(hipEventCreateWithFlags(&g.step_ev, hipEventDisableTiming | hipEventDisableSystemFence));
  else if (g.step_last != st)
    HIP_TRY(hipStreamWaitEvent(st, g.step_ev, 0));
  hipError_t e = hipModuleLaunchKernel(g.dec_step, grid, 1, 1, 256, 1, 1, 0, st, args,
                                       nullptr);
  if (e != hipSuccess) return hip_fail(e, "launch of dec_step");
  HIP_TRY(hipEventRecord(g.step_ev, st));
  g.step_last = st;
  return Q8_OK;
}

// Whether a step over a cache of max_seq positions runs as one launch: the mode
// asks for it and the device holds the grid (per phase otherwise, the same bits).
bool use_single(int64_t max_seq) {
  return g.step_single.load(std::memory_order_relaxed) == 1 && g.dec_step != nullptr &&
         g.step_slots >= step_grid(max_seq);
}

// Status bit 1 of a scratch: a single-launch step gave up waiting for a
// hand-off (its outputs are not valid).  Reads the word on `st` (which the
// caller has just synchronized or is about to: the copy is stream-ordered).
int check_not_aborted(void* scratch, hipStream_t st, const char* when) {
  uint32_t status = 0;
  HIP_TRY(hipMemcpyAsync(&status, mb(scratch) + kScrStatus, sizeof(status),
                         hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (status & 2u)
    return fail(Q8_ERR_STEP_ABORTED,
                "%s: a single-launch decode step gave up waiting for a hand-off (status bit 1); "
                "its outputs are invalid; qwen3_scratch_reset clears the scratch", when);
  return Q8_OK;
}

// The status word of a scratch, read on `st` after everything before it.
int read_status(const void* scratch, hipStream_t st, uint32_t* status) {
  *status = 0;
  HIP_TRY(hipMemcpyAsync(status, cb(scratch) + kScrStatus, sizeof(*status), hipMemcpyDeviceToHost,
                         st));
  HIP_TRY(hipStreamSynchronize(st));
  return Q8_OK;
}

// After a single-launch step gave up (status bit 1: its outputs are invalid,
// it wrote neither token nor position, and every single launch queued behind
// it on this scratch returned at its start): bit 1 cleared and bit 2 (a step
// was re-run per phase) set on `st`, which is then synchronized, so the
// caller can re-run the steps that did nothing with the per-phase launches
// (the same bits).  Counts the fallback.
int recover_from_abort(void* scratch, hipStream_t st, uint32_t status) {
  const uint32_t v = (status & ~2u) | 4u;
  HIP_TRY(hipMemcpyAsync(mb(scratch) + kScrStatus, &v, sizeof(v), hipMemcpyHostToDevice, st));
  HIP_TRY(hipStreamSynchronize(st));
  g.step_fallbacks.fetch_add(1);
  return Q8_OK;
}

int check_decode_ready() {
  int rc = check_ready();
  if (rc) return rc;
  if (!g.dec_module)
    return fail(Q8_ERR_CODE_OBJECT, "decode_gfx950.hsaco was not found or lacks a kernel");
  return Q8_OK;
}

int validate_weights(const qwen3_weights* w) {
  if (!w) return fail(Q8_ERR_NULL_POINTER, "null weights struct");
  const void* ptrs[] = {w->token_embd, w->attn_norm, w->ffn_norm, w->q_norm, w->k_norm,
                        w->wq,         w->wk,        w->wv,       w->wo,     w->wgu,
                        w->wdn,        w->output_norm, w->output_w};
  for (const void* p : ptrs) {
    if (!p) return fail(Q8_ERR_NULL_POINTER, "null weight pointer");
    if (!aligned(p, 16)) return fail(Q8_ERR_MISALIGNED, "weights must be 16-byte aligned");
  }
  if (w->prefill_f16 && !aligned(w->prefill_f16, 256))
    return fail(Q8_ERR_MISALIGNED, "prefill_f16 must be 256-byte aligned");
  return Q8_OK;
}

int validate_cache(void* k_cache, void* v_cache, int64_t max_seq) {
  if (!k_cache || !v_cache) return fail(Q8_ERR_NULL_POINTER, "null KV cache");
  if (!aligned(k_cache, 16) || !aligned(v_cache, 16))
    return fail(Q8_ERR_MISALIGNED, "KV cache must be 16-byte aligned");
  if (max_seq < 1 || max_seq > (1LL << 24))
    return fail(Q8_ERR_BAD_SHAPE, "max_seq %lld outside [1, 2^24]", (long long)max_seq);
  return Q8_OK;
}

int launch_layer(const qwen3_weights* w, int layer, void* k_cache, void* v_cache, int64_t max_seq,
                 const int32_t* pos, const void* h_in, void* h_out, void* scratch,
                 hipStream_t st) {
  const int64_t bpl_q = 2048LL * 1024 / 32 * 34, bpl_kv = 1024LL * 1024 / 32 * 34;
  const int64_t bpl_o = 1024LL * 2048 / 32 * 34, bpl_gu = 6144LL * 1024 / 32 * 34;
  const int64_t bpl_dn = 1024LL * 3072 / 32 * 34;
  const void* wq = cb(w->wq) + layer * bpl_q;
  const void* wk = cb(w->wk) + layer * bpl_kv;
  const void* wv = cb(w->wv) + layer * bpl_kv;
  const void* wo = cb(w->wo) + layer * bpl_o;
  const void* wgu = cb(w->wgu) + layer * bpl_gu;
  const void* wdn = cb(w->wdn) + layer * bpl_dn;
  const void* an = cb(w->attn_norm) + layer * 2048;
  const void* fn = cb(w->ffn_norm) + layer * 2048;
  const void* qn = cb(w->q_norm) + layer * 256;
  const void* kn = cb(w->k_norm) + layer * 256;
  void* kc = mb(k_cache) + (int64_t)layer * max_seq * kKvRow * 2;
  void* vc = mb(v_cache) + (int64_t)layer * max_seq * kKvRow * 2;
  void* q = mb(scratch) + kScrQ;
  void* k = mb(scratch) + kScrK;
  void* v = mb(scratch) + kScrV;
  void* attn = mb(scratch) + kScrAttn;
  void* res = mb(scratch) + kScrRes;
  void* act = mb(scratch) + kScrAct;
  void* part = mb(scratch) + kScrPart;
  void* xn = mb(scratch) + kScrXn;
  void* qr = mb(scratch) + kScrQr;
  void* fnx = mb(scratch) + kScrFn;
  const void* hin = h_in;
  int ms = (int)max_seq;
  int rc;
  {
    void* args[] = {&wq, &wk, &wv, &hin, &an, &q, &k, &v, &xn};
    if ((rc = launch(g.dec_qkv, 1024, 64, args, st))) return rc;
  }
  {
    const void* pp = pos;
    void* args[] = {&q, &k, &v, &qn, &kn, &pp, &ms, &kc, &vc, &part, &qr};
    if ((rc = launch(g.dec_attn, 8 * kAttnGroupsHost, 256, args, st))) return rc;
  }
  {
    const void* pp = pos;
    void* args[] = {&wo, &part, &hin, &res, &attn, &pp, &ms};
    if ((rc = launch(g.dec_o, 64, 256, args, st))) return rc;
  }
  {
    void* args[] = {&wgu, &res, &fn, &act, &fnx};
    if ((rc = launch(g.dec_gu, 768, 64, args, st))) return rc;
  }
  {
    void* args[] = {&wdn, &act, &res, &h_out};
    if ((rc = launch(g.dec_dn, 256, 64, args, st))) return rc;
  }
  return Q8_OK;
}

int launch_head(const qwen3_weights* w, const void* h, void* logits, int32_t* token,
                int32_t* pos, int advance, int64_t max_seq, void* scratch, hipStream_t st,
                int32_t* out = nullptr) {
  const void* W = w->output_w;
  const void* on = w->output_norm;
  void* ws = mb(scratch) + kScrKey;
  void* status = mb(scratch) + kScrStatus;
  void* xn = mb(scratch) + kScrOn;
  int rc;
  {
    void* args[] = {&W, &h, &on, &logits, &ws, &xn};
    if ((rc = launch(g.dec_vocab, (uint32_t)vocab_grid(), 256, args, st))) return rc;
  }
  int adv = advance ? 1 : 0;
  int ms = (int)max_seq;
  void* args[] = {&ws, &token, &pos, &adv, &ms, &status, &out};
  return launch(g.dec_final, 1, 64, args, st);
}

int launch_embed(const qwen3_weights* w, const int32_t* token, void* h, hipStream_t st) {
  const void* t = token;
  const void* e = w->token_embd;
  void* args[] = {&t, &e, &h};
  return launch(g.dec_embed, 1, 128, args, st);
}

// Embedding of *token_in, the 28 layers at *pos; the final hidden state is
// left in the scratch's h_a.
int launch_body(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                const int32_t* token_in, const int32_t* pos, void* scratch, hipStream_t st,
                void** h_final) {
  void* ha = mb(scratch) + kScrHA;
  void* hb = mb(scratch) + kScrHB;
  int rc = launch_embed(w, token_in, ha, st);
  if (rc) return rc;
  for (int l = 0; l < kLayers; ++l) {
    if ((rc = launch_layer(w, l, k_cache, v_cache, max_seq, pos, ha, hb, scratch, st))) return rc;
    std::swap(ha, hb);
  }
  *h_final = ha;
  return Q8_OK;
}

// ---- batched prompt ingestion ----

// What the q/k/v products write (layout shared with prefill_kernels.hip).
struct QkvOut {
  void *q, *k, *v, *q_roped, *k_cache, *v_cache;
  const void *qn_w, *kn_w, *rope;
  int start;
};

// Argument block of pf_gemm_q8* (layout shared with prefill_kernels.hip).
struct GemmArgs {
  const void* x;
  const void* w;
  void* y;
  const void* r;
  int M, K;
  int n_tiles;
  int ldx, ldy, ldr;
  int up_row;
  const void *wk, *wv;  // q/k/v: the further weights
  QkvOut qkv;
  float* part;  // split-K partial sums (pf_gemm_q8_part*)
  int splits;
};

// Workspace regions, f16 elements per token: h, h1 (residual), xn
// (rms_norm(h, attn_norm)), q, k, v, q_roped, attention output, SwiGLU
// output, fn (rms_norm(h1, ffn_norm)).
// Then the attention's split partials (f32 slots of kPfAttnSlotFloats for
// pf_attn_pair_cap(n) pairs x 8 kv heads), then the RoPE table (per token
// the 64 cosines, then the 64 sines, f32).
constexpr int kPfTokenRegions = 10;
constexpr int kPfRegions = 12;
constexpr int kPfRopeRegion = 11;
constexpr int kPfCols[kPfTokenRegions] = {1024, 1024, 1024, 2048, 1024, 1024, 2048, 2048, 3072, 1024};
constexpr int32_t kPfMaxTokens = 1 << 20;

// (query block, split) pairs the partial slots hold: 2 per query block + 64
int64_t pf_attn_pair_cap(int32_t n) { return 2LL * ((n + 31) / 32) + 64; }

size_t pf_region_bytes(int32_t n, int i) {
  size_t b;
  if (i < kPfTokenRegions)
    b = (size_t)n * kPfCols[i] * 2;
  else if (i == kPfRopeRegion)
    b = (size_t)n * 128 * 4;
  else
    b = (size_t)pf_attn_pair_cap(n) * kKvHeads * kPfAttnSlotFloats * 4;
  return (b + 255) / 256 * 256;
}

// Positions per attention split, in blocks of 32.  A query block's positions
// are walked one block after another (about 0.6 us each), so without splits
// the longest query block sets the time; each split costs a partial written
// and merged, and the first one the merge's launch.  nb = blocks of the longest
// query block.
//   No splits up to nb = 8, or 16 from 8 query blocks on (256 workgroups with
//   the 8 kv heads): 300 tokens from position 0 (nb 10) 67.9 us a layer
//   against 69.8 with splits of 8, 512 tokens (16) 69.9 against 70.2.
//   From 32 query blocks on (1000 tokens) a third of nb, at least 8: flat
//   within 2 % over 2 .. 32 blocks (1021 tokens 105.3 at 8, 2048 tokens 176.3
//   at 22).
//   Between, about 0.6 sqrt(nb), which balances the walk against the merge, at
//   least 2, or 8 from 8 query blocks on.  Layer, against a third of nb: 1
//   token after 300 / 1000 / 6000 positions 33.6 / 35.6 / 73.0 -> 29.4 / 32.2
//   / 39.8 us, 33 tokens 40.2 / 47.2 (1700) / 79.0 -> 36.5 / 40.4 / 47.9, 100
//   tokens after 6000 85.2 -> 60.0, 300 after 6000 114.6 -> 101.5.
// Raised where the partial slots would not hold the splits.
int32_t pf_attn_split_default(int32_t nqb, int32_t nb) {
  if (nb <= (nqb >= 8 ? 16 : 8)) return nb;
  if (nqb >= 32) return std::max(8, (nb + 2) / 3);
  int32_t s = nqb >= 8 ? 8 : 2;
  while (25LL * s * s < 9LL * nb) ++s;
  return s;
}

int32_t pf_attn_split_blocks(int32_t n, int32_t p0, int chunk_local) {
  const PfSplitGeometry G = pf_split_geometry(n, p0, chunk_local ? p0 : 0);
  const int64_t cap = pf_attn_pair_cap(n);
  const int32_t nb_max = std::max(G.nb_last, G.c + G.nqb - 2);
  const int32_t set_split = g.pf_attn_split.load(std::memory_order_relaxed);
  const int32_t s0 = set_split > 0 ? set_split : pf_attn_split_default(G.nqb, nb_max);
  int32_t lo_s = std::min(s0, nb_max), hi_s = nb_max;
  // smallest S >= lo_s whose pairs fit (at S = nb_max there are nqb pairs)
  while (lo_s < hi_s) {
    const int32_t mid = lo_s + (hi_s - lo_s) / 2;
    if (pf_pairs_total(G, mid) <= cap)
      hi_s = mid;
    else
      lo_s = mid + 1;
  }
  return lo_s;
}

size_t pf_workspace_bytes(int32_t n) {
  size_t b = 0;
  for (int i = 0; i < kPfRegions; ++i) b += pf_region_bytes(n, i);
  return b;
}

// fn covers 64 tokens per workgroup; fn_m32 (may be null) the same product
// over 32 tokens (same operations per output element, so the same bits).  The
// 32-token tile is used where the 64-token grid would leave the device with
// fewer than 2 workgroups per CU.
int launch_gemm(hipFunction_t fn, hipFunction_t fn_m32, const void* x, int ldx, const void* wl,
                int K, int n_out, int tile_cols, void* y, int ldy, const void* r, int ldr,
                int up_row, int M, hipStream_t st, float* part = nullptr, int splits = 1,
                const void* wk = nullptr, const void* wv = nullptr, const QkvOut* qkv = nullptr) {
  GemmArgs a{x, wl, y, r, M, K, n_out / tile_cols, ldx, ldy, ldr, up_row, wk, wv,
             qkv ? *qkv : QkvOut{}, part, splits};
  // the kernel maps workgroups to n tiles in groups of 8 (one per XCD)
  if (n_out % tile_cols != 0 || a.n_tiles % 8 != 0 || K % 256 != 0)
    return fail(Q8_ERR_BAD_SHAPE, "prefill GEMM shape N=%d K=%d", n_out, K);
  int rows = 64;
  if (fn_m32) {
    const int set_rows = g.pf_tile_rows.load(std::memory_order_relaxed);
    if (set_rows == 32)
      rows = 32;
    else if (set_rows == 0 && ((int64_t)M + 63) / 64 * a.n_tiles < 2LL * g.compute_units)
      rows = 32;
  }
  if (rows == 32) fn = fn_m32;
  const int64_t mt = ((int64_t)M + rows - 1) / rows;
  const int64_t grid = mt * a.n_tiles * splits;
  if (grid > 0x7fffffff) return fail(Q8_ERR_BAD_SHAPE, "prefill GEMM grid too large");
  void* args[] = {&a};
  return launch(fn, (uint32_t)grid, 256, args, st);
}

// Argument block of pf_gemm_f16* (layout shared with prefill_kernels.hip).
struct GemmF16Args {
  const void* x;
  const void* w;
  void* y;
  const void* r;
  float* part;
  int M, K;
  int n_tiles;
  int ldx, ldy, ldr;
  int splits;
  QkvOut qkv;
};

// The f16 layer matrices (qwen3_weights.prefill_f16), f16 elements per
// layer: q/k/v rows [4096, 1024] (q rows, then k, then v), attn_o [1024,
// 2048], gate/up [6144, 1024] in groups of 16 gate rows + the matching 16 up
// rows, ffn_down [1024, 3072].
constexpr int64_t kPfF16Qkv = 0;
constexpr int64_t kPfF16O = 4096LL * 1024;
constexpr int64_t kPfF16Gu = kPfF16O + 1024LL * 2048;
constexpr int64_t kPfF16Dn = kPfF16Gu + 6144LL * 1024;
constexpr int64_t kPfF16Layer = kPfF16Dn + 1024LL * 3072;
constexpr size_t kPfF16Bytes = (size_t)kLayers * kPfF16Layer * 2;

struct F16Tile {
  hipFunction_t fn;
  int bm, bn;   // token rows x W rows per workgroup
  int ks;       // k per stage (K per split must be a multiple)
  int per_cu;   // chosen when the grid gives every CU at least this many workgroups
  int threads = 256;
};

// One pf_gemm_f16* launch.  Tile: the first of `tiles` whose grid gives every
// CU at least its per_cu workgroups (the last one regardless); a gemm_rows
// setting (qwen3_set_prefill_tiling) picks the first tile of that many token
// rows instead (the next larger where the GEMM has none).  Every tile gives
// the same bits.
int launch_gemm_f16(std::initializer_list<F16Tile> tiles, const void* x, int ldx, const void* wm,
                    int K, int n_w, void* y, int ldy, const void* r, int ldr, int M,
                    hipStream_t st, float* part = nullptr, int splits = 1,
                    const QkvOut* qkv = nullptr) {
  auto grid_of = [&](const F16Tile& t) {
    return ((int64_t)M + t.bm - 1) / t.bm * (n_w / t.bn) * splits;
  };
  const F16Tile* pick = nullptr;
  const int set_rows = g.pf_tile_rows.load(std::memory_order_relaxed);
  if (set_rows > 0) {
    for (const F16Tile& t : tiles)
      if (t.bm >= set_rows && (!pick || t.bm < pick->bm)) pick = &t;
  } else {
    for (const F16Tile& t : tiles)
      if (!pick && grid_of(t) >= (int64_t)t.per_cu * g.compute_units) pick = &t;
  }
  if (!pick) pick = tiles.end() - 1;
  const int bn = pick->bn;
  // the kernel maps workgroups to n tiles in groups of 8 (one per XCD)
  if (n_w % (8 * bn) != 0 || splits < 1 || K % (pick->ks * splits) != 0)
    return fail(Q8_ERR_BAD_SHAPE, "prefill f16 GEMM shape N=%d K=%d splits=%d", n_w, K, splits);
  GemmF16Args a{x, wm, y, r, part, M, K, n_w / bn, ldx, ldy, ldr, splits,
                qkv ? *qkv : QkvOut{}};
  const int64_t grid = grid_of(*pick);
  if (grid > 0x7fffffff) return fail(Q8_ERR_BAD_SHAPE, "prefill GEMM grid too large");
  void* args[] = {&a};
  return launch(pick->fn, (uint32_t)grid, (uint32_t)pick->threads, args, st);
}

// y = r + x W^T for N = 1024 (attn_o, ffn_down).  Where 32-token tiles would
// leave CUs idle (short prompts), K is split into equal ranges of whole stages
// (the fewest that fill the CUs), each range's f32 sums go to `part`, and
// pf_res_reduce adds them in order with the residual; where they fill the CUs
// once but not twice (about 512-1023 tokens), K is split in two, since one
// workgroup per CU walking all of K hides too little load latency; where
// 128 x 128 tiles cover the CUs once in two K ranges but not in one (about
// 2048-4095 tokens), K is split in two for those tiles (over f16 weights 513
// to 2560 tokens instead finish in one launch, see below).  The split
// count depends on M only, so every token tile gives the same bits.  With
// norm_w set and K split, the reduce also writes norm_out = rms_norm(y,
// norm_w) (pf_res_reduce_norm, the bits of a separate pf_rmsnorm) and
// *normed becomes true; otherwise the caller runs the norm itself.
int launch_gemm_res(const void* x, int ldx, const void* wl, int K, void* y, const void* r,
                    int M, void* part, size_t part_bytes, hipStream_t st,
                    const void* norm_w = nullptr, void* norm_out = nullptr,
                    bool* normed = nullptr, const void* wf16 = nullptr) {
  if (normed) *normed = false;
  constexpr int kN = 1024;
  const int n_tiles = kN / 64;
  const int stages = K / 256;
  int splits = 1;
  const int64_t wgs32 = ((int64_t)M + 31) / 32 * n_tiles;
  const int64_t wgs128 = ((int64_t)M + 127) / 128 * (kN / 128);
  if (g.pf_gemm_part && g.pf_gemm_part_m32 && g.pf_res_reduce) {
    if (wgs32 < g.compute_units) {
      splits = stages;
      for (int d = 1; d <= stages; ++d)
        if (stages % d == 0 && wgs32 * d >= g.compute_units) {
          splits = d;
          break;
        }
    } else if (wgs32 < 2 * g.compute_units && stages % 2 == 0) {
      splits = 2;
    } else if (wgs128 < g.compute_units && 2 * wgs128 >= g.compute_units && stages % 2 == 0) {
      splits = 2;
    }
    if ((size_t)splits * M * kN * 4 > part_bytes) splits = 1;
  }
  // One round of workgroups that finish their outputs themselves, where there
  // is such a grid (figures beside the kernels; whole prompts of 640 / 1021
  // tokens with other weights each time 2527 / 2922 -> 2336 / 2761 us, ffn_down
  // alone 2416 / 2823); a norm that follows is the caller's.  The 128 x 64
  // kernel, one workgroup a CU, also where a second round is at most a quarter
  // full (2049 to 2560 tokens on 256 CUs): layer of 2049 / 2304 / 2560 tokens
  // 201 / 226 / 239 us against 210 / 232 / 246 with the split product, prompt of
  // 2049 5.67 against 5.79 ms.  Fuller second rounds win a layer by itself (2561
  // / 3072 / 3500 tokens 245 / 277 / 323 against 251 / 280 / 319) but no prompt,
  // whose weights come from HBM (2560 / 2688 / 3072 tokens 6.78 / 7.01 / 7.76
  // against 6.79 / 7.00 / 7.60 ms).
  if (wf16 && splits <= 2 && g.pf_tile_rows.load(std::memory_order_relaxed) == 0) {
    const int64_t wgs64 = ((int64_t)M + 63) / 64 * (kN / 64);
    const int64_t wgs128n = ((int64_t)M + 127) / 128 * (kN / 64);
    const int k = K == 2048 ? 0 : 1;
    if (M > 512 && wgs64 <= g.compute_units)
      return launch_gemm_f16({{g.pf_f16_res_pipe[0][k][splits - 1], 64, 64, 64, 0}}, x, ldx, wf16,
                             K, kN, y, kN, r, kN, M, st);
    if (M > 512 && 4 * wgs128n <= 5LL * g.compute_units)
      return launch_gemm_f16({{g.pf_f16_res_pipe[1][k][splits - 1], 128, 64, 64, 0, 512}}, x, ldx,
                             wf16, K, kN, y, kN, r, kN, M, st);
  }
  // with a norm to form, even an unsplit K goes through the f32 sums and the
  // reduce (which adds the residual exactly as the GEMM epilogue would):
  // 1024 tokens 4.24 -> 4.13 ms, 2048 tokens 7.69 -> 7.61 ms
  if (splits == 1 && !(norm_w && g.pf_gemm_part && (size_t)M * kN * 4 <= part_bytes)) {
    if (wf16)
      return launch_gemm_f16({{g.pf_f16_res_22, 64, 64, 128, 2},
                              {g.pf_f16_res_12k, 32, 64, 256, 0}},
                             x, ldx, wf16, K, kN, y, kN, r, kN, M, st);
    return launch_gemm(g.pf_gemm_res, g.pf_gemm_res_m32, x, ldx, wl, K, kN, 64, y, kN, r, kN, 0,
                       M, st);
  }
  int rc = wf16 ? launch_gemm_f16({{g.pf_f16_part_44k, 128, 128, 128, 1},
                                   {g.pf_f16_part_22, 64, 64, 128, 2},
                                   {g.pf_f16_part_22k, 64, 64, 256, 1},
                                   {g.pf_f16_part_12k, 32, 64, 256, 0}},
                                  x, ldx, wf16, K, kN, nullptr, kN, nullptr, 0, M, st,
                                  static_cast<float*>(part), splits)
                : launch_gemm(g.pf_gemm_part, g.pf_gemm_part_m32, x, ldx, wl, K, kN, 64, nullptr,
                              kN, nullptr, 0, 0, M, st, static_cast<float*>(part),
                              splits);
  if (rc) return rc;
  const void* pp = part;
  int sp = splits, mm = M, nn = kN, ld = kN;
  if (norm_w && splits <= kPfMaxSplits) {
    void* args[] = {&pp, &sp, &mm, &r, &y, &norm_w, &norm_out};
    if ((rc = launch(g.pf_res_reduce_norm, (uint32_t)M, 256, args, st))) return rc;
    if (normed) *normed = true;
    return Q8_OK;
  }
  void* args[] = {&pp, &sp, &mm, &nn, &r, &ld, &y, &ld};
  return launch(g.pf_res_reduce, (uint32_t)(((int64_t)M * kN + 255) / 256), 256, args, st);
}

// Argument blocks of the row products (layouts shared with prefill_rows.h).
struct RowsQkvArgs {
  const void *h, *norm_w;
  const void* w[3];
  void *xn, *q, *k, *v, *q_roped, *k_cache, *v_cache;
  const void *qn_w, *kn_w;
  void* rope;
  int M, start, rope_ready;
};
struct RowsNormArgs {
  const void *h, *norm_w;
  const void* w[3];
  void *x, *y[3], *rope;
  int M, start;
};
struct RowsResArgs {
  const void *x, *w, *r;
  void* y;
  int M;
};

// Most tokens the row products serve.  At 128 tokens a layer takes 39.9 us with
// them and 50.6 with the tiled GEMMs, at 160 tokens (where a workgroup's token
// rows are normalised by twice as many workgroups as the device has CUs) 60 and
// 57; the q/k/v one alone 54.0 at 160 tokens, against 50.9 with a separate norm
// and the tiled one that ends in RoPE.
constexpr int32_t kPfRowsMax = 128;

// Weights the attention launch's further workgroups bring into the caches
// (layout shared with prefill_kernels.hip).
constexpr int kPfTouchMats = 7;
struct PfTouch {
  const void* base[kPfTouchMats];
  int tile_bytes[kPfTouchMats];
  int tiles[kPfTouchMats];
};

// attn_o, gate/up, ffn_down and, above 128 tokens (where the next layer's q/k/v
// product is long enough away for nothing to be evicted: 128 tokens 1177 us a
// prompt without, 1189 with; 300 tokens 1765 and 1729), the next layer's q, k
// and v, in the tiles their products will use for n tokens.  A tile that is
// taken to be another only lands in another XCD's L2.
PfTouch touch_plan(const qwen3_weights* w, int layer, int32_t n) {
  PfTouch t{};
  int mats = 0;
  auto add = [&](const uint8_t* base, int row_bytes, int rows, int tile_rows) {
    t.base[mats] = base;
    t.tile_bytes[mats] = row_bytes * tile_rows;
    t.tiles[mats++] = rows / tile_rows;
  };
  const bool rows = n <= kPfRowsMax, next = !rows && layer + 1 < kLayers;
  const int rows_gu = n <= 32 ? 32 : (n <= 64 ? 64 : 96);
  if (w->prefill_f16) {
    const uint8_t* f = cb(w->prefill_f16) + (int64_t)layer * kPfF16Layer * 2;
    const int res = rows ? 16 : (n > 2560 ? 128 : 64);
    add(f + kPfF16O * 2, 2 * 2048, 1024, res);
    add(f + kPfF16Gu * 2, 2 * 1024, 6144, rows ? rows_gu : (n > 1792 ? 192 : (n > 640 ? 128 : 64)));
    add(f + kPfF16Dn * 2, 2 * 3072, 1024, res);
    if (next) add(f + (kPfF16Layer + kPfF16Qkv) * 2, 2 * 1024, 4096, 128);
  } else {
    const int64_t l = layer, r1 = 1088, r2 = 2176, r3 = 3264;  // row bytes of K = 1024, 2048, 3072
    const uint8_t* gu = cb(w->wgu) + l * 6144 * r1;
    const int res = rows ? 16 : 64, half = rows ? rows_gu / 2 : 32;
    add(cb(w->wo) + l * 1024 * r2, (int)r2, 1024, res);
    add(gu, (int)r1, 3072, half);
    add(gu + 3072 * r1, (int)r1, 3072, half);
    add(cb(w->wdn) + l * 1024 * r3, (int)r3, 1024, res);
    if (next) {
      add(cb(w->wq) + (l + 1) * 2048 * r1, (int)r1, 2048, 128);
      add(cb(w->wk) + (l + 1) * 1024 * r1, (int)r1, 1024, 128);
      add(cb(w->wv) + (l + 1) * 1024 * r1, (int)r1, 1024, 128);
    }
  }
  return t;
}

int launch_rows(hipFunction_t fn, int n, int tokens, int n_tiles, int threads, void* block,
                hipStream_t st) {
  void* args[] = {block};
  return launch(fn, (uint32_t)((n + tokens - 1) / tokens * n_tiles), (uint32_t)threads, args, st);
}

// One layer.  xn_ready: the workspace's xn already holds rms_norm(h,
// attn_norm of this layer) (written by the previous layer's last reduce).
// next_norm (the next layer's attn_norm, or null): if ffn_down's reduce can
// also form the next layer's xn it does so and *next_xn_ready becomes true.
// whole_prompt: the other layers run before and after, so the attention launch
// also brings the following weights into the caches (a layer by itself may find
// them there: 512 tokens 62.4 us a layer over and over, 64.1 with).
int launch_prefill_layer(const qwen3_weights* w, int layer, void* k_cache, void* v_cache,
                         int64_t max_seq, int32_t n, int32_t p0, int chunk_local,
                         void* const (&ws)[kPfRegions], hipStream_t st, bool xn_ready = false,
                         const void* next_norm = nullptr, bool* next_xn_ready = nullptr,
                         bool rope_ready = false, bool whole_prompt = false) {
  const int64_t bpl_q = 2048LL * 1024 / 32 * 34, bpl_kv = 1024LL * 1024 / 32 * 34;
  const int64_t bpl_o = 1024LL * 2048 / 32 * 34, bpl_gu = 6144LL * 1024 / 32 * 34;
  const int64_t bpl_dn = 1024LL * 3072 / 32 * 34;
  const void* an = cb(w->attn_norm) + layer * 2048;
  const void* fn = cb(w->ffn_norm) + layer * 2048;
  const void* qn = cb(w->q_norm) + layer * 256;
  const void* kn = cb(w->k_norm) + layer * 256;
  void* kc = mb(k_cache) + (int64_t)layer * max_seq * kKvRow * 2;
  void* vc = mb(v_cache) + (int64_t)layer * max_seq * kKvRow * 2;
  void *h = ws[0], *h1 = ws[1], *xn = ws[2], *q = ws[3], *k = ws[4], *v = ws[5], *qr = ws[6],
       *attn = ws[7], *act = ws[8], *fnx = ws[9], *part = ws[10], *rope = ws[kPfRopeRegion];
  int rc;
  // f16 layer matrices when the caller made them, else the Q8_0 stacks
  const uint8_t* f16l =
      w->prefill_f16 ? cb(w->prefill_f16) + (int64_t)layer * kPfF16Layer * 2 : nullptr;
  const int q8 = f16l ? 0 : 1;
  const bool rows = n <= kPfRowsMax;
  const void* wq = f16l ? (const void*)(f16l + kPfF16Qkv * 2) : cb(w->wq) + layer * bpl_q;
  const void* wk = cb(w->wk) + layer * bpl_kv;
  const void* wv = cb(w->wv) + layer * bpl_kv;
  if (n <= 64) {
    // 16 columns a workgroup fill the CUs with one token tile; from 17 tokens
    // on 32 columns halve the times a row is normalised (24 tokens 38.5 -> 38.2
    // us a layer, 64 tokens 46.1 -> 44.1)
    RowsNormArgs a{h, an, {wq, wk, wv}, xn, {q, k, v}, rope_ready ? nullptr : rope, n, p0};
    const int i = n <= 16 ? 0 : 1;
    if ((rc = launch_rows(g.pf_rows_qkv[i][q8], n, 16, 256 >> i, 512, &a, st))) return rc;
  } else if (rows) {
    // a whole head a workgroup, so RoPE and the cache writes fit behind it:
    // 32 workgroups per token tile, enough from about 65 tokens (64 tokens
    // 44.1 against 44.9 us a layer, 96 tokens 46.9 against 46.2)
    RowsQkvArgs a{h, an, {wq, wk, wv}, xn, q, k, v, qr, kc, vc, qn, kn, rope, n, p0,
                  rope_ready ? 1 : 0};
    if ((rc = launch_rows(g.pf_rows_qkv_rope[q8], n, 16, 32, 512, &a, st))) return rc;
  }
  // rms_norm, with the RoPE table of the prompt's positions (the same for
  // every layer) where it is not there yet
  auto norm = [&](const void* in, const void* weight, void* out, bool table) {
    int start = p0;
    void* args[] = {&in, &weight, &out, &n, &start, &rope};
    const uint32_t wgs = (uint32_t)((n + 3) / 4);
    return launch(g.pf_norm, table ? 2 * wgs : wgs, 64, args, st);
  };
  if (!rows) {
    if (!xn_ready && (rc = norm(h, an, xn, !rope_ready))) return rc;
    const QkvOut out{q, k, v, qr, kc, vc, qn, kn, rope, p0};
    // f16: q, k, v as one [4096, 1024] matrix, a head (128 columns) a tile.
    // Where 64-token tiles give each CU at most one workgroup (512 tokens), the
    // eight-wave one with six stages in LDS: 300 / 512 tokens 60.4 / 63.0 us a
    // layer against 65.1 / 65.9 (640 tokens 85.4 against 83.8).  A gemm_rows
    // setting picks among the others.
    if (f16l && (int64_t)(n + 63) / 64 * 32 <= g.compute_units &&
        g.pf_tile_rows.load(std::memory_order_relaxed) == 0)
      rc = launch_gemm_f16({{g.pf_f16_qkv_22p, 64, 128, 64, 0, 512}}, xn, 1024, wq, 1024, 4096,
                           nullptr, 0, nullptr, 0, n, st, nullptr, 1, &out);
    else if (f16l)
      rc = launch_gemm_f16({{g.pf_f16_qkv_44, 128, 128, 64, 2}, {g.pf_f16_qkv_24, 64, 128, 64, 0}},
                           xn, 1024, wq, 1024, 4096, nullptr, 0, nullptr, 0, n, st, nullptr, 1,
                           &out);
    else
      rc = launch_gemm(g.pf_gemm_qkv, g.pf_gemm_qkv_m32, xn, 1024, wq, 1024, 4096, 128, nullptr, 0,
                       nullptr, 0, 0, n, st, nullptr, 1, wk, wv, &out);
    if (rc) return rc;
  }
  if (n <= 64) {
    int start = p0;
    void* args[] = {&q, &k, &v, &start, &qn, &kn, &rope, &qr, &kc, &vc};
    if ((rc = launch(g.pf_rope, (uint32_t)n, 256, args, st))) return rc;
  }
  {
    int start = p0, cl = chunk_local ? 1 : 0, nn = n;
    int sb = pf_attn_split_blocks(n, p0, chunk_local);
    const PfSplitGeometry G = pf_split_geometry(n, p0, cl ? p0 : 0);
    const int64_t pairs = pf_pairs_total(G, sb);
    if (pairs > pf_attn_pair_cap(n))
      return fail(Q8_ERR_BAD_SHAPE, "attention splits exceed the workspace");  // not reached
    PfTouch touch = whole_prompt ? touch_plan(w, layer, n) : PfTouch{};
    const uint32_t touch_wgs = !whole_prompt ? 0 : (n <= 64 ? 256 : 128);
    int attn_wgs = (int)(8 * pairs);
    void* args[] = {&qr, &kc, &vc, &nn, &start, &cl, &sb, &part, &attn, &attn_wgs, &touch};
    // 1-D grids, kv head = workgroup mod 8: one head per XCD
    if ((rc = launch(g.pf_attn, (uint32_t)attn_wgs + touch_wgs, 256, args, st))) return rc;
    if (pairs > G.nqb) {  // some query block has several splits
      void* margs[] = {&part, &nn, &start, &cl, &sb, &attn};
      if ((rc = launch(g.pf_attn_merge, (uint32_t)(32 * G.nqb), 256, margs, st))) return rc;
    }
  }
  // the attention partials are consumed by now: their region holds the
  // split-K sums of attn_o and ffn_down
  const size_t part_bytes = pf_region_bytes(n, kPfTokenRegions);
  bool fn_done = false;
  if (rows) {
    // attn_o, gate/up and ffn_down as row products: 16 tokens a workgroup while
    // that leaves CUs to fill, then 32; gate/up with 16, 16, 32 and 48 gate and
    // up rows (each step where the next was measured faster: 32 / 64 / 128
    // tokens)
    const int i = n <= 64 ? 0 : 1;
    RowsResArgs ao{attn, f16l ? (const void*)(f16l + kPfF16O * 2) : cb(w->wo) + layer * bpl_o, h,
                   h1, n};
    if ((rc = launch_rows(g.pf_rows_o[i][q8], n, 16 << i, 64, 512, &ao, st))) return rc;
    RowsNormArgs gu{h1, fn,
                    {f16l ? (const void*)(f16l + kPfF16Gu * 2) : cb(w->wgu) + layer * bpl_gu,
                     nullptr, nullptr},
                    fnx, {act, nullptr, nullptr}, nullptr, n, 0};
    const int j = n <= 16 ? 0 : (n <= 32 ? 1 : (n <= 64 ? 2 : 3));
    const int gu_tiles[4] = {192, 192, 96, 64};
    if ((rc = launch_rows(g.pf_rows_gu[j][q8], n, j == 0 ? 16 : 32, gu_tiles[j], 512, &gu, st)))
      return rc;
    RowsResArgs ad{act, f16l ? (const void*)(f16l + kPfF16Dn * 2) : cb(w->wdn) + layer * bpl_dn,
                   h1, h, n};
    return launch_rows(g.pf_rows_dn[i][q8], n, 16 << i, 64, 768, &ad, st);
  }
  if ((rc = launch_gemm_res(attn, 2048, cb(w->wo) + layer * bpl_o, 2048, h1, h, n, part,
                            part_bytes, st, fn, fnx, &fn_done,
                            f16l ? f16l + kPfF16O * 2 : nullptr)))
    return rc;
  if (!fn_done) {
    if ((rc = norm(h1, fn, fnx, false))) return rc;
  }
  if (f16l)
    rc = launch_gemm_f16({{g.pf_f16_sw_46w, 256, 192, 64, 1, 512},
                          {g.pf_f16_sw_44, 128, 128, 64, 2}, {g.pf_f16_sw_24, 64, 128, 64, 2},
                          {g.pf_f16_sw_22, 64, 64, 64, 0}},
                         fnx, 1024, f16l + kPfF16Gu * 2, 1024, 6144, act, 3072, nullptr, 0, n, st);
  else
    rc = launch_gemm(g.pf_gemm_swiglu, nullptr, fnx, 1024, cb(w->wgu) + layer * bpl_gu, 1024, 3072,
                     32, act, 3072, nullptr, 0, 3072, n, st);
  if (rc) return rc;
  return launch_gemm_res(act, 3072, cb(w->wdn) + layer * bpl_dn, 3072, h, h1, n, part, part_bytes,
                         st, next_norm, xn, next_xn_ready, f16l ? f16l + kPfF16Dn * 2 : nullptr);
}

int check_prefill_ready() {
  int rc = check_decode_ready();
  if (rc) return rc;
  if (!g.pf_module)
    return fail(Q8_ERR_CODE_OBJECT, "prefill_gfx950.hsaco was not found or lacks a kernel");
  return Q8_OK;
}

int validate_step_args(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                       const int32_t* token, const int32_t* pos, const void* scratch) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if ((rc = validate_cache(k_cache, v_cache, max_seq))) return rc;
  if (!token || !pos || !scratch) return fail(Q8_ERR_NULL_POINTER, "null token, pos or scratch");
  if (!aligned(token, 4) || !aligned(pos, 4) || !aligned(scratch, 256))
    return fail(Q8_ERR_MISALIGNED, "token/pos 4, scratch 256-byte alignment");
  return Q8_OK;
}

}  // namespace

extern "C" {

size_t qwen3_scratch_bytes(void) { return kScrBytes; }
size_t qwen3_scratch_status_offset(void) { return kScrStatus; }

int64_t qwen3_scratch_offset(const char* name) {
  if (!name) return -1;
  const std::string n(name);
  if (n == "q") return (int64_t)kScrQ;
  if (n == "k") return (int64_t)kScrK;
  if (n == "v") return (int64_t)kScrV;
  if (n == "attn") return (int64_t)kScrAttn;
  if (n == "res") return (int64_t)kScrRes;
  if (n == "act") return (int64_t)kScrAct;
  if (n == "xn") return (int64_t)kScrXn;
  if (n == "q_roped") return (int64_t)kScrQr;
  if (n == "fn") return (int64_t)kScrFn;
  if (n == "on") return (int64_t)kScrOn;
  if (n == "part") return (int64_t)kScrPart;
  return -1;
}

int qwen3_scratch_reset(void* scratch, void* stream) {
  if (!scratch) return fail(Q8_ERR_NULL_POINTER, "null scratch");
  if (!aligned(scratch, 256)) return fail(Q8_ERR_MISALIGNED, "scratch must be 256-byte aligned");
  int rc = check_ready();
  if (rc) return rc;
  if ((rc = check_decode_ready())) return rc;
  void* p = scratch;
  uint32_t n = (uint32_t)(kScrBytes / 4);
  void* args[] = {&p, &n};
  return launch(g.dec_clear, 64, 256, args, static_cast<hipStream_t>(stream));
}

int qwen3_set_step_mode(int mode) {
  if (mode != 0 && mode != 1) return fail(Q8_ERR_BAD_ARGUMENT, "step mode %d not in {0, 1}", mode);
  int rc = check_decode_ready();
  if (rc) return rc;
  if (mode == 1 && g.step_slots < kStepWgs)
    return fail(Q8_ERR_BAD_ARGUMENT, "this device cannot run the single-launch step "
                "(needs its 448 workgroups resident at once, two per CU)");
  std::lock_guard<std::mutex> lock(g.mu);
  g.step_single = mode;
  return Q8_OK;
}

int qwen3_set_step_spin_limit(uint32_t polls) {
  std::lock_guard<std::mutex> lock(g.mu);
  g.step_spin_limit = polls == 0 ? kDefaultSpinLimit : polls;
  return Q8_OK;
}

int qwen3_step_fallback_count(uint64_t* count) {
  if (!count) return fail(Q8_ERR_NULL_POINTER, "null count");
  *count = g.step_fallbacks.load();
  return Q8_OK;
}

int qwen3_debug_force_step_abort(int64_t after) {
  if (after < -1) return fail(Q8_ERR_BAD_ARGUMENT, "after %lld < -1", (long long)after);
  std::lock_guard<std::mutex> lock(g.mu);
  g.force_abort_in = after;
  return Q8_OK;
}

int qwen3_check_status(const void* scratch, uint32_t* status, void* stream) {
  if (!scratch || !status) return fail(Q8_ERR_NULL_POINTER, "null scratch or status");
  if (!aligned(scratch, 256)) return fail(Q8_ERR_MISALIGNED, "scratch must be 256-byte aligned");
  int rc = check_ready();
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  *status = 0;
  HIP_TRY(hipMemcpyAsync(status, cb(scratch) + kScrStatus, sizeof(*status), hipMemcpyDeviceToHost,
                         st));
  HIP_TRY(hipStreamSynchronize(st));
  if (*status & 2u)
    return fail(Q8_ERR_STEP_ABORTED,
                "a single-launch decode step gave up waiting for a hand-off (status bit 1); "
                "its outputs are invalid; qwen3_scratch_reset clears the scratch");
  return Q8_OK;
}

int qwen3_get_step_mode(int* mode) {
  if (!mode) return fail(Q8_ERR_NULL_POINTER, "null mode");
  int rc = check_decode_ready();
  if (rc) return rc;
  *mode = use_single(1) ? 1 : 0;
  return Q8_OK;
}

int qwen3_set_prefill_tiling(int gemm_rows, int attn_split_blocks) {
  if (gemm_rows != 0 && gemm_rows != 32 && gemm_rows != 64 && gemm_rows != 128)
    return fail(Q8_ERR_BAD_ARGUMENT, "prefill GEMM rows %d not in {0, 32, 64, 128}", gemm_rows);
  if (attn_split_blocks < 0)
    return fail(Q8_ERR_BAD_ARGUMENT, "attention split of %d blocks", attn_split_blocks);
  int rc = check_prefill_ready();
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(g.mu);
  g.pf_tile_rows = gemm_rows;
  g.pf_attn_split = attn_split_blocks;
  return Q8_OK;
}

int qwen3_decode_embed(const qwen3_weights* w, const int32_t* token, void* h_out, void* stream) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if (!token || !h_out) return fail(Q8_ERR_NULL_POINTER, "null token or h_out");
  if (!aligned(token, 4) || !aligned(h_out, 16))
    return fail(Q8_ERR_MISALIGNED, "token needs 4-byte, h_out 16-byte alignment");
  if ((rc = check_decode_ready())) return rc;
  return launch_embed(w, token, h_out, static_cast<hipStream_t>(stream));
}

int qwen3_decode_layer(const qwen3_weights* w, int layer, void* k_cache, void* v_cache,
                       int64_t max_seq, const int32_t* pos, const void* h_in, void* h_out,
                       void* scratch, void* stream) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if (layer < 0 || layer >= kLayers)
    return fail(Q8_ERR_LAYER_RANGE, "layer %d outside [0, %d)", layer, kLayers);
  if ((rc = validate_cache(k_cache, v_cache, max_seq))) return rc;
  if (!pos || !h_in || !h_out || !scratch) return fail(Q8_ERR_NULL_POINTER, "null argument");
  if (!aligned(pos, 4) || !aligned(h_in, 16) || !aligned(h_out, 16) || !aligned(scratch, 256))
    return fail(Q8_ERR_MISALIGNED, "pos 4, h 16, scratch 256-byte alignment required");
  if (h_in == h_out) return fail(Q8_ERR_BAD_ARGUMENT, "h_in and h_out must differ");
  if ((rc = check_decode_ready())) return rc;
  return launch_layer(w, layer, k_cache, v_cache, max_seq, pos, h_in, h_out, scratch,
                      static_cast<hipStream_t>(stream));
}

int qwen3_decode_head(const qwen3_weights* w, const void* h, void* logits, int32_t* token,
                      int32_t* pos, int advance, int64_t max_seq, void* scratch, void* stream) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if (!h || !token || !pos || !scratch) return fail(Q8_ERR_NULL_POINTER, "null argument");
  if (!aligned(h, 16) || !aligned(token, 4) || !aligned(pos, 4) || !aligned(scratch, 256) ||
      (logits && !aligned(logits, 2)))
    return fail(Q8_ERR_MISALIGNED, "h 16, token/pos 4, scratch 256, logits 2-byte alignment");
  if (max_seq < 1) return fail(Q8_ERR_BAD_SHAPE, "max_seq must be >= 1");
  if ((rc = check_decode_ready())) return rc;
  return launch_head(w, h, logits, token, pos, advance, max_seq, scratch,
                     static_cast<hipStream_t>(stream));
}

int qwen3_decode_step(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                      int32_t* token, int32_t* pos, void* logits, int advance, void* scratch,
                      void* stream) {
  int rc = validate_step_args(w, k_cache, v_cache, max_seq, token, pos, scratch);
  if (rc) return rc;
  if (logits && !aligned(logits, 2)) return fail(Q8_ERR_MISALIGNED, "logits 2-byte alignment");
  if ((rc = check_decode_ready())) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (use_single(max_seq))
    return launch_step(w, k_cache, v_cache, max_seq, token, token, pos, logits, nullptr, advance,
                       1, scratch, st);
  void* h = nullptr;
  if ((rc = launch_body(w, k_cache, v_cache, max_seq, token, pos, scratch, st, &h))) return rc;
  return launch_head(w, h, logits, token, pos, advance, max_seq, scratch, st);
}

int qwen3_decode_step_checked(const qwen3_weights* w, void* k_cache, void* v_cache,
                              int64_t max_seq, int32_t* token, int32_t* pos, void* logits,
                              int advance, void* scratch, void* stream) {
  int rc = validate_step_args(w, k_cache, v_cache, max_seq, token, pos, scratch);
  if (rc) return rc;
  if (logits && !aligned(logits, 2)) return fail(Q8_ERR_MISALIGNED, "logits 2-byte alignment");
  if ((rc = check_decode_ready())) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if ((rc = check_not_aborted(scratch, st, "before qwen3_decode_step_checked"))) return rc;
  if (use_single(max_seq)) {
    if ((rc = launch_step(w, k_cache, v_cache, max_seq, token, token, pos, logits, nullptr,
                          advance, 1, scratch, st)))
      return rc;
    uint32_t status = 0;
    if ((rc = read_status(scratch, st, &status))) return rc;
    if ((status & 2u) == 0) return Q8_OK;
    // the launch gave up (token and position untouched): the same step per phase
    if ((rc = recover_from_abort(scratch, st, status))) return rc;
  }
  void* h = nullptr;
  if ((rc = launch_body(w, k_cache, v_cache, max_seq, token, pos, scratch, st, &h))) return rc;
  if ((rc = launch_head(w, h, logits, token, pos, advance, max_seq, scratch, st))) return rc;
  HIP_TRY(hipStreamSynchronize(st));
  return Q8_OK;
}

int qwen3_prefill(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                  const int32_t* prompt, int32_t n_prompt, int32_t* token, int32_t* pos,
                  void* scratch, void* stream) {
  int rc = validate_step_args(w, k_cache, v_cache, max_seq, token, pos, scratch);
  if (rc) return rc;
  if (!prompt) return fail(Q8_ERR_NULL_POINTER, "null prompt");
  if (!aligned(prompt, 4)) return fail(Q8_ERR_MISALIGNED, "prompt 4-byte alignment");
  if (n_prompt < 1 || n_prompt > max_seq)
    return fail(Q8_ERR_BAD_SHAPE, "n_prompt %d outside [1, max_seq]", n_prompt);
  if ((rc = check_decode_ready())) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  void* status = mb(scratch) + kScrStatus;
  int ms = (int)max_seq;
  int32_t i0 = 0;  // the first prompt token the per-phase launches take
  if (use_single(max_seq)) {
    // the position before and after, so a step that gave up can be resumed
    int32_t p0 = 0, p1 = 0;
    HIP_TRY(hipMemcpyAsync(&p0, pos, sizeof(p0), hipMemcpyDeviceToHost, st));
    if ((rc = check_not_aborted(scratch, st, "before qwen3_prefill"))) return rc;
    for (int32_t i = 0; i < n_prompt; ++i) {
      const bool last = i + 1 == n_prompt;
      if ((rc = launch_step(w, k_cache, v_cache, max_seq, prompt + i, token, pos, nullptr, nullptr,
                            1, last ? 1 : 0, scratch, st)))
        return rc;
    }
    HIP_TRY(hipMemcpyAsync(&p1, pos, sizeof(p1), hipMemcpyDeviceToHost, st));
    uint32_t sw = 0;
    if ((rc = read_status(scratch, st, &sw))) return rc;
    if ((sw & 2u) == 0) return Q8_OK;
    // Each completed step moved the position by one; the step that gave up
    // and those behind it did nothing.  With the cache full (bit 0) the
    // position no longer counts the steps, and nothing is re-run.
    if ((sw & 1u) != 0 || p1 < p0 || p1 - p0 >= n_prompt)
      return fail(Q8_ERR_STEP_ABORTED,
                  "qwen3_prefill: a single-launch step gave up waiting for a hand-off (status bit "
                  "1) and the position cannot tell which steps completed; qwen3_scratch_reset "
                  "clears the scratch");
    if ((rc = recover_from_abort(scratch, st, sw))) return rc;
    i0 = p1 - p0;
  }
  for (int32_t i = i0; i < n_prompt; ++i) {
    void* h = nullptr;
    if ((rc = launch_body(w, k_cache, v_cache, max_seq, prompt + i, pos, scratch, st, &h)))
      return rc;
    if (i + 1 < n_prompt) {
      void* args[] = {&pos, &ms, &status};
      if ((rc = launch(g.dec_adv, 1, 64, args, st))) return rc;
    } else {
      if ((rc = launch_head(w, h, nullptr, token, pos, 1, max_seq, scratch, st))) return rc;
    }
  }
  return Q8_OK;
}

// qwen3_generate's host-visible copy of the loop state after a batch, and
// the pinned slots and events it uses, released on every return path once
// the stream has drained (no copy into a slot is left in flight).
struct GenReadback {
  int32_t token;
  int32_t pos;
  uint32_t status;
  uint32_t pad;
};
struct GenResources {
  hipStream_t st;
  GenReadback* rb = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  explicit GenResources(hipStream_t s) : st(s) {}
  GenResources(const GenResources&) = delete;
  GenResources& operator=(const GenResources&) = delete;
  ~GenResources() {
    (void)hipStreamSynchronize(st);
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (rb) (void)hipHostFree(rb);
  }
};

int qwen3_generate(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                   int32_t* token, int32_t* pos, int32_t max_new, int32_t eos_id,
                   int32_t* out_tokens, int32_t* n_generated, void* scratch, void* stream) {
  int rc = validate_step_args(w, k_cache, v_cache, max_seq, token, pos, scratch);
  if (rc) return rc;
  if (!out_tokens || !n_generated) return fail(Q8_ERR_NULL_POINTER, "null out_tokens or n_generated");
  if (!aligned(out_tokens, 4)) return fail(Q8_ERR_MISALIGNED, "out_tokens 4-byte alignment");
  if (max_new < 0) return fail(Q8_ERR_BAD_SHAPE, "max_new %d < 0", max_new);
  if ((rc = check_decode_ready())) return rc;
  *n_generated = 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  int32_t p0 = 0;
  HIP_TRY(hipMemcpyAsync(&p0, pos, sizeof(p0), hipMemcpyDeviceToHost, st));
  if ((rc = check_not_aborted(scratch, st, "before qwen3_generate"))) return rc;
  if (p0 < 0 || (int64_t)p0 + max_new > max_seq)
    return fail(Q8_ERR_BAD_SHAPE, "positions %d + %d new tokens exceed max_seq %lld", p0, max_new,
                (long long)max_seq);
  // One batch stays queued behind the one being checked, so the device does
  // not wait for the host's check between batches: after batch k's steps, its
  // token, position and status are copied into pinned host slot k % 2 and an
  // event is recorded; batch k + 1 is launched before the host waits for that
  // event.  When batch k ends the loop (its last token is EOS, or a step gave
  // up), batch k + 1 -- already queued -- is waited for and the token,
  // position and status are put back to their values after batch k, so
  // everything the caller can observe is what a loop without the queued batch
  // leaves (out_tokens slots past *n_generated aside).  Cache rows past the
  // restored position are never read before a later step rewrites them.
  GenResources res(st);
  HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&res.rb), 2 * sizeof(GenReadback),
                        hipHostMallocDefault));
  for (hipEvent_t& e : res.ev) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  uint32_t* status = reinterpret_cast<uint32_t*>(mb(scratch) + kScrStatus);
  // the step mode, once for the call; per-phase for the rest of it after a
  // single launch gave up
  bool single = use_single(max_seq);
  // steps first + from .. first + count - 1 of a batch (from = 0: all)
  auto launch_batch = [&](int32_t first, int32_t count, int slot, int32_t from) -> int {
    for (int32_t b = from; b < count; ++b) {
      int brc;
      if (single) {
        if ((brc = launch_step(w, k_cache, v_cache, max_seq, token, token, pos, nullptr,
                               out_tokens + first + b, 1, 1, scratch, st)))
          return brc;
        continue;
      }
      void* h = nullptr;
      if ((brc = launch_body(w, k_cache, v_cache, max_seq, token, pos, scratch, st, &h))) return brc;
      if ((brc = launch_head(w, h, nullptr, token, pos, 1, max_seq, scratch, st,
                             out_tokens + first + b)))
        return brc;
    }
    GenReadback* r = &res.rb[slot];
    HIP_TRY(hipMemcpyAsync(&r->token, token, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(&r->pos, pos, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(&r->status, status, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipEventRecord(res.ev[slot], st));
    return Q8_OK;
  };
  int32_t first = 0;
  int32_t count = max_new < kGenerateBatch ? max_new : kGenerateBatch;
  int slot = 0;
  if (count > 0 && (rc = launch_batch(first, count, slot, 0))) return rc;
  while (count > 0) {
    const int32_t next = first + count;
    const int32_t next_count = max_new - next < kGenerateBatch ? max_new - next : kGenerateBatch;
    if (next_count > 0 && (rc = launch_batch(next, next_count, 1 - slot, 0))) return rc;
    HIP_TRY(hipEventSynchronize(res.ev[slot]));
    const GenReadback r = res.rb[slot];
    bool aborted = (r.status & 2u) != 0;
    if (aborted && single) {
      // A single launch of this batch gave up: it and every single launch
      // behind it (the rest of the batch, the queued batch) returned at their
      // start, so the position counts the steps that completed.  Re-run this
      // batch from there per phase (the same bits) and check it again.
      if (next_count > 0) HIP_TRY(hipEventSynchronize(res.ev[1 - slot]));
      const int32_t done = r.pos - p0;
      if (done >= first && done < next) {
        if ((rc = recover_from_abort(scratch, st, r.status))) return rc;
        single = false;
        if ((rc = launch_batch(first, count, slot, done - first))) return rc;
        continue;  // the next batch is queued again at the top
      }
    }
    // the batch's steps must all have completed; otherwise its tokens are not
    // valid and n_generated stays at the previous batch
    if (!aborted) *n_generated = next;
    if (aborted || r.token == eos_id) {
      if (next_count > 0) {  // undo the queued batch
        HIP_TRY(hipEventSynchronize(res.ev[1 - slot]));
        res.rb[1 - slot] = r;
        GenReadback* u = &res.rb[1 - slot];
        HIP_TRY(hipMemcpyAsync(token, &u->token, sizeof(int32_t), hipMemcpyHostToDevice, st));
        HIP_TRY(hipMemcpyAsync(pos, &u->pos, sizeof(int32_t), hipMemcpyHostToDevice, st));
        HIP_TRY(hipMemcpyAsync(status, &u->status, sizeof(uint32_t), hipMemcpyHostToDevice, st));
        HIP_TRY(hipStreamSynchronize(st));
      }
      if (aborted)
        return fail(Q8_ERR_STEP_ABORTED,
                    "qwen3_generate: a single-launch decode step gave up waiting for a hand-off "
                    "(status bit 1); its outputs are invalid; qwen3_scratch_reset clears the "
                    "scratch");
      break;
    }
    first = next;
    count = next_count;
    slot = 1 - slot;
  }
  return Q8_OK;
}

int64_t qwen3_prefill_workspace_offset(int32_t n_prompt, const char* name) {
  static const char* const kNames[kPfRegions] = {"h", "res",     "xn",   "q",   "k",  "v",
                                                 "q_roped", "attn", "act", "fn", "attn_part", "rope"};
  if (!name || n_prompt < 1 || n_prompt > kPfMaxTokens) return -1;
  int64_t off = 0;
  for (int i = 0; i < kPfRegions; ++i) {
    if (std::strcmp(name, kNames[i]) == 0) return off;
    off += (int64_t)pf_region_bytes(n_prompt, i);
  }
  return -1;
}

int qwen3_prefill_layer(const qwen3_weights* w, int layer, void* k_cache, void* v_cache,
                        int64_t max_seq, int32_t n_tokens, int32_t start_pos, int chunk_local,
                        void* workspace, size_t workspace_bytes, void* stream) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if ((rc = validate_cache(k_cache, v_cache, max_seq))) return rc;
  if (layer < 0 || layer >= kLayers)
    return fail(Q8_ERR_LAYER_RANGE, "layer %d outside [0, %d)", layer, kLayers);
  if (!workspace) return fail(Q8_ERR_NULL_POINTER, "null workspace");
  if (!aligned(workspace, 256)) return fail(Q8_ERR_MISALIGNED, "workspace 256-byte alignment");
  if (n_tokens < 1 || n_tokens > kPfMaxTokens || start_pos < 0 ||
      (int64_t)start_pos + n_tokens > max_seq)
    return fail(Q8_ERR_BAD_SHAPE, "tokens [%d, %d + %d) outside the cache of %lld", start_pos,
                start_pos, n_tokens, (long long)max_seq);
  if (workspace_bytes < pf_workspace_bytes(n_tokens))
    return fail(Q8_ERR_BAD_SHAPE, "workspace of %zu bytes < %zu needed for %d tokens",
                workspace_bytes, pf_workspace_bytes(n_tokens), n_tokens);
  if ((rc = check_prefill_ready())) return rc;
  void* ws[kPfRegions];
  size_t off = 0;
  for (int i = 0; i < kPfRegions; ++i) {
    ws[i] = mb(workspace) + off;
    off += pf_region_bytes(n_tokens, i);
  }
  return launch_prefill_layer(w, layer, k_cache, v_cache, max_seq, n_tokens, start_pos,
                              chunk_local, ws, static_cast<hipStream_t>(stream));
}

size_t qwen3_prefill_workspace_bytes(int32_t n_prompt) {
  if (n_prompt < 1 || n_prompt > kPfMaxTokens) return 0;
  return pf_workspace_bytes(n_prompt);
}

size_t qwen3_prefill_matrices_bytes(void) { return kPfF16Bytes; }

int qwen3_prefill_matrices_expand(const qwen3_weights* w, void* matrices, size_t bytes,
                                  void* stream) {
  int rc = validate_weights(w);
  if (rc) return rc;
  if (!matrices) return fail(Q8_ERR_NULL_POINTER, "null matrices buffer");
  if (!aligned(matrices, 256)) return fail(Q8_ERR_MISALIGNED, "matrices must be 256-byte aligned");
  if (bytes < kPfF16Bytes)
    return fail(Q8_ERR_BAD_SHAPE, "matrices buffer of %zu bytes, %zu needed", bytes, kPfF16Bytes);
  if ((rc = check_prefill_ready())) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // (Q8_0 stack, its rows and K, first destination row in the layer's f16 matrices)
  struct Part {
    const void* src;
    int rows, K;
    int64_t dst;
    int gu_half;
  } parts[] = {{w->wq, 2048, 1024, kPfF16Qkv, 0},
               {w->wk, 1024, 1024, kPfF16Qkv + 2048LL * 1024, 0},
               {w->wv, 1024, 1024, kPfF16Qkv + 3072LL * 1024, 0},
               {w->wo, 1024, 2048, kPfF16O, 0},
               {w->wgu, 6144, 1024, kPfF16Gu, 3072},
               {w->wdn, 1024, 3072, kPfF16Dn, 0}};
  for (const Part& p : parts) {
    const void* src = p.src;
    long long src_layer = (long long)p.rows * p.K / 32 * 34;
    int rows = p.rows, K = p.K, gu = p.gu_half;
    void* dst = mb(matrices) + p.dst * 2;
    long long dst_layer = kPfF16Layer;
    void* args[] = {&src, &src_layer, &rows, &K, &gu, &dst, &dst_layer};
    const uint32_t blocks = (uint32_t)(((int64_t)rows * K / 32 + 255) / 256);
    if ((rc = launch2(g.pf_expand, blocks, kLayers, 256, args, st))) return rc;
  }
  return Q8_OK;
}

int qwen3_prefill_batched(const qwen3_weights* w, void* k_cache, void* v_cache, int64_t max_seq,
                          const int32_t* prompt, int32_t n_prompt, int32_t* token, int32_t* pos,
                          void* logits, int chunk_local, void* workspace, size_t workspace_bytes,
                          void* scratch, void* stream) {
  int rc = validate_step_args(w, k_cache, v_cache, max_seq, token, pos, scratch);
  if (rc) return rc;
  if (!prompt || !workspace) return fail(Q8_ERR_NULL_POINTER, "null prompt or workspace");
  if (!aligned(prompt, 4) || !aligned(workspace, 256) || (logits && !aligned(logits, 16)))
    return fail(Q8_ERR_MISALIGNED, "prompt 4, workspace 256, logits 16-byte alignment");
  if (n_prompt < 1 || n_prompt > max_seq || n_prompt > kPfMaxTokens)
    return fail(Q8_ERR_BAD_SHAPE, "n_prompt %d outside [1, min(max_seq, 2^20)]", n_prompt);
  if (workspace_bytes < pf_workspace_bytes(n_prompt))
    return fail(Q8_ERR_BAD_SHAPE, "workspace of %zu bytes < %zu needed for %d tokens",
                workspace_bytes, pf_workspace_bytes(n_prompt), n_prompt);
  if ((rc = check_prefill_ready())) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  int32_t p0 = 0;
  HIP_TRY(hipMemcpyAsync(&p0, pos, sizeof(p0), hipMemcpyDeviceToHost, st));
  if ((rc = check_not_aborted(scratch, st, "before qwen3_prefill_batched"))) return rc;
  if (p0 < 0 || (int64_t)p0 + n_prompt > max_seq)
    return fail(Q8_ERR_BAD_SHAPE, "positions %d + %d prompt tokens exceed max_seq %lld", p0,
                n_prompt, (long long)max_seq);
  void* ws[kPfRegions];
  size_t off = 0;
  for (int i = 0; i < kPfRegions; ++i) {
    ws[i] = mb(workspace) + off;
    off += pf_region_bytes(n_prompt, i);
  }
  {
    const void* tp = prompt;
    const void* e = w->token_embd;
    void* h = ws[0];
    void* args[] = {&tp, &e, &h};
    if ((rc = launch(g.pf_embed, (uint32_t)n_prompt, 128, args, st))) return rc;
  }
  bool xn_ready = false;
  for (int l = 0; l < kLayers; ++l) {
    const void* next_norm = l + 1 < kLayers ? cb(w->attn_norm) + (l + 1) * 2048 : nullptr;
    if ((rc = launch_prefill_layer(w, l, k_cache, v_cache, max_seq, n_prompt, p0, chunk_local, ws,
                                   st, xn_ready, next_norm, &xn_ready, l > 0, true)))
      return rc;
  }
  {
    int last = p0 + n_prompt - 1;
    void* args[] = {&pos, &last};
    if ((rc = launch(g.pf_set_pos, 1, 64, args, st))) return rc;
  }
  const void* h_last = cb(ws[0]) + (size_t)(n_prompt - 1) * 2048;
  return launch_head(w, h_last, logits, token, pos, 1, max_seq, scratch, st);
}

}  // extern "C"
