// libmxfa.so: C ABI over the gfx950 code object mxfa_kernels.hsaco.
//
// Replaces the reference's launch path (mu_schedule(fa_entry, nullptr, occupancy),
// lib/src/mu_schedule.cpp:83-104, started from main() in
// kernels/flash_attention_mx_gqa/kernel.cpp:186-191) with hipModuleLaunchKernel on
// the caller's stream.  One hipModule per device is loaded lazily (or by
// mxfa_init) and kept until mxfa_shutdown.  Host code only: built with g++ against
// libamdhip64; the kernels are compiled separately by hipcc --genco.
#include "mxfa.h"

#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <string_view>
#include <unordered_map>

#include "mxfa_args.h"

namespace {

thread_local std::string g_err;

mxfa_status fail(mxfa_status st, const std::string& msg) {
  g_err = msg;
  return st;
}

#define MXFA_HIP(call)                                                                         \
  do {                                                                                         \
    hipError_t e_ = (call);                                                                    \
    if (e_ != hipSuccess) return fail(MXFA_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

const char* const kKernelNames[] = {
    "mxfa_quant_rows_e4m3",    "mxfa_quant_rows_e3m2",    "mxfa_quant_cols_e4m3", "mxfa_quant_cols_e3m2",
    "mxfa_softmax_requant_rows",     "mxfa_fill_normal_f32",
    "mxfa_decode_d64",         "mxfa_decode_d128",        "mxfa_decode_d256",     "mxfa_decode_d64_softcap",
    "mxfa_decode_d128_softcap", "mxfa_decode_d256_softcap", "mxfa_decode_combine", "mxfa_kv_append_e4m3",
    "mxfa_kv_append_e3m2",     "mxfa_kv_tail_update",     "mxfa_quant_rows_r4",
    "mxfa_decode_d64_r2", "mxfa_decode_d128_r2",
    "mxfa_decode_d256_r2",     "mxfa_decode_d64_softcap_r2", "mxfa_decode_d128_softcap_r2",
    "mxfa_decode_d256_softcap_r2", "mxfa_gemm", "mxfa_gemm_ae3m2", "mxfa_gemm_be3m2", "mxfa_gemm_ae3m2_be3m2",
    "mxfa_k_to_bf16",          "mxfa_prefill3_d64",       "mxfa_prefill3_d128",   "mxfa_prefill3_d64_softcap",
    "mxfa_prefill3_d128_softcap", "mxfa_prefill3_d64_r2", "mxfa_prefill3_d128_r2", "mxfa_prefill3_d64_softcap_r2",
    "mxfa_prefill3_d128_softcap_r2",
    "mxfa_prefill3_d256",      "mxfa_prefill3_d256_softcap", "mxfa_prefill3_d256_r2", "mxfa_prefill3_d256_softcap_r2",
    "mxfa_prefill3_trace_d64", "mxfa_prefill3_trace_d128", "mxfa_prefill3_trace_d256",
    "mxfa_prefill3_trace_d64_softcap", "mxfa_prefill3_trace_d128_softcap", "mxfa_prefill3_trace_d256_softcap",
    "mxfa_prefill3_trace_d64_r2", "mxfa_prefill3_trace_d128_r2", "mxfa_prefill3_trace_d256_r2",
    "mxfa_prefill3_trace_d64_softcap_r2", "mxfa_prefill3_trace_d128_softcap_r2", "mxfa_prefill3_trace_d256_softcap_r2",
    "mxfa_gemm_dma", "mxfa_gemm_skinny_t1", "mxfa_gemm_skinny_t2",
    "mxfa_prefill3n_d64", "mxfa_prefill3n_d128", "mxfa_prefill3n_d256", "mxfa_prefill3n_d64_softcap",
    "mxfa_prefill3n_d128_softcap", "mxfa_prefill3n_d256_softcap", "mxfa_prefill3n_d64_r2", "mxfa_prefill3n_d128_r2",
    "mxfa_prefill3n_d256_r2", "mxfa_prefill3n_d64_softcap_r2", "mxfa_prefill3n_d128_softcap_r2",
    "mxfa_prefill3n_d256_softcap_r2",
    "mxfa_prefill3n_d64_e3m2", "mxfa_prefill3n_d128_e3m2", "mxfa_prefill3n_d256_e3m2",
    "mxfa_prefill3n_d64_softcap_e3m2", "mxfa_prefill3n_d128_softcap_e3m2", "mxfa_prefill3n_d256_softcap_e3m2",
    "mxfa_prefill3n_d64_r2_e3m2", "mxfa_prefill3n_d128_r2_e3m2", "mxfa_prefill3n_d256_r2_e3m2",
    "mxfa_prefill3n_d64_softcap_r2_e3m2", "mxfa_prefill3n_d128_softcap_r2_e3m2", "mxfa_prefill3n_d256_softcap_r2_e3m2",
    "mxfa_quant_cols_e3m2_blk", "mxfa_kv_append_e3m2_blk",
    "mxfa_gemm_mid_dma", "mxfa_gemm_small_dma", "mxfa_gemm_mid_ae3m2", "mxfa_gemm_mid_be3m2", "mxfa_gemm_mid_ae3m2_be3m2",
    "mxfa_prefill_max_d64",    "mxfa_prefill_max_d128",   "mxfa_prefill_max_d256",  "mxfa_prefill_max_d64_softcap",
    "mxfa_prefill_max_d128_softcap", "mxfa_prefill_max_d256_softcap",
#define MXFA_SPLIT_NAMES4(D, V) \
  "mxfa_prefill3s_d" #D V, "mxfa_prefill3s_d" #D "_softcap" V, "mxfa_prefill3s_d" #D "_r2" V, "mxfa_prefill3s_d" #D "_softcap_r2" V
#define MXFA_SPLIT_NAMES(D) MXFA_SPLIT_NAMES4(D, ""), MXFA_SPLIT_NAMES4(D, "_e3m2"), MXFA_SPLIT_NAMES4(D, "_blk")
    MXFA_SPLIT_NAMES(64), MXFA_SPLIT_NAMES(128), MXFA_SPLIT_NAMES(256),
#define MXFA_BLK_NAMES(D)                                                                                      \
  "mxfa_prefill3_d" #D "_blk", "mxfa_prefill3_d" #D "_softcap_blk", "mxfa_prefill3_d" #D "_r2_blk",            \
      "mxfa_prefill3_d" #D "_softcap_r2_blk", "mxfa_prefill3n_d" #D "_blk", "mxfa_prefill3n_d" #D "_softcap_blk", \
      "mxfa_prefill3n_d" #D "_r2_blk", "mxfa_prefill3n_d" #D "_softcap_r2_blk"
    MXFA_BLK_NAMES(64), MXFA_BLK_NAMES(128), MXFA_BLK_NAMES(256),
#define MXFA_DECODE_BLK_NAMES(D)                                                            \
  "mxfa_decode_d" #D "_blk", "mxfa_decode_d" #D "_softcap_blk", "mxfa_decode_d" #D "_r2_blk", \
      "mxfa_decode_d" #D "_softcap_r2_blk"
    MXFA_DECODE_BLK_NAMES(64), MXFA_DECODE_BLK_NAMES(128), MXFA_DECODE_BLK_NAMES(256),
};
constexpr int kNumKernels = sizeof(kKernelNames) / sizeof(kKernelNames[0]);

struct DeviceModule {
  hipModule_t mod = nullptr;
  hipFunction_t fn[kNumKernels] = {};
  void* decode_scratch = nullptr;     // this device's address of mxfa_decode_scratch
  size_t decode_scratch_bytes = 0;
};

std::mutex g_mu;
std::unordered_map<int, DeviceModule> g_mods;

std::string code_object_path() {
  if (const char* env = getenv("MXFA_HSACO")) return env;
  Dl_info info;
  if (dladdr(reinterpret_cast<void*>(&mxfa_version), &info) && info.dli_fname) {
    std::string p(info.dli_fname);
    size_t slash = p.rfind('/');
    return (slash == std::string::npos ? std::string(".") : p.substr(0, slash)) + "/mxfa_kernels.hsaco";
  }
  return "mxfa_kernels.hsaco";
}

// Module of the current device (loaded on first use).
mxfa_status module_for_current(DeviceModule** out) {
  int dev = -1;
  MXFA_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_mods.find(dev);
  if (it != g_mods.end()) {
    *out = &it->second;
    return MXFA_OK;
  }
  hipDeviceProp_t prop;
  MXFA_HIP(hipGetDeviceProperties(&prop, dev));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(MXFA_ERR_UNSUPPORTED, std::string("device ") + std::to_string(dev) + " is " + prop.gcnArchName +
                                          "; libmxfa is built for gfx950 (MI355X) only");
  DeviceModule dm;
  std::string path = code_object_path();
  hipError_t e = hipModuleLoad(&dm.mod, path.c_str());
  if (e != hipSuccess) return fail(MXFA_ERR_MODULE, "hipModuleLoad(" + path + "): " + hipGetErrorString(e));
  for (int i = 0; i < kNumKernels; i++) {
    e = hipModuleGetFunction(&dm.fn[i], dm.mod, kKernelNames[i]);
    if (e != hipSuccess) {
      (void)hipModuleUnload(dm.mod);
      return fail(MXFA_ERR_MODULE, std::string("kernel ") + kKernelNames[i] + " missing from " + path);
    }
  }
  // The device address of the decode scratch array in this device's copy of the module (the
  // module-API form of hipGetSymbolAddress): taken here, with the device current, and only
  // this address is ever passed to a kernel.
  hipDeviceptr_t sp = nullptr;
  e = hipModuleGetGlobal(&sp, &dm.decode_scratch_bytes, dm.mod, "mxfa_decode_scratch");
  if (e != hipSuccess || !sp || dm.decode_scratch_bytes < MXFA_DECODE_SCRATCH_BYTES) {
    (void)hipModuleUnload(dm.mod);
    return fail(MXFA_ERR_MODULE, std::string("hipModuleGetGlobal(mxfa_decode_scratch) in ") + path + ": " +
                                     (e != hipSuccess ? hipGetErrorString(e) : "missing or too small"));
  }
  dm.decode_scratch = reinterpret_cast<void*>(sp);
  auto res = g_mods.emplace(dev, dm);
  *out = &res.first->second;
  return MXFA_OK;
}

// Module of the current device if it is already loaded (never loads: no allocation).
mxfa_status loaded_module_for_current(DeviceModule** out) {
  int dev = -1;
  MXFA_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_mods.find(dev);
  if (it == g_mods.end())
    return fail(MXFA_ERR_MODULE, "no code object loaded on device " + std::to_string(dev) +
                                     ": call mxfa_init() on it before mxfa_decode_noalloc");
  *out = &it->second;
  return MXFA_OK;
}

// (a hashed index: walking the two hundred names cost half a microsecond per launch)
hipFunction_t fn_by_name(DeviceModule* dm, const char* name) {
  static const std::unordered_map<std::string_view, int> index = [] {
    std::unordered_map<std::string_view, int> m;
    for (int i = 0; i < kNumKernels; i++) m.emplace(kKernelNames[i], i);
    return m;
  }();
  const auto it = index.find(name);
  return it == index.end() ? nullptr : dm->fn[it->second];
}

// MXFA_PREFILL_LDS_PAD=<bytes>: that much dynamic LDS added to every prefill launch, which
// lowers how many workgroups share a CU without changing the code object (an occupancy
// measurement; unset, the launches use their static LDS only)
unsigned prefill_lds_pad(const char* name) {
  if (std::strncmp(name, "mxfa_prefill3", 13) != 0) return 0;
  const char* env = getenv("MXFA_PREFILL_LDS_PAD");
  const long v = env ? atol(env) : 0;
  return v > 0 && v <= 96 * 1024 ? (unsigned)v : 0;
}

mxfa_status launch(DeviceModule* dm, const char* name, dim3 grid, dim3 block, void** args, void* stream) {
  hipFunction_t f = fn_by_name(dm, name);
  if (!f) return fail(MXFA_ERR_MODULE, std::string("unknown kernel ") + name);
  MXFA_HIP(hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, block.x, block.y, block.z, prefill_lds_pad(name),
                                 reinterpret_cast<hipStream_t>(stream), args, nullptr));
  return MXFA_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// A launch's x extent in work-items (grid.x * block.x) is a 32-bit count in the dispatch
// packet: a call that would need more is refused before any device work.
mxfa_status check_grid(int64_t blocks, int threads) {
  if (blocks * threads > (int64_t)UINT32_MAX)
    return fail(MXFA_ERR_UNSUPPORTED, "the call needs more than 2^32 work-items in one launch: split it");
  return MXFA_OK;
}

mxfa_status check_params(const mxfa_attn_params* p, bool decode) {
  if (!p) return fail(MXFA_ERR_INVALID_ARG, "params is NULL");
  if (p->batch < 1 || p->num_q_heads < 1 || p->num_kv_heads < 1 || p->seq_q < 1 || p->seq_k < 1)
    return fail(MXFA_ERR_INVALID_ARG, "batch, heads, seq_q and seq_k must be >= 1");
  if (p->num_q_heads % p->num_kv_heads)
    return fail(MXFA_ERR_INVALID_ARG, "num_q_heads must be a multiple of num_kv_heads");
  if (p->head_dim % 32) return fail(MXFA_ERR_INVALID_ARG, "head_dim must be a multiple of 32");
  if (p->head_dim != 64 && p->head_dim != 128 && p->head_dim != 256)
    return fail(MXFA_ERR_UNSUPPORTED, "head_dim must be 64, 128 or 256");
  if (p->seq_k % 32) return fail(MXFA_ERR_INVALID_ARG, "seq_k must be a multiple of 32 (V scale blocks)");
  if (p->q_pos0 < 0 || p->window < 0) return fail(MXFA_ERR_INVALID_ARG, "q_pos0 and window must be >= 0");
  if (!(p->softmax_scale > 0.0f) || !std::isfinite(p->softmax_scale))
    return fail(MXFA_ERR_INVALID_ARG, "softmax_scale must be finite and > 0");
  if (!(p->softcap >= 0.0f) || !std::isfinite(p->softcap)) return fail(MXFA_ERR_INVALID_ARG, "softcap must be finite and >= 0");
  if (p->v_fmt != MXFA_FMT_E4M3 && p->v_fmt != MXFA_FMT_E3M2 && p->v_fmt != MXFA_FMT_E3M2_BLK)
    return fail(MXFA_ERR_INVALID_ARG, "v_fmt must be E4M3, E3M2 or E3M2_BLK");
  if (p->block_n != 0 && p->block_n != 64) return fail(MXFA_ERR_UNSUPPORTED, "block_n must be 0 (default) or 64");
  if (p->p_rule != MXFA_P_R1 && p->p_rule != MXFA_P_R2) return fail(MXFA_ERR_INVALID_ARG, "p_rule must be R1 or R2");
  if (p->kv_stride != 0 && (p->kv_stride < p->seq_k || p->kv_stride % 32))
    return fail(MXFA_ERR_INVALID_ARG, "kv_stride must be 0 or a multiple of 32 that is >= seq_k");
  if (decode) {
    if (p->seq_q != 1) return fail(MXFA_ERR_INVALID_ARG, "decode needs seq_q == 1");
    if (p->num_q_heads / p->num_kv_heads > 32)
      return fail(MXFA_ERR_UNSUPPORTED, "decode supports at most 32 query heads per KV head");
  }
  // Per (batch, KV head) the kernels address K/V (and the workspace's bf16 K, 2 bytes per
  // element) through buffer resources of seq_k * 2 * head_dim bytes with 32-bit signed byte
  // offsets: keep that range below 2^31.
  if ((int64_t)p->seq_k * 2 * p->head_dim > (int64_t)INT32_MAX)
    return fail(MXFA_ERR_UNSUPPORTED, "seq_k * head_dim exceeds the kernels' 32-bit K/V range (2^30 elements per head)");
  int64_t qelems = (int64_t)p->batch * p->num_q_heads * p->seq_q * p->head_dim;
  int64_t kelems = (int64_t)p->batch * p->num_kv_heads * (p->kv_stride ? p->kv_stride : p->seq_k) * p->head_dim;
  if (qelems > (int64_t)1 << 40 || kelems > (int64_t)1 << 40) return fail(MXFA_ERR_INVALID_ARG, "tensor too large");
  return MXFA_OK;
}

mxfa_status check_ptrs(const void* const* ptrs, int n) {
  for (int i = 0; i < n; i++) {
    if (!ptrs[i]) return fail(MXFA_ERR_INVALID_ARG, "NULL tensor pointer");
    if (!aligned16(ptrs[i])) return fail(MXFA_ERR_INVALID_ARG, "tensor pointers must be 16-byte aligned");
  }
  return MXFA_OK;
}

FaArgs make_args(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* qs, const uint8_t* k, const uint8_t* ks,
                 const uint8_t* v, const uint8_t* vs, float* o) {
  FaArgs a;
  std::memset(&a, 0, sizeof a);
  a.q = q; a.qs = qs; a.k = k; a.ks = ks; a.v = v; a.vs = vs; a.o = o;
  a.B = p->batch; a.Hq = p->num_q_heads; a.Hkv = p->num_kv_heads; a.Sq = p->seq_q; a.Sk = p->seq_k;
  a.Skc = p->kv_stride ? p->kv_stride : p->seq_k;
  a.q_pos0 = p->q_pos0; a.window = p->window; a.causal = p->causal ? 1 : 0; a.v_e3m2 = p->v_fmt == MXFA_FMT_E3M2;
  a.group = p->num_q_heads / p->num_kv_heads;
  const float log2e = 1.4426950408889634f;
  a.c_log2 = p->softmax_scale * log2e;
  if (p->softcap > 0.0f) {
    a.sc_u = p->softmax_scale / p->softcap;
    a.cap_log2 = p->softcap * log2e;
  }
  return a;
}

// Kernel name for a parameter set; v_suffix adds the V-format suffix of the prefill kernels
// ("_e3m2": E3M2 codes rewritten in LDS, "_blk": block-packed E3M2 read as fp6).
const char* kernel_name(const char* kind, const mxfa_attn_params* p, bool v_suffix = false) {
  static thread_local char buf[64];
  const char* vs = !v_suffix ? "" : p->v_fmt == MXFA_FMT_E3M2 ? "_e3m2" : p->v_fmt == MXFA_FMT_E3M2_BLK ? "_blk" : "";
  std::snprintf(buf, sizeof buf, "mxfa_%s_d%d%s%s%s", kind, p->head_dim, p->softcap > 0.0f ? "_softcap" : "",
                p->p_rule == MXFA_P_R2 ? "_r2" : "", vs);
  return buf;
}

// Split-KV plan: the 64-key blocks of each (b, KV head) are dealt to n_parts interleaved
// partials (partial i: blocks i, i + n_parts, ...), one wave each, four to a workgroup.
// Interleaving puts the partial waves of a head, which share a workgroup, on adjacent blocks at
// the same time (measured on c5: 188 us vs 204 us for contiguous chunks at 2048 waves).
//
// At most about kDecodeWaves partial waves per call -- two per SIMD of the 256-CU chip, at the two
// workgroups per CU of D <= 128; half as many at D = 256, whose kernel fits one workgroup per CU
// (measured on B32 Hq16 Hkv8 L8192 D256: 0.169 ms at 1,024 waves, 0.182 at 2,048).  At most 4
// partials are rounded up to 1, 2 or 4 so that a head's partials fill whole 4-wave workgroups and
// merge inside them.  The workspace is sized for this many; MXFA_DECODE_WAVES overrides the target
// and then exactly so many are used.
constexpr int64_t kDecodeWaves = 2048;

int64_t decode_wave_override() {
  const char* env = getenv("MXFA_DECODE_WAVES");
  const long long v = env ? atoll(env) : 0;
  return v > 0 ? v : 0;
}

int decode_parts_max(const mxfa_attn_params* p) {
  const int64_t bk = (int64_t)p->batch * p->num_kv_heads;
  const int64_t blocks = (p->seq_k + 63) / 64;
  int64_t target = decode_wave_override();
  if (target == 0) target = p->head_dim == 256 ? kDecodeWaves / 2 : kDecodeWaves;
  int64_t n = (target + bk - 1) / bk;
  if (n == 3) n = 4;
  if (n > blocks) n = blocks;
  if (n < 1) n = 1;
  return (int)n;
}

// Of those, no more than the blocks that the query sees: with a window in a longer cache the other
// partials are empty (window 4,096 in a cache of 60,000 keys: 65 of 938 blocks visible, 256 partials
// 14.1 us a call, 65 12.6).  Each visible block is then a partial of its own in either plan, so O
// differs by the order of the merge's fp32 sums only.  Not where a head's partials share a workgroup
// at D = 256 (one workgroup per CU) in any case: fewer of them only put the visible blocks on fewer
// CUs (batch 32, Hkv 8, 2 blocks visible: 11.6 us in 4 partials, 12.9 in 2).  (Fewer partials than that can be faster
// -- 96 heads of 47 blocks at D = 256, 264 workgroups on 256 CUs in 11 partials each: 50.2 us, in 10
// 32.7 -- but change the running maxima that P is quantized against.)
int decode_parts(const mxfa_attn_params* p) {
  const int nmax = decode_parts_max(p);
  if (p->window <= 0 || decode_wave_override() || (p->head_dim == 256 && nmax <= 4)) return nmax;
  const int hi = p->causal ? std::min(p->seq_k - 1, p->q_pos0) : p->seq_k - 1;
  const int lo = std::max(0, p->q_pos0 - p->window + 1);
  const int vis = hi >= lo ? hi / 64 - lo / 64 + 1 : 1;
  return std::min(nmax, vis == 3 ? 4 : vis);
}

}  // namespace

extern "C" {

int32_t mxfa_version(void) { return MXFA_VERSION; }

const char* mxfa_status_string(mxfa_status st) {
  switch (st) {
    case MXFA_OK: return "ok";
    case MXFA_ERR_INVALID_ARG: return "invalid argument";
    case MXFA_ERR_UNSUPPORTED: return "unsupported";
    case MXFA_ERR_HIP: return "HIP error";
    case MXFA_ERR_MODULE: return "code object error";
    case MXFA_ERR_WORKSPACE: return "workspace too small";
  }
  return "unknown status";
}

const char* mxfa_last_error(void) { return g_err.c_str(); }

mxfa_status mxfa_init(void) {
  DeviceModule* dm;
  return module_for_current(&dm);
}

void mxfa_shutdown(void) {
  std::lock_guard<std::mutex> lk(g_mu);
  for (auto& kv : g_mods) (void)hipModuleUnload(kv.second.mod);
  g_mods.clear();
}

mxfa_status mxfa_quantize_rows(const float* x, int64_t rows, int32_t cols, mxfa_fmt fmt, uint8_t* codes,
                               uint8_t* scales, void* stream) {
  if (rows < 0 || cols <= 0 || cols % 32) return fail(MXFA_ERR_INVALID_ARG, "cols must be a positive multiple of 32");
  if (fmt != MXFA_FMT_E4M3 && fmt != MXFA_FMT_E3M2) return fail(MXFA_ERR_INVALID_ARG, "bad fmt");
  if (rows == 0) return MXFA_OK;
  if (!x || !codes || !scales) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  if (!aligned16(x) || (reinterpret_cast<uintptr_t>(codes) & 3u))
    return fail(MXFA_ERR_INVALID_ARG, "x must be 16-byte and codes 4-byte aligned");
  int64_t nblocks = rows * (int64_t)cols / 32;
  if (mxfa_status st = check_grid((nblocks * 8 + 255) / 256, 256)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  // One block per thread for a small x, four where there are enough of them to fill the chip.  us for
  // one and four, x from the MALL (from HBM): E4M3 131,072 blocks 6.4 and 6.9 (6.1 and 6.4), 230,000 9.1
  // and 10.1 (8.8 and 9.6), 524,288 16.5 and 16.3 (17.2 and 17.3); E3M2, whose table each workgroup
  // fills once, 131,072 9.6 and 8.4 (9.1 and 7.7).
  int per_thread = nblocks >= (fmt == MXFA_FMT_E4M3 ? 524288 : 131072) ? 4 : 1;
  dim3 grid((unsigned)((nblocks + 32 * per_thread - 1) / (32 * per_thread)));
  void* args[] = {(void*)&x, &nblocks, &codes, &scales, &per_thread};
  return launch(dm, fmt == MXFA_FMT_E4M3 ? "mxfa_quant_rows_e4m3" : "mxfa_quant_rows_e3m2", grid, dim3(256), args, stream);
}

mxfa_status mxfa_quantize_rows_r4(const float* x, int64_t rows, int32_t cols, uint8_t* codes, uint8_t* scales,
                                  void* stream) {
  if (rows < 0 || cols <= 0 || cols % 32) return fail(MXFA_ERR_INVALID_ARG, "cols must be a positive multiple of 32");
  if (rows == 0) return MXFA_OK;
  if (!x || !codes || !scales) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  if (!aligned16(x) || (reinterpret_cast<uintptr_t>(codes) & 3u))
    return fail(MXFA_ERR_INVALID_ARG, "x must be 16-byte and codes 4-byte aligned");
  int64_t nblocks = rows * (int64_t)cols / 32;
  if (mxfa_status st = check_grid((nblocks * 8 + 255) / 256, 256)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  void* args[] = {(void*)&x, &nblocks, &codes, &scales};
  return launch(dm, "mxfa_quant_rows_r4", dim3((unsigned)((nblocks * 8 + 255) / 256)), dim3(256), args, stream);
}

mxfa_status mxfa_quantize_cols(const float* x, int64_t mats, int32_t rows, int32_t cols, mxfa_fmt fmt, uint8_t* codes,
                               uint8_t* scales, void* stream) {
  if (mats < 0 || rows <= 0 || rows % 32 || cols <= 0 || cols % 4)
    return fail(MXFA_ERR_INVALID_ARG, "rows must be a positive multiple of 32 and cols of 4");
  if (fmt != MXFA_FMT_E4M3 && fmt != MXFA_FMT_E3M2 && fmt != MXFA_FMT_E3M2_BLK) return fail(MXFA_ERR_INVALID_ARG, "bad fmt");
  if (mats == 0) return MXFA_OK;
  if (!x || !codes || !scales) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  if (!aligned16(x) || (reinterpret_cast<uintptr_t>(codes) & 3u) || (reinterpret_cast<uintptr_t>(scales) & 3u))
    return fail(MXFA_ERR_INVALID_ARG, "x must be 16-byte, codes and scales 4-byte aligned");
  // one wave per (matrix, 32-row block, 128 columns), four waves per workgroup
  const int64_t units = mats * (rows / 32) * ((cols + 127) / 128);
  if (mxfa_status st = check_grid((units + 3) / 4, 256)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  dim3 grid((unsigned)((units + 3) / 4));
  void* args[] = {(void*)&x, &mats, &rows, &cols, &codes, &scales};
  return launch(dm, fmt == MXFA_FMT_E4M3 ? "mxfa_quant_cols_e4m3" : fmt == MXFA_FMT_E3M2 ? "mxfa_quant_cols_e3m2"
                                                                                        : "mxfa_quant_cols_e3m2_blk",
                grid, dim3(256), args, stream);
}

mxfa_status mxfa_kv_append(const mxfa_kv_params* p, const float* k_new, const float* v_new, int32_t pos0, int32_t n_new,
                           uint8_t* k_cache, uint8_t* k_sc, uint8_t* v_cache, uint8_t* v_sc, float* v_tail,
                           void* stream) {
  if (!p) return fail(MXFA_ERR_INVALID_ARG, "params is NULL");
  if (p->batch < 1 || p->num_kv_heads < 1) return fail(MXFA_ERR_INVALID_ARG, "batch and num_kv_heads must be >= 1");
  if (p->head_dim < 32 || p->head_dim % 32) return fail(MXFA_ERR_INVALID_ARG, "head_dim must be a positive multiple of 32");
  if (p->max_len < 32 || p->max_len % 32) return fail(MXFA_ERR_INVALID_ARG, "max_len must be a positive multiple of 32");
  if (p->v_fmt != MXFA_FMT_E4M3 && p->v_fmt != MXFA_FMT_E3M2 && p->v_fmt != MXFA_FMT_E3M2_BLK)
    return fail(MXFA_ERR_INVALID_ARG, "bad v_fmt");
  if (pos0 < 0 || n_new < 0 || (int64_t)pos0 + n_new > p->max_len)
    return fail(MXFA_ERR_INVALID_ARG, "need 0 <= pos0 and pos0 + n_new <= max_len");
  if (n_new == 0) return MXFA_OK;
  const void* ptrs[] = {k_new, v_new, k_cache, k_sc, v_cache, v_sc, v_tail};
  for (const void* q : ptrs)
    if (!q) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  for (const void* q : ptrs)
    if (!aligned16(q)) return fail(MXFA_ERR_INVALID_ARG, "buffers must be 16-byte aligned");
  const int64_t bk = (int64_t)p->batch * p->num_kv_heads;
  int D = p->head_dim, L = p->max_len, n = n_new, pos = pos0;
  // one launch: K (8 lanes per 32-block) then V (one wave per 32 columns of a touched
  // 32-token block)
  int64_t kblocks = bk * n * (D / 32);
  const int64_t kgroups64 = (kblocks * 8 + 255) / 256;
  const int end = pos0 + n_new;
  int ntouch = (end - 1) / 32 - pos0 / 32 + 1;
  int64_t vunits = bk * ntouch * (D / 32);
  const int64_t vgroups = (vunits + 3) / 4;
  if (mxfa_status st = check_grid(kgroups64 + vgroups, 256)) return st;
  int kgroups = (int)kgroups64;
  if (mxfa_status st = check_grid((bk * 32 * (D / 4) + 255) / 256, 256)) return st;   // the tail update
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  void* args[] = {(void*)&k_new, (void*)&v_new, &v_tail, &kblocks, &kgroups, &vunits, &ntouch,
                  &n, &L, &D, &pos, &k_cache, &k_sc, &v_cache, &v_sc};
  if (mxfa_status st = launch(dm, p->v_fmt == MXFA_FMT_E4M3   ? "mxfa_kv_append_e4m3"
                                  : p->v_fmt == MXFA_FMT_E3M2 ? "mxfa_kv_append_e3m2"
                                                              : "mxfa_kv_append_e3m2_blk",
                              dim3((unsigned)(kgroups + vgroups)), dim3(256), args, stream))
    return st;
  if (end % 32 == 0 || ntouch == 1) return MXFA_OK;   // no open block, or its tail is already written
  // the block left open after a multi-block append keeps its fp32 values for the next one
  int64_t tthreads = bk * 32 * (D / 4);
  void* ta[] = {(void*)&v_new, &v_tail, &tthreads, &n, &D, &pos};
  return launch(dm, "mxfa_kv_tail_update", dim3((unsigned)((tthreads + 255) / 256)), dim3(256), ta, stream);
}

mxfa_status mxfa_softmax_requant(const float* s, const float* row_max, float c, int64_t rows, int32_t cols,
                                 int32_t p_rule, float* p, uint8_t* codes, uint8_t* scales, float* row_sum,
                                 void* stream) {
  if (rows < 0 || cols <= 0 || cols % 32) return fail(MXFA_ERR_INVALID_ARG, "cols must be a positive multiple of 32");
  if (p_rule != MXFA_P_R1 && p_rule != MXFA_P_R2) return fail(MXFA_ERR_INVALID_ARG, "p_rule must be R1 or R2");
  if (!(c > 0.0f) || !std::isfinite(c)) return fail(MXFA_ERR_INVALID_ARG, "c must be finite and > 0");
  if (rows == 0) return MXFA_OK;
  if (!s || !row_max || !p || !codes || !scales || !row_sum) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  if (!aligned16(s) || (reinterpret_cast<uintptr_t>(codes) & 3u))
    return fail(MXFA_ERR_INVALID_ARG, "s must be 16-byte and codes 4-byte aligned");
  if (mxfa_status st = check_grid((rows + 255) / 256, 256)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  dim3 grid((unsigned)((rows + 255) / 256));
  int cols_i = cols;
  int rule = p_rule;
  void* args[] = {(void*)&s, (void*)&row_max, &c, &rows, &cols_i, &p, &codes, &scales, &row_sum, &rule};
  return launch(dm, "mxfa_softmax_requant_rows", grid, dim3(256), args, stream);
}

mxfa_status mxfa_gemm(const mxfa_gemm_params* p, const uint8_t* a, const uint8_t* a_sc, const uint8_t* b,
                      const uint8_t* b_sc, void* c, void* stream) {
  if (!p) return fail(MXFA_ERR_INVALID_ARG, "params is NULL");
  if (p->m < 1 || p->n < 1 || p->k < 1) return fail(MXFA_ERR_INVALID_ARG, "m, n and k must be >= 1");
  if (p->k % 32) return fail(MXFA_ERR_INVALID_ARG, "k must be a multiple of 32 (scale blocks)");
  if (p->k % 64 || p->m % 16 || p->n % 16)
    return fail(MXFA_ERR_UNSUPPORTED, "mxfa_gemm needs k % 64 == 0, m % 16 == 0 and n % 16 == 0");
  if (p->a_fmt != MXFA_FMT_E4M3 && p->a_fmt != MXFA_FMT_E3M2) return fail(MXFA_ERR_INVALID_ARG, "bad a_fmt");
  if (p->b_fmt != MXFA_FMT_E4M3 && p->b_fmt != MXFA_FMT_E3M2) return fail(MXFA_ERR_INVALID_ARG, "bad b_fmt");
  if (p->c_fmt != MXFA_C_F32 && p->c_fmt != MXFA_C_BF16) return fail(MXFA_ERR_INVALID_ARG, "bad c_fmt");
  const int64_t lim = (int64_t)1 << 31;
  if (p->m * p->k >= lim || p->k * p->n >= lim)
    return fail(MXFA_ERR_UNSUPPORTED, "mxfa_gemm operands are limited to 2^31 elements");
  if (p->n >= ((int64_t)1 << 22))   // a 256-row tile of C stays under 2^32 bytes
    return fail(MXFA_ERR_UNSUPPORTED, "mxfa_gemm needs n < 4194304");
  const void* ptrs[] = {a, a_sc, b, b_sc, c};
  if (mxfa_status st = check_ptrs(ptrs, 5)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  GemmArgs g;
  std::memset(&g, 0, sizeof g);
  g.a = a; g.sa = a_sc; g.b = b; g.sb = b_sc; g.c = static_cast<uint8_t*>(c);
  g.c_bf16 = p->c_fmt == MXFA_C_BF16;
  g.M = (int)p->m; g.N = (int)p->n; g.K = (int)p->k;
  g.a_e3m2 = p->a_fmt == MXFA_FMT_E3M2;
  g.b_e3m2 = p->b_fmt == MXFA_FMT_E3M2;
  static const char* const names[2][2] = {{"mxfa_gemm", "mxfa_gemm_be3m2"},
                                          {"mxfa_gemm_ae3m2", "mxfa_gemm_ae3m2_be3m2"}};
  const int64_t tm = (p->m + 255) / 256, tn = (p->n + 255) / 256;
  g.tiles_n = (int)tn;
  // MXFA_GEMM selects a kernel for comparison: big or dma the 256 x 256 tiles (big also below M =
  // 128), reg their register-staged form, mid the 128 x 128 tiles
  const char* sel = getenv("MXFA_GEMM");
  auto selected = [&](const char* name) { return sel && std::strcmp(sel, name) == 0; };
  const bool e4m3 = !g.a_e3m2 && !g.b_e3m2;
  // M <= 64 with E4M3 operands (the batched-decode projection): the skinny kernel, one workgroup per
  // 32-column strip (its LDS holds all of SA and the strip's SB: (k / 32) (m + 32) <= 96 KiB), while
  // the strips fit the chip at once (us, strips and 64 x 64 tiles, weights from HBM: N = 10,240, K = 512
  // M = 16 8.8 and 5.0, M = 32 9.3 and 5.2; K = 4,096 32.3 and 22.8, 34.1 and 23.6; K = 14,336 89 and 72,
  // 93 and 77) and, above M = 32, only for a long K.  Up to there the tiles are faster on weights that
  // the caches hold and the strips on weights from HBM (us, M = 64, N = 4,096: K = 4,096 11.2 and 7.6
  // cached, 21.0 and 20.8 from HBM; 6,144 13.9 and 9.4, 28.2 and 30.3; 8,192 23.1 and 22.4, 35.5 and
  // 38.5; N = 2,048, K = 8,192 18.9 and 14.6, 34.4 and 39.1), above it the strips either way (K =
  // 14,336, N = 4,096, cached: M = 16 30.6 and 35.1, 32 32.0 and 36.4, 64 38.9 and 40.7).
  const int64_t strips = (p->n + 31) / 32;
  if (e4m3 && p->m <= 64 && (p->k / 32) * (p->m + 32) <= 96 * 1024 && strips <= 256 && (p->m <= 32 || p->k > 8192) &&
      !selected("big") && !selected("reg") && !selected("mid")) {
    void* args[] = {&g};
    return launch(dm, p->m <= 32 ? "mxfa_gemm_skinny_t1" : "mxfa_gemm_skinny_t2", dim3((unsigned)strips), dim3(256), args,
                  stream);
  }
  // 64 x 64 tiles while there is a CU for each (E4M3; us for 64 and 128 tiles at K = 4,096: M = 128, N =
  // 6,144 13.3 and 18.3, M = 256, N = 4,096 9.9 and 13.6, M = N = 1,024 10.2 and 17.1; more than one
  // round, M = 400, N = 4,096: 20.4 and 14.0)
  const int64_t tiles64 = (p->m + 63) / 64 * ((p->n + 63) / 64);
  if (!sel && e4m3 && tiles64 <= 256) {
    g.tiles_n = (int)((p->n + 63) / 64);
    void* args[] = {&g};
    return launch(dm, "mxfa_gemm_small_dma", dim3((unsigned)tiles64), dim3(256), args, stream);
  }
  // 128 x 128 tiles (the same sums in the same order) while the 256 x 256 tiles are at most two
  // rounds over the CUs and the smaller ones at most twice as many: a K step of 128 takes 0.3 us
  // against 1.1.  N = 6,144, K = 4,096: M = 400 16 against 43 us, 1,024 (384 tiles of 128) 36 against
  // 44; 2,048 (768, three rounds against one) 57 against 47.  With E3M2 operands (two workgroups
  // per CU): M = 400 35 against 69 us, 1,024 50 against 69.  A second round of them pays from k = 1,024
  // on, or where the 256 x 256 tiles would be the register-staged ones (k % 128 = 64): M = 1,024, N =
  // 6,144, 256 and 128 tiles: k = 128 8.8 and 10.1 us, 192 12.6 and 10.2, 384 11.1 and 11.8, 768 16.2 and
  // 17.3, 1,024 20.0 and 20.6, 2,048 34.0 and 31.9; N = 5,120 1,024 19.7 and 19.1.
  const int64_t tiles128 = (p->m + 127) / 128 * ((p->n + 127) / 128);
  const int64_t rounds256 = (tm * tn + 255) / 256;
  if (selected("mid") || (!sel && rounds256 <= 2 &&
                          (e4m3 ? tiles128 <= 256 || ((p->k >= 1024 || p->k % 128) && (tiles128 + 255) / 256 <= 2 * rounds256)
                                : (tiles128 + 511) / 512 <= rounds256))) {
    g.tiles_n = (int)((p->n + 127) / 128);
    const char* mid = e4m3         ? "mxfa_gemm_mid_dma"
                      : !g.a_e3m2  ? "mxfa_gemm_mid_be3m2"
                      : !g.b_e3m2  ? "mxfa_gemm_mid_ae3m2"
                                   : "mxfa_gemm_mid_ae3m2_be3m2";
    void* args[] = {&g};
    return launch(dm, mid, dim3((unsigned)tiles128), dim3(256), args, stream);
  }
  // The 256 x 256 kernels are built for one workgroup size (their launch bounds): 256 or 512
  // threads.  E4M3 operands with whole K steps (k % 128 == 0) take the LDS-DMA kernel.
  const bool dma = e4m3 && p->k % 128 == 0 && !selected("reg");
  const char* name = dma ? "mxfa_gemm_dma" : names[g.a_e3m2][g.b_e3m2];
  int threads = 0;
  MXFA_HIP(hipFuncGetAttribute(&threads, HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK, fn_by_name(dm, name)));
  if (threads != 256 && threads != 512)
    return fail(MXFA_ERR_MODULE, std::string(name) + " has an unexpected workgroup size " + std::to_string(threads));
  void* args[] = {&g};
  return launch(dm, name, dim3((unsigned)(tm * tn)), dim3((unsigned)threads), args, stream);
}

mxfa_status mxfa_fill_normal(float* x, int64_t n, uint64_t seed, float outlier_p, float outlier_mul, void* stream) {
  if (n < 0) return fail(MXFA_ERR_INVALID_ARG, "n must be >= 0");
  if (n == 0) return MXFA_OK;
  if (!x) return fail(MXFA_ERR_INVALID_ARG, "NULL pointer");
  if (mxfa_status st = check_grid((n + 255) / 256, 256)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  dim3 grid((unsigned)((n + 255) / 256));
  void* args[] = {&x, &n, &seed, &outlier_p, &outlier_mul};
  return launch(dm, "mxfa_fill_normal_f32", grid, dim3(256), args, stream);
}

}  // extern "C"

namespace {
// The merge of a.n_qblk partials of each of `rows` output rows (mxfa_decode_combine).
mxfa_status launch_combine(DeviceModule* dm, FaArgs& a, int64_t rows, int D, void* stream) {
  const int nparts = a.n_qblk;
  void* args[] = {&a};
  // Groups of 16 threads per workgroup of the merge: 4 up to 32 partials, where more threads
  // cost more than their partials in flight give (24 partials of 128 heads 4.0 us against 4.1 with
  // 16 groups and 5.0 with 64; 16 partials of 2,048 heads 6.2, 8.6 and 28), then 16 (64 partials of
  // 128 heads 3.3 against 4.5 with 4) and above 128 partials 32 (256 of 32 heads 5.2 against
  // 11.2 and 6.0 with 4 and 16).
  if (nparts <= 4)
    return launch(dm, "mxfa_decode_combine", dim3((unsigned)rows), dim3((unsigned)(D / 4)), args, stream);
  return launch(dm, "mxfa_decode_combine", dim3((unsigned)rows, (unsigned)(D / 64)),
                dim3(nparts <= 32 ? 64 : nparts <= 128 ? 256 : 512), args, stream);
}

// Workgroup shape of the prefill kernels: nw waves, hpw query heads (of one KV head) per
// workgroup, nw / hpw 32-query waves each.
FaArgs prefill_args(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k,
                    const uint8_t* k_sc, const uint8_t* v, const uint8_t* v_sc, float* o, int nw, dim3& grid) {
  FaArgs a = make_args(p, q, q_sc, k, k_sc, v, v_sc, o);
  a.hpw = 1;
  for (int h = nw; h > 1; h /= 2)
    if (a.group % h == 0) {
      a.hpw = h;
      break;
    }
  a.qpw = 32 * (nw / a.hpw);
  a.n_qblk = (p->seq_q + a.qpw - 1) / a.qpw;
  grid = dim3((unsigned)a.n_qblk, (unsigned)(p->batch * p->num_kv_heads * (a.group / a.hpw)));
  return a;
}

// Wave-blocks (32 queries x 64 keys) of one launch of the prefill3 grid: every wave of a
// workgroup walks the workgroup's key blocks [j0, j1) (the kernels' own loop bounds).
int64_t prefill3_wave_blocks(const FaArgs& a, const mxfa_attn_params* p) {
  const int nkb = (p->seq_k + 63) / 64;
  int64_t per_group = 0;
  for (int qblk = 0; qblk < a.n_qblk; qblk++) {
    const int q0 = qblk * a.qpw, qmax = std::min(q0 + a.qpw, p->seq_q) - 1;
    const int j0 = p->window > 0 ? std::max(0, p->q_pos0 + q0 - p->window + 1) / 64 : 0;
    const int j1 = p->causal ? std::min(nkb, std::max(0, p->q_pos0 + qmax) / 64 + 1) : nkb;
    per_group += 4 * std::max(0, j1 - j0);
  }
  return per_group * p->batch * p->num_kv_heads * (a.group / a.hpw);
}

// mxfa_prefill_ws widens K to bf16 once, into the workspace, by a pre-pass -- or leaves it to
// the workspace-free kernel, whose workgroups widen each block they read in LDS: each K
// element about 16 * wave_blocks / (B * Hkv * Sk) times.  Measured (same box): at 8.5 (MHA,
// S = 2048) the in-LDS form is 3.4% faster; at 49 (Gemma shape) 2-4% and at 65 (GQA-4, S =
// 4096) 6.5% slower.  Below 32 the call runs the workspace-free kernel (the workspace is
// then not touched).
bool prefill_ws_widens_in_lds(const FaArgs& a, const mxfa_attn_params* p) {
  return 16 * prefill3_wave_blocks(a, p) < (int64_t)32 * p->batch * p->num_kv_heads * p->seq_k;
}

// Waves per workgroup of the workspace kernel (mxfa_prefill3_*).
int prefill3_waves(const mxfa_attn_params*) { return 4; }

// Workspace of mxfa_prefill_ws: the bf16 copy of K, then (E3M2 V) the E4M3 copy of V.
size_t prefill3_kbf_bytes(const mxfa_attn_params* p) {
  return (size_t)p->batch * p->num_kv_heads * p->seq_k * p->head_dim * 2;
}
size_t prefill3_workspace(const mxfa_attn_params* p) {
  const size_t v = p->v_fmt == MXFA_FMT_E3M2 ? (size_t)p->batch * p->num_kv_heads * p->seq_k * p->head_dim : 0;
  return prefill3_kbf_bytes(p) + v;
}

// Whether n ranges of a call's `longest` key blocks take less time than one walk over them, by an
// estimate in us fitted to 1,377 calls (D = 64, 128, 256; 1 to 512 rows, batch 1 to 64, 1,000 to 32,768
// keys), each timed both ways: a block takes `block` in a workgroup that has its CU nearly to
// itself; one walk slows down by 0.9 per workgroup and CU, n ranges by `share` (their waves hide
// each other's latency); the maxima add a third; two more launches and the ramp cost 8 us, the
// partials 3 MB per us written and read.  Of the 1,133 calls that the other rules split it leaves
// out 51: 40 are slower split (1.9 times at most), 5 gain more than 4% (13% at most).  Of the calls
// still split the worst loses 4%.
bool split_pays(const mxfa_attn_params* p, int64_t items, int longest, int n, int64_t partial_bytes) {
  const double block = (p->head_dim == 256 ? 2.8 : p->head_dim == 128 ? 1.8 : 1.3) *
                       (1.0 + (p->softcap > 0.0f ? 0.3 : 0.0) + (p->p_rule == MXFA_P_R2 ? 0.15 : 0.0));
  const double share = p->head_dim == 256 ? 0.8 : p->head_dim == 128 ? 0.6 : 0.5;
  const double per_cu = items / 256.0;
  const double one = block * longest * std::max(1.0, 0.9 * per_cu);
  const double split = 8.0 + 4.0 / 3.0 * block * ((longest + n - 1) / n) * std::max(1.0, share * per_cu * n) +
                       2.0 * partial_bytes / 3e6;
  return split < one;
}

// Key ranges per query block of a mxfa_prefill_ws call (1: not split).  A few rows against a long
// cache (a prompt chunk, drafted tokens to verify) give a grid of `items` workgroups that leaves
// most of the chip idle for the whole walk over the keys.  Split, three launches: the row maxima
// of every range but the last (prefill_max_impl), the attention kernel per range, starting from
// the maximum of the ranges before it -- so every P and its code are the unsplit call's -- and
// the merge of the partials.  O differs from the unsplit call's by the order of fp32 sums only
// (rel-L2 3e-7 at most over 60 random calls, 6e-7 at 131,072 keys in 128 ranges, 1.3e-5 at 8,000,000 in
// 1,000).  Measured, unsplit -> split (ranges):
//   Hq 32, Hkv 8, D = 128:  200 rows x 32,768 keys 1,009 -> 207 us (13), 8 x 8,192 254 -> 28 (32),
//     8 x 1,024 36 -> 18 (11), batch 8 of 8 x 4,096 131 -> 47 (12), 512 x 16,384 391 -> 258 (3)
//   Hq 16, Hkv 8, D = 256:  256 x 16,384 631 -> 123 (16), 30 x 2,048 softcap 111 -> 30 (16), 256 x
//     32,768 with a window of 4,096, softcap and 6-bit V 192 -> 68 (16)
//   Hq 16, Hkv 16, D = 64:  300 x 16,384 402 -> 75 (21)
// - as many ranges as fill the slots the kernel's registers leave (two workgroups per CU at D =
//   256, three at 128, four at 64), and not more than sqrt(8 x key blocks): a range's time falls
//   with their number, the merge's grows (128 blocks: 61, 28, 30 us with 8, 32, 48 ranges; 32
//   blocks: 24, 19, 21 with 8, 16, 24);
// - as many partials as the workspace of the plan holds in place of the operand copies;
// - at least 3: with 2 ranges the maxima (a third of the pass) and the merge eat the gain once
//   there is a workgroup for most CUs (256 items: 131 against 132 us); up to 128 items 2 still win
//   (32 x 8,192 x 8 rows 207 against 254 us);
// - from 16 visible key blocks on (8 rows; 8 blocks: 20 -> 18 us only), and for more than one query
//   tile per head (32 rows) in calls of more than 5,120 keys: shorter ones keep their
//   bit-identity with mxfa_prefill, at the price of what 64 rows x 4,096 keys could gain (103 ->
//   40 us);
// - where the split is estimated to be the faster form (split_pays): many rows over a short range
//   spend more on writing and merging the partials than the shorter walk saves (batch 32 of 32
//   rows x 1,000 keys, D = 64: 26 -> 51 us split; batch 24, D = 128: 39 -> 60; batch 20, D = 256:
//   50 -> 77).
int prefill_splits(const FaArgs& a, const mxfa_attn_params* p, int64_t items) {
  const int64_t slots = p->head_dim == 256 ? 512 : p->head_dim == 128 ? 768 : 1024;
  const int nkb = (p->seq_k + 63) / 64;
  int longest = 0;
  for (int qblk = 0; qblk < a.n_qblk && slots / items > 1; qblk++) {
    const int q0 = qblk * a.qpw, qmax = std::min(q0 + a.qpw, p->seq_q) - 1;
    const int j0 = p->window > 0 ? std::max(0, p->q_pos0 + q0 - p->window + 1) / 64 : 0;
    const int j1 = p->causal ? std::min(nkb, std::max(0, p->q_pos0 + qmax) / 64 + 1) : nkb;
    longest = std::max(longest, j1 - j0);
  }
  if (longest < 16 || (p->seq_q > 32 && p->seq_k <= 5120)) return 1;
  const int64_t row_bytes = (int64_t)p->batch * p->num_q_heads * p->seq_q * (p->head_dim + 3) * (int64_t)sizeof(float);
  int64_t n = std::min(slots / items, (int64_t)std::sqrt(8.0 * longest));
  n = std::min(n, (int64_t)prefill3_workspace(p) / row_bytes);
  return (n >= 3 || (n == 2 && items <= 128)) && split_pays(p, items, longest, (int)n, n * row_bytes) ? (int)n : 1;
}

}  // namespace

extern "C" {

mxfa_status mxfa_prefill(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k,
                         const uint8_t* k_sc, const uint8_t* v, const uint8_t* v_sc, float* o, void* stream) {
  if (mxfa_status st = check_params(p, false)) return st;
  const void* ptrs[] = {q, q_sc, k, k_sc, v, v_sc, o};
  if (mxfa_status st = check_ptrs(ptrs, 7)) return st;
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  dim3 grid;
  FaArgs a = prefill_args(p, q, q_sc, k, k_sc, v, v_sc, o, 4, grid);
  void* args[] = {&a};
  // the workspace kernel's design in its workspace-free form: K widened to bf16 in LDS, E3M2
  // V read as E5M2
  return launch(dm, kernel_name("prefill3n", p, true), grid, dim3(256), args, stream);
}

mxfa_status mxfa_prefill_plan(const mxfa_attn_params* p, size_t* workspace_bytes) {
  if (mxfa_status st = check_params(p, false)) return st;
  if (!workspace_bytes) return fail(MXFA_ERR_INVALID_ARG, "workspace_bytes is NULL");
  *workspace_bytes = prefill3_workspace(p);
  return MXFA_OK;
}

}  // extern "C"

namespace {
// The workspace prefill (mxfa_prefill_ws), or with tr set its stage trace: the one
// workgroup that holds query rows 32 * tr->q_tile .. + 31 of head tr->bh.
struct TraceReq {
  int32_t bh, q_tile;
  float *s_out, *ml_out;
  uint8_t *p_out, *ps_out;
};

mxfa_status prefill_ws_impl(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k,
                            const uint8_t* k_sc, const uint8_t* v, const uint8_t* v_sc, float* o, void* workspace,
                            size_t workspace_bytes, void* stream, const TraceReq* tr) {
  const void* ptrs[] = {q, q_sc, k, k_sc, v, v_sc, o};
  if (mxfa_status st = check_ptrs(ptrs, 7)) return st;
  const size_t need = prefill3_workspace(p);
  if (!workspace || workspace_bytes < need)
    return fail(MXFA_ERR_WORKSPACE, "prefill workspace needs " + std::to_string(need) + " bytes");
  if (!aligned16(workspace)) return fail(MXFA_ERR_INVALID_ARG, "workspace must be 16-byte aligned");
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  const int nw = prefill3_waves(p);
  dim3 grid;
  FaArgs a = prefill_args(p, q, q_sc, k, k_sc, v, v_sc, o, nw, grid);
  const int nsplit = tr ? 1 : prefill_splits(a, p, (int64_t)grid.x * grid.y);
  if (nsplit > 1) {
    // the workspace holds the partials instead of the operand copies: O, (m, l), row maxima
    const int64_t rows = (int64_t)p->batch * p->num_q_heads * p->seq_q;
    a.nsplit = nsplit;
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = a.part_o + rows * nsplit * p->head_dim;
    a.part_max = a.part_ml + rows * nsplit * 2;
    const unsigned items = grid.x * grid.y;
    void* args[] = {&a};
    char name[64];
    std::snprintf(name, sizeof name, "mxfa_prefill_max_d%d%s", p->head_dim, p->softcap > 0.0f ? "_softcap" : "");
    if (mxfa_status st = launch(dm, name, dim3(items * (unsigned)(nsplit - 1)), dim3(256), args, stream)) return st;
    if (mxfa_status st = launch(dm, kernel_name("prefill3s", p, true), dim3(items * (unsigned)nsplit), dim3(256), args, stream))
      return st;
    a.n_qblk = nsplit;
    return launch_combine(dm, a, rows, p->head_dim, stream);
  }
  if (!tr && prefill_ws_widens_in_lds(a, p)) {
    void* args[] = {&a};
    return launch(dm, kernel_name("prefill3n", p, true), grid, dim3(256), args, stream);
  }
  uint8_t* kbf = static_cast<uint8_t*>(workspace);
  // (E3M2 V codes one per byte: widened to E4M3 by the pre-pass; block-packed E3M2 V is read
  // by the kernel as it is)
  uint8_t* vws = p->v_fmt == MXFA_FMT_E3M2 ? kbf + prefill3_kbf_bytes(p) : nullptr;
  a.kbf = kbf;
  a.vws = vws;
  // bf16 K (and E4M3 V) in one launch: 16 pieces of 8 codes per thread, one (batch, KV head)
  // per grid row
  int D = p->head_dim, Sk = p->seq_k, Skc = a.Skc;
  const int64_t pieces = (int64_t)Sk * (D / 8);    // per (batch, KV head)
  if (pieces > INT32_MAX - 256 * 16) return fail(MXFA_ERR_UNSUPPORTED, "seq_k * head_dim / 8 exceeds the workspace pre-pass's range");
  const dim3 cgrid((unsigned)((pieces + 256 * 16 - 1) / (256 * 16)), (unsigned)(p->batch * p->num_kv_heads));
  void* cargs[] = {(void*)&k, (void*)&k_sc, (void*)&v, &D, &Sk, &Skc, &kbf, &vws};
  if (mxfa_status st = launch(dm, "mxfa_k_to_bf16", cgrid, dim3(256), cargs, stream)) return st;
  void* args[] = {&a};
  if (!tr) return launch(dm, kernel_name("prefill3", p, p->v_fmt == MXFA_FMT_E3M2_BLK), grid, dim3((unsigned)(64 * nw)),
                         args, stream);
  // the item (qx, qy) of the traced rows, as the kernel's own mapping assigns them
  const int b = tr->bh / p->num_q_heads, head = tr->bh % p->num_q_heads;
  const int kvh = head / a.group, hc = (head % a.group) / a.hpw;
  const int qblk = 32 * tr->q_tile / a.qpw;
  a.tr_qy = (b * p->num_kv_heads + kvh) * (a.group / a.hpw) + hc;
  a.tr_qx = p->causal ? a.n_qblk - 1 - qblk : qblk;
  a.tr_head = head;
  a.tr_q0 = 32 * tr->q_tile;
  a.tr_s = tr->s_out;
  a.tr_ml = tr->ml_out;
  a.tr_p = tr->p_out;
  a.tr_ps = tr->ps_out;
  return launch(dm, kernel_name("prefill3_trace", p), dim3(1), dim3((unsigned)(64 * nw)), args, stream);
}
}  // namespace

extern "C" {

mxfa_status mxfa_prefill_ws(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k,
                            const uint8_t* k_sc, const uint8_t* v, const uint8_t* v_sc, float* o, void* workspace,
                            size_t workspace_bytes, void* stream) {
  if (mxfa_status st = check_params(p, false)) return st;
  return prefill_ws_impl(p, q, q_sc, k, k_sc, v, v_sc, o, workspace, workspace_bytes, stream, nullptr);
}

mxfa_status mxfa_prefill_trace(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k,
                               const uint8_t* k_sc, const uint8_t* v, const uint8_t* v_sc, float* o,
                               void* workspace, size_t workspace_bytes, int32_t bh, int32_t q_tile, float* s_out,
                               float* ml_out, uint8_t* p_out, uint8_t* ps_out, void* stream) {
  if (mxfa_status st = check_params(p, false)) return st;
  if (bh < 0 || bh >= p->batch * p->num_q_heads || q_tile < 0 || 32 * q_tile >= p->seq_q)
    return fail(MXFA_ERR_INVALID_ARG, "bh or q_tile out of range");
  if (!s_out || !ml_out || !p_out || !ps_out) return fail(MXFA_ERR_INVALID_ARG, "NULL trace buffer");
  if (p->v_fmt == MXFA_FMT_E3M2_BLK) return fail(MXFA_ERR_UNSUPPORTED, "the stage trace reads V as E4M3 or E3M2 codes");
  const TraceReq tr = {bh, q_tile, s_out, ml_out, p_out, ps_out};
  return prefill_ws_impl(p, q, q_sc, k, k_sc, v, v_sc, o, workspace, workspace_bytes, stream, &tr);
}

mxfa_status mxfa_decode_plan(const mxfa_attn_params* p, int32_t* n_parts, size_t* workspace_bytes) {
  if (mxfa_status st = check_params(p, true)) return st;
  if (n_parts) *n_parts = decode_parts(p);
  // sized for the most partials a call of this shape could take, so that it never shrinks with a
  // longer cache
  if (workspace_bytes)
    *workspace_bytes = (size_t)p->batch * p->num_q_heads * decode_parts_max(p) * (p->head_dim + 2) * sizeof(float) + 256;
  return MXFA_OK;
}

}  // extern "C"

namespace {

// The decode launches of mxfa_decode and mxfa_decode_noalloc (arguments already checked;
// workspace holds the partials of the two-launch path).
mxfa_status decode_launch(DeviceModule* dm, const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc,
                          const uint8_t* k_cache, const uint8_t* k_sc, const uint8_t* v_cache, const uint8_t* v_sc,
                          float* o, void* workspace, void* stream) {
  FaArgs a = make_args(p, q, q_sc, k_cache, k_sc, v_cache, v_sc, o);
  const int nparts = decode_parts(p);
  a.n_qblk = nparts;
  int64_t nbh = (int64_t)p->batch * p->num_q_heads;
  a.part_o = reinterpret_cast<float*>(workspace);
  a.part_ml = a.part_o + nbh * nparts * p->head_dim;
  // 4 waves per workgroup over the linear (b, KV head, chunk) items
  const int nw = 4;
  const int64_t items = (int64_t)p->batch * p->num_kv_heads * nparts;
  const dim3 grid((unsigned)((items + nw - 1) / nw));
  // When every head's partials fit in one workgroup (nparts divides its 4 waves) and the
  // valid columns' partials fit the waves' V slots (group <= 16), the kernel merges them
  // itself (same formula and order as mxfa_decode_combine) and no combine launch follows.
  // MXFA_DECODE_COMBINE=kernel selects the combine kernel always (the two paths give
  // bit-identical O; the switch exists to test exactly that).
  const char* comb = getenv("MXFA_DECODE_COMBINE");
  const bool force_kernel = comb && std::strcmp(comb, "kernel") == 0;
  a.fuse_combine = !force_kernel && nw % nparts == 0 && a.group <= 16;
  void* args[] = {&a};
  if (mxfa_status st = launch(dm, kernel_name("decode", p, p->v_fmt == MXFA_FMT_E3M2_BLK), grid, dim3(64 * nw), args,
                              stream))
    return st;
  if (a.fuse_combine) return MXFA_OK;
  return launch_combine(dm, a, nbh, p->head_dim, stream);
}

}  // namespace

extern "C" {

mxfa_status mxfa_decode(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc, const uint8_t* k_cache,
                        const uint8_t* k_sc, const uint8_t* v_cache, const uint8_t* v_sc, float* o, void* workspace,
                        size_t workspace_bytes, void* stream) {
  if (mxfa_status st = check_params(p, true)) return st;
  const void* ptrs[] = {q, q_sc, k_cache, k_sc, v_cache, v_sc, o};
  if (mxfa_status st = check_ptrs(ptrs, 7)) return st;
  size_t need = 0;
  int32_t sl = 0;
  mxfa_decode_plan(p, &sl, &need);
  if (!workspace || workspace_bytes < need)
    return fail(MXFA_ERR_WORKSPACE, "decode workspace must be at least " + std::to_string(need) + " bytes");
  if (!aligned16(workspace)) return fail(MXFA_ERR_INVALID_ARG, "workspace must be 16-byte aligned");
  DeviceModule* dm;
  if (mxfa_status st = module_for_current(&dm)) return st;
  return decode_launch(dm, p, q, q_sc, k_cache, k_sc, v_cache, v_sc, o, workspace, stream);
}

mxfa_status mxfa_decode_noalloc(const mxfa_attn_params* p, const uint8_t* q, const uint8_t* q_sc,
                                const uint8_t* k_cache, const uint8_t* k_sc, const uint8_t* v_cache,
                                const uint8_t* v_sc, float* o, void* stream) {
  if (mxfa_status st = check_params(p, true)) return st;
  const void* ptrs[] = {q, q_sc, k_cache, k_sc, v_cache, v_sc, o};
  if (mxfa_status st = check_ptrs(ptrs, 7)) return st;
  size_t need = 0;
  int32_t sl = 0;
  mxfa_decode_plan(p, &sl, &need);
  if (need > MXFA_DECODE_SCRATCH_BYTES)
    return fail(MXFA_ERR_WORKSPACE, "mxfa_decode_noalloc: the partials of this shape need " + std::to_string(need) +
                                        " bytes, above the " + std::to_string(MXFA_DECODE_SCRATCH_BYTES) +
                                        "-byte device scratch; use mxfa_decode with a workspace");
  DeviceModule* dm;
  if (mxfa_status st = loaded_module_for_current(&dm)) return st;
  return decode_launch(dm, p, q, q_sc, k_cache, k_sc, v_cache, v_sc, o, dm->decode_scratch, stream);
}

}  // extern "C"
