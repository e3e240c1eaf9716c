// zlm_gpu_hip.cpp -- host side of the MI355X backend: the C ABI declared in
// include/zlm_gpu_hip.h over the HIP runtime.
//
// The kernels live in gfx950 code objects next to this library, loaded with
// hipModuleLoad: zlm_kernels_gfx950.hsaco (layout, dequant, quantizer, GEMM,
// decode glue; $ZLM_HIP_CODE_OBJECT overrides its path) and one
// zlm_gemv_<quant>_gfx950.hsaco per quant with that quant's GEMV forms.  One HIP
// stream per device carries every copy and launch in order, so a burst's
// shared activation and a resident's layout conversion are ordered before the
// kernels that read them without extra synchronisation.
//
// Contract behaviour follows the reference Vulkan device
// (src/gpu/backend/vulkan/root.zig, pipeline.zig); the differences are
// deliberate hardening of the invariants that device leaves implicit:
//   * the 8-slot ring refuses a 9th in-flight submit instead of silently
//     reusing a slot (reference pipeline.zig:1353-1355 wraps unconditionally);
//     handles carry a generation, so a stale handle is refused by wait;
//   * a burst member must pass the same x pointer and length as the burst's
//     first submit (reference pipeline.zig:264-276 only documents it).
#include "zlm_gpu_hip.h"

#include "zlm_static_scratch.h"

#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <link.h>
#include <time.h>

#include <algorithm>
#include <cctype>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <unordered_map>
#include <string>
#include <vector>

namespace {

constexpr int kRing = ZLM_RING_SIZE;
constexpr uint32_t kNoLayout = 0xffffffffu;
// Library scratch kinds a captured graph can reference.
constexpr uint32_t kUsesAttn = 1u;  // the attention partials
constexpr uint32_t kUsesGemm = 2u;  // the GEMM's quantized activations and the residents' GEMM tiles
constexpr uint32_t kQ4kRecords = 0xfffffffeu;
constexpr uint32_t kQ6kRecords = 0xfffffffdu;

// Supported GEMV quants and their GGUF block geometry (the contract's
// blockElems/blockBytes, reference gpu/backend/root.zig:198-220: the float
// types count one element per block).
struct QuantInfo {
    uint32_t type;
    uint32_t block_elems;
    uint32_t block_bytes;
    uint32_t payload_bytes;  // bytes per block in the device layout (scales split out)
    uint32_t scale_offset;   // offset of the f16 scales inside the raw block, kNoLayout (raw layout),
                             // kQ4kRecords (zlm_repack_q4_k) or kQ6kRecords (zlm_repack_q6_k)
    int slot;                // index into the kernel tables
    uint32_t scale_count;    // 16-bit words per block in the scale area (q4_1: d and m; q4_k / q6_k:
                             // their 20- / 84-byte records)
    uint32_t chunk_elems;    // elements per 16-byte payload chunk of a row (the GEMV's unit)
    uint32_t kblock;         // elements per kernel block: the kernels take nb = k / kblock
};

const QuantInfo kQuants[] = {
    {ZLM_GGML_Q4_0, 32, 18, 16, 0, 0, 1, 32, 32},
    {ZLM_GGML_Q8_0, 32, 34, 32, 0, 1, 1, 16, 32},
    {ZLM_GGML_Q4_K, 256, 144, 128, kQ4kRecords, 2, 10, 32, 256},
    {ZLM_GGML_Q6_K, 256, 210, 128, kQ6kRecords, 3, 42, 32, 256},
    {ZLM_GGML_Q4_1, 32, 20, 16, 0, 4, 2, 32, 32},
    {ZLM_GGML_F32, 1, 4, 4, kNoLayout, 5, 0, 4, 32},
    {ZLM_GGML_F16, 1, 2, 2, kNoLayout, 6, 0, 8, 32},
    {ZLM_GGML_BF16, 1, 2, 2, kNoLayout, 7, 0, 8, 32},
};
constexpr int kNumQuants = 8;
const char* const kQuantNames[kNumQuants] = {"q4_0", "q8_0", "q4_k", "q6_k", "q4_1", "f32", "f16", "bf16"};

const QuantInfo* quant_info(uint32_t quant) {
    const uint32_t t = quant & 0xffu;
    for (const QuantInfo& q : kQuants)
        if (q.type == t) return &q;
    return nullptr;
}

uint32_t variant_of(uint32_t quant) { return (quant >> 8) & 0xffu; }

// A fused op's quant code carrying the op's `variant` argument (a GpuVariant
// code; 0 keeps whatever variant the quant code itself carries).
uint32_t with_variant(uint32_t quant, uint32_t variant) {
    return variant ? ((quant & 0xffu) | ((variant & 0xffu) << 8)) : quant;
}

// GEMV kernels: 4 waves (256 threads) per workgroup unless an instance's launch
// bounds say otherwise; k up to 32768.
constexpr size_t kMaxK = 32768;

// GpuVariant -> rows per wave tile.  The reference's variants are Vulkan
// spec-constant axes (gpu/kernels/grid.zig:41-53): `u4`/`u8` (its 8-row group)
// select the 4-row tile, `un2`/`un4` the 2-row tile, every other variant the
// default 1-row tile (the fastest measured on gfx950 for the benchmark
// shapes).  A variant never changes results beyond fp32 summation order.
int rt_for_variant(uint32_t v) {
    switch (v) {
    case ZLM_VARIANT_U4:
    case ZLM_VARIANT_U8:
        return 4;
    case ZLM_VARIANT_UN2:
    case ZLM_VARIANT_UN4:
        return 2;
    default:
        return 1;
    }
}

// A resolved GEMV kernel: rows per tile and exact steps (0 = generic).
struct GemvKernel {
    hipFunction_t fn = nullptr;
    int rt = 0;
    int steps = 0;
    int threads = 256;     // the kernel's launch bounds
    int waves_per_cu = 0;  // grid target of a prefetching instance; 0 = gemv_grid's rule
    bool struct_args = false;  // takes one GemvArgs (fused forms, prefetching instances)
    int role = 0;              // kernel_role(): the form it computes, or kRoleMulti
    bool split = false;        // split-K: the workgroup's waves share each tile of rt rows
    bool xq = false;           // sums in another order than the batch kernel (int8-plane x or split-K)
};

struct Slot {
    hipEvent_t done = nullptr;
    float* h_y = nullptr;  // pinned; the result kernel writes it through h_y_dev
    float* h_y_dev = nullptr;
    size_t y_cap = 0;
    float* d_x = nullptr;
    float* h_x = nullptr;
    float* h_x_dev = nullptr;
    size_t x_cap = 0;
    float* h_bx = nullptr;  // pinned; a burst's activation when this slot is its first member
    float* h_bx_dev = nullptr;
    size_t bx_cap = 0;
    bool pending = false;
    uint32_t gen = 0;
    size_t rows = 0;
};

}  // namespace

struct zlm_resident {
    uint64_t bytes = 0;
    uint8_t* raw = nullptr;        // device copy of the raw blocks, until converted
    uint8_t* payload = nullptr;    // device layout payload
    uint16_t* scales = nullptr;    // device layout scales (split quants)
    uint32_t layout = kNoLayout;   // GGML type of the device layout
    uint64_t blocks = 0;           // whole blocks in the layout
    // The prefill GEMM's tiled copy of a Q4_0 / Q8_0 weight ([rows/32][nb][32]
    // [16 or 32 B] + scales [rows/32][nb][32]), built on the first GEMM for a
    // given nb.
    uint8_t* gemm_payload = nullptr;
    void* gemm_scales = nullptr;  // f16 (q4_0, q8_0) or float2 (scale, min) (q4_1, q4_k)
    uint64_t gemm_nb = 0;
    uint64_t gemm_rt = 0;  // 32-row tiles
    uint64_t tiles_due = 0;  // row length (blocks) whose tiles the next capture builds (build_tiles_due); 0 = none
    uint64_t layout_alloc = 0;  // device bytes of the layout allocation
    uint64_t gemm_alloc = 0;    // device bytes of the GEMM tile allocation
    zlm_device* owner = nullptr;
};

struct zlm_device {
    bool avail = false;
    int ordinal = 0;
    int cus = 0;
    char name[256] = "off";
    std::string err;

    hipModule_t mod = nullptr;          // zlm_kernels_gfx950.hsaco
    hipModule_t gemv_mod[kNumQuants] = {};  // zlm_gemv_<quant>_gfx950.hsaco, by QuantInfo::slot
    std::map<std::string, GemvKernel> gemv;  // by entry-point name; null fn = absent
    std::unordered_map<uint64_t, const GemvKernel*> picks;  // kernel picked per shape class (pick_key)
    hipFunction_t repack = nullptr;
    hipFunction_t repack_q4_k = nullptr;
    hipFunction_t repack_q6_k = nullptr;
    hipFunction_t dequant[kNumQuants] = {};
    hipFunction_t quantize_q8 = nullptr;
    hipFunction_t quantize_q8_tiled = nullptr;
    hipFunction_t tile_q4_0 = nullptr;
    hipFunction_t tile_q8_0 = nullptr;
    hipFunction_t tile_q4_1 = nullptr;
    hipFunction_t tile_q4_k = nullptr;
    hipFunction_t gemm_q4_1 = nullptr;
    hipFunction_t gemm_q4_k = nullptr;
    hipFunction_t copy16 = nullptr;
    hipFunction_t gemm_small_q4_0 = nullptr;  // m <= kGemmSmallM: split-K, one 32-token tile
    hipFunction_t gemm_small_q8_0 = nullptr;
    hipFunction_t gemm_small_q4_1 = nullptr;
    hipFunction_t gemm_small_q4_k = nullptr;
    // the tiled GEMMs with each tile's blocks split over two wave groups
    hipFunction_t gemm_q4_0_k2 = nullptr;
    hipFunction_t gemm_q8_0_k2 = nullptr;
    hipFunction_t gemm_q4_0_k4 = nullptr;
    hipFunction_t gemm_q8_0_k4 = nullptr;
    hipFunction_t gemm_q4_0 = nullptr;  // unsplit
    hipFunction_t gemm_q8_0 = nullptr;
    hipFunction_t gemm_q4_1_k2 = nullptr;
    hipFunction_t gemm_q4_k_k2 = nullptr;
    // the wide fp6 GEMM (q4_1 / q4_k; 128-token x 192-row tiles, 12 waves) and its activations
    hipFunction_t quantize_fp6 = nullptr;
    hipFunction_t gemm_wide = nullptr;
    // 3 to 8 tokens by a tall weight, from the GEMV layout: k up to 4096, up to 8192
    hipFunction_t gemm_tall[kNumQuants][2] = {};
    hipFunction_t qk_norm_rope_kv = nullptr;
    hipFunction_t attn_partial = nullptr;
    hipFunction_t attn_combine = nullptr;
    hipFunction_t attn_combine_wide = nullptr;
    hipFunction_t attn_decode = nullptr;
    hipFunction_t synth_blocks = nullptr;
    hipFunction_t synth_f16 = nullptr;

    // attention partials (per q head and 64-position split: 128 acc + m + l)
    float* attn_part = nullptr;
    size_t attn_part_cap = 0;
    bool capturing = false;
    // Library scratch a capture recorded (kUses* bits, collected while the
    // capture is open) and, per kind, the captured graphs not yet destroyed
    // that reference it: a graph replays with the addresses it was captured
    // with.
    uint32_t capture_uses = 0;
    // static LDS bytes per kernel (launch checks) and the optional launch log
    std::unordered_map<hipFunction_t, uint32_t> lds_bytes;
    bool log_launches = false;
    std::vector<zlm_launch_record> launch_log;
    int attn_graphs = 0;
    int gemm_graphs = 0;
    // this device's address of the fixed static scratch (the no-alloc entry
    // point's partials); null if the lookup at init failed
    float* static_scratch = nullptr;
    std::string static_scratch_err;

    // prefill scratch: quantized activations (qx, dx, sums) and staged x/out
    uint8_t* q_scratch = nullptr;
    uint64_t q_scratch_cap = 0;
    uint64_t q_scratch_refused = UINT64_MAX;  // fewest bytes an optional growth was refused (grow_gemm_scratch)
    std::vector<zlm_resident*> tiles_due;  // the residents with tiles_due set
    hipStream_t stream = nullptr;

    Slot slots[kRing];
    int next_slot = 0;

    // synchronous-op staging (pinned host halves mapped for the device: x is
    // copied in by the copy kernel, y written by the GEMV itself)
    float* d_x = nullptr;
    float* h_x = nullptr;
    float* h_x_dev = nullptr;
    size_t x_cap = 0;
    float* d_y = nullptr;
    float* h_y = nullptr;
    float* h_y_dev = nullptr;
    size_t y_cap = 0;
    uint8_t* s_raw = nullptr;  // streamed-weight staging (raw blocks)
    uint64_t s_raw_cap = 0;
    uint8_t* s_lay = nullptr;  // streamed-weight staging (device layout)
    uint64_t s_lay_cap = 0;

    // the fused MLP's ffn_mid (device only)
    float* d_mid = nullptr;
    size_t mid_cap = 0;

    // burst-shared activation (device; staged through the first member's slot)
    float* d_bx = nullptr;
    size_t bx_cap = 0;
    const float* burst_src = nullptr;
    size_t burst_len = 0;
    bool burst_open = false;
};

namespace {

bool fail(zlm_device* d, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (d) d->err = buf;
    return false;
}

bool ok(zlm_device* d, hipError_t e, const char* what) {
    if (e == hipSuccess) return true;
    return fail(d, "%s: %s", what, hipGetErrorString(e));
}

// Directory of this library (the code objects sit beside it).
std::string library_dir() {
    Dl_info info;
    if (dladdr(reinterpret_cast<void*>(&zlm_gpu_init), &info) && info.dli_fname) {
        std::string p(info.dli_fname);
        size_t slash = p.rfind('/');
        return (slash == std::string::npos) ? "." : p.substr(0, slash);
    }
    return ".";
}

void unload_modules(zlm_device* d) {
    if (d->mod) hipModuleUnload(d->mod);
    d->mod = nullptr;
    for (hipModule_t& m : d->gemv_mod) {
        if (m) hipModuleUnload(m);
        m = nullptr;
    }
    d->picks.clear();
    d->gemv.clear();
}

// The quants the tall kernel has (below, enqueue_gemm_tall).
bool gemm_tall_type(uint32_t type) { return type == ZLM_GGML_Q4_0 || type == ZLM_GGML_Q4_1 || type == ZLM_GGML_Q4_K; }

bool load_kernels(zlm_device* d) {
    const std::string dir = library_dir();
    const char* env = getenv("ZLM_HIP_CODE_OBJECT");
    const std::string path = env ? std::string(env) : dir + "/zlm_kernels_gfx950.hsaco";
    if (!ok(d, hipModuleLoad(&d->mod, path.c_str()), path.c_str())) return false;
    char nm[128];
    for (int q = 0; q < kNumQuants; q++) {
        const std::string gp = dir + "/zlm_gemv_" + kQuantNames[q] + "_gfx950.hsaco";
        if (!ok(d, hipModuleLoad(&d->gemv_mod[q], gp.c_str()), gp.c_str())) return false;
    }
    for (int q = 0; q < kNumQuants; q++) {
        snprintf(nm, sizeof nm, "zlm_dequant_%s", kQuantNames[q]);
        if (!ok(d, hipModuleGetFunction(&d->dequant[q], d->mod, nm), nm)) return false;
    }
    if (!ok(d, hipModuleGetFunction(&d->repack, d->mod, "zlm_repack_split"), "zlm_repack_split")) return false;
    if (!ok(d, hipModuleGetFunction(&d->repack_q4_k, d->mod, "zlm_repack_q4_k"), "zlm_repack_q4_k")) return false;
    if (!ok(d, hipModuleGetFunction(&d->repack_q6_k, d->mod, "zlm_repack_q6_k"), "zlm_repack_q6_k")) return false;
    if (!ok(d, hipModuleGetFunction(&d->quantize_q8, d->mod, "zlm_quantize_q8"), "zlm_quantize_q8")) return false;
    if (!ok(d, hipModuleGetFunction(&d->quantize_q8_tiled, d->mod, "zlm_quantize_q8_tiled"), "quantize tiled"))
        return false;
    if (!ok(d, hipModuleGetFunction(&d->tile_q4_0, d->mod, "zlm_tile_q4_0"), "zlm_tile_q4_0")) return false;
    if (!ok(d, hipModuleGetFunction(&d->copy16, d->mod, "zlm_copy16"), "zlm_copy16")) return false;
    if (!ok(d, hipModuleGetFunction(&d->tile_q8_0, d->mod, "zlm_tile_q8_0"), "zlm_tile_q8_0")) return false;
    if (!ok(d, hipModuleGetFunction(&d->tile_q4_1, d->mod, "zlm_tile_q4_1"), "zlm_tile_q4_1")) return false;
    if (!ok(d, hipModuleGetFunction(&d->tile_q4_k, d->mod, "zlm_tile_q4_k"), "zlm_tile_q4_k")) return false;
    if (!ok(d, hipModuleGetFunction(&d->gemm_q4_1, d->mod, "zlm_gemm_q4_1_q8"), "zlm_gemm_q4_1_q8")) return false;
    if (!ok(d, hipModuleGetFunction(&d->gemm_q4_k, d->mod, "zlm_gemm_q4_k_q8"), "zlm_gemm_q4_k_q8")) return false;
    const struct {
        hipFunction_t* f;
        const char* name;
    } more[] = {{&d->gemm_q4_0, "zlm_gemm_q4_0_q8"},
                {&d->gemm_q8_0, "zlm_gemm_q8_0_q8"},
                {&d->gemm_q4_0_k2, "zlm_gemm_q4_0_q8_k2"},
                {&d->gemm_q4_0_k4, "zlm_gemm_q4_0_q8_k4"},
                {&d->gemm_q8_0_k4, "zlm_gemm_q8_0_q8_k4"},
                {&d->gemm_q8_0_k2, "zlm_gemm_q8_0_q8_k2"},
                {&d->gemm_q4_1_k2, "zlm_gemm_q4_1_q8_k2"},
                {&d->gemm_q4_k_k2, "zlm_gemm_q4_k_q8_k2"},
                {&d->quantize_fp6, "zlm_quantize_fp6_tiled"},
                {&d->gemm_wide, "zlm_gemm_wide"},
                {&d->gemm_small_q4_0, "zlm_gemm_small_q4_0_q8"},
                {&d->gemm_small_q8_0, "zlm_gemm_small_q8_0_q8"},
                {&d->gemm_small_q4_1, "zlm_gemm_small_q4_1_q8"},
                {&d->gemm_small_q4_k, "zlm_gemm_small_q4_k_q8"},
                {&d->qk_norm_rope_kv, "zlm_qk_norm_rope_kv"},
                {&d->attn_partial, "zlm_attn_partial"},
                {&d->attn_combine, "zlm_attn_combine"},
                {&d->attn_combine_wide, "zlm_attn_combine_wide"},
                {&d->attn_decode, "zlm_attn_decode"},
                {&d->synth_blocks, "zlm_synth_blocks"},
                {&d->synth_f16, "zlm_synth_f16"}};
    for (const auto& m : more)
        if (!ok(d, hipModuleGetFunction(m.f, d->mod, m.name), m.name)) return false;
    for (const QuantInfo& qi : kQuants) {
        if (!gemm_tall_type(qi.type)) continue;
        for (int tier = 0; tier < 2; tier++) {
            char nm[64];
            snprintf(nm, sizeof nm, "zlm_gemm_tall_%s_g%d", kQuantNames[qi.slot], tier ? 8 : 4);
            if (!ok(d, hipModuleGetFunction(&d->gemm_tall[qi.slot][tier], d->mod, nm), nm)) return false;
        }
    }
    return true;
}

// A device buffer and a pinned host buffer of n floats, and the host
// buffer's device-side address (kernels read or write it directly); all three
// are replaced together when the buffer grows.
bool ensure_pair(zlm_device* d, float*& dev, float*& host, size_t& cap, size_t n, float*& host_dev) {
    if (cap >= n && dev && host && host_dev) return true;
    if (dev) hipFree(dev);
    if (host) hipHostFree(host);
    dev = nullptr;
    host = nullptr;
    host_dev = nullptr;
    cap = 0;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&dev), n * sizeof(float)), "hipMalloc")) return false;
    if (!ok(d, hipHostMalloc(reinterpret_cast<void**>(&host), n * sizeof(float), hipHostMallocDefault),
            "hipHostMalloc")) {
        hipFree(dev);
        dev = nullptr;
        return false;
    }
    void* p = nullptr;
    if (!ok(d, hipHostGetDevicePointer(&p, host, 0), "host buffer device address")) {
        hipFree(dev);
        hipHostFree(host);
        dev = nullptr;
        host = nullptr;
        return false;
    }
    host_dev = static_cast<float*>(p);
    cap = n;
    return true;
}

// A device buffer of n floats (contents not kept when it grows).
bool ensure_dev(zlm_device* d, float*& dev, size_t& cap, size_t n) {
    if (cap >= n && dev) return true;
    if (dev) {
        hipStreamSynchronize(d->stream);
        hipFree(dev);
    }
    dev = nullptr;
    cap = 0;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&dev), n * sizeof(float)), "hipMalloc")) return false;
    cap = n;
    return true;
}

// A pinned host buffer of n floats and its device-side address (kernels write
// it directly).
bool ensure_host(zlm_device* d, float*& host, float*& host_dev, size_t& cap, size_t n) {
    if (cap >= n && host && host_dev) return true;
    if (host) hipHostFree(host);
    host = nullptr;
    host_dev = nullptr;
    cap = 0;
    if (!ok(d, hipHostMalloc(reinterpret_cast<void**>(&host), n * sizeof(float), hipHostMallocDefault),
            "hipHostMalloc"))
        return false;
    void* p = nullptr;
    if (!ok(d, hipHostGetDevicePointer(&p, host, 0), "host buffer device address")) {
        hipHostFree(host);
        host = nullptr;
        return false;
    }
    host_dev = static_cast<float*>(p);
    cap = n;
    return true;
}

// Library scratch that a captured graph can reference -- the attention
// partials (kUsesAttn), the GEMM's quantized activations and the residents'
// GEMM tiles (kUsesGemm) -- is never freed or replaced while a capture is open
// or a captured graph that used it exists.  Growth then fails with the
// reason, and the caller falls back.
bool may_replace_scratch(zlm_device* d, uint32_t kind, const char* what) {
    if (d->capturing) return fail(d, "%s must be sized by an eager call before capture", what);
    const int live = kind == kUsesAttn ? d->attn_graphs : d->gemm_graphs;
    if (live > 0)
        return fail(d, "%s cannot be replaced while %d captured graph(s) use it; destroy them first", what, live);
    return true;
}

// The contract's host-buffer ops copy x and results through host memory on
// the calling thread, so they cannot be recorded into a graph; under capture
// they fail (the *_enqueue entry points are the capturable forms).
bool contract_ready(zlm_device* d) {
    if (!d || !d->avail) return false;
    if (d->capturing) return fail(d, "host-buffer ops cannot run under graph capture; use the enqueue forms");
    return true;
}

bool ensure_bytes(zlm_device* d, uint8_t*& p, uint64_t& cap, uint64_t n) {
    if (cap >= n && p) return true;
    if (p) {
        hipStreamSynchronize(d->stream);
        hipFree(p);
    }
    p = nullptr;
    cap = 0;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&p), n ? n : 1), "hipMalloc")) return false;
    cap = n;
    return true;
}

// Growth of the GEMM activation scratch for a call that also runs in what there
// is: the larger buffer is allocated before the old one is given up, a refusal
// leaves the scratch and the error text as they were, and the size is not asked
// for again until this library gives device memory back (memory_given_back).
bool grow_gemm_scratch(zlm_device* d, uint64_t n) {
    if (n <= d->q_scratch_cap) return true;
    if (d->capturing || d->gemm_graphs > 0 || n >= d->q_scratch_refused) return false;
    uint8_t* p = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&p), n) != hipSuccess) {
        hipGetLastError();
        d->q_scratch_refused = n;
        return false;
    }
    if (d->q_scratch) {
        hipStreamSynchronize(d->stream);
        hipFree(d->q_scratch);
    }
    d->q_scratch = p;
    d->q_scratch_cap = n;
    return true;
}

void memory_given_back(zlm_device* d) { d->q_scratch_refused = UINT64_MAX; }

// Every kernel launch of the library: the dispatch checked on the host
// against what an AQL kernel-dispatch packet can carry (workgroup of 1..1024
// work-items, a whole number of 64-lane waves; each grid dimension's work-item
// count, workgroups x workgroup size, below 2^32; the kernel's static LDS
// within the CU's 160 KiB), so a launch outside them fails here with its
// parameters instead of reaching the queue; then recorded in the launch log
// when that is on.
constexpr uint64_t kMaxLds = 160 * 1024;
constexpr size_t kLaunchLogMax = 1 << 16;

uint32_t static_lds(zlm_device* d, hipFunction_t f) {
    auto it = d->lds_bytes.find(f);
    if (it != d->lds_bytes.end()) return it->second;
    int v = 0;
    if (hipFuncGetAttribute(&v, HIP_FUNC_ATTRIBUTE_SHARED_SIZE_BYTES, f) != hipSuccess) {
        hipGetLastError();
        v = 0;
    }
    d->lds_bytes.emplace(f, static_cast<uint32_t>(v));
    return static_cast<uint32_t>(v);
}

bool launch3(zlm_device* d, hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned block, void** args,
             const char* what) {
    if (!f) return fail(d, "%s: kernel not loaded", what);
    const uint32_t lds = static_lds(d, f);
    const bool dims_ok = gx > 0 && gy > 0 && gz > 0 && block >= 64 && block <= 1024 && block % 64 == 0;
    const uint64_t wx = static_cast<uint64_t>(gx) * block;
    if (!dims_ok || wx >= (1ull << 32) || gy > 65536 || gz > 65536 || lds > kMaxLds)
        return fail(d, "%s: launch outside the dispatch limits (grid %u x %u x %u, block %u, LDS %u bytes)", what,
                    gx, gy, gz, block, lds);
    if (d->log_launches && d->launch_log.size() < kLaunchLogMax)
        d->launch_log.push_back({what, gx, gy, gz, block, lds});
    return ok(d, hipModuleLaunchKernel(f, gx, gy, gz, block, 1, 1, 0, d->stream, args, nullptr), what);
}

bool launch(zlm_device* d, hipFunction_t f, unsigned grid, unsigned block, void** args, const char* what) {
    return launch3(d, f, grid, 1, 1, block, args, what);
}

// Bytes of the device layout of `nblk` blocks: payload rounded to 256 B, then scales.
uint64_t layout_bytes(const QuantInfo* qi, uint64_t nblk) {
    const uint64_t p = (nblk * qi->payload_bytes + 255) & ~static_cast<uint64_t>(255);
    return p + nblk * 2 * qi->scale_count + 256;
}

// Enqueue the raw -> device-layout conversion of `nblk` blocks into `dst`.
bool convert_blocks(zlm_device* d, const uint8_t* raw, uint64_t nblk, const QuantInfo* qi, uint8_t* dst,
                    uint16_t** scales_out) {
    const uint64_t p = (nblk * qi->payload_bytes + 255) & ~static_cast<uint64_t>(255);
    uint16_t* scales = reinterpret_cast<uint16_t*>(dst + p);
    *scales_out = scales;
    if (nblk == 0) return true;
    uint64_t n = nblk;
    const unsigned grid = static_cast<unsigned>((nblk + 255) / 256);
    if (qi->scale_offset == kQ4kRecords || qi->scale_offset == kQ6kRecords) {
        void* args[] = {&raw, &dst, &scales, &n};
        return launch(d, qi->scale_offset == kQ4kRecords ? d->repack_q4_k : d->repack_q6_k, grid, 256, args,
                      "repack records");
    }
    uint32_t bb = qi->block_bytes, so = qi->scale_offset, ns = qi->scale_count;
    void* args[] = {&raw, &dst, &scales, &n, &bb, &so, &ns};
    return launch(d, d->repack, grid, 256, args, "repack");
}

// Convert a resident's raw blocks into the device layout of `qi` (once; the
// raw copy is released).  A resident keeps one layout for its lifetime.
bool ensure_layout(zlm_device* d, zlm_resident* r, const QuantInfo* qi) {
    if (r->layout == qi->type) return true;
    if (r->layout != kNoLayout) return fail(d, "resident already holds a type-%u layout", r->layout);
    if (!r->raw) return fail(d, "resident has no raw bytes");
    if (d->capturing) return fail(d, "a resident's first op must run eagerly before capture (layout conversion)");
    const uint64_t nblk = r->bytes / qi->block_bytes;
    if (qi->scale_offset == kNoLayout) {  // f32 / f16 / bf16: the raw rows are the layout
        r->payload = r->raw;
        r->raw = nullptr;
        r->scales = nullptr;
        r->layout_alloc = r->bytes;
    } else {
        uint8_t* dst = nullptr;
        if (!ok(d, hipMalloc(reinterpret_cast<void**>(&dst), layout_bytes(qi, nblk)), "hipMalloc layout"))
            return false;
        r->layout_alloc = layout_bytes(qi, nblk);
        uint16_t* scales = nullptr;
        if (!convert_blocks(d, r->raw, nblk, qi, dst, &scales)) {
            hipFree(dst);
            return false;
        }
        hipStreamSynchronize(d->stream);
        hipFree(r->raw);
        r->raw = nullptr;
        r->payload = dst;
        r->scales = scales;
    }
    r->layout = qi->type;
    r->blocks = nblk;
    return true;
}

// Look up (and cache) a GEMV entry point by name in its quant's code object;
// the block size is the kernel's launch bound.
// What a GEMV entry point computes and how it takes its arguments, read from
// its name zlm_gemv_<quant>_<rest>: <rest> "multi_..." is the batch kernel,
// "tok2_..." the two-token GEMV, "q8tok..." the int-path token GEMV,
// "pair_" / "normpair_" / "norm_" / "resid_" a fused form (ZLM_FORM_*),
// anything else the plain GEMV.  Only the plain exact-steps and generic
// instances (r<RT>_s<STEPS>, r<RT>_g) take separate arguments; every other instance
// takes one GemvArgs.  The host checks a cached kernel's role before each
// launch, so a kernel picked for one form can never be launched as another.
constexpr int kRoleMulti = 16;
constexpr int kRoleTok2 = 17;
constexpr int kRoleQ8Tok = 18;

void kernel_role(const char* name, int slot, int* role, bool* struct_args) {
    const char* rest = name + strlen("zlm_gemv_") + strlen(kQuantNames[slot]) + 1;
    static const struct {
        const char* prefix;
        int role;
    } kForms[] = {{"multi_", kRoleMulti},
                  {"tok2_", kRoleTok2},
                  {"q8tok", kRoleQ8Tok},
                  {"pair_", ZLM_FORM_PAIR},
                  {"normpair_", ZLM_FORM_NORMPAIR},
                  {"norm_", ZLM_FORM_NORM},
                  {"resid_", ZLM_FORM_RESID}};
    for (const auto& f : kForms) {
        if (strncmp(rest, f.prefix, strlen(f.prefix)) == 0) {
            *role = f.role;
            *struct_args = true;
            return;
        }
    }
    *role = ZLM_FORM_PLAIN;
    // r<digits>_s<digits> or r<digits>_g, nothing after
    const char* p = rest;
    bool separate = *p == 'r';
    if (separate) {
        p++;
        separate = isdigit(static_cast<unsigned char>(*p));
        while (isdigit(static_cast<unsigned char>(*p))) p++;
        separate = separate && *p == '_';
        if (separate) {
            p++;
            if (*p == 'g') {
                p++;
            } else if (*p == 's' && isdigit(static_cast<unsigned char>(p[1]))) {
                p++;
                while (isdigit(static_cast<unsigned char>(*p))) p++;
            } else {
                separate = false;
            }
            separate = separate && *p == '\0';
        }
    }
    *struct_args = !separate;
}

const GemvKernel* find_gemv(zlm_device* d, int slot, const char* name, int rt, int steps, int waves_per_cu = 0,
                            bool struct_args = false, bool split = false, bool xq = false) {
    auto it = d->gemv.find(name);
    if (it == d->gemv.end()) {
        GemvKernel g;
        if (hipModuleGetFunction(&g.fn, d->gemv_mod[slot], name) == hipSuccess) {
            g.rt = rt;
            g.steps = steps;
            g.waves_per_cu = waves_per_cu;
            bool by_name = false;
            kernel_role(name, slot, &g.role, &by_name);
            g.struct_args = by_name;
            (void)struct_args;
            g.split = split;
            g.xq = xq || split;
            int mt = 0;
            if (hipFuncGetAttribute(&mt, HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK, g.fn) == hipSuccess && mt >= 64)
                g.threads = mt;
            else
                hipGetLastError();
        } else {
            g.fn = nullptr;
            hipGetLastError();
        }
        it = d->gemv.emplace(name, g).first;
    }
    return it->second.fn ? &it->second : nullptr;
}

// The prefetching instances' name suffixes, the grid's waves per CU, the
// fewest rows a suffix is taken for (_tallq / _tallq1 / _tall: the lm_heads,
// with int8-plane x in two- or one-row tiles, or with fp32 x) and whether x
// is staged as int8 planes (a summation the batch kernel does not share).
struct PfSuffix {
    const char* suffix;
    int waves_per_cu;
    size_t min_rows;
    bool xq;
    int rt;  // rows per wave tile of the plain (r<rt>) instance
};
constexpr PfSuffix kPfSuffixes[] = {{"_tallq", 16, 65536, true, 2},     {"_tallq1", 16, 65536, true, 1},
                                    {"_tall", 16, 65536, false, 1},
                                    {"_pf", 8, 0, false, 1},         {"_pfw16", 16, 0, false, 1},
                                    {"_pfq", 8, 0, true, 1},         {"_pfqw16", 16, 0, true, 1}};

// The split-K instances' name suffixes: _sk<RT> (RT rows per tile) for any
// row of ceil(chunks / 64) == steps, _sk<RT>x for exact rows only (chunks ==
// 64 * steps); one workgroup per CU.
constexpr int kSkRows[] = {2, 4};

// Whether a launch of `rows` rows at a row length of 4097-8192 elements takes
// the split-K instance (rows of 3-4 chunk steps; q8_0 5-8).  Measured on
// gfx950 (alternating runs, rows 1024-28672 x k 5120-8192, weights rotated
// past the Infinity Cache): q4_0 and q4_k gain at every row count (4096 x
// 8192 Q4_0 9.2 -> 7.4 us, 14336 x 8192 21.6 -> 16.6 us), q8_0 and q6_k up
// to 8192 rows (4096 x 8192 Q6_K 10.9 -> 9.1 us) but lose 2-10% from 14336
// rows; 65536 rows and more keep the one-wave-per-row instances.
bool split_mid_rows(const QuantInfo* qi, size_t rows) {
    if (rows <= 8192) return true;
    return rows < 65536 && (qi->type == ZLM_GGML_Q4_0 || qi->type == ZLM_GGML_Q4_K);
}

const GemvKernel* find_split(zlm_device* d, const QuantInfo* qi, size_t k, const char* form, size_t rows) {
    const size_t chunks = k / qi->chunk_elems;
    const int steps = static_cast<int>((chunks + 63) / 64);
    const bool exact = chunks % 64 == 0;
    const bool mid = qi->type == ZLM_GGML_Q8_0 ? (steps >= 5 && steps <= 8) : (steps >= 3 && steps <= 4);
    if (mid && !split_mid_rows(qi, rows)) return nullptr;
    char nm[96];
    for (int rt : kSkRows) {
        if (exact) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_s%d_sk%dx", kQuantNames[qi->slot], form, steps, rt);
            if (const GemvKernel* g = find_gemv(d, qi->slot, nm, rt, steps, 0, true, true)) return g;
        }
        snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_s%d_sk%d", kQuantNames[qi->slot], form, steps, rt);
        if (const GemvKernel* g = find_gemv(d, qi->slot, nm, rt, steps, 0, true, true)) return g;
    }
    return nullptr;
}

// The GEMV kernel for a shape: for a 1-row tile the split-K instance of the
// shape if the quant has one, else the prefetching instance of the exact step
// count if the quant has one (zlm_gemv_<quant>_r2_s<steps>_tallq or
// _r1_s<steps>_tall from 65536 rows, then _r1_s<steps> with _pf, _pfw16, _pfq,
// _pfqw16); else the
// instance whose step count equals ceil(chunks per row / 64) with the
// requested row tile, else with a 1-row tile, else the generic bounded
// instance.  Chunks per row: k / chunk_elems (k/16 for q8_0, k/32 for q4_0,
// q4_1 and the K-quants, k/8 for f16 / bf16, k/4 for f32).
// Whether the residual form takes two-row tiles: q4_0 rows of 2 chunk steps
// (k <= 4096) in launches of at most 8192 rows (the decode step's o
// projection: 1.619 -> 1.605 ms per decode token on gfx950).  The plain form
// at the same shape measured slower with two-row tiles (4.63 -> 5.27 us at
// 4096 x 4096) and keeps one.  Two-row tiles sum each row in the same
// per-lane order and reduction as one-row tiles, so results do not change.
bool resid_two_rows(const QuantInfo* qi, int steps, size_t rows) {
    return qi->type == ZLM_GGML_Q4_0 && steps == 2 && rows <= 8192;
}

// The pick functions below depend on the shape only through (quant, k, row
// tile or form, rows >= 65536, rows >= 32768, rows <= 8192); the device
// caches their result per class so an op's host path is one hash lookup (the
// name lookups cost ~1 us per launch, most of a small GEMV's enqueue).
// The kernel picked per shape class: (k, quant slot, what is picked, its
// parameter, row-count class) in disjoint bit fields.
enum PickKind : uint64_t { kPickPlain = 0, kPickForm = 1, kPickPairTile = 2, kPickTok2 = 3, kPickQ8Tok = 4 };

uint64_t pick_key(const QuantInfo* qi, size_t k, PickKind kind, int param, size_t rows) {
    const uint64_t rows_class = rows >= 65536 ? 2 : rows >= 32768 ? 3 : rows <= 8192 ? 1 : 0;
    return (static_cast<uint64_t>(k) << 24) | (static_cast<uint64_t>(qi->slot) << 16) |
           (static_cast<uint64_t>(kind) << 12) | (static_cast<uint64_t>(param & 0x3ff) << 2) | rows_class;
}

const GemvKernel* pick_gemv_named(zlm_device* d, const QuantInfo* qi, size_t k, int rt, size_t rows);

// Whether a launch of `form` over rows of 3-4 chunk steps (4097-8192
// elements, the 32-element-chunk quants) takes the generic two-step
// instance over an 8192-element x tile (zlm_gemv_<quant>_<form>_g8k) instead
// of the exact-steps one.  Measured on gfx950 (alternating runs, graph
// replays, k 5120-8192, weights rotated past the Infinity Cache):
// - norm and resid: faster for q4_0 / q4_1 / q4_k / q6_k (e.g. q4_k resid
//   8192 x 8192 18.2 -> 15.5 us);
// - pair and normpair: q4_1 and q6_k (q6_k 32768 x 8192 gate_up 117 -> 88
//   us), q4_0 at 3 steps only (20480 x 5120 59 -> 35 us; 1-4% slower at 4),
//   not q4_k (equal at 3 steps, 2% slower at 4);
// - plain (rows the split-K instances do not take), below 65536 rows: q4_1,
//   and q6_k at 3 steps (q4_1 14336 x 8192 21.8 -> 18.0 us); q6_k at 4 steps
//   was faster at 14336 rows but slower from 28672.
// Launches of 65536 rows and more take the lm_head instances instead (the
// prefetching _tallq / _tallq1 / _tall suffixes, plain and RMSNorm-fused)
// where the quant has one for the step count, else the exact-steps instances
// (e.g. q6_k 152064 x 5120: 190 us exact-steps, 161 us g8k, 134 us
// _r2_s3_tallq; q4_0 / q4_k plain were slower with g8k there; the pair and
// residual forms were not measured at that size).
bool use_g8k(const QuantInfo* qi, uint32_t form, int steps, size_t rows) {
    if (steps != 3 && steps != 4) return false;
    const uint32_t t = qi->type;
    if (t != ZLM_GGML_Q4_0 && t != ZLM_GGML_Q4_1 && t != ZLM_GGML_Q4_K && t != ZLM_GGML_Q6_K) return false;
    if (rows >= 65536) return false;
    if (form == ZLM_FORM_PLAIN) return t == ZLM_GGML_Q4_1 || (t == ZLM_GGML_Q6_K && steps == 3);
    if (form == ZLM_FORM_NORM || form == ZLM_FORM_RESID) return true;
    return t == ZLM_GGML_Q4_1 || t == ZLM_GGML_Q6_K || (t == ZLM_GGML_Q4_0 && steps == 3);
}

const GemvKernel* pick_gemv(zlm_device* d, const QuantInfo* qi, size_t k, int rt, size_t rows) {
    const uint64_t key = pick_key(qi, k, kPickPlain, rt, rows);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const GemvKernel* g = pick_gemv_named(d, qi, k, rt, rows);
    d->picks.emplace(key, g);
    return g;
}

const GemvKernel* pick_gemv_named(zlm_device* d, const QuantInfo* qi, size_t k, int rt, size_t rows) {
    const size_t chunks = k / qi->chunk_elems;
    const int steps = static_cast<int>((chunks + 63) / 64);
    const char* qn = kQuantNames[qi->slot];
    char nm[96];
    if (rt == 1) {
        if (const GemvKernel* g = find_split(d, qi, k, "r1", rows)) return g;
        if (use_g8k(qi, ZLM_FORM_PLAIN, steps, rows)) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_r1_g8k", qn);
            if (const GemvKernel* g = find_gemv(d, qi->slot, nm, 1, steps, 0, true)) return g;
        }
        for (const PfSuffix& v : kPfSuffixes) {
            if (rows < v.min_rows) continue;
            snprintf(nm, sizeof nm, "zlm_gemv_%s_r%d_s%d%s", qn, v.rt, steps, v.suffix);
            if (const GemvKernel* g = find_gemv(d, qi->slot, nm, v.rt, steps, v.waves_per_cu, true, false, v.xq))
                return g;
        }
    }
    snprintf(nm, sizeof nm, "zlm_gemv_%s_r%d_s%d", qn, rt, steps);
    if (const GemvKernel* g = find_gemv(d, qi->slot, nm, rt, steps)) return g;
    snprintf(nm, sizeof nm, "zlm_gemv_%s_r1_s%d", qn, steps);
    if (const GemvKernel* g = find_gemv(d, qi->slot, nm, 1, steps)) return g;
    snprintf(nm, sizeof nm, "zlm_gemv_%s_r1_g", qn);
    return find_gemv(d, qi->slot, nm, 1, 0);
}

// The two-token GEMV for matMul at m = 2: zlm_gemv_<quant>_tok2_g<T>, the
// smallest tier T in {4, 8, 16} whose x tiles hold k <= 1024*T floats, or
// null (the quant has none, or k > 16384), and the caller runs one GEMV per
// token.  At the 4096- and 8192-float tiers the wave tile holds two rows
// (_r2; q4_k at 4096 four, _r4), which halves the x reads from LDS per row;
// the results are bit for bit those of one-row tiles (the same per-lane sums
// and reduction tree).  Measured on gfx950 (alternating runs, weights rotated
// past the Infinity Cache): Q4_K 262144 x 3840 192 -> 163 us (170 with two
// rows), Q8_0 151936 x 4096 122 -> 109 us, Q4_1 151936 x 4096 106 -> 101 us,
// Q8_0 12288 x 4096 15.5 -> 13.4 us, Q4_0 4096 x 4096 7.4 -> 6.6 us, Q4_K
// 4096 x 8192 11.5 -> 10.5 us.  Four rows measured slower at q4_0 / q8_0
// (Q4_0 4096 x 8192 12.8 against 10.1 us); the 16-wave tier's two-row form
// (capped at 128 VGPRs) was slower too (Q8_0 4096 x 12288 19.5 against 15.5
// us), so it keeps one row.
constexpr size_t kTok2MaxK = 16384;

const GemvKernel* pick_tok2(zlm_device* d, const QuantInfo* qi, size_t k) {
    const uint64_t key = pick_key(qi, k, kPickTok2, 0, 0);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const GemvKernel* g = nullptr;
    if (k <= kTok2MaxK) {
        const int tier = k <= 4096 ? 4 : k <= 8192 ? 8 : 16;
        char nm[96];
        const int rt = tier == 16 ? 1 : (qi->type == ZLM_GGML_Q4_K && tier == 4) ? 4 : 2;
        if (rt > 1) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_tok2_g%d_r%d", kQuantNames[qi->slot], tier, rt);
            g = find_gemv(d, qi->slot, nm, rt, 0);
        }
        if (!g) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_tok2_g%d", kQuantNames[qi->slot], tier);
            g = find_gemv(d, qi->slot, nm, 1, 0);
        }
    }
    d->picks.emplace(key, g);
    return g;
}

// Validate resident `r` as a rows x k weight of quant `qi` and make sure its
// device layout exists.
bool check_resident(zlm_device* d, zlm_resident* r, const QuantInfo* qi, size_t rows, size_t k) {
    if (!r) return fail(d, "null resident");
    if (rows == 0 || k == 0 || k % qi->block_elems != 0 || k % qi->kblock != 0)
        return fail(d, "bad shape rows=%zu k=%zu", rows, k);
    if (rows > 0xffffffffu) return fail(d, "rows too large");
    if (k > kMaxK) return fail(d, "k=%zu exceeds the LDS-staged activation capacity", k);
    const uint64_t nb = k / qi->block_elems;
    if (r->bytes < rows * nb * qi->block_bytes) return fail(d, "resident too short");
    if (!ensure_layout(d, r, qi)) return false;
    if (r->blocks < rows * nb) return fail(d, "resident layout too short");
    return true;
}

// Grid of a GEMV launch: one wave per tile up to a per-CU cap.  Measured on
// gfx950: rows up to k = 4096 for q8_0, 8192 for the others (the float types
// follow the same x-size rule) run best at 4 workgroups per CU; wider rows
// stage a larger x in LDS and one workgroup per CU looping over tiles is best.  Tall launches (>= 64K row
// tiles, the lm_heads) with a 4096-float x capacity (19 KB of LDS) run 8
// workgroups per CU: 262144 x 3840 q6_k 222 -> 190 us.  steps 0 = the generic
// instance (32768-float x capacity, one workgroup per CU).
// A prefetching instance (waves_per_cu set) runs that many waves per CU; a
// split-K instance one workgroup (one tile at a time) per CU.
unsigned gemv_grid(const zlm_device* d, const QuantInfo* qi, uint64_t tiles, const GemvKernel* gk) {
    if (gk->split) return static_cast<unsigned>(std::min<uint64_t>(tiles, static_cast<uint64_t>(d->cus)));
    const uint64_t waves = static_cast<uint64_t>(gk->threads / 64);
    const uint64_t wgs = (tiles + waves - 1) / waves;
    const int steps = gk->steps;
    const uint64_t xk = static_cast<uint64_t>(steps) * 64 * qi->chunk_elems;  // elements of x a row covers
    const bool small_x = steps > 0 && xk <= 4096;
    const bool wide = steps == 0 || xk > (qi->type == ZLM_GGML_Q8_0 ? 4096u : 8192u);
    uint64_t cap = static_cast<uint64_t>(d->cus) * (wide ? 1 : (small_x && tiles >= 65536) ? 8 : 4);
    if (gk->waves_per_cu > 0)
        cap = std::max<uint64_t>(1, static_cast<uint64_t>(d->cus) * static_cast<uint64_t>(gk->waves_per_cu) / waves);
    return static_cast<unsigned>(std::min<uint64_t>(wgs, cap));
}

// Validate a GEMV over resident `r` and pick its kernel.
bool prepare_gemv(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k, hipFunction_t* f,
                  unsigned* grid, unsigned* block, const GemvKernel** picked = nullptr) {
    if (!d || !d->avail) return fail(d, "device unavailable");
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu);
    if (!check_resident(d, r, qi, rows, k)) return false;
    const GemvKernel* gk = pick_gemv(d, qi, k, rt_for_variant(variant_of(quant)), rows);
    if (!gk) return fail(d, "no GEMV kernel for quant %u k=%zu", qi->type, k);
    *f = gk->fn;
    *grid = gemv_grid(d, qi, (rows + gk->rt - 1) / gk->rt, gk);
    *block = static_cast<unsigned>(gk->threads);
    if (picked) *picked = gk;
    return true;
}

// Kernel-argument block of the fused forms; the same layout as GemvArgs in
// gemv_impl.h (passed by value as the kernel's only argument).
struct GemvArgsHost {
    const uint8_t* w0;
    const uint16_t* d0;
    const uint8_t* w1;
    const uint16_t* d1;
    const float* x;
    const float* xw;
    float* y;
    const float* res;
    uint32_t rows;
    uint32_t nb;
    float eps;
    uint32_t act;
    uint32_t m;  // the token forms: rows of x and y
};
static_assert(sizeof(GemvArgsHost) == 88, "GemvArgs layout");

bool enqueue_gemv(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k, const float* x_dev,
                  float* y_dev) {
    hipFunction_t f;
    unsigned grid, block;
    const GemvKernel* gk = nullptr;
    if (!prepare_gemv(d, r, quant, rows, k, &f, &grid, &block, &gk)) return false;
    const QuantInfo* qi = quant_info(quant);
    if (gk->role != ZLM_FORM_PLAIN) return fail(d, "internal: picked kernel (role %d) is not a plain GEMV", gk->role);
    const uint8_t* w = r->payload;
    const uint16_t* s = r->scales;
    uint32_t rows32 = static_cast<uint32_t>(rows), nb = static_cast<uint32_t>(k / qi->kblock);
    if (gk->struct_args) {
        GemvArgsHost a = {w, s, w, s, x_dev, x_dev, y_dev, y_dev, rows32, nb, 0.0f, 0u, 1u};
        void* args[] = {&a};
        return launch(d, f, grid, block, args, "gemv");
    }
    void* args[] = {&w, &s, &x_dev, &y_dev, &rows32, &nb};
    return launch(d, f, grid, block, args, "gemv");
}

// Both tokens of an m = 2 product in one launch: y_dev[t * rows + r] = row r
// . x_dev[t * k ..], t = 0, 1.  Returns false without an error when there is
// no two-token instance for the shape (*ran = false); the caller then runs
// one GEMV per token.  Workgroups per CU: 4, or as many as the two x tiles
// leave room for in LDS.
bool enqueue_gemv_tok2(zlm_device* d, zlm_resident* r, const QuantInfo* qi, size_t rows, size_t k,
                       const float* x_dev, float* y_dev, bool* ran) {
    *ran = false;
    const GemvKernel* gk = pick_tok2(d, qi, k);
    if (!gk) return true;
    if (gk->role != kRoleTok2 || !gk->struct_args)
        return fail(d, "internal: picked kernel (role %d) is not the two-token GEMV", gk->role);
    const uint32_t lds = static_lds(d, gk->fn);
    const uint64_t per_cu = std::max<uint64_t>(1, std::min<uint64_t>(4, kMaxLds / std::max<uint32_t>(lds, 1)));
    const uint64_t waves = static_cast<uint64_t>(gk->threads / 64);
    const uint64_t tiles = (rows + gk->rt - 1) / gk->rt;
    const uint64_t wgs = (tiles + waves - 1) / waves;
    const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(wgs, static_cast<uint64_t>(d->cus) * per_cu));
    const uint8_t* w = r->payload;
    const uint16_t* s = r->scales;
    GemvArgsHost a = {w, s, w, s, x_dev, x_dev, y_dev, y_dev, static_cast<uint32_t>(rows),
                      static_cast<uint32_t>(k / qi->kblock), 0.0f, 0u, 2u};
    void* args[] = {&a};
    *ran = true;
    return launch(d, gk->fn, grid, static_cast<unsigned>(gk->threads), args, "gemv two tokens");
}

// The int path for 3 <= m <= kQ8TokM tokens and k <= kQ8TokMaxK (and for
// 5 <= m <= 8 where pick_q8tok8 below has an instance) in one pass
// over the weights (zlm_gemv_<quant>_q8tok4_g<T>: T = 4 or 8 for k <= 4096
// or 8192; every workgroup quantizes the m activation rows itself), or null:
// the caller runs the small-M GEMM.  Measured on gfx950 (m = 3-4, against
// the quantizer + small-M GEMM): 4096 x 4096 Q4_0 9.9 -> 7.4 us, Q4_K 13.2 ->
// 7.7 us, 12288 x 4096 Q8_0 19.4 -> 14.7 us, the 262144 x 3840 Q4_K lm_head
// 269 -> 194 us; eight token slots were slower than the GEMM on most shapes.
// From 32768 rows the nibble quants take two-row tiles (_r2; bit for bit the
// one-row results): Q4_K 262144 x 3840 175 -> 155 us, Q4_0 151936 x 4096 91
// -> 80 us, Q4_1 the same shape 95 -> 85 us, Q4_0 32768 x 4096 26.7 -> 25.1
// us.  Below that they idle waves: the grid holds one 16-wave workgroup per
// CU, so 4096 rows are 2048 two-row tiles for 4096 waves (7.3 -> 8.8 us).
// q4_1 and q4_k also run k 8193-16384 here (zlm_gemv_<quant>_q8tok4_g16,
// one-row tiles), where their min-carrying GEMM is slower: Q4_K 3840 x 15360
// 34.4 -> 25.7 us, Q4_1 4096 x 12288 28.8 -> 20.5 us (m = 3, 4; alternating
// runs).  For q4_0 the tier measured slower than the GEMM (4096 x 12288:
// 19.3 -> 20.4 us) and q8_0 about even (23.8 -> 23.1 us).
constexpr size_t kQ8TokM = 4;
constexpr size_t kQ8TokMaxK = 8192;

// m = 5..8: the eight-slot instance (zlm_gemv_<quant>_q8tok8_g4) for q4_1 at
// k <= 4096, and for q4_k there up to 8192 rows, or null (the small-M GEMM
// runs).  Measured on gfx950 against the quantizer + small-M GEMM (m = 5 and
// 8, alternating runs): Q4_K 4096 x 4096 13.3 -> 11.9 us, 1024 x 4096 13.0
// -> 11.1 us; Q4_1 4096 x 4096 13.3 -> 11.7 us, 12288 x 4096 22.4 -> 20.4
// us, 151936 x 4096 173 -> 143 us.  Slower: Q4_K 15360 x 3840 (21.9 ->
// 26.3 us) and 4096 x 8192 (21.1 -> 23.4), Q4_0 and Q8_0 (4096 x 4096 Q4_0
// 9.9 -> 11.2 us), whose GEMMs carry no min term.
constexpr size_t kQ8Tok8M = 8;

const GemvKernel* pick_q8tok8(zlm_device* d, const QuantInfo* qi, size_t k, size_t rows) {
    const uint64_t key = pick_key(qi, k, kPickQ8Tok, static_cast<int>(kQ8Tok8M), rows);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const GemvKernel* g = nullptr;
    if (k <= 4096 && (qi->type == ZLM_GGML_Q4_1 || (qi->type == ZLM_GGML_Q4_K && rows <= 8192))) {
        char nm[96];
        snprintf(nm, sizeof nm, "zlm_gemv_%s_q8tok8_g4", kQuantNames[qi->slot]);
        g = find_gemv(d, qi->slot, nm, 1, 0);
    }
    d->picks.emplace(key, g);
    return g;
}

const GemvKernel* pick_q8tok(zlm_device* d, const QuantInfo* qi, size_t k, size_t rows) {
    const int ntok = static_cast<int>(kQ8TokM);
    const uint64_t key = pick_key(qi, k, kPickQ8Tok, ntok, rows);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const GemvKernel* g = nullptr;
    if (k <= kQ8TokMaxK) {
        char nm[96];
        if (rows >= 32768 && qi->type != ZLM_GGML_Q8_0) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_q8tok%d_g%d_r2", kQuantNames[qi->slot], ntok, k <= 4096 ? 4 : 8);
            g = find_gemv(d, qi->slot, nm, 2, 0);
        }
        if (!g) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_q8tok%d_g%d", kQuantNames[qi->slot], ntok, k <= 4096 ? 4 : 8);
            g = find_gemv(d, qi->slot, nm, 1, 0);
        }
    } else if (k <= 2 * kQ8TokMaxK && (qi->type == ZLM_GGML_Q4_1 || qi->type == ZLM_GGML_Q4_K)) {
        // q4_1 / q4_k, k 8193-16384: the 16384-float tier (the min-carrying
        // GEMM is the slower route there)
        char nm[96];
        snprintf(nm, sizeof nm, "zlm_gemv_%s_q8tok%d_g16", kQuantNames[qi->slot], ntok);
        g = find_gemv(d, qi->slot, nm, 1, 0);
    }
    d->picks.emplace(key, g);
    return g;
}

// Enqueue the int-path token GEMV (y_dev[t * rows + r], t < m) where an
// instance covers (m, k); *ran = false otherwise.  One 16-wave workgroup per
// CU, each looping over row tiles.
bool enqueue_gemv_q8tok(zlm_device* d, zlm_resident* r, const QuantInfo* qi, size_t rows, size_t k, size_t m,
                        const float* x_dev, float* y_dev, bool* ran) {
    *ran = false;
    if (m < 3 || m > kQ8Tok8M) return true;
    const GemvKernel* gk = m <= kQ8TokM ? pick_q8tok(d, qi, k, rows) : pick_q8tok8(d, qi, k, rows);
    if (!gk) return true;
    if (gk->role != kRoleQ8Tok || !gk->struct_args)
        return fail(d, "internal: picked kernel (role %d) is not the int token GEMV", gk->role);
    const uint64_t waves = static_cast<uint64_t>(gk->threads / 64);
    const uint64_t tiles = (rows + gk->rt - 1) / gk->rt;
    const uint64_t wgs = (tiles + waves - 1) / waves;
    const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(wgs, static_cast<uint64_t>(d->cus)));
    const uint8_t* w = r->payload;
    const uint16_t* s = r->scales;
    GemvArgsHost a = {w, s, w, s, x_dev, x_dev, y_dev, y_dev, static_cast<uint32_t>(rows),
                      static_cast<uint32_t>(k / qi->kblock), 0.0f, 0u, static_cast<uint32_t>(m)};
    void* args[] = {&a};
    *ran = true;
    return launch(d, gk->fn, grid, static_cast<unsigned>(gk->threads), args, "gemv int tokens");
}

// ---- fused GEMV forms (prologue/epilogue variants of the same kernel) ----

const char* const kFormNames[] = {"plain", "pair", "norm", "normpair", "resid"};

bool form_is_pair(uint32_t form) { return form == ZLM_FORM_PAIR || form == ZLM_FORM_NORMPAIR; }
bool form_is_norm(uint32_t form) { return form == ZLM_FORM_NORM || form == ZLM_FORM_NORMPAIR; }

// Kernel-argument block of the batch kernel (GemvMultiArgs in gemv_impl.h).
constexpr int kMultiMax = 8;
struct GemvMultiArgsHost {
    const uint8_t* w[kMultiMax];
    const uint16_t* d[kMultiMax];
    float* y[kMultiMax];
    uint32_t first[kMultiMax + 1];
    const float* x;
    uint32_t n;
    uint32_t nb;
};
static_assert(sizeof(GemvMultiArgsHost) == 248, "GemvMultiArgs layout");
static_assert(kMultiMax == kRing, "a batch holds at most RingSize ops");
static_assert(ZLM_NOALLOC_ATTN_HEAD_SPLITS == ZLM_STATIC_SCRATCH_HEAD_SPLITS, "no-alloc scratch size");

// Enqueue up to kMultiMax GEMVs that share quant `qi`, k and x_dev as one
// launch of the batch kernel, op i's rows into ys[i].  The residents are
// validated by the caller (check_resident).
bool enqueue_multi(zlm_device* d, const QuantInfo* qi, size_t k, const float* x_dev, zlm_resident* const* res,
                   const size_t* rows, float* const* ys, size_t n) {
    const size_t chunks = k / qi->chunk_elems;
    const int steps = static_cast<int>((chunks + 63) / 64);
    const char* qn = kQuantNames[qi->slot];
    char nm[96];
    snprintf(nm, sizeof nm, "zlm_gemv_%s_multi_s%d", qn, steps);
    const GemvKernel* gk = find_gemv(d, qi->slot, nm, 1, steps);
    if (!gk) {
        snprintf(nm, sizeof nm, "zlm_gemv_%s_multi_g", qn);
        gk = find_gemv(d, qi->slot, nm, 1, 0);
    }
    if (!gk) return fail(d, "no batch GEMV kernel for quant %u", qi->type);
    if (gk->role != kRoleMulti) return fail(d, "internal: picked kernel (role %d) is not the batch GEMV", gk->role);
    GemvMultiArgsHost a = {};
    uint64_t total = 0;
    for (size_t i = 0; i < n; i++) {
        a.w[i] = res[i]->payload;
        a.d[i] = res[i]->scales;
        a.y[i] = ys[i];
        a.first[i] = static_cast<uint32_t>(total);
        total += rows[i];
    }
    if (total > 0xffffffffu) return fail(d, "batch too large");
    for (size_t i = n; i <= static_cast<size_t>(kMultiMax); i++) a.first[i] = static_cast<uint32_t>(total);
    a.x = x_dev;
    a.n = static_cast<uint32_t>(n);
    a.nb = static_cast<uint32_t>(k / qi->kblock);
    void* args[] = {&a};
    return launch(d, gk->fn, gemv_grid(d, qi, total, gk), static_cast<unsigned>(gk->threads), args, "gemv batch");
}

// Whether a same-quant batch at this k runs as one launch of the batch
// kernel: its rows equal the single-op kernel's bit for bit (same per-lane
// order) unless the single op runs split-K or on int8-plane x.
bool batch_one_launch(zlm_device* d, const QuantInfo* qi, size_t k) {
    const GemvKernel* g = pick_gemv(d, qi, k, 1, 0);
    return g && !g->xq;
}

// The fused-form kernel for a shape: the split-K or two-row-tile instance
// (resid form) or the prefetching exact-steps instance if the quant has one,
// else the exact-steps instance, else the generic one.
const GemvKernel* pick_gemvx_named(zlm_device* d, const QuantInfo* qi, size_t k, uint32_t form, size_t rows);

const GemvKernel* pick_gemvx(zlm_device* d, const QuantInfo* qi, size_t k, uint32_t form, size_t rows) {
    const uint64_t key = pick_key(qi, k, kPickForm, static_cast<int>(form), rows);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const GemvKernel* g = pick_gemvx_named(d, qi, k, form, rows);
    d->picks.emplace(key, g);
    return g;
}

const GemvKernel* pick_gemvx_named(zlm_device* d, const QuantInfo* qi, size_t k, uint32_t form, size_t rows) {
    const size_t chunks = k / qi->chunk_elems;
    const int steps = static_cast<int>((chunks + 63) / 64);
    const int rt = form_is_pair(form) ? 2 : 1;
    const char* qn = kQuantNames[qi->slot];
    char nm[96];
    if (form == ZLM_FORM_RESID) {
        if (const GemvKernel* g = find_split(d, qi, k, kFormNames[form], rows)) return g;
        if (resid_two_rows(qi, steps, rows)) {
            snprintf(nm, sizeof nm, "zlm_gemv_%s_resid_s%d_r2", qn, steps);
            if (const GemvKernel* g = find_gemv(d, qi->slot, nm, 2, steps)) return g;
        }
    }
    if (use_g8k(qi, form, steps, rows)) {
        snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_g8k", qn, kFormNames[form]);
        if (const GemvKernel* g = find_gemv(d, qi->slot, nm, rt, steps, 0, true)) return g;
    }
    for (const PfSuffix& v : kPfSuffixes) {
        if (rows < v.min_rows) continue;
        snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_s%d%s", qn, kFormNames[form], steps, v.suffix);
        // the suffix's rows per tile, times the gate and up rows of a pair form
        if (const GemvKernel* g = find_gemv(d, qi->slot, nm, v.rt * rt, steps, v.waves_per_cu, true, false, v.xq))
            return g;
    }
    snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_s%d", qn, kFormNames[form], steps);
    if (const GemvKernel* g = find_gemv(d, qi->slot, nm, rt, steps)) return g;
    snprintf(nm, sizeof nm, "zlm_gemv_%s_%s_g", qn, kFormNames[form]);
    return find_gemv(d, qi->slot, nm, rt, 0);
}

// The gate_up pair form with `rp` output rows per wave tile (2 or 4), the tile
// a GpuVariant selects (rt_for_variant); built for q4_0, q4_1 and q8_0, the
// quants the reference grid lists gate_up variants for
// (gpu/kernels/grid.zig:150-254).  Null where no such instance exists: the
// default tile runs.
const GemvKernel* pick_pair_tile(zlm_device* d, const QuantInfo* qi, size_t k, int rp, size_t rows) {
    const uint64_t key = pick_key(qi, k, kPickPairTile, rp, rows);
    auto it = d->picks.find(key);
    if (it != d->picks.end()) return it->second;
    const size_t chunks = k / qi->chunk_elems;
    const int steps = static_cast<int>((chunks + 63) / 64);
    const char* qn = kQuantNames[qi->slot];
    char nm[96];
    snprintf(nm, sizeof nm, "zlm_gemv_%s_pair_s%d_r%d", qn, steps, rp);
    const GemvKernel* g = find_gemv(d, qi->slot, nm, 2 * rp, steps);
    if (!g) {
        snprintf(nm, sizeof nm, "zlm_gemv_%s_pair_g_r%d", qn, rp);
        g = find_gemv(d, qi->slot, nm, 2 * rp, 0);
    }
    d->picks.emplace(key, g);
    return g;
}

// Enqueue one GEMV op on device buffers: validate the residents, pick the
// kernel of the op's form and launch it on the device stream.
bool enqueue_op(zlm_device* d, const zlm_gemv_op& op) {
    if (!d || !d->avail) return fail(d, "device unavailable");
    if (op.form > ZLM_FORM_RESID) return fail(d, "unknown GEMV form %u", op.form);
    if (op.form == ZLM_FORM_PLAIN) {
        if (!op.x || !op.y) return fail(d, "null buffer");
        return enqueue_gemv(d, op.w, op.quant, op.rows, op.k, op.x, op.y);
    }
    const QuantInfo* qi = quant_info(op.quant);
    if (!qi) return fail(d, "unsupported quant %u", op.quant & 0xffu);
    const bool pair = form_is_pair(op.form);
    if (!op.x || !op.y || (form_is_norm(op.form) && !op.norm_w) || (op.form == ZLM_FORM_RESID && !op.res))
        return fail(d, "null buffer");
    if (pair && op.act > ZLM_ACT_GELU) return fail(d, "unknown activation %u", op.act);
    if (!check_resident(d, op.w, qi, op.rows, op.k)) return false;
    if (pair && !check_resident(d, op.w_up, qi, op.rows, op.k)) return false;
    const int vrp = op.form == ZLM_FORM_PAIR ? rt_for_variant(variant_of(op.quant)) : 1;
    const GemvKernel* gk = vrp > 1 ? pick_pair_tile(d, qi, op.k, vrp, op.rows) : nullptr;
    if (!gk) gk = pick_gemvx(d, qi, op.k, op.form, op.rows);
    if (!gk) return fail(d, "no %s GEMV kernel for quant %u k=%zu", kFormNames[op.form], qi->type, op.k);
    if (gk->role != static_cast<int>(op.form) || !gk->struct_args)
        return fail(d, "internal: picked kernel (role %d) does not compute the %s form", gk->role,
                    kFormNames[op.form]);
    GemvArgsHost a = {};
    a.w0 = op.w->payload;
    a.d0 = op.w->scales;
    a.w1 = pair ? op.w_up->payload : op.w->payload;
    a.d1 = pair ? op.w_up->scales : op.w->scales;
    a.x = op.x;
    a.xw = form_is_norm(op.form) ? op.norm_w : op.x;
    a.y = op.y;
    a.res = op.form == ZLM_FORM_RESID ? op.res : op.y;
    a.rows = static_cast<uint32_t>(op.rows);
    a.nb = static_cast<uint32_t>(op.k / qi->kblock);
    a.eps = op.eps;
    a.act = op.act;
    a.m = 1;
    void* args[] = {&a};
    const uint64_t per_tile = static_cast<uint64_t>(pair ? gk->rt / 2 : gk->rt);  // output rows per tile
    const uint64_t tiles = (op.rows + per_tile - 1) / per_tile;
    return launch(d, gk->fn, gemv_grid(d, qi, tiles, gk), static_cast<unsigned>(gk->threads), args,
                  kFormNames[op.form]);
}

zlm_resident* new_resident(zlm_device* d, const void* bytes, size_t len) {
    zlm_resident* r = new (std::nothrow) zlm_resident();
    if (!r) return nullptr;
    r->owner = d;
    r->bytes = len;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&r->raw), len ? len : 1), "hipMalloc resident")) {
        delete r;
        return nullptr;
    }
    if (len && !ok(d, hipMemcpy(r->raw, bytes, len, hipMemcpyHostToDevice), "upload resident")) {
        hipFree(r->raw);
        delete r;
        return nullptr;
    }
    return r;
}

void release_resident_memory(zlm_resident* r) {
    if (r->raw) hipFree(r->raw);
    if (r->payload) hipFree(r->payload);
    if (r->gemm_payload) hipFree(r->gemm_payload);
    r->raw = nullptr;
    r->payload = nullptr;
    r->scales = nullptr;
    r->layout = kNoLayout;
    r->blocks = 0;
    r->layout_alloc = 0;
    r->gemm_alloc = 0;
    r->gemm_payload = nullptr;
    r->gemm_scales = nullptr;
    r->gemm_nb = 0;
    r->gemm_rt = 0;
}

// Copy n floats from a pinned host buffer (its device address `src`) into
// device memory on the stream: the library's copy kernel reading the host
// memory directly (one dependent launch; cheaper than a DMA copy at these
// sizes), or a DMA copy when n is not whole 16-byte units.
bool stage_in(zlm_device* d, float* dst, const float* src, const float* src_host, size_t n) {
    if (n % 4 == 0) {
        const uint4* s4 = reinterpret_cast<const uint4*>(src);
        uint4* d4 = reinterpret_cast<uint4*>(dst);
        uint64_t n16 = n / 4;
        void* args[] = {&s4, &d4, &n16};
        return launch(d, d->copy16, static_cast<unsigned>(std::min<uint64_t>((n16 + 255) / 256, 1024)), 256, args,
                      "stage x");
    }
    return ok(d, hipMemcpyAsync(dst, src_host, n * sizeof(float), hipMemcpyHostToDevice, d->stream), "stage x");
}

// Stage host x into the synchronous-op device buffer.
bool stage_x_sync(zlm_device* d, const float* x, size_t n) {
    if (!ensure_pair(d, d->d_x, d->h_x, d->x_cap, n, d->h_x_dev)) return false;
    memcpy(d->h_x, x, n * sizeof(float));
    return stage_in(d, d->d_x, d->h_x_dev, d->h_x, n);
}

// Wait for the synchronous op whose result kernel wrote d->h_y (through its
// device address), then copy it out.
bool finish_sync(zlm_device* d, float* out, size_t n) {
    if (!ok(d, hipStreamSynchronize(d->stream), "sync")) return false;
    memcpy(out, d->h_y, n * sizeof(float));
    return true;
}

int find_free_slot(zlm_device* d) {
    for (int i = 0; i < kRing; i++) {
        const int s = (d->next_slot + i) % kRing;
        if (!d->slots[s].pending) return s;
    }
    return -1;
}

int32_t make_handle(zlm_device* d, int s) {
    Slot& sl = d->slots[s];
    sl.gen = (sl.gen + 1) & 0x0fffffffu;
    sl.pending = true;
    d->next_slot = (s + 1) % kRing;
    return static_cast<int32_t>((sl.gen << 3) | static_cast<uint32_t>(s));
}

// Launch a resident GEMV reading device x into slot `s`, then queue the read-back.
bool submit_into_slot(zlm_device* d, int s, zlm_resident* r, uint32_t quant, size_t rows, size_t k,
                      const float* x_dev) {
    Slot& sl = d->slots[s];
    size_t ycap = sl.y_cap;
    if (!ensure_host(d, sl.h_y, sl.h_y_dev, ycap, rows)) return false;
    sl.y_cap = ycap;
    if (!sl.done && !ok(d, hipEventCreateWithFlags(&sl.done, hipEventDisableTiming), "event")) return false;
    // the GEMV writes the slot's pinned host buffer directly (no read-back copy)
    if (!enqueue_gemv(d, r, quant, rows, k, x_dev, sl.h_y_dev)) return false;
    if (!ok(d, hipEventRecord(sl.done, d->stream), "record")) return false;
    sl.rows = rows;
    return true;
}

double now_ns() {
    timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return static_cast<double>(ts.tv_sec) * 1e9 + static_cast<double>(ts.tv_nsec);
}

// Matrix products by token count m: up to kGemmGemvM tokens the fp path (the
// production GEMV's arithmetic, as zlm's CPU runs small batches through its fp
// batched GEMV, reference form/single.zig:258-292; cheaper than the int path's
// quantizer + GEMM there): one token the GEMV, two the two-token GEMV (one
// pass over the weights, k <= 16384; beyond it one GEMV per token).  From 3
// tokens the int path: 3-8 tokens by a tall weight the tall kernel
// (gemm_tall_pays); 3-4 tokens the int-path token GEMV where it covers k; up
// to one 32-token tile the split-K small-M int GEMM (zlm_gemm_small_*: 16
// waves per workgroup for q4_0 / q8_0, 8 for q4_1 / q4_k; one workgroup per
// 32-row x 32-token tile); beyond it whichever of that kernel and the
// 128 x 64 tiled int GEMM (each tile's blocks split over four or two wave
// groups, or not) the cost model below predicts faster, or for q4_1 / q4_k the
// wide fp6 GEMM where its rounds fill the chip (gemm_wide_pays).
constexpr size_t kGemmGemvM = 2;
constexpr size_t kGemmSmallM = 32;

// Whether the quant's tiles carry a min term.
bool gemm_has_min(uint32_t type) { return type == ZLM_GGML_Q4_1 || type == ZLM_GGML_Q4_K; }

// Predicted microseconds of the int GEMM kernels for rows x k x m, fitted to
// gfx950 measurements (256 CUs; 10 shapes, 3840-15360 rows, k 3840-15360,
// m 33-512, weights rotated past the Infinity Cache).  On those 100 points
// the picks below lose 3.7 us in all against the fastest kernel, 3.0 of it
// at 12288 x 4096 x 512 (below).
// - The small-M kernel: a fixed part plus a rate per (32-row tile, 32-token
//   tile, 32-element block): 7 us + 0.15 ns (q4_0, q8_0), 6 us + 0.25 ns (the
//   min-carrying q4_1, q4_k: 8-wave workgroups).
// - The tiled kernel: each wave walks a tile's whole block range, so its time
//   is a per-block cost set by n = its workgroups per CU (rounded up): 3 us +
//   c(n) us per block.  q4_0 / q8_0: split over four wave groups (*split =
//   4, 16-wave workgroups, a quarter of the blocks per wave) at n = 1,
//   c = 0.195; over two (*split = 2, 8-wave workgroups) at n = 2, c = 0.345;
//   unsplit from n = 3, c = 0.19n (12288 x 4096 x 512: the two-way split measured
//   2-3% faster there but re-read 1.3x the HBM bytes).  q4_1 / q4_k: split
//   over two at n = 1, c = 0.26 (one resident workgroup per CU: 159 VGPRs and
//   64 KB of LDS; four groups do not fit); unsplit past that, c = 0.475 /
//   0.67 / 0.22n at n = 2 / 3 / >= 4.
double gemm_small_us(const QuantInfo* qi, size_t rows, size_t m, size_t nb, int cus) {
    const double units = static_cast<double>((rows + 31) / 32) * static_cast<double>((m + 31) / 32) *
                         static_cast<double>(nb) * 256.0 / cus;
    return gemm_has_min(qi->type) ? 6.0 + 0.25e-3 * units : 7.0 + 0.15e-3 * units;
}

double gemm_tiled_us(const QuantInfo* qi, size_t rows, size_t m, size_t nb, int cus, int* split) {
    const uint64_t wgs = static_cast<uint64_t>((rows + 63) / 64) * static_cast<uint64_t>((m + 127) / 128);
    const uint64_t n = std::max<uint64_t>(1, (wgs + static_cast<uint64_t>(cus) - 1) / static_cast<uint64_t>(cus));
    const double dn = static_cast<double>(n);
    double c;
    if (!gemm_has_min(qi->type)) {
        *split = n == 1 ? 4 : n == 2 ? 2 : 1;
        c = n == 1 ? 0.195 : n == 2 ? 0.345 : 0.19 * dn;
    } else if (n == 1) {
        *split = 2;
        c = 0.26;
    } else {
        *split = 1;
        c = n == 2 ? 0.475 : n == 3 ? 0.67 : 0.22 * dn;
    }
    return 3.0 + c * static_cast<double>(nb);
}

// - The wide fp6 kernel (q4_1, q4_k): rounds of one 128-token x 192-row
//   workgroup per CU, 6 us + 0.6 us per block and round with its quantizer
//   (4.5 us of them at 512 tokens, which the tiled prediction leaves out).  It has no
//   smaller tile for what is left over, so where its last round is emptier the tiled
//   kernels take over (15360 x 3840 x 512, 320 workgroups: 107 and 139); the line is
//   seven eighths of all rounds' CUs, the range it was measured on.
//   What it gains depends on the clocks: a prefill is tens of milliseconds of
//   products, whose steady clocks favour it, a product after a pause runs both forms
//   faster and the tiled one more so.  Measured, tiled -> wide, steady (400 products on
//   end) and one after a pause, us:
//     one round (40 products on end): 12288 x 1536 x 512 45.5 -> 42.7, 45.6 -> 45.4;
//     12288 x 4096 x 512 96 -> 92, 99 -> 98; 49152 x 4096 x 128 106 -> 92, 106 -> 96;
//     several rounds: 24576 x 1024 x 2048 182 -> 183, 188 -> 207; 12288 x 1536 x 2048 134 ->
//     133, 147 -> 155; 12288 x 2048 x 2048 175 -> 171, 190 -> 199; 12288 x 3072 x 2048 255 ->
//     245, 274 -> 284; 24576 x 3072 x 512 131 -> 121, 143 -> 144; 15360 x 3840 x 1999 386 ->
//     366, 404 -> 418; 12288 x 4096 x 1024 171 -> 161, 183 -> 186.
//   So several rounds take it from kGemmWideRoundsNb blocks a row, where the steady gain
//   (4-7%) outweighs the single product's loss (1-4%); below, it is the other way round
//   (49152 x 256 x 896 loses 20% in either).
//   Rows longer than kGemmWideMaxNb blocks keep to the other kernels (the wide
//   kernel's offsets are 32-bit).
constexpr uint64_t kGemmWideMaxNb = 1u << 18, kGemmWideRoundsNb = 96;

bool gemm_wide_pays(const QuantInfo* qi, size_t rows, size_t m, size_t nb, int cus, double tiled_us) {
    if (!gemm_has_min(qi->type) || nb > kGemmWideMaxNb) return false;
    const uint64_t c = static_cast<uint64_t>(cus);
    const uint64_t wgs = static_cast<uint64_t>((rows + 191) / 192) * static_cast<uint64_t>((m + 127) / 128);
    const uint64_t n = (wgs + c - 1) / c;
    if (n > 1 && nb < kGemmWideRoundsNb) return false;
    return 8 * wgs >= 7 * n * c && 6.0 + 0.6 * static_cast<double>(n * nb) < tiled_us;
}

// Whether the split-K kernel runs the product; if not, *tiled_us is the tiled
// kernels' prediction and *split their split.
bool gemm_runs_small(const QuantInfo* qi, size_t rows, size_t m, size_t nb, int cus, double* tiled_us, int* split) {
    *tiled_us = gemm_tiled_us(qi, rows, m, nb, cus, split);
    return m <= kGemmSmallM || gemm_small_us(qi, rows, m, nb, cus) < *tiled_us;
}

// The quants with a prefill GEMM.
bool gemm_supported(uint32_t type) {
    return type == ZLM_GGML_Q4_0 || type == ZLM_GGML_Q8_0 || type == ZLM_GGML_Q4_1 || type == ZLM_GGML_Q4_K;
}

// Bytes of the GEMM's tiled copy of a weight of `rows` rows and nb 32-element
// blocks per row: per 32-row tile and block, 16 (nibbles) or 32 (q8_0) bytes a
// row plus the row's scale (f16) or (scale, min) float pair.
uint64_t gemm_tile_bytes(uint32_t type, uint64_t rows, uint64_t nb) {
    const uint64_t rt = (rows + 31) / 32;
    return rt * nb * 32 * (type == ZLM_GGML_Q8_0 ? 32 : 16) + rt * nb * 32 * (gemm_has_min(type) ? 8 : 2);
}

// Bytes of the GEMM's quantized activations: m tokens, padded to whole 32-token
// tiles, of nb blocks (32 quants, a scale and for the min-carrying types a sum).
uint64_t gemm_scratch_bytes(uint32_t type, uint64_t m, uint64_t nb) {
    return (m + 31) / 32 * 32 * nb * (32 + (gemm_has_min(type) ? 8 : 4));
}

void free_gemm_tiles(zlm_resident* r) {
    if (r->gemm_payload) hipFree(r->gemm_payload);
    r->gemm_payload = nullptr;
    r->gemm_scales = nullptr;
    r->gemm_nb = 0;
    r->gemm_rt = 0;
    r->gemm_alloc = 0;
}

void forget_tiles_due(zlm_device* d, zlm_resident* r) {
    if (r->tiles_due == 0) return;
    r->tiles_due = 0;
    auto& due = d->tiles_due;
    const auto it = std::find(due.begin(), due.end(), r);
    if (it != due.end()) due.erase(it);
}

// Build (once per row length) the GEMM's tiled copy of a resident weight, over
// all whole rows it holds, rows padded to 32; nb = 32-element blocks per row:
//   q4_0 / q8_0  payload [rt][nb][32 rows][16 / 32 B] + f16 scales [rt][nb][32]
//                (from the split layout);
//   q4_1 / q4_k  payload [rt][nb][32 rows][16 B nibbles] + (scale, min) float2
//                [rt][nb][32] (q4_1 from its split layout, q4_k from its
//                qs payload and records).
// The resident's layout type never changes, so nb keys the copy.
bool ensure_gemm_tiles(zlm_device* d, zlm_resident* r, const QuantInfo* qi, uint64_t nb) {
    if (r->gemm_payload && r->gemm_nb == nb) return true;
    if (d->capturing) return fail(d, "a resident's GEMM tiles must be built by an eager matMul before capture");
    if (r->gemm_payload && !may_replace_scratch(d, kUsesGemm, "a resident's GEMM tiles")) return false;
    if (r->gemm_payload) hipStreamSynchronize(d->stream);
    free_gemm_tiles(r);
    const uint64_t wblocks = nb * 32 / qi->block_elems;  // layout blocks per row
    const uint64_t rows_total = r->blocks / wblocks;
    const uint64_t rt = (rows_total + 31) / 32;
    if (rt == 0 || rt * 32 > 0xffffffffu) return fail(d, "GEMM weight shape out of range");
    const uint64_t pbytes = rt * nb * 32 * (qi->type == ZLM_GGML_Q8_0 ? 32 : 16);
    const uint64_t sbytes = gemm_tile_bytes(qi->type, rows_total, nb) - pbytes;
    uint8_t* p = nullptr;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&p), pbytes + sbytes), "hipMalloc gemm tiles")) return false;
    r->gemm_alloc = pbytes + sbytes;
    uint8_t* payload = r->payload;
    uint16_t* scales = r->scales;
    uint8_t* tp = p;
    void* ts = p + pbytes;
    uint32_t rows32 = static_cast<uint32_t>(rows_total), nb32 = static_cast<uint32_t>(nb),
             rt32 = static_cast<uint32_t>(rt);
    const uint64_t n = rt * 32 * nb;
    const unsigned grid = static_cast<unsigned>((n + 255) / 256);
    bool good;
    {
        void* args[] = {&payload, &scales, &tp, &ts, &rows32, &nb32, &rt32};
        hipFunction_t tile = qi->type == ZLM_GGML_Q8_0   ? d->tile_q8_0
                             : qi->type == ZLM_GGML_Q4_1 ? d->tile_q4_1
                             : qi->type == ZLM_GGML_Q4_K ? d->tile_q4_k
                                                         : d->tile_q4_0;
        good = launch(d, tile, grid, 256, args, "tile weights");
    }
    if (!good) {
        hipFree(p);
        return false;
    }
    r->gemm_payload = tp;
    r->gemm_scales = ts;
    r->gemm_nb = nb;
    r->gemm_rt = rt;
    forget_tiles_due(d, r);
    return true;
}

// A capture can build nothing, so the eager matMul before it builds the tiles and
// the activation scratch that it needs, for up to 32 tokens whatever the eager
// call's own number.  The tall kernel needs neither; a resident that it ran 5 to 8
// tokens of is noted here instead, and the next capture's begin prepares it, so
// that only callers who capture hold the tiled copy.  What memory does not allow
// is left out: a captured call that needs it fails with the reason, as it would
// without an eager call.
void note_tiles_due(zlm_device* d, zlm_resident* r, uint64_t nb) {
    if (d->capturing || r->tiles_due == nb || (r->gemm_payload && r->gemm_nb == nb)) return;
    if (r->tiles_due == 0) d->tiles_due.push_back(r);
    r->tiles_due = nb;
}

void build_tiles_due(zlm_device* d) {
    const std::string err = d->err;
    while (!d->tiles_due.empty()) {
        zlm_resident* r = d->tiles_due.back();
        const uint64_t nb = r->tiles_due;
        forget_tiles_due(d, r);
        const QuantInfo* qi = quant_info(r->layout);
        if (!grow_gemm_scratch(d, gemm_scratch_bytes(qi->type, kGemmSmallM, nb)) || !ensure_gemm_tiles(d, r, qi, nb))
            hipGetLastError();
    }
    d->err = err;
}

// The tall kernel (16-row tiles of the GEMV layout, a wave each, one 16-wave
// workgroup per CU; no tiled copy, no quantizer launch) runs m = 3..8 where there
// are at least eight tiles a CU: a tile is one wave's, so a call takes at least as
// long as a tile, 1.6 us per 256 elements.  Measured, the route before it and it, us:
//   m = 5 to 8: q4_k 32768 x 1024 15 and 10, x 4096 36 and 21, x 8192 72 and 49; q4_1
//   32768 x 4096 37 and 23, x 8192 73 and 51; q4_0 65536 x 4096 42 and 33, x 8192 95 and
//   73.  Fewer rows stay where they were: it still gains there (q4_k and q4_1 16384 x
//   4096 23 and 17, 22 and 20; q4_0 32768 x 4096 30 and 24), until a CU has two to four
//   tiles (8192 x 4096 q4_k 16 and 17, q4_1 15 and 19; q4_0 16384 x 4096 14 and 17).
//   m = 3 and 4, where the int token GEMV is closer: q4_k 65536 x 4096 42 and 32, 65536 x
//   8192 80 and 75, 32768 x 8192 46 and 50; q4_0 and q4_1 win only with short rows (q4_0
//   262144 x 2048 69 and 64, 65536 x 2048 22 and 19; 151936 x 4096 73 and 76, 65536 x 8192
//   63 and 68).
// k % 64: q4_0 and q4_1 scales are loaded in pairs.
bool gemm_tall_pays(const QuantInfo* qi, size_t rows, size_t k, size_t m) {
    if (!gemm_tall_type(qi->type) || m < 3 || m > 8 || k > 8192 || k % 64) return false;
    if (m <= 4) return rows >= 65536 && (qi->type == ZLM_GGML_Q4_K || k <= 2048);
    return rows >= (qi->type == ZLM_GGML_Q4_0 ? 65536 : 32768);
}

bool enqueue_gemm_tall(zlm_device* d, zlm_resident* r, const QuantInfo* qi, size_t rows, size_t k, size_t m,
                       const float* x_dev, float* out_dev) {
    const uint8_t* w = r->payload;
    const uint16_t* s = r->scales;
    uint32_t rows32 = static_cast<uint32_t>(rows), m32 = static_cast<uint32_t>(m), nb32 = static_cast<uint32_t>(k / 32);
    void* args[] = {&w, &s, const_cast<float**>(&x_dev), &out_dev, &rows32, &m32, &nb32};
    // tiles are dealt to the workgroups first and to their waves second
    const uint64_t tiles = (static_cast<uint64_t>(rows) + 15) / 16;
    const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(tiles, static_cast<uint64_t>(d->cus)));
    return launch(d, d->gemm_tall[qi->slot][k <= 4096 ? 0 : 1], grid, 1024, args, "gemm tall");
}

// Enqueue the matrix product out_dev[t*rows + r] over a resident Q4_0, Q8_0, Q4_1
// or Q4_K weight and device activations x_dev (m x k, token-major): a few tokens
// straight from the device layout, more by quantizing x to q8 blocks into the device
// scratch (plus dx*sum(q) for the min-carrying types) and a GEMM over the tiled
// weights.
bool enqueue_gemm(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k, size_t m,
                  const float* x_dev, float* out_dev) {
    if (!d || !d->avail) return fail(d, "device unavailable");
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu);
    if (!gemm_supported(qi->type)) return fail(d, "no GEMM kernel for quant %u", qi->type);
    if (!r || rows == 0 || k == 0 || m == 0 || k % qi->block_elems || k % 32) return fail(d, "bad GEMM shape");
    if (rows > 0x7fffffffu || m > 0x7fffffffu || k / 32 > 0xffffffu) return fail(d, "GEMM shape too large");
    const uint64_t nb = k / 32, wblocks = k / qi->block_elems;
    if (r->bytes < rows * wblocks * qi->block_bytes) return fail(d, "resident too short");
    if (!ensure_layout(d, r, qi)) return false;
    if (r->blocks < rows * wblocks) return fail(d, "resident layout too short");
    if (m <= kGemmGemvM) {  // fp GEMVs (no activation quantizer, no tiled weight copy)
        if (m == 2) {  // both tokens in one pass over the weights where an instance fits k
            bool ran = false;
            if (!check_resident(d, r, qi, rows, k)) return false;
            if (!enqueue_gemv_tok2(d, r, qi, rows, k, x_dev, out_dev, &ran)) return false;
            if (ran) return true;
        }
        for (size_t t = 0; t < m; t++)
            if (!enqueue_gemv(d, r, quant, rows, k, x_dev + t * k, out_dev + t * rows)) return false;
        return true;
    }
    if (gemm_tall_pays(qi, rows, k, m)) {
        if (m > kQ8TokM && !pick_q8tok8(d, qi, k, rows)) note_tiles_due(d, r, nb);
        return enqueue_gemm_tall(d, r, qi, rows, k, m, x_dev, out_dev);
    }
    {  // a few tokens: the int path in one pass over the GEMV layout, no tiled copy or quantizer launch
        bool ran = false;
        if (!enqueue_gemv_q8tok(d, r, qi, rows, k, m, x_dev, out_dev, &ran)) return false;
        if (ran) return true;
    }
    if (!ensure_gemm_tiles(d, r, qi, nb)) return false;
    if (r->gemm_rt * 32 < rows) return fail(d, "GEMM tiles too short");
    const bool with_min = gemm_has_min(qi->type);
    int split = 1;
    double tiled_us = 0.0;
    const bool small = gemm_runs_small(qi, rows, m, nb, d->cus, &tiled_us, &split);
    const uint64_t mt = (static_cast<uint64_t>(m) + 31) / 32;
    const uint64_t qbytes = mt * 32 * k;  // a multiple of 1024
    const uint64_t fbytes = mt * 32 * nb * 4;
    const uint64_t need = gemm_scratch_bytes(qi->type, m, nb);
    // The wide kernel's activations: records of 128 tokens and two blocks, 1.4 times
    // the tiled form's bytes.  Where the scratch cannot grow for the records (under
    // capture, beside a graph that uses it, memory spent), or a launch could not cover
    // them, the tiled kernels run.
    const uint64_t gt = (static_cast<uint64_t>(m) + 127) / 128, records = gt * ((nb + 1) / 2);
    const bool wide = !small && records < (1u << 21) && gemm_wide_pays(qi, rows, m, nb, d->cus, tiled_us) &&
                      grow_gemm_scratch(d, records * 14336);
    if (need > d->q_scratch_cap && !may_replace_scratch(d, kUsesGemm, "the GEMM activation scratch")) return false;
    if (!ensure_bytes(d, d->q_scratch, d->q_scratch_cap, need)) return false;
    if (d->capturing) d->capture_uses |= kUsesGemm;
    int8_t* qx = reinterpret_cast<int8_t*>(d->q_scratch);
    float* dx = reinterpret_cast<float*>(d->q_scratch + qbytes);
    float* ds = with_min ? reinterpret_cast<float*>(d->q_scratch + qbytes + fbytes) : nullptr;
    uint32_t rows32 = static_cast<uint32_t>(rows), m32 = static_cast<uint32_t>(m), nb32 = static_cast<uint32_t>(nb),
             mt32 = static_cast<uint32_t>(mt);
    if (wide) {
        const uint8_t* wq = r->gemm_payload;
        const void* ws = r->gemm_scales;
        void* qargs[] = {const_cast<float**>(&x_dev), &qx, &m32, &nb32};
        // 256 slots a record, eight threads each
        if (!launch(d, d->quantize_fp6, static_cast<unsigned>(records * 8), 256, qargs, "quantize tiled")) return false;
        void* args[] = {&wq, &ws, &qx, &out_dev, &rows32, &m32, &nb32};
        return launch3(d, d->gemm_wide, static_cast<unsigned>((rows + 191) / 192), static_cast<unsigned>(gt), 1, 768, args,
                       "gemm wide");
    }
    {
        const uint64_t n = mt * 32 * nb * 8;  // eight threads per (token, block)
        void* args[] = {const_cast<float**>(&x_dev), &qx, &dx, &m32, &nb32, &mt32, &ds};
        if (!launch(d, d->quantize_q8_tiled, static_cast<unsigned>((n + 255) / 256), 256, args, "quantize tiled"))
            return false;
    }
    const uint8_t* wq = r->gemm_payload;
    const void* ws = r->gemm_scales;
    if (small) {
        // the split-K kernel, a workgroup per 32-row tile and 32-token tile
        const float* dsa = ds ? ds : dx;
        void* args[] = {&wq, &ws, &qx, &dx, &dsa, &out_dev, &rows32, &m32, &nb32};
        hipFunction_t f = qi->type == ZLM_GGML_Q4_0   ? d->gemm_small_q4_0
                          : qi->type == ZLM_GGML_Q8_0 ? d->gemm_small_q8_0
                          : qi->type == ZLM_GGML_Q4_1 ? d->gemm_small_q4_1
                                                      : d->gemm_small_q4_k;
        const unsigned threads = with_min ? 8 * 64 : 16 * 64;
        return launch3(d, f, static_cast<unsigned>((rows + 31) / 32), mt32, 1, threads, args, "gemm small");
    }
    const unsigned gx = static_cast<unsigned>((rows + 63) / 64), gy = static_cast<unsigned>((m + 127) / 128);
    const bool use_k2 = split == 2;
    const char* what = split == 4 ? "gemm k4" : use_k2 ? "gemm k2" : "gemm";
    const unsigned threads = 256u * static_cast<unsigned>(split);
    if (with_min) {
        void* args[] = {&wq, &ws, &qx, &dx, &ds, &out_dev, &rows32, &m32, &nb32, &mt32};
        hipFunction_t f = qi->type == ZLM_GGML_Q4_1 ? (use_k2 ? d->gemm_q4_1_k2 : d->gemm_q4_1)
                                                    : (use_k2 ? d->gemm_q4_k_k2 : d->gemm_q4_k);
        return launch3(d, f, gx, gy, 1, threads, args, what);
    }
    void* args[] = {&wq, &ws, &qx, &dx, &out_dev, &rows32, &m32, &nb32, &mt32};
    if (split == 4)
        return launch3(d, qi->type == ZLM_GGML_Q8_0 ? d->gemm_q8_0_k4 : d->gemm_q4_0_k4, gx, gy, 1, threads, args, what);
    hipFunction_t f = qi->type == ZLM_GGML_Q8_0 ? (use_k2 ? d->gemm_q8_0_k2 : d->gemm_q8_0)
                                                : (use_k2 ? d->gemm_q4_0_k2 : d->gemm_q4_0);
    return launch3(d, f, gx, gy, 1, threads, args, what);
}

}  // namespace

// ======================= the backend contract =======================

extern "C" zlm_device* zlm_gpu_init(void) {
    zlm_device* d = new (std::nothrow) zlm_device();
    if (!d) return nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1) {
        fail(d, "no HIP device");
        return d;
    }
    if (hipSetDevice(0) != hipSuccess) {
        fail(d, "hipSetDevice failed");
        return d;
    }
    hipDeviceProp_t props;
    if (hipGetDeviceProperties(&props, 0) != hipSuccess) {
        fail(d, "hipGetDeviceProperties failed");
        return d;
    }
    if (strncmp(props.gcnArchName, "gfx950", 6) != 0) {
        fail(d, "device %s is not gfx950", props.gcnArchName);
        return d;
    }
    d->cus = props.multiProcessorCount;
    snprintf(d->name, sizeof d->name, "%.200s (%.40s)", props.name, props.gcnArchName);
    if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
        fail(d, "hipStreamCreate failed");
        snprintf(d->name, sizeof d->name, "off");
        return d;
    }
    if (!load_kernels(d)) {
        std::string why = d->err;
        unload_modules(d);
        hipStreamDestroy(d->stream);
        d->stream = nullptr;
        snprintf(d->name, sizeof d->name, "off");
        d->err = why;
        return d;
    }
    // The fixed scratch of the no-alloc entry point: this device's address of
    // the array, looked up once with the device current.
    const hipError_t se = zlm_static_scratch_address(&d->static_scratch);
    if (se != hipSuccess) {
        d->static_scratch = nullptr;
        d->static_scratch_err = hipGetErrorString(se);
    }
    d->avail = true;
    d->err.clear();
    return d;
}

extern "C" void zlm_gpu_deinit(zlm_device* d) {
    if (!d) return;
    if (d->avail) {
        hipStreamSynchronize(d->stream);
        for (Slot& s : d->slots) {
            if (s.done) hipEventDestroy(s.done);
            if (s.h_y) hipHostFree(s.h_y);
            if (s.d_x) hipFree(s.d_x);
            if (s.h_x) hipHostFree(s.h_x);
            if (s.h_bx) hipHostFree(s.h_bx);
        }
        if (d->d_x) hipFree(d->d_x);
        if (d->h_x) hipHostFree(d->h_x);
        if (d->d_y) hipFree(d->d_y);
        if (d->h_y) hipHostFree(d->h_y);
        if (d->attn_part) hipFree(d->attn_part);
        if (d->d_mid) hipFree(d->d_mid);
        if (d->d_bx) hipFree(d->d_bx);
        if (d->s_raw) hipFree(d->s_raw);
        if (d->q_scratch) hipFree(d->q_scratch);
        if (d->s_lay) hipFree(d->s_lay);
        unload_modules(d);
        hipStreamDestroy(d->stream);
    }
    delete d;
}

extern "C" bool zlm_gpu_available(const zlm_device* d) { return d && d->avail; }

extern "C" const char* zlm_gpu_backend_name(const zlm_device* d) { return (d && d->avail) ? "hip" : "off"; }

extern "C" const char* zlm_gpu_device_name(const zlm_device* d) { return (d && d->avail) ? d->name : "off"; }

extern "C" bool zlm_gpu_is_uma(const zlm_device*) { return false; }

extern "C" zlm_resident* zlm_gpu_upload_resident(zlm_device* d, const void* bytes, size_t len) {
    if (!contract_ready(d)) return nullptr;
    if (!bytes && len) return nullptr;
    return new_resident(d, bytes, len);
}

extern "C" void zlm_gpu_free_resident(zlm_device* d, zlm_resident* r) {
    if (!r) return;
    if (d && d->avail) hipStreamSynchronize(d->stream);
    if (d) memory_given_back(d);
    if (d) forget_tiles_due(d, r);
    release_resident_memory(r);
    delete r;
}

extern "C" uint64_t zlm_gpu_resident_bytes(const zlm_resident* r) { return r ? r->bytes : 0; }

extern "C" bool zlm_gpu_resident_read_raw(zlm_device* d, const zlm_resident* r, void* dst, size_t len) {
    if (!contract_ready(d) || !r || !dst) return false;
    if (!r->raw) return fail(d, "resident holds no raw bytes (its first op converted them)");
    if (len != r->bytes) return fail(d, "resident holds %llu raw bytes, not %zu", (unsigned long long)r->bytes, len);
    return ok(d, hipMemcpy(dst, r->raw, len, hipMemcpyDeviceToHost), "read raw bytes");
}

extern "C" uint64_t zlm_gpu_resident_device_bytes(const zlm_resident* r) {
    if (!r) return 0;
    return (r->raw ? r->bytes : 0) + r->layout_alloc + r->gemm_alloc;
}

extern "C" uint64_t zlm_gpu_layout_bytes(uint32_t quant, size_t rows, size_t k, bool with_gemm) {
    const QuantInfo* qi = quant_info(quant);
    if (!qi || rows == 0 || k == 0 || k % qi->block_elems) return 0;
    const uint64_t nblk = static_cast<uint64_t>(rows) * (k / qi->block_elems);
    uint64_t b = qi->scale_offset == kNoLayout ? nblk * qi->block_bytes : layout_bytes(qi, nblk);
    if (with_gemm && gemm_supported(qi->type) && k % 32 == 0) b += gemm_tile_bytes(qi->type, rows, k / 32);
    return b;
}

extern "C" bool zlm_gpu_release_gemm_tiles(zlm_device* d, zlm_resident* r) {
    if (!d || !d->avail || !r) return false;
    if (r->gemm_payload && !may_replace_scratch(d, kUsesGemm, "a resident's GEMM tiles")) return false;
    if (r->gemm_payload) hipStreamSynchronize(d->stream);
    memory_given_back(d);
    free_gemm_tiles(r);
    forget_tiles_due(d, r);
    return true;
}

extern "C" bool zlm_gpu_mat_vec_resident(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k,
                                         const float* x, size_t x_len, float* out, size_t out_len) {
    if (!contract_ready(d)) return false;
    if (!x || !out || x_len != k || out_len < rows) return fail(d, "bad buffers");
    hipFunction_t f;
    unsigned g, b;
    if (!prepare_gemv(d, r, quant, rows, k, &f, &g, &b)) return false;
    if (!ensure_pair(d, d->d_y, d->h_y, d->y_cap, rows, d->h_y_dev)) return false;
    if (!stage_x_sync(d, x, k)) return false;
    if (!enqueue_gemv(d, r, quant, rows, k, d->d_x, d->h_y_dev)) return false;
    return finish_sync(d, out, rows);
}

extern "C" bool zlm_gpu_mat_vec(zlm_device* d, uint32_t quant, const void* w, size_t w_len, size_t rows, size_t k,
                                const float* x, size_t x_len, float* out, size_t out_len) {
    if (!contract_ready(d)) return false;
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu);
    if (!w || !x || !out || x_len != k || out_len < rows) return fail(d, "bad buffers");
    if (rows == 0 || k == 0 || k % qi->block_elems != 0) return fail(d, "bad shape");
    const uint64_t nblk = static_cast<uint64_t>(rows) * (k / qi->block_elems);
    const uint64_t need = nblk * qi->block_bytes;
    if (w_len < need) return fail(d, "weight too short");
    // Stage the raw blocks, convert them into the reusable layout buffer and
    // run the resident GEMV over a transient view of it.
    if (!ensure_bytes(d, d->s_raw, d->s_raw_cap, need)) return false;
    if (!ok(d, hipMemcpyAsync(d->s_raw, w, need, hipMemcpyHostToDevice, d->stream), "stage weights")) return false;
    zlm_resident view;
    view.owner = d;
    view.bytes = need;
    view.layout = qi->type;
    view.blocks = nblk;
    if (qi->scale_offset == kNoLayout) {
        view.payload = d->s_raw;
    } else {
        if (!ensure_bytes(d, d->s_lay, d->s_lay_cap, layout_bytes(qi, nblk))) return false;
        if (!convert_blocks(d, d->s_raw, nblk, qi, d->s_lay, &view.scales)) return false;
        view.payload = d->s_lay;
    }
    const bool ran = zlm_gpu_mat_vec_resident(d, &view, quant, rows, k, x, x_len, out, out_len);
    view.payload = nullptr;  // the staging buffers stay owned by the device
    view.scales = nullptr;
    return ran;
}

extern "C" int32_t zlm_gpu_mat_vec_resident_async(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows,
                                                  size_t k, const float* x, size_t x_len) {
    if (!contract_ready(d)) return ZLM_NULL_HANDLE;
    if (!x || x_len != k) return fail(d, "bad x"), ZLM_NULL_HANDLE;
    hipFunction_t f;
    unsigned g, b;
    if (!prepare_gemv(d, r, quant, rows, k, &f, &g, &b)) return ZLM_NULL_HANDLE;
    const int s = find_free_slot(d);
    if (s < 0) return fail(d, "ring full: %d dispatches in flight", kRing), ZLM_NULL_HANDLE;
    Slot& sl = d->slots[s];
    size_t xcap = sl.x_cap;
    if (!ensure_pair(d, sl.d_x, sl.h_x, xcap, k, sl.h_x_dev)) return ZLM_NULL_HANDLE;
    sl.x_cap = xcap;
    memcpy(sl.h_x, x, k * sizeof(float));
    if (!stage_in(d, sl.d_x, sl.h_x_dev, sl.h_x, k)) return ZLM_NULL_HANDLE;
    if (!submit_into_slot(d, s, r, quant, rows, k, sl.d_x)) return ZLM_NULL_HANDLE;
    return make_handle(d, s);
}

namespace {

// The burst-shared activation (reference pipeline.zig:1422-1484): `first`
// stages x into the device-owned buffer, later members must pass the same x
// pointer and length and reuse it.  Returns the device copy, or null.  x goes
// through the pinned buffer of slot `s`, the burst's first member: that
// slot's completion event follows the copy on the stream, and the slot is
// only reused after a wait on it, so the pinned buffer is never overwritten
// while the copy may still read it (no event of its own).
const float* stage_burst(zlm_device* d, const float* x, size_t x_len, bool first, int s) {
    if (first) {
        Slot& sl = d->slots[s];
        if (!ensure_host(d, sl.h_bx, sl.h_bx_dev, sl.bx_cap, x_len)) return nullptr;
        if (!ensure_dev(d, d->d_bx, d->bx_cap, x_len)) return nullptr;
        memcpy(sl.h_bx, x, x_len * sizeof(float));
        if (!stage_in(d, d->d_bx, sl.h_bx_dev, sl.h_bx, x_len)) {
            d->burst_open = false;
            return nullptr;
        }
        d->burst_src = x;
        d->burst_len = x_len;
        d->burst_open = true;
    } else if (!d->burst_open || x != d->burst_src || x_len != d->burst_len) {
        fail(d, "burst member does not match the burst's activation");
        return nullptr;
    }
    return d->d_bx;
}

// A burst op that fails after stage_burst: its slot stays free, so the copy
// from that slot's pinned buffer must finish before the slot can be staged
// into again, and the burst is closed (later members are refused).  Returns
// the null handle.
int32_t burst_failed(zlm_device* d, bool first) {
    if (first) hipStreamSynchronize(d->stream);
    d->burst_open = false;
    return ZLM_NULL_HANDLE;
}

// Make slot `s` ready to receive `rows` floats (its result kernel writes the
// pinned host buffer through sl.h_y_dev).
bool prepare_slot(zlm_device* d, int s, size_t rows) {
    Slot& sl = d->slots[s];
    size_t ycap = sl.y_cap;
    if (!ensure_host(d, sl.h_y, sl.h_y_dev, ycap, rows)) return false;
    sl.y_cap = ycap;
    if (!sl.done && !ok(d, hipEventCreateWithFlags(&sl.done, hipEventDisableTiming), "event")) return false;
    return true;
}

// Queue slot `s`'s completion event (its result is already in host memory
// when the event completes).
bool finish_slot(zlm_device* d, int s, size_t rows) {
    Slot& sl = d->slots[s];
    if (!ok(d, hipEventRecord(sl.done, d->stream), "record")) return false;
    sl.rows = rows;
    return true;
}

// The fused MLP behind both MLP contract ops: gate_up (pair form) into the
// device-side ffn_mid, then the down GEMV into slot `s`.
bool enqueue_mlp(zlm_device* d, int s, zlm_resident* rg, zlm_resident* ru, zlm_resident* rd, uint32_t gu_quant,
                 uint32_t down_quant, size_t rows, size_t k, size_t ffn, const float* x_dev, uint32_t act) {
    if (!ensure_dev(d, d->d_mid, d->mid_cap, ffn)) return false;
    zlm_gemv_op gu = {};
    gu.form = ZLM_FORM_PAIR;
    gu.quant = gu_quant;
    gu.w = rg;
    gu.w_up = ru;
    gu.rows = ffn;
    gu.k = k;
    gu.x = x_dev;
    gu.act = act;
    gu.y = d->d_mid;
    if (!enqueue_op(d, gu)) return false;
    return enqueue_gemv(d, rd, down_quant, rows, ffn, d->d_mid, d->slots[s].h_y_dev);
}

}  // namespace

extern "C" int32_t zlm_gpu_mat_vec_resident_burst_async(zlm_device* d, zlm_resident* r, uint32_t quant,
                                                        size_t rows, size_t k, const float* x, size_t x_len,
                                                        bool first) {
    if (!contract_ready(d)) return ZLM_NULL_HANDLE;
    if (!x || x_len != k) return fail(d, "bad x"), ZLM_NULL_HANDLE;
    hipFunction_t f;
    unsigned g, b;
    if (!prepare_gemv(d, r, quant, rows, k, &f, &g, &b)) return ZLM_NULL_HANDLE;
    const int s = find_free_slot(d);
    if (s < 0) return fail(d, "ring full: %d dispatches in flight", kRing), ZLM_NULL_HANDLE;
    const float* xd = stage_burst(d, x, x_len, first, s);
    if (!xd) return ZLM_NULL_HANDLE;
    if (!submit_into_slot(d, s, r, quant, rows, k, xd)) return burst_failed(d, first);
    return make_handle(d, s);
}

extern "C" bool zlm_gpu_wait_resident(zlm_device* d, int32_t h, float* out, size_t out_len, size_t rows) {
    if (!contract_ready(d) || h < 0) return false;
    const int s = h & (kRing - 1);
    const uint32_t gen = static_cast<uint32_t>(h) >> 3;
    Slot& sl = d->slots[s];
    if (!sl.pending || sl.gen != gen) return fail(d, "stale or unknown handle %d", h);
    if (!out || out_len < rows || rows > sl.rows) return fail(d, "bad output buffer");
    if (!ok(d, hipEventSynchronize(sl.done), "wait")) return false;
    memcpy(out, sl.h_y, rows * sizeof(float));
    sl.pending = false;
    return true;
}

extern "C" bool zlm_gpu_mat_vec_resident_batch(zlm_device* d, size_t k, const float* x, size_t x_len,
                                               const zlm_resident_op* ops, size_t n) {
    if (!contract_ready(d)) return false;
    if (!ops || n == 0 || n > kRing || !x || x_len != k) return fail(d, "bad batch");
    size_t total = 0;
    for (size_t i = 0; i < n; i++) {
        hipFunction_t f;
        unsigned g, b;
        if (ops[i].rows == 0 || !ops[i].out || ops[i].out_len < ops[i].rows) return fail(d, "bad batch op %zu", i);
        if (!prepare_gemv(d, ops[i].res, ops[i].quant, ops[i].rows, k, &f, &g, &b)) return false;
        total += ops[i].rows;
    }
    if (!ensure_pair(d, d->d_y, d->h_y, d->y_cap, total, d->h_y_dev)) return false;
    if (!stage_x_sync(d, x, k)) return false;
    // Ops of one quant go out as one launch of the batch kernel; a mixed batch,
    // or one whose shape has a split-K single-op kernel (another summation
    // order), runs op by op.
    bool same = n > 1 && batch_one_launch(d, quant_info(ops[0].quant), k);
    for (size_t i = 1; i < n; i++) same = same && (ops[i].quant & 0xffu) == (ops[0].quant & 0xffu);
    size_t off = 0;
    if (same) {
        zlm_resident* res[kMultiMax];
        size_t rows[kMultiMax];
        float* ys[kMultiMax];
        for (size_t i = 0; i < n; i++) {
            res[i] = ops[i].res;
            rows[i] = ops[i].rows;
            ys[i] = d->d_y + off;
            off += ops[i].rows;
        }
        if (!enqueue_multi(d, quant_info(ops[0].quant), k, d->d_x, res, rows, ys, n)) {
            hipStreamSynchronize(d->stream);
            return false;
        }
    } else {
        for (size_t i = 0; i < n; i++) {
            if (!enqueue_gemv(d, ops[i].res, ops[i].quant, ops[i].rows, k, d->d_x, d->d_y + off)) {
                hipStreamSynchronize(d->stream);
                return false;
            }
            off += ops[i].rows;
        }
    }
    if (!ok(d, hipMemcpyAsync(d->h_y, d->d_y, total * sizeof(float), hipMemcpyDeviceToHost, d->stream), "read y") ||
        !ok(d, hipStreamSynchronize(d->stream), "sync"))
        return false;
    off = 0;
    for (size_t i = 0; i < n; i++) {
        memcpy(ops[i].out, d->h_y + off, ops[i].rows * sizeof(float));
        off += ops[i].rows;
    }
    return true;
}

// How a host matMul's x and y cross: small ones are bound by the DMA copies' own
// start and end (6 and 9 us), not by their bytes, so the copy kernel pulls x and the
// product stores y straight into pinned host memory, as in the GEMV ops; large ones
// by the bytes, which the DMA engine moves better.  Measured, us of the whole call,
// x and y by DMA and by kernel:
//   both: q4_0 4096 x 4096 x 4 37 and 26, 12288 x 4096 x 8 61 and 47, 12288 x 4096 x 2
//   44 and 33; q4_k 12288 x 4096 x 24 124 and 105, 262144 x 3840 x 5 435 and 347.
//   x: 768 KiB 95 and 92 (q4_0 4096 x 4096 x 48, y by DMA), 1 MiB 122 and 124 (x 64),
//   2 MiB 207 and 220 (x 128).  With y by DMA the copy kernel saves 0-5 us up to 64 KiB
//   of x and nothing past it.
// Where y's line lies depends on how the product's waves store it, few rows at a
// time and the sooner the shorter the rows are (us by DMA and direct, x by kernel):
//   one token: 32768 x 1024 41 and 37; 65536 x 2048 58 and 61, 131072 x 1024 q4_0 86
//   and 99, q4_k 83 and 93; but with longer rows 131072 x 3072 82 and 74, 262144 x 3840
//   q4_k 177 and 153 (q8_0 131072 x 3072 112 and 122, 262144 x 3840 241 and 224);
//   two tokens: 65536 x 2048 74 and 71; q4_0 131072 x 1024 134 and 138, q8_0 105 and 106,
//   but q8_0 131072 x 3072 148 and 142, and q4_k (four-row tiles) 126 and 118;
//   the token GEMV: q8_0 131072 x 1024 x 4 168 and 159, 262144 x 1024 x 4 310 and 316;
//   262144 x 4096 x 4 445 and 387;
//   the tall kernel: q4_0 262144 x 1024 x 4 264 and 261, x 8 514 and 521, 262144 x 4096 x
//   8 558 and 511;
//   the small-M GEMM: 12288 x 4096 x 64 q4_0 240 and 226, 100000 x 1024 x 31 676 and
//   659; 65536 x 4096 x 50 (12.5 MiB of y) 840 and 845;
//   the tiled GEMMs: 0-3% less direct, and as much between runs of one form (megabytes
//   of y out of the pinned buffer), so theirs goes by DMA.
constexpr size_t kMatMulStageBytes = 896u << 10, kMatMulStageDmaBytes = 64u << 10;

static bool mat_mul_direct(zlm_device* d, const QuantInfo* qi, size_t rows, size_t k, size_t m) {
    if (!qi || !gemm_supported(qi->type)) return false;  // refused further down
    const size_t kib = (m * rows * sizeof(float) + 1023) >> 10;
    if (m == 1) return kib <= (k >= (qi->type == ZLM_GGML_Q8_0 ? 3840 : 3072) ? 1024 : 160);
    if (m <= kGemmGemvM)
        return kib <= (qi->type == ZLM_GGML_Q4_K || (qi->type == ZLM_GGML_Q8_0 && k >= 2048) ? 1024 : 512);
    if (gemm_tall_pays(qi, rows, k, m)) return kib <= (k < 2048 ? 4096 : 12288);
    if (m <= kQ8Tok8M && (m <= kQ8TokM ? pick_q8tok(d, qi, k, rows) : pick_q8tok8(d, qi, k, rows)))
        return kib <= (k < 4096 ? 3072 : 12288);
    double us;
    int split;
    return kib <= 12288 && gemm_runs_small(qi, rows, m, k / 32, d->cus, &us, &split);
}

extern "C" bool zlm_gpu_mat_mul_resident(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k,
                                         size_t m, const float* x, size_t x_len, float* out, size_t out_len) {
    if (!contract_ready(d)) return false;
    if (!x || !out || m == 0 || x_len != m * k || out_len < m * rows) return fail(d, "bad buffers");
    if (!ensure_pair(d, d->d_x, d->h_x, d->x_cap, m * k, d->h_x_dev)) return false;
    if (!ensure_pair(d, d->d_y, d->h_y, d->y_cap, m * rows, d->h_y_dev)) return false;
    const bool direct = mat_mul_direct(d, quant_info(quant), rows, k, m);
    if (m * k * sizeof(float) <= (direct ? kMatMulStageBytes : kMatMulStageDmaBytes)) {
        if (!stage_x_sync(d, x, m * k)) return false;
    } else {
        memcpy(d->h_x, x, m * k * sizeof(float));
        if (!ok(d, hipMemcpyAsync(d->d_x, d->h_x, m * k * sizeof(float), hipMemcpyHostToDevice, d->stream), "stage x"))
            return false;
    }
    if (!enqueue_gemm(d, r, quant, rows, k, m, d->d_x, direct ? d->h_y_dev : d->d_y)) {
        hipStreamSynchronize(d->stream);
        return false;
    }
    if (!direct &&
        !ok(d, hipMemcpyAsync(d->h_y, d->d_y, m * rows * sizeof(float), hipMemcpyDeviceToHost, d->stream), "read y"))
        return false;
    return finish_sync(d, out, m * rows);
}

extern "C" bool zlm_gpu_mat_mul_batch(zlm_device* d, uint32_t quant, const void* w, size_t w_len, size_t rows,
                                      size_t k, size_t m, const float* x, size_t x_len, float* out, size_t out_len) {
    if (!contract_ready(d)) return false;
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu);
    if (!gemm_supported(qi->type)) return fail(d, "no GEMM kernel for quant %u", qi->type);
    if (!w || rows == 0 || k == 0 || k % qi->block_elems) return fail(d, "bad shape");
    const uint64_t nblk = static_cast<uint64_t>(rows) * (k / qi->block_elems);
    const uint64_t need = nblk * qi->block_bytes;
    if (w_len < need) return fail(d, "weight too short");
    if (!ensure_bytes(d, d->s_raw, d->s_raw_cap, need)) return false;
    if (!ok(d, hipMemcpyAsync(d->s_raw, w, need, hipMemcpyHostToDevice, d->stream), "stage weights")) return false;
    zlm_resident view;
    view.owner = d;
    view.bytes = need;
    view.layout = qi->type;
    view.blocks = nblk;
    if (!ensure_bytes(d, d->s_lay, d->s_lay_cap, layout_bytes(qi, nblk))) return false;
    if (!convert_blocks(d, d->s_raw, nblk, qi, d->s_lay, &view.scales)) return false;
    view.payload = d->s_lay;
    const bool ran = zlm_gpu_mat_mul_resident(d, &view, quant, rows, k, m, x, x_len, out, out_len);
    forget_tiles_due(d, &view);
    free_gemm_tiles(&view);
    view.payload = nullptr;
    view.scales = nullptr;
    return ran;
}

// The variant argument of the fused ops selects Vulkan shader variants in the
// reference; here it selects the pair kernel's row tile (rt_for_variant: one,
// two or four gate/up row pairs per wave tile, for q4_0, q4_1 and q8_0 where
// those instances exist).  Results differ only by fp32 summation order.
extern "C" int32_t zlm_gpu_mat_vec_gate_up_resident_burst_async(zlm_device* d, zlm_resident* rg, zlm_resident* ru,
                                                                uint32_t quant, size_t rows, size_t k,
                                                                const float* x, size_t x_len, uint32_t act,
                                                                uint32_t variant, bool first) {
    if (!contract_ready(d)) return ZLM_NULL_HANDLE;
    if (!x || x_len != k) return fail(d, "bad x"), ZLM_NULL_HANDLE;
    if (act > ZLM_ACT_GELU) return fail(d, "unknown activation %u", act), ZLM_NULL_HANDLE;
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu), ZLM_NULL_HANDLE;
    if (!check_resident(d, rg, qi, rows, k) || !check_resident(d, ru, qi, rows, k)) return ZLM_NULL_HANDLE;
    const int s = find_free_slot(d);
    if (s < 0) return fail(d, "ring full: %d dispatches in flight", kRing), ZLM_NULL_HANDLE;
    if (!prepare_slot(d, s, rows)) return ZLM_NULL_HANDLE;
    const float* xd = stage_burst(d, x, x_len, first, s);
    if (!xd) return ZLM_NULL_HANDLE;
    zlm_gemv_op op = {};
    op.form = ZLM_FORM_PAIR;
    op.quant = with_variant(quant, variant);
    op.w = rg;
    op.w_up = ru;
    op.rows = rows;
    op.k = k;
    op.x = xd;
    op.act = act;
    op.y = d->slots[s].h_y_dev;
    if (!enqueue_op(d, op) || !finish_slot(d, s, rows)) return burst_failed(d, first);
    return make_handle(d, s);
}

extern "C" int32_t zlm_gpu_mat_vec_mlp_pair_resident_burst_async(zlm_device* d, zlm_resident* rg,
                                                                 zlm_resident* ru, zlm_resident* rd,
                                                                 uint32_t gu_quant, uint32_t down_quant,
                                                                 size_t rows, size_t k, size_t ffn, const float* x,
                                                                 size_t x_len, uint32_t act, uint32_t variant,
                                                                 bool first) {
    if (!contract_ready(d)) return ZLM_NULL_HANDLE;
    if (!x || x_len != k) return fail(d, "bad x"), ZLM_NULL_HANDLE;
    if (act > ZLM_ACT_GELU) return fail(d, "unknown activation %u", act), ZLM_NULL_HANDLE;
    const QuantInfo* gq = quant_info(gu_quant);
    const QuantInfo* dq = quant_info(down_quant);
    if (!gq || !dq) return fail(d, "unsupported quant"), ZLM_NULL_HANDLE;
    if (!check_resident(d, rg, gq, ffn, k) || !check_resident(d, ru, gq, ffn, k) ||
        !check_resident(d, rd, dq, rows, ffn))
        return ZLM_NULL_HANDLE;
    const int s = find_free_slot(d);
    if (s < 0) return fail(d, "ring full: %d dispatches in flight", kRing), ZLM_NULL_HANDLE;
    if (!prepare_slot(d, s, rows)) return ZLM_NULL_HANDLE;
    const float* xd = stage_burst(d, x, x_len, first, s);
    if (!xd) return ZLM_NULL_HANDLE;
    if (!enqueue_mlp(d, s, rg, ru, rd, with_variant(gu_quant, variant), down_quant, rows, k, ffn, xd, act) ||
        !finish_slot(d, s, rows))
        return burst_failed(d, first);
    return make_handle(d, s);
}

// The reference's single-dispatch fused MLP (one workgroup, vulkan
// pipeline.zig:1565-1635) is the same computation as the two-kernel form; on
// gfx950 the two full-grid kernels are the faster shape, so both ops run it.
extern "C" int32_t zlm_gpu_mat_vec_mlp_resident_burst_async(zlm_device* d, zlm_resident* rg, zlm_resident* ru,
                                                            zlm_resident* rd, uint32_t quant, size_t rows, size_t k,
                                                            size_t ffn, const float* x, size_t x_len, uint32_t act,
                                                            uint32_t variant, bool first) {
    return zlm_gpu_mat_vec_mlp_pair_resident_burst_async(d, rg, ru, rd, quant, quant, rows, k, ffn, x, x_len, act,
                                                         variant, first);
}

extern "C" void zlm_gpu_sync(zlm_device* d) {
    if (d && d->avail) hipStreamSynchronize(d->stream);
}

// ---- probeGpu (reference gpu/backend/root.zig:357-498) ----
// Each rate is min-of-5 host wall time of one contract op (as the reference
// measures it: staging, dispatch and read-back included), in GB/s over the
// weight bytes.  Variants are measured interleaved and the fastest recorded;
// every GpuVariant maps to one of this backend's row tiles (rt_for_variant).
// Every quant the backend runs is probed (q4_0, q4_1, q8_0, q4_k, q6_k, f32,
// f16, bf16) and the fused gate_up over q4_0, q8_0 and q4_1, as the
// reference's probe does; the gate_up variants map to the fused kernel's row
// tiles the same way (one, two or four output rows per wave tile).

namespace {

constexpr int kProbeSamples = 5;
constexpr size_t kProbeMaxRows = 12 * 1024;
constexpr size_t kProbeMaxK = 4 * 1024;
constexpr uint32_t kAllVariants[] = {ZLM_VARIANT_PLAIN, ZLM_VARIANT_U4, ZLM_VARIANT_U8, ZLM_VARIANT_SUB,
                                     ZLM_VARIANT_UN2,   ZLM_VARIANT_UN4, ZLM_VARIANT_W32, ZLM_VARIANT_W128};

// IEEE binary16 bits of a binary32 value (round to nearest even; subnormal
// results rounded the same way, overflow to infinity, NaN kept quiet).
uint16_t f32_to_f16_bits(uint32_t f) {
    const uint32_t sign = (f >> 16) & 0x8000u;
    const uint32_t exp = (f >> 23) & 0xffu;
    uint32_t man = f & 0x7fffffu;
    if (exp == 0xffu) return static_cast<uint16_t>(sign | 0x7c00u | (man ? 0x200u : 0u));
    const int e = static_cast<int>(exp) - 127 + 15;
    if (e >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
    if (e <= 0) {  // subnormal (or zero) half
        if (e < -10) return static_cast<uint16_t>(sign);
        man |= 0x800000u;
        const int shift = 14 - e;  // 24-bit significand down to the subnormal's 10 bits
        const uint32_t q = man >> shift, rem = man & ((1u << shift) - 1), halfway = 1u << (shift - 1);
        const uint32_t r = q + ((rem > halfway || (rem == halfway && (q & 1u))) ? 1u : 0u);
        return static_cast<uint16_t>(sign | r);
    }
    const uint32_t q = man >> 13, rem = man & 0x1fffu;
    uint32_t h = (static_cast<uint32_t>(e) << 10) | q;
    if (rem > 0x1000u || (rem == 0x1000u && (q & 1u))) h++;  // may carry into the exponent (and to inf)
    return static_cast<uint16_t>(sign | h);
}

// fillWeights (gpu/backend/root.zig:734-786): random bytes with the scale
// fields overwritten (q4_0/q8_0 d = 0.05, q4_1 d = 0.05 and m = 0.02, q4_k
// d = 0.05 and dmin = 0.02, q6_k d = 0.02); the float types the ramp
// f32(i % 13) * 0.05 - 0.3 (f16 rounded, bf16 truncated).  The bytes come from
// a splitmix64 stream, not Zig's PRNG.
std::vector<uint8_t> probe_weights(uint32_t type, size_t rows, size_t k) {
    const QuantInfo* qi = quant_info(type);
    const size_t nblk = rows * (k / qi->block_elems);
    std::vector<uint8_t> w(nblk * qi->block_bytes);
    if (qi->scale_offset == kNoLayout) {
        for (size_t i = 0; i < nblk; i++) {
            const float v = static_cast<float>(i % 13) * 0.05f - 0.3f;
            if (type == ZLM_GGML_F32) {
                memcpy(w.data() + 4 * i, &v, 4);
            } else {
                uint32_t bits;
                memcpy(&bits, &v, 4);
                uint16_t h;
                h = type == ZLM_GGML_BF16 ? static_cast<uint16_t>(bits >> 16) : f32_to_f16_bits(bits);
                memcpy(w.data() + 2 * i, &h, 2);
            }
        }
        return w;
    }
    uint64_t z = 0x9e3779b97f4a7c15ull;
    for (size_t i = 0; i < w.size(); i += 8) {
        z += 0x9E3779B97F4A7C15ull;
        uint64_t r = z;
        r = (r ^ (r >> 30)) * 0xBF58476D1CE4E5B9ull;
        r = (r ^ (r >> 27)) * 0x94D049BB133111EBull;
        r ^= r >> 31;
        for (size_t j = 0; j < 8 && i + j < w.size(); j++) w[i + j] = static_cast<uint8_t>(r >> (8 * j));
    }
    const uint16_t h005 = 0x2A66, h002 = 0x251F;  // f16(0.05), f16(0.02)
    for (size_t b = 0; b < nblk; b++) {
        uint8_t* blk = w.data() + b * qi->block_bytes;
        auto put = [&](size_t off, uint16_t v) {
            blk[off] = static_cast<uint8_t>(v & 0xff);
            blk[off + 1] = static_cast<uint8_t>(v >> 8);
        };
        if (type == ZLM_GGML_Q4_0 || type == ZLM_GGML_Q8_0) put(0, h005);
        if (type == ZLM_GGML_Q4_1 || type == ZLM_GGML_Q4_K) {
            put(0, h005);
            put(2, h002);
        }
        if (type == ZLM_GGML_Q6_K) put(208, h002);
    }
    return w;
}

uint8_t fastest(const double* rates) {
    uint8_t best = ZLM_VARIANT_PLAIN;
    double rate = 0.0;
    for (uint32_t v : kAllVariants)
        if (rates[v] > rate) {
            rate = rates[v];
            best = static_cast<uint8_t>(v);
        }
    return best;
}

// Interleaved min-of-N resident GEMV rates of every variant (probeResidentVariants).
void probe_resident_variants(zlm_device* d, uint32_t type, size_t rows, size_t k, const float* x, float* out,
                             double* rates) {
    for (int v = 0; v < 8; v++) rates[v] = 0.0;
    if (k % quant_info(type)->block_elems) return;
    std::vector<uint8_t> w = probe_weights(type, rows, k);
    zlm_resident* r = zlm_gpu_upload_resident(d, w.data(), w.size());
    if (!r) return;
    double best[8];
    for (double& b : best) b = 1e300;
    for (uint32_t v : kAllVariants) zlm_gpu_mat_vec_resident(d, r, ZLM_QUANT(type, v), rows, k, x, k, out, rows);
    for (int i = 0; i < kProbeSamples; i++)
        for (uint32_t v : kAllVariants) {
            const double t0 = now_ns();
            const bool ran = zlm_gpu_mat_vec_resident(d, r, ZLM_QUANT(type, v), rows, k, x, k, out, rows);
            const double t1 = now_ns();
            if (ran && t1 > t0) best[v] = std::min(best[v], t1 - t0);
        }
    for (uint32_t v : kAllVariants)
        if (best[v] < 1e300) rates[v] = static_cast<double>(w.size()) / best[v];
    zlm_gpu_free_resident(d, r);
}

// Interleaved min-of-N fused gate_up rates over both weights' bytes (probeGateUpRates).
void probe_gate_up(zlm_device* d, uint32_t type, size_t rows, size_t k, const float* x, float* out, double* rates) {
    for (int v = 0; v < 8; v++) rates[v] = 0.0;
    std::vector<uint8_t> w = probe_weights(type, rows, k);
    zlm_resident* rg = zlm_gpu_upload_resident(d, w.data(), w.size());
    zlm_resident* ru = zlm_gpu_upload_resident(d, w.data(), w.size());
    if (rg && ru) {
        double best[8];
        for (double& b : best) b = 1e300;
        for (int i = 0; i <= kProbeSamples; i++)  // the first pass warms up
            for (uint32_t v : kAllVariants) {
                const double t0 = now_ns();
                const int32_t h =
                    zlm_gpu_mat_vec_gate_up_resident_burst_async(d, rg, ru, type, rows, k, x, k, ZLM_ACT_GELU, v, true);
                const bool ran = h != ZLM_NULL_HANDLE && zlm_gpu_wait_resident(d, h, out, rows, rows);
                const double t1 = now_ns();
                if (i > 0 && ran && t1 > t0) best[v] = std::min(best[v], t1 - t0);
            }
        for (uint32_t v : kAllVariants)
            if (best[v] < 1e300) rates[v] = 2.0 * static_cast<double>(w.size()) / best[v];
    }
    if (rg) zlm_gpu_free_resident(d, rg);
    if (ru) zlm_gpu_free_resident(d, ru);
}

}  // namespace

extern "C" void zlm_gpu_probe(zlm_device* d, size_t rows_in, size_t k_in, size_t m_in, zlm_probe* out) {
    if (!out) return;
    memset(out, 0, sizeof *out);
    if (!contract_ready(d)) return;
    const size_t rows = std::min(rows_in, kProbeMaxRows);
    size_t k = std::min(k_in, kProbeMaxK);
    k -= k % 32;
    const size_t m = std::max<size_t>(m_in, 2);
    if (rows == 0 || k == 0) return;
    std::vector<float> x(k), y(rows), xm(m * k), ym(m * rows);
    for (size_t i = 0; i < k; i++) x[i] = static_cast<float>(static_cast<int>((i * 7 + 3) % 17) - 8) * 0.125f;
    for (size_t j = 0; j < m; j++)
        for (size_t i = 0; i < k; i++) xm[j * k + i] = x[i] * static_cast<float>(j + 1);
    const std::vector<uint8_t> w = probe_weights(ZLM_GGML_Q4_0, rows, k);
    const uint32_t q40 = ZLM_QUANT(ZLM_GGML_Q4_0, ZLM_VARIANT_PLAIN);
    // warm-up of the streamed and GEMM paths, then min-of-N of each
    zlm_gpu_mat_vec(d, q40, w.data(), w.size(), rows, k, x.data(), k, y.data(), rows);
    zlm_gpu_mat_mul_batch(d, q40, w.data(), w.size(), rows, k, m, xm.data(), m * k, ym.data(), m * rows);
    double best_s = 1e300, best_m = 1e300;
    for (int i = 0; i < kProbeSamples; i++) {
        double t0 = now_ns();
        bool ran = zlm_gpu_mat_vec(d, q40, w.data(), w.size(), rows, k, x.data(), k, y.data(), rows);
        double t1 = now_ns();
        if (ran && t1 > t0) best_s = std::min(best_s, t1 - t0);
        t0 = now_ns();
        ran = zlm_gpu_mat_mul_batch(d, q40, w.data(), w.size(), rows, k, m, xm.data(), m * k, ym.data(), m * rows);
        t1 = now_ns();
        if (ran && t1 > t0) best_m = std::min(best_m, t1 - t0);
    }
    const double wb = static_cast<double>(w.size());
    if (best_s < 1e300) out->gemv_streamed_gbps = wb / best_s;
    if (best_m < 1e300) out->matmul_gbps = wb / best_m;

    double rates[8];
    probe_resident_variants(d, ZLM_GGML_Q4_0, rows, k, x.data(), y.data(), rates);
    out->gemv_gbps = rates[ZLM_VARIANT_PLAIN];
    out->q4_0_u4_gbps = rates[ZLM_VARIANT_U4];
    out->q4_0_sub_gbps = rates[ZLM_VARIANT_SUB];
    out->q4_0_un2_gbps = rates[ZLM_VARIANT_UN2];
    out->q4_0_un4_gbps = rates[ZLM_VARIANT_UN4];
    out->q4_0_w32_gbps = rates[ZLM_VARIANT_W32];
    out->q4_0_w128_gbps = rates[ZLM_VARIANT_W128];
    out->q4_0_variant = fastest(rates);

    probe_gate_up(d, ZLM_GGML_Q4_0, rows, k, x.data(), y.data(), rates);
    out->gate_up_gbps = rates[ZLM_VARIANT_PLAIN];
    out->gate_up_u4_gbps = rates[ZLM_VARIANT_U4];
    out->gate_up_variant = fastest(rates);
    probe_gate_up(d, ZLM_GGML_Q8_0, rows, k, x.data(), y.data(), rates);
    out->gate_up_q8_0_variant = fastest(rates);

    // the K-quants need k in whole 256-element super-blocks
    const size_t kk = k - k % 256;
    if (kk) {
        probe_resident_variants(d, ZLM_GGML_Q4_K, rows, kk, x.data(), y.data(), rates);
        out->q4_k_gbps = rates[ZLM_VARIANT_PLAIN];
        out->q4_k_u4_gbps = rates[ZLM_VARIANT_U4];
        out->q4_k_variant = fastest(rates);
        probe_resident_variants(d, ZLM_GGML_Q6_K, rows, kk, x.data(), y.data(), rates);
        out->q6_k_variant = fastest(rates);
    }
    probe_resident_variants(d, ZLM_GGML_Q8_0, rows, k, x.data(), y.data(), rates);
    out->q8_0_variant = fastest(rates);
    probe_resident_variants(d, ZLM_GGML_Q4_1, rows, k, x.data(), y.data(), rates);
    out->q4_1_variant = fastest(rates);
    probe_gate_up(d, ZLM_GGML_Q4_1, rows, k, x.data(), y.data(), rates);
    out->gate_up_q4_1_variant = fastest(rates);
    probe_resident_variants(d, ZLM_GGML_F32, rows, k, x.data(), y.data(), rates);
    out->f32_variant = fastest(rates);
    probe_resident_variants(d, ZLM_GGML_F16, rows, k, x.data(), y.data(), rates);
    out->f16_variant = fastest(rates);
    probe_resident_variants(d, ZLM_GGML_BF16, rows, k, x.data(), y.data(), rates);
    out->bf16_variant = fastest(rates);
    zlm_gpu_sync(d);
}

extern "C" bool zlm_gpu_probe_rates(zlm_device* d, uint32_t ggml_type, bool gate_up, size_t rows_in, size_t k_in,
                                    double* rates) {
    if (!rates) return false;
    for (int v = 0; v < 8; v++) rates[v] = 0.0;
    if (!contract_ready(d)) return false;
    const QuantInfo* qi = quant_info(ggml_type);
    if (!qi || variant_of(ggml_type) != 0) return fail(d, "unsupported quant %u", ggml_type);
    const size_t rows = std::min(rows_in, kProbeMaxRows);
    size_t k = std::min(k_in, kProbeMaxK);
    k -= k % std::max<size_t>(32, qi->block_elems);
    if (rows == 0 || k == 0) return fail(d, "probe shape out of range");
    std::vector<float> x(k), y(rows);
    for (size_t i = 0; i < k; i++) x[i] = static_cast<float>(static_cast<int>((i * 7 + 3) % 17) - 8) * 0.125f;
    if (gate_up) probe_gate_up(d, qi->type, rows, k, x.data(), y.data(), rates);
    else probe_resident_variants(d, qi->type, rows, k, x.data(), y.data(), rates);
    for (int v = 0; v < 8; v++)
        if (!(rates[v] > 0.0)) return fail(d, "variant %d of quant %u was not measured", v, qi->type);
    return true;
}

// ======================= device-level entry points =======================

extern "C" const char* zlm_gpu_last_error(const zlm_device* d) { return d ? d->err.c_str() : "null device"; }

extern "C" int zlm_gpu_cu_count(const zlm_device* d) { return (d && d->avail) ? d->cus : 0; }

extern "C" bool zlm_gpu_vram_info(zlm_device* d, uint64_t* free_bytes, uint64_t* total_bytes) {
    if (!d || !d->avail || !free_bytes || !total_bytes) return false;
    size_t f = 0, t = 0;
    if (!ok(d, hipMemGetInfo(&f, &t), "hipMemGetInfo")) return false;
    *free_bytes = f;
    *total_bytes = t;
    return true;
}

extern "C" void* zlm_gpu_dev_malloc(zlm_device* d, size_t bytes) {
    if (!d || !d->avail) return nullptr;
    void* p = nullptr;
    if (!ok(d, hipMalloc(&p, bytes ? bytes : 1), "hipMalloc")) return nullptr;
    return p;
}

extern "C" void zlm_gpu_dev_free(zlm_device* d, void* p) {
    if (!d || !d->avail || !p) return;
    hipStreamSynchronize(d->stream);
    hipFree(p);
    memory_given_back(d);
}

extern "C" bool zlm_gpu_dev_upload(zlm_device* d, void* dst, const void* src, size_t n) {
    if (!d || !d->avail) return false;
    if (!ok(d, hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, d->stream), "upload")) return false;
    return ok(d, hipStreamSynchronize(d->stream), "sync");
}

extern "C" bool zlm_gpu_dev_download(zlm_device* d, void* dst, const void* src, size_t n) {
    if (!d || !d->avail) return false;
    if (!ok(d, hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, d->stream), "download")) return false;
    return ok(d, hipStreamSynchronize(d->stream), "sync");
}

extern "C" bool zlm_gpu_dev_copy_enqueue(zlm_device* d, void* dst, const void* src, size_t bytes) {
    if (!d || !d->avail || !dst || !src) return false;
    if (bytes % 16 || reinterpret_cast<uintptr_t>(dst) % 16 || reinterpret_cast<uintptr_t>(src) % 16)
        return fail(d, "dev_copy needs 16-byte granules");
    if (bytes == 0) return true;
    uint64_t n16 = bytes / 16;
    const unsigned grid = static_cast<unsigned>(std::min<uint64_t>((n16 + 255) / 256, static_cast<uint64_t>(d->cus) * 8));
    void* args[] = {const_cast<void**>(&src), &dst, &n16};
    return launch(d, d->copy16, grid, 256, args, "copy");
}

extern "C" bool zlm_gpu_dev_copy(zlm_device* d, void* dst, const void* src, size_t bytes) {
    return zlm_gpu_dev_copy_enqueue(d, dst, src, bytes) && ok(d, hipStreamSynchronize(d->stream), "sync");
}

extern "C" bool zlm_gpu_mat_vec_enqueue(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k,
                                        const float* x_dev, float* y_dev) {
    if (!d || !d->avail) return false;
    return enqueue_gemv(d, r, quant, rows, k, x_dev, y_dev);
}

extern "C" bool zlm_gpu_mat_vec_batch_enqueue(zlm_device* d, zlm_resident* const* res, uint32_t quant,
                                              const size_t* rows, size_t n, size_t k, const float* x_dev,
                                              float* const* y_dev) {
    if (!d || !d->avail) return false;
    if (!res || !rows || !y_dev || !x_dev || n == 0 || n > static_cast<size_t>(kMultiMax)) return fail(d, "bad batch");
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant %u", quant & 0xffu);
    for (size_t i = 0; i < n; i++) {
        if (!y_dev[i]) return fail(d, "null y");
        if (!check_resident(d, res[i], qi, rows[i], k)) return false;
    }
    if (n > 1 && batch_one_launch(d, qi, k)) return enqueue_multi(d, qi, k, x_dev, res, rows, y_dev, n);
    for (size_t i = 0; i < n; i++)
        if (!enqueue_gemv(d, res[i], quant, rows[i], k, x_dev, y_dev[i])) return false;
    return true;
}

extern "C" bool zlm_gpu_mat_mul_enqueue(zlm_device* d, zlm_resident* r, uint32_t quant, size_t rows, size_t k,
                                        size_t m, const float* x_dev, float* out_dev) {
    if (!d || !d->avail) return false;
    return enqueue_gemm(d, r, quant, rows, k, m, x_dev, out_dev);
}

extern "C" bool zlm_gpu_time_mat_mul(zlm_device* d, zlm_resident* const* res, size_t n_res, uint32_t quant,
                                     size_t rows, size_t k, size_t m, const float* x_dev, float* out_dev, int iters,
                                     double* ms) {
    if (!contract_ready(d) || !res || n_res == 0 || iters < 1 || !ms) return false;
    for (size_t i = 0; i < n_res; i++)  // layouts and scratch outside the timed region
        if (!enqueue_gemm(d, res[i], quant, rows, k, m, x_dev, out_dev)) return false;
    hipEvent_t e0, e1;
    if (!ok(d, hipEventCreate(&e0), "event")) return false;
    if (!ok(d, hipEventCreate(&e1), "event")) {
        hipEventDestroy(e0);
        return false;
    }
    bool good = ok(d, hipEventRecord(e0, d->stream), "record");
    for (int i = 0; good && i < iters; i++) good = enqueue_gemm(d, res[i % n_res], quant, rows, k, m, x_dev, out_dev);
    good = good && ok(d, hipEventRecord(e1, d->stream), "record") && ok(d, hipEventSynchronize(e1), "sync");
    float t = 0.0f;
    good = good && ok(d, hipEventElapsedTime(&t, e0, e1), "elapsed");
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    *ms = t;
    return good;
}

extern "C" bool zlm_gpu_time_mat_vec(zlm_device* d, zlm_resident* const* res, size_t n_res, uint32_t quant,
                                     size_t rows, size_t k, const float* x_dev, float* y_dev, int iters,
                                     double* ms) {
    if (!contract_ready(d) || !res || n_res == 0 || iters < 1 || !ms) return false;
    for (size_t i = 0; i < n_res; i++) {  // converts layouts outside the timed region
        hipFunction_t f;
        unsigned g, b;
        if (!prepare_gemv(d, res[i], quant, rows, k, &f, &g, &b)) return false;
    }
    hipEvent_t e0, e1;
    if (!ok(d, hipEventCreate(&e0), "event") || !ok(d, hipEventCreate(&e1), "event")) return false;
    bool good = ok(d, hipEventRecord(e0, d->stream), "record");
    for (int i = 0; good && i < iters; i++) good = enqueue_gemv(d, res[i % n_res], quant, rows, k, x_dev, y_dev);
    good = good && ok(d, hipEventRecord(e1, d->stream), "record") && ok(d, hipEventSynchronize(e1), "sync");
    float t = 0.0f;
    good = good && ok(d, hipEventElapsedTime(&t, e0, e1), "elapsed");
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    *ms = t;
    return good;
}

extern "C" bool zlm_gpu_time_gemv_sequence(zlm_device* d, const zlm_gemv_desc* descs, size_t n, int iters,
                                           double* ms) {
    if (!contract_ready(d) || !descs || n == 0 || iters < 1 || !ms) return false;
    for (size_t i = 0; i < n; i++) {  // converts layouts outside the timed region
        hipFunction_t f;
        unsigned g, b;
        if (!prepare_gemv(d, descs[i].res, descs[i].quant, descs[i].rows, descs[i].k, &f, &g, &b)) return false;
    }
    hipEvent_t e0, e1;
    if (!ok(d, hipEventCreate(&e0), "event")) return false;
    if (!ok(d, hipEventCreate(&e1), "event")) {
        hipEventDestroy(e0);
        return false;
    }
    bool good = ok(d, hipEventRecord(e0, d->stream), "record");
    for (int it = 0; good && it < iters; it++)
        for (size_t i = 0; good && i < n;) {
            size_t j = i + 1;  // [i, j): one launch
            while (descs[j - 1].with_next && j < n && j - i < static_cast<size_t>(kMultiMax)) j++;
            if (j - i == 1) {
                good = enqueue_gemv(d, descs[i].res, descs[i].quant, descs[i].rows, descs[i].k, descs[i].x_dev,
                                    descs[i].y_dev);
            } else {
                zlm_resident* res[kMultiMax];
                size_t rows[kMultiMax];
                float* ys[kMultiMax];
                for (size_t t = i; t < j; t++) {
                    res[t - i] = descs[t].res;
                    rows[t - i] = descs[t].rows;
                    ys[t - i] = descs[t].y_dev;
                }
                good = zlm_gpu_mat_vec_batch_enqueue(d, res, descs[i].quant, rows, j - i, descs[i].k, descs[i].x_dev,
                                                     ys);
            }
            i = j;
        }
    good = good && ok(d, hipEventRecord(e1, d->stream), "record") && ok(d, hipEventSynchronize(e1), "sync");
    float t = 0.0f;
    good = good && ok(d, hipEventElapsedTime(&t, e0, e1), "elapsed");
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    *ms = t;
    return good;
}

// ---- the contract path as zlm's executor drives it (timing) ----

extern "C" bool zlm_gpu_time_contract_gemv(zlm_device* d, zlm_resident* const* res, size_t n_res, uint32_t quant,
                                           size_t rows, size_t k, int iters, double* us) {
    if (!contract_ready(d) || !res || n_res == 0 || iters < 1 || !us) return false;
    std::vector<float> x(k), y(rows);
    for (size_t i = 0; i < k; i++) x[i] = static_cast<float>(static_cast<int>((i * 7 + 3) % 17) - 8) * 0.125f;
    for (size_t i = 0; i < n_res; i++)  // layouts converted outside the timed region
        if (!zlm_gpu_mat_vec_resident(d, res[i], quant, rows, k, x.data(), k, y.data(), rows)) return false;
    const double t0 = now_ns();
    for (int it = 0; it < iters; it++) {
        const int32_t h =
            zlm_gpu_mat_vec_resident_burst_async(d, res[it % n_res], quant, rows, k, x.data(), k, true);
        if (h == ZLM_NULL_HANDLE || !zlm_gpu_wait_resident(d, h, y.data(), rows, rows)) return false;
    }
    *us = (now_ns() - t0) / 1e3 / iters;
    return true;
}

extern "C" bool zlm_gpu_time_contract_gemv_split(zlm_device* d, zlm_resident* const* res, size_t n_res,
                                                 uint32_t quant, size_t rows, size_t k, int iters, double* out) {
    if (!contract_ready(d) || !res || n_res == 0 || iters < 1 || !out) return false;
    std::vector<float> x(k), y(rows);
    for (size_t i = 0; i < k; i++) x[i] = static_cast<float>(static_cast<int>((i * 7 + 3) % 17) - 8) * 0.125f;
    for (size_t i = 0; i < n_res; i++)
        if (!zlm_gpu_mat_vec_resident(d, res[i], quant, rows, k, x.data(), k, y.data(), rows)) return false;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (!ok(d, hipEventCreate(&e0), "event") || !ok(d, hipEventCreate(&e1), "event")) {
        if (e0) hipEventDestroy(e0);
        return false;
    }
    double total = 0, submit = 0, wait = 0, gpu = 0;
    bool good = true;
    for (int it = 0; it < iters && good; it++) {
        const double t0 = now_ns();
        good = ok(d, hipEventRecord(e0, d->stream), "record");
        const int32_t h =
            zlm_gpu_mat_vec_resident_burst_async(d, res[it % n_res], quant, rows, k, x.data(), k, true);
        good = good && h != ZLM_NULL_HANDLE && ok(d, hipEventRecord(e1, d->stream), "record");
        const double t1 = now_ns();
        good = good && zlm_gpu_wait_resident(d, h, y.data(), rows, rows);
        const double t2 = now_ns();
        float ms = 0.0f;
        good = good && ok(d, hipEventSynchronize(e1), "sync") && ok(d, hipEventElapsedTime(&ms, e0, e1), "elapsed");
        total += t2 - t0;
        submit += t1 - t0;
        wait += t2 - t1;
        gpu += ms * 1e6;
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (!good) return false;
    out[0] = total / 1e3 / iters;
    out[1] = submit / 1e3 / iters;
    out[2] = wait / 1e3 / iters;
    out[3] = gpu / 1e3 / iters;
    return true;
}

extern "C" bool zlm_gpu_time_contract_decode(zlm_device* d, const zlm_contract_layer* layers, size_t n_layers,
                                             uint32_t quant, size_t hidden, size_t q_rows, size_t kv_rows,
                                             size_t ffn, zlm_resident* lm_head, uint32_t lm_quant, size_t vocab,
                                             int iters, double* ms) {
    if (!contract_ready(d) || !layers || n_layers == 0 || !lm_head || iters < 1 || !ms) return false;
    std::vector<float> x(hidden), qo(q_rows), ko(kv_rows), vo(kv_rows), ho(hidden), mo(hidden), logits(vocab);
    for (size_t i = 0; i < hidden; i++) x[i] = static_cast<float>(static_cast<int>((i * 7 + 3) % 17) - 8) * 0.125f;
    for (size_t i = 0; i < q_rows; i++) qo[i] = x[i % hidden];
    auto step = [&]() -> bool {
        for (size_t l = 0; l < n_layers; l++) {
            const zlm_contract_layer& L = layers[l];
            // q, k, v share the normed hidden state: one burst, then the drain
            const int32_t hq = zlm_gpu_mat_vec_resident_burst_async(d, L.q, quant, q_rows, hidden, x.data(), hidden,
                                                                    true);
            const int32_t hk = zlm_gpu_mat_vec_resident_burst_async(d, L.k, quant, kv_rows, hidden, x.data(),
                                                                    hidden, false);
            const int32_t hv = zlm_gpu_mat_vec_resident_burst_async(d, L.v, quant, kv_rows, hidden, x.data(),
                                                                    hidden, false);
            if (hq == ZLM_NULL_HANDLE || hk == ZLM_NULL_HANDLE || hv == ZLM_NULL_HANDLE) return false;
            if (!zlm_gpu_wait_resident(d, hq, qo.data(), q_rows, q_rows) ||
                !zlm_gpu_wait_resident(d, hk, ko.data(), kv_rows, kv_rows) ||
                !zlm_gpu_wait_resident(d, hv, vo.data(), kv_rows, kv_rows))
                return false;
            // (the CPU's attention would run here; its output stands in as q's rows)
            const int32_t ho_h = zlm_gpu_mat_vec_resident_burst_async(d, L.o, quant, hidden, q_rows, qo.data(),
                                                                      q_rows, true);
            if (ho_h == ZLM_NULL_HANDLE || !zlm_gpu_wait_resident(d, ho_h, ho.data(), hidden, hidden)) return false;
            // (residual add and the FFN RMSNorm on the CPU) then the fused MLP pair
            const int32_t hm = zlm_gpu_mat_vec_mlp_pair_resident_burst_async(
                d, L.gate, L.up, L.down, quant, quant, hidden, hidden, ffn, x.data(), hidden, ZLM_ACT_SILU,
                ZLM_VARIANT_PLAIN, true);
            if (hm == ZLM_NULL_HANDLE || !zlm_gpu_wait_resident(d, hm, mo.data(), hidden, hidden)) return false;
        }
        return zlm_gpu_mat_vec_resident(d, lm_head, lm_quant, vocab, hidden, x.data(), hidden, logits.data(), vocab);
    };
    if (!step()) return false;  // layouts converted outside the timed region
    const double t0 = now_ns();
    for (int it = 0; it < iters; it++)
        if (!step()) return false;
    *ms = (now_ns() - t0) / 1e6 / iters;
    return true;
}

extern "C" bool zlm_gpu_gemv_op_enqueue(zlm_device* d, const zlm_gemv_op* op) {
    if (!d || !d->avail) return false;
    if (!op) return fail(d, "null op");
    return enqueue_op(d, *op);
}

// ---- decode-step glue, graphs and synthetic data ----

extern "C" bool zlm_gpu_qk_norm_rope_kv_enqueue(zlm_device* d, const float* qkv, float* q_out, const float* q_norm_w,
                                                const float* k_norm_w, uint32_t n_heads, uint32_t n_kv_heads,
                                                uint32_t head_dim, float eps, float freq_base, const int32_t* pos,
                                                uint16_t* k_cache, uint16_t* v_cache, uint32_t max_seq) {
    if (!d || !d->avail) return false;
    if (!qkv || !q_out || !q_norm_w || !k_norm_w || !pos || !k_cache || !v_cache) return fail(d, "null buffer");
    if (n_heads == 0 || n_kv_heads == 0 || head_dim == 0 || head_dim % 2 || head_dim > 256 || max_seq == 0)
        return fail(d, "bad attention shape");
    uint16_t* kc = k_cache;
    uint16_t* vc = v_cache;
    void* args[] = {&qkv, &q_out, &q_norm_w, &k_norm_w, &n_heads, &n_kv_heads, &head_dim, &eps, &freq_base,
                    &pos, &kc, &vc, &max_seq};
    return launch(d, d->qk_norm_rope_kv, n_heads + 2 * n_kv_heads, 64, args, "qk norm rope");
}

namespace {

// Size the attention partials (floats).  Allocation happens on an eager call;
// a call under capture that would need it fails.
bool ensure_attn_scratch(zlm_device* d, size_t need) {
    if (need > d->attn_part_cap) {
        if (!may_replace_scratch(d, kUsesAttn, "the attention scratch")) return false;
        if (d->attn_part) {
            hipStreamSynchronize(d->stream);
            hipFree(d->attn_part);
        }
        d->attn_part = nullptr;
        d->attn_part_cap = 0;
        if (!ok(d, hipMalloc(reinterpret_cast<void**>(&d->attn_part), need * sizeof(float)), "hipMalloc attn"))
            return false;
        d->attn_part_cap = need;
    }
    if (d->capturing) d->capture_uses |= kUsesAttn;
    return true;
}

}  // namespace

namespace {

// The split merge: one 256-thread workgroup per q head up to 64 splits
// (4096 positions), beyond that the wide merge: two workgroups per head (64
// dims each) of one wave per 32 splits (at most 16 waves).
bool enqueue_attn_merge(zlm_device* d, float* part, uint32_t nsplit, uint32_t n_heads, float* out) {
    void* args[] = {&part, &nsplit, &out};
    if (nsplit > 64) {
        const unsigned waves = std::min<unsigned>(16u, (nsplit + 31) / 32);
        return launch3(d, d->attn_combine_wide, n_heads, 2, 1, 64 * waves, args, "attention combine wide");
    }
    return launch(d, d->attn_combine, n_heads, 256, args, "attention combine");
}

bool check_attn_decode(zlm_device* d, const float* qkv, const float* q_norm_w, const float* k_norm_w,
                       uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim, const int32_t* pos,
                       const uint16_t* k_cache, const uint16_t* v_cache, uint32_t max_seq, const float* out) {
    if (!qkv || !q_norm_w || !k_norm_w || !pos || !k_cache || !v_cache || !out) return fail(d, "null buffer");
    if (head_dim != 128) return fail(d, "attention supports head_dim 128 (got %u)", head_dim);
    if (n_kv_heads == 0 || n_heads % n_kv_heads || n_heads / n_kv_heads > 4 || max_seq == 0)
        return fail(d, "attention supports 1-4 q heads per kv head");
    return true;
}

// The fused attention launch and the merge, with the partials in `part`
// (n_heads * nsplit * 130 floats).
bool enqueue_attn_decode(zlm_device* d, const float* qkv, const float* q_norm_w, const float* k_norm_w,
                         uint32_t n_heads, uint32_t n_kv_heads, float eps, float freq_base, const int32_t* pos,
                         uint16_t* k_cache, uint16_t* v_cache, uint32_t max_seq, float scale, float* out,
                         float* part, uint32_t nsplit) {
    {
        void* args[] = {&qkv, &q_norm_w, &k_norm_w, &n_heads, &n_kv_heads, &eps, &freq_base, &pos, &k_cache,
                        &v_cache, &max_seq, &scale, &part, &nsplit};
        if (!launch3(d, d->attn_decode, n_kv_heads, nsplit, 1, 256, args, "attention decode")) return false;
    }
    return enqueue_attn_merge(d, part, nsplit, n_heads, out);
}

}  // namespace

extern "C" bool zlm_gpu_attention_decode_window_enqueue(zlm_device* d, const float* qkv, const float* q_norm_w,
                                                        const float* k_norm_w, uint32_t n_heads, uint32_t n_kv_heads,
                                                        uint32_t head_dim, float eps, float freq_base,
                                                        const int32_t* pos, uint16_t* k_cache, uint16_t* v_cache,
                                                        uint32_t max_seq, uint32_t window, float scale, float* out) {
    if (!d || !d->avail) return false;
    if (!check_attn_decode(d, qkv, q_norm_w, k_norm_w, n_heads, n_kv_heads, head_dim, pos, k_cache, v_cache, max_seq,
                           out))
        return false;
    if (window == 0 || window > max_seq) return fail(d, "attention window %u outside 1..max_seq %u", window, max_seq);
    const uint32_t nsplit = static_cast<uint32_t>((static_cast<uint64_t>(window) + 63) / 64);
    if (!ensure_attn_scratch(d, static_cast<size_t>(n_heads) * nsplit * 130)) return false;
    return enqueue_attn_decode(d, qkv, q_norm_w, k_norm_w, n_heads, n_kv_heads, eps, freq_base, pos, k_cache, v_cache,
                               max_seq, scale, out, d->attn_part, nsplit);
}

extern "C" bool zlm_gpu_attention_decode_enqueue(zlm_device* d, const float* qkv, const float* q_norm_w,
                                                 const float* k_norm_w, uint32_t n_heads, uint32_t n_kv_heads,
                                                 uint32_t head_dim, float eps, float freq_base, const int32_t* pos,
                                                 uint16_t* k_cache, uint16_t* v_cache, uint32_t max_seq, float scale,
                                                 float* out) {
    return zlm_gpu_attention_decode_window_enqueue(d, qkv, q_norm_w, k_norm_w, n_heads, n_kv_heads, head_dim, eps,
                                                   freq_base, pos, k_cache, v_cache, max_seq, max_seq, scale, out);
}

extern "C" bool zlm_gpu_attention_decode_enqueue_noalloc(zlm_device* d, const float* qkv, const float* q_norm_w,
                                                         const float* k_norm_w, uint32_t n_heads, uint32_t n_kv_heads,
                                                         uint32_t head_dim, float eps, float freq_base,
                                                         const int32_t* pos, uint16_t* k_cache, uint16_t* v_cache,
                                                         uint32_t max_seq, float scale, float* out) {
    if (!d || !d->avail) return false;
    if (!d->static_scratch)
        return fail(d, "static scratch unavailable (lookup at init failed: %s)", d->static_scratch_err.c_str());
    if (!check_attn_decode(d, qkv, q_norm_w, k_norm_w, n_heads, n_kv_heads, head_dim, pos, k_cache, v_cache, max_seq,
                           out))
        return false;
    const uint32_t nsplit = static_cast<uint32_t>((static_cast<uint64_t>(max_seq) + 63) / 64);
    const uint64_t head_splits = static_cast<uint64_t>(n_heads) * nsplit;
    if (head_splits > ZLM_STATIC_SCRATCH_HEAD_SPLITS)
        return fail(d, "no-alloc attention holds at most %u head-splits (n_heads * ceil(max_seq / 64)); got %u * %u",
                    ZLM_STATIC_SCRATCH_HEAD_SPLITS, n_heads, nsplit);
    return enqueue_attn_decode(d, qkv, q_norm_w, k_norm_w, n_heads, n_kv_heads, eps, freq_base, pos, k_cache, v_cache,
                               max_seq, scale, out, d->static_scratch, nsplit);
}

extern "C" bool zlm_gpu_attention_enqueue(zlm_device* d, const float* q, const uint16_t* k_cache,
                                          const uint16_t* v_cache, uint32_t n_heads, uint32_t n_kv_heads,
                                          uint32_t head_dim, const int32_t* pos, uint32_t max_seq, float scale,
                                          float* out) {
    if (!d || !d->avail) return false;
    if (!q || !k_cache || !v_cache || !pos || !out) return fail(d, "null buffer");
    if (head_dim != 128) return fail(d, "attention supports head_dim 128 (got %u)", head_dim);
    if (n_kv_heads == 0 || n_heads % n_kv_heads || n_heads / n_kv_heads > 4 || max_seq == 0)
        return fail(d, "attention supports 1-4 q heads per kv head");
    uint32_t nsplit = (max_seq + 63) / 64;
    if (!ensure_attn_scratch(d, static_cast<size_t>(n_heads) * nsplit * 130)) return false;
    float* part = d->attn_part;
    {
        void* args[] = {&q, &k_cache, &v_cache, &n_heads, &n_kv_heads, &pos, &max_seq, &scale, &part, &nsplit};
        if (!launch3(d, d->attn_partial, n_kv_heads, nsplit, 1, 256, args, "attention")) return false;
    }
    return enqueue_attn_merge(d, part, nsplit, n_heads, out);
}

struct zlm_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    zlm_device* owner = nullptr;
    uint32_t uses = 0;  // kUses* bits: library scratch the graph references
};

// Whether a profiler library (rocprofiler-sdk, as rocprofv3 preloads it, or
// the older librocprofiler64) is mapped into this process (maps_path: a
// /proc/<pid>/maps-format file; null = this process's own).  The HIP runtime's
// own librocprofiler-register and torch's roctracer/roctx are always mapped
// and do not count.  1 or 0, or -1 where the file could not be read to its end.
int profiler_in_maps(const char* maps_path) {
    FILE* f = fopen(maps_path ? maps_path : "/proc/self/maps", "r");
    if (!f) return -1;
    char line[4096];
    bool found = false;
    while (!found && fgets(line, sizeof line, f))
        found = strstr(line, "librocprofiler-sdk") != nullptr || strstr(line, "librocprofiler64") != nullptr;
    const bool whole = !ferror(f);
    fclose(f);
    return found ? 1 : whole ? 0 : -1;
}

// profiler_in_maps(nullptr), the maps read again only when the loader has added
// or removed objects since: reading them costs 0.4 ms in a process with torch
// loaded, most of a small model's step; the loader's counters (of all its
// namespaces) cost 0.1 us.  A map that could not be read counts as none for this
// call and is read again at the next.
bool profiler_in_process() {
    struct Counts {
        unsigned long long adds, subs;
    } now = {0, 0};
    dl_iterate_phdr(
        [](dl_phdr_info* info, size_t size, void* out) {
            if (size >= offsetof(dl_phdr_info, dlpi_subs) + sizeof info->dlpi_subs)
                *static_cast<Counts*>(out) = {info->dlpi_adds, info->dlpi_subs};
            return 1;  // the counters are the same in every entry
        },
        &now);
    static std::mutex mu;
    static Counts seen = {0, 0};
    static bool found = false;
    std::lock_guard<std::mutex> lock(mu);
    if (now.adds == 0 || now.adds != seen.adds || now.subs != seen.subs) {
        const int read = profiler_in_maps(nullptr);
        if (read < 0) return false;
        found = read == 1;
        seen = now;
    }
    return found;
}

extern "C" bool zlm_gpu_capture_begin(zlm_device* d) {
    if (!d || !d->avail) return false;
    if (d->capturing) return fail(d, "already capturing");
    build_tiles_due(d);
    if (!ok(d, hipStreamBeginCapture(d->stream, hipStreamCaptureModeRelaxed), "begin capture")) return false;
    d->capturing = true;
    d->capture_uses = 0;
    return true;
}

extern "C" zlm_graph* zlm_gpu_capture_end(zlm_device* d) {
    if (!d || !d->avail || !d->capturing) return nullptr;
    d->capturing = false;
    zlm_graph* g = new (std::nothrow) zlm_graph();
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(d->stream, &graph);
    if (!g || !ok(d, e, "end capture") || !graph) {
        if (graph) hipGraphDestroy(graph);
        delete g;
        return nullptr;
    }
    g->graph = graph;
    if (!ok(d, hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0), "instantiate")) {
        hipGraphDestroy(graph);
        delete g;
        return nullptr;
    }
    g->owner = d;
    g->uses = d->capture_uses;
    if (g->uses & kUsesAttn) d->attn_graphs++;
    if (g->uses & kUsesGemm) d->gemm_graphs++;
    return g;
}

// Graph launches queued ahead of the GPU by one zlm_gpu_graph_launch call:
// before launch i the host waits for launch i - kGraphsInFlight to finish, so
// a long run of replays never holds more than this many graphs' dispatches
// (a decode step is ~220 kernels) in the stream's queue at once.
constexpr int kGraphsInFlight = 4;

extern "C" bool zlm_gpu_profiler_loaded(const char* maps_path) {
    return maps_path ? profiler_in_maps(maps_path) == 1 : profiler_in_process();
}

extern "C" bool zlm_gpu_kernel_convention(const char* name, int32_t* role, bool* struct_args) {
    if (!name || !role || !struct_args) return false;
    for (int q = 0; q < kNumQuants; q++) {
        const std::string prefix = std::string("zlm_gemv_") + kQuantNames[q] + "_";
        if (strncmp(name, prefix.c_str(), prefix.size()) != 0) continue;
        int r = 0;
        bool st = false;
        kernel_role(name, q, &r, &st);
        *role = r;
        *struct_args = st;
        return true;
    }
    return false;
}

extern "C" bool zlm_gpu_launch_log(zlm_device* d, bool enable) {
    if (!d || !d->avail) return false;
    d->log_launches = enable;
    d->launch_log.clear();
    return true;
}

extern "C" size_t zlm_gpu_launch_log_read(const zlm_device* d, zlm_launch_record* out, size_t max) {
    if (!d || !d->avail) return 0;
    const size_t n = std::min(max, d->launch_log.size());
    if (out)
        for (size_t i = 0; i < n; i++) out[i] = d->launch_log[i];
    return d->launch_log.size();
}

extern "C" uint64_t zlm_gpu_scratch_device_bytes(const zlm_device* d) {
    if (!d || !d->avail) return 0;
    uint64_t b = (d->x_cap + d->y_cap + d->bx_cap + d->mid_cap + d->attn_part_cap) * sizeof(float) +
                 d->q_scratch_cap + d->s_raw_cap + d->s_lay_cap;
    for (const Slot& sl : d->slots) b += sl.x_cap * sizeof(float);
    return b;
}

extern "C" bool zlm_gpu_graph_launch(zlm_device* d, zlm_graph* g, int iters, double* ms) {
    if (!d || !d->avail || !g || iters < 1) return false;
    if (g->owner != d) return fail(d, "graph was captured on another device handle");
    // Replays of a captured decode step aborted inside hipGraphLaunch ("invalid
    // AQL packet") when the process ran under rocprofv3's kernel trace, while
    // the same replays without the profiler run clean; the cause is not known,
    // so replays are refused while a rocprofiler library is in the process
    // (profile the same kernels from eager launches instead).
    if (profiler_in_process())
        return fail(d, "graph replay refused: a rocprofiler library is loaded in this process "
                       "(replays under the kernel tracer aborted); trace eager launches instead");
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipEvent_t done[kGraphsInFlight] = {};
    bool good = true;
    const bool bounded = iters > kGraphsInFlight;  // fewer replays never wait for one
    if (bounded)
        for (hipEvent_t& e : done) good = good && ok(d, hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
    if (good && ms) {
        good = ok(d, hipEventCreate(&e0), "event") && ok(d, hipEventCreate(&e1), "event") &&
               ok(d, hipEventRecord(e0, d->stream), "record");
    }
    for (int i = 0; i < iters && good; i++) {
        hipEvent_t e = done[i % kGraphsInFlight];
        if (i >= kGraphsInFlight) good = ok(d, hipEventSynchronize(e), "graph wait");
        good = good && ok(d, hipGraphLaunch(g->exec, d->stream), "graph launch") &&
               (!bounded || ok(d, hipEventRecord(e, d->stream), "record"));
    }
    if (good && ms) good = ok(d, hipEventRecord(e1, d->stream), "record");
    good = ok(d, hipStreamSynchronize(d->stream), "sync") && good;
    if (good && ms) {
        float t = 0.0f;
        good = ok(d, hipEventElapsedTime(&t, e0, e1), "elapsed");
        *ms = t;
    }
    for (hipEvent_t e : {e0, e1})
        if (e) hipEventDestroy(e);
    for (hipEvent_t e : done)
        if (e) hipEventDestroy(e);
    return good;
}

extern "C" void zlm_gpu_graph_destroy(zlm_device* d, zlm_graph* g) {
    if (!g) return;
    if (d && d->avail) hipStreamSynchronize(d->stream);
    if (d && d == g->owner) {
        if (g->uses & kUsesAttn) d->attn_graphs--;
        if (g->uses & kUsesGemm) d->gemm_graphs--;
    }
    if (g->exec) hipGraphExecDestroy(g->exec);
    if (g->graph) hipGraphDestroy(g->graph);
    delete g;
}

extern "C" zlm_resident* zlm_gpu_synth_resident(zlm_device* d, uint32_t ggml_type, size_t nblocks, uint64_t seed,
                                                float scale) {
    if (!d || !d->avail) return nullptr;
    if (ggml_type != ZLM_GGML_Q4_0 && ggml_type != ZLM_GGML_Q8_0) {
        fail(d, "synthetic blocks exist for q4_0 and q8_0");
        return nullptr;
    }
    const QuantInfo* qi = quant_info(ggml_type);
    zlm_resident* r = new (std::nothrow) zlm_resident();
    if (!r) return nullptr;
    r->owner = d;
    r->bytes = nblocks * qi->block_bytes;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&r->raw), r->bytes ? r->bytes : 1), "hipMalloc resident")) {
        delete r;
        return nullptr;
    }
    uint8_t* raw = r->raw;
    uint64_t n = nblocks;
    void* args[] = {&raw, &ggml_type, &n, &seed, &scale};
    if (nblocks && (!launch(d, d->synth_blocks, static_cast<unsigned>((nblocks + 255) / 256), 256, args, "synth") ||
                    !ok(d, hipStreamSynchronize(d->stream), "sync"))) {
        hipFree(r->raw);
        delete r;
        return nullptr;
    }
    return r;
}

extern "C" bool zlm_gpu_synth_f16(zlm_device* d, uint16_t* dst, size_t n, uint64_t seed, float scale) {
    if (!d || !d->avail) return false;
    if (!dst) return fail(d, "null buffer");
    if (n == 0) return true;
    uint64_t nn = n;
    void* args[] = {&dst, &nn, &seed, &scale};
    return launch(d, d->synth_f16, static_cast<unsigned>((n + 255) / 256), 256, args, "synth f16") &&
           ok(d, hipStreamSynchronize(d->stream), "sync");
}

extern "C" bool zlm_gpu_dequant_resident(zlm_device* d, zlm_resident* r, uint32_t quant, size_t n, float* out) {
    if (!d || !d->avail || !r || !out) return false;
    const QuantInfo* qi = quant_info(quant);
    if (!qi) return fail(d, "unsupported quant");
    if (n % qi->block_elems) return fail(d, "n must be whole blocks");
    const uint64_t nblk = n / qi->block_elems;
    if (r->bytes < nblk * qi->block_bytes) return fail(d, "resident too short");
    if (!ensure_layout(d, r, qi)) return false;
    float* dev_out = nullptr;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&dev_out), (n ? n : 1) * sizeof(float)), "hipMalloc")) return false;
    bool good = true;
    if (nblk) {
        uint64_t nb = nblk;
        void* args[] = {&r->payload, &r->scales, &dev_out, &nb};
        good = launch(d, d->dequant[qi->slot], static_cast<unsigned>((nblk + 255) / 256), 256, args, "dequant");
    }
    good = good && ok(d, hipMemcpyAsync(out, dev_out, n * sizeof(float), hipMemcpyDeviceToHost, d->stream), "read") &&
           ok(d, hipStreamSynchronize(d->stream), "sync");
    hipFree(dev_out);
    return good;
}

extern "C" bool zlm_gpu_quantize_act_q8(zlm_device* d, const float* x, size_t n, int8_t* qx, float* dx,
                                        int32_t* sums) {
    if (!d || !d->avail || !x || !qx || !dx || !sums || n % 32) return false;
    const size_t nblk = n / 32;
    if (nblk == 0) return true;
    char* buf = nullptr;
    const size_t xb = n * 4, qb = (n + 15) & ~size_t(15), db = nblk * 4;
    if (!ok(d, hipMalloc(reinterpret_cast<void**>(&buf), xb + qb + 2 * db + 64), "hipMalloc")) return false;
    float* dxx = reinterpret_cast<float*>(buf);
    int8_t* dq = reinterpret_cast<int8_t*>(buf + xb);
    float* ddx = reinterpret_cast<float*>(buf + xb + qb);
    int32_t* ds = reinterpret_cast<int32_t*>(buf + xb + qb + db);
    uint64_t nb = nblk;
    void* args[] = {&dxx, &dq, &ddx, &ds, &nb};
    bool good = ok(d, hipMemcpyAsync(dxx, x, xb, hipMemcpyHostToDevice, d->stream), "upload") &&
                launch(d, d->quantize_q8, static_cast<unsigned>((nblk + 255) / 256), 256, args, "quantize") &&
                ok(d, hipMemcpyAsync(qx, dq, n, hipMemcpyDeviceToHost, d->stream), "read qx") &&
                ok(d, hipMemcpyAsync(dx, ddx, db, hipMemcpyDeviceToHost, d->stream), "read dx") &&
                ok(d, hipMemcpyAsync(sums, ds, db, hipMemcpyDeviceToHost, d->stream), "read sums") &&
                ok(d, hipStreamSynchronize(d->stream), "sync");
    hipFree(buf);
    return good;
}
