// HIP backend behind SimdOnnx's backend surface (include/sox_backend.h).
//
//   HipBackend          (VkBackend,  Backends/Vulkan/VkBackend.cs:11-267)
//   HipGraphModel       (VkGraphModel, Backends/Vulkan/VkGraph.cs:44-1233)
//   HipInferenceSession (VkInferenceSession, Backends/Vulkan/VkSession.cs:63-571)
//
// Everything here talks to the GPU only through the thin C ABI of include/sox_hip.h (the calls a
// managed host would P/Invoke): code objects embedded in this library are loaded with
// sox_module_load (hipModuleLoadData) and every dispatch is a sox_launch
// (hipModuleLaunchKernel) of a kernarg block laid out by include/sox_abi.h.
#include "../../../include/sox_backend.h"

#include <elf.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <exception>
#include <map>
#include <set>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "../../../include/sox_abi.h"

// ---- embedded code objects (generated by the build: one .incbin per .hsaco) ----
struct SoxResource {
    const char* name;
    const unsigned char* start;
    const unsigned char* end;
};
#include "resources_table.inc"

namespace {

thread_local std::string g_err;

struct SoxError : std::runtime_error {
    int code;
    SoxError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

[[noreturn]] void fail(int code, const std::string& msg) { throw SoxError(code, msg); }
[[noreturn]] void unsupported(const std::string& msg) { fail(SOX_E_UNSUPPORTED, "HIP: " + msg); }

void check(int rc, const char* what) {
    if (rc != SOX_OK) fail(rc, std::string(what) + ": " + sox_error_string(rc));
}

template <class F> int guarded(F&& f) {
    try {
        f();
        return SOX_OK;
    } catch (const SoxError& e) {
        g_err = e.what();
        return e.code;
    } catch (const std::exception& e) {
        g_err = e.what();
        return SOX_E_INVALID;
    }
}

// IEEE binary16 round-to-nearest-even (the (Half) cast of GpuPack.Build, Extensions.cs:315).
uint16_t f32_to_f16_bits(float f) {
    _Float16 h = (_Float16)f;
    uint16_t b;
    memcpy(&b, &h, 2);
    return b;
}

float f16_bits_to_f32(uint16_t b) {
    _Float16 h;
    memcpy(&h, &b, 2);
    return (float)h;
}

// Over n values: the bits, and the rounded values as floats. With F16C where the CPU has it (a library call per value
// without: creating the recognizer graph 84 ms, 25 with); the library itself runs on any CPU.
#if defined(__x86_64__)
__attribute__((target("f16c"))) void f32_to_f16_f16c(const float* x, uint16_t* y, int64_t n) {
    for (int64_t i = 0; i < n; i++) {
        const _Float16 h = (_Float16)x[i];
        memcpy(y + i, &h, 2);
    }
}
__attribute__((target("f16c"))) void round_f16_f16c(const float* x, float* y, int64_t n) {
    for (int64_t i = 0; i < n; i++) y[i] = (float)(_Float16)x[i];
}
bool has_f16c() {
    static const bool has = __builtin_cpu_supports("f16c");
    return has;
}
#endif
void f32_to_f16_n(const float* x, uint16_t* y, int64_t n) {
#if defined(__x86_64__)
    if (has_f16c()) return f32_to_f16_f16c(x, y, n);
#endif
    for (int64_t i = 0; i < n; i++) y[i] = f32_to_f16_bits(x[i]);
}
void round_f16_n(const float* x, float* y, int64_t n) {
#if defined(__x86_64__)
    if (has_f16c()) return round_f16_f16c(x, y, n);
#endif
    for (int64_t i = 0; i < n; i++) y[i] = f16_bits_to_f32(f32_to_f16_bits(x[i]));
}

// bfloat16 round-to-nearest-even: the upper half of the fp32 pattern after adding 0x7fff plus the
// lowest kept bit (ties to even); NaN keeps a quiet NaN.
uint16_t f32_to_bf16_bits(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

float bf16_bits_to_f32(uint16_t b) {
    const uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

int64_t prod(const std::vector<int>& v) {
    int64_t n = 1;
    for (int d : v) n *= d;
    return n;
}

}  // namespace

// ================================================================================================
// Plan
// ================================================================================================
struct PlanValue {
    std::vector<int> shape, layout;  // layout empty = identity
    int buf = -1;
    std::vector<float> floats;
    bool is_const = false;
    std::string name;
    int64_t count() const { return prod(shape); }
    std::vector<int> phys() const {
        if (layout.empty()) return shape;
        std::vector<int> p(shape.size());
        for (size_t i = 0; i < shape.size(); i++) p[i] = shape[layout[i]];
        return p;
    }
};

struct PlanNode {
    int op = 0;
    std::vector<int> in, out;
    std::vector<uint8_t> params;
    std::string ext;
    template <class P> const P& p() const {
        if (params.size() < sizeof(P)) fail(SOX_E_INVALID, "node params record too short");
        return *reinterpret_cast<const P*>(params.data());
    }
};

struct sox_plan {
    std::vector<PlanValue> values;
    std::vector<PlanNode> nodes;
    std::vector<int64_t> buf_offset;
    int64_t arena_floats = 0;
    std::vector<int> inputs;
    int output = -1;
};

// ================================================================================================
// Backend
// ================================================================================================
struct ExtEntry {
    sox_ext_emit_fn emit;
    sox_ext_consts_fn consts;
    void* user;
};

// Whether the AMDGPU code object `img` (an ELF image) defines kernel `name`: its symbol table holds
// the kernel's descriptor symbol "<name>.kd". Every read is bounds-checked against the image size.
static bool code_object_defines(const unsigned char* img, size_t size, const std::string& name) {
    Elf64_Ehdr eh;
    if (size < sizeof eh) return false;
    memcpy(&eh, img, sizeof eh);
    if (memcmp(eh.e_ident, ELFMAG, SELFMAG) != 0 || eh.e_ident[EI_CLASS] != ELFCLASS64) return false;
    if (eh.e_shentsize != sizeof(Elf64_Shdr) || eh.e_shoff > size ||
        (uint64_t)eh.e_shnum * sizeof(Elf64_Shdr) > size - eh.e_shoff)
        return false;
    auto section = [&](uint32_t i) {
        Elf64_Shdr sh;
        memcpy(&sh, img + eh.e_shoff + (uint64_t)i * sizeof sh, sizeof sh);
        return sh;
    };
    const std::string want = name + ".kd";
    for (uint32_t i = 0; i < eh.e_shnum; i++) {
        const Elf64_Shdr sh = section(i);
        if ((sh.sh_type != SHT_SYMTAB && sh.sh_type != SHT_DYNSYM) || sh.sh_link >= eh.e_shnum) continue;
        const Elf64_Shdr st = section(sh.sh_link);
        if (sh.sh_offset > size || sh.sh_size > size - sh.sh_offset || st.sh_offset > size ||
            st.sh_size > size - st.sh_offset)
            continue;
        const char* strs = reinterpret_cast<const char*>(img + st.sh_offset);
        for (uint64_t k = 0; k + sizeof(Elf64_Sym) <= sh.sh_size; k += sizeof(Elf64_Sym)) {
            Elf64_Sym sym;
            memcpy(&sym, img + sh.sh_offset + k, sizeof sym);
            if (sym.st_name >= st.sh_size) continue;
            const size_t room = (size_t)(st.sh_size - sym.st_name);
            if (want.size() < room && memcmp(strs + sym.st_name, want.c_str(), want.size() + 1) == 0) return true;
        }
    }
    return false;
}

struct sox_backend {
    sox_device_info info{};
    std::vector<void*> modules;
    std::map<std::string, void*> fns;
    std::map<std::string, ExtEntry> exts;
    std::mutex mu;
    bool lost = false;
    // Built by sox_backend_create_offline: no device is touched. Graphs lower completely (rewrites,
    // const packing, dispatch records) against the embedded code objects' symbol tables, but cannot
    // run: kernel handles are stand-ins and nothing is uploaded.
    bool offline = false;
    std::map<std::string, std::string> offline_fns;  // kernel name -> stand-in handle (its map node)
    void* dummy = nullptr;  // 256 zero bytes for unused bindings
    void* scratch = nullptr;  // this device's static scratch (sox_scratch), for the allocation-free entry points
    size_t scratch_bytes = 0;
    // the scratch's users: one at a time on the host, and each stream waits for the previous user's
    // kernels (an event recorded after them; not for work captured into a graph)
    std::mutex scratch_mu;
    void* scratch_ev = nullptr;
    bool scratch_used = false;

    void need_device(const char* what) const {
        if (offline) fail(SOX_E_UNSUPPORTED, std::string(what) + ": the backend was created without a device");
    }

    void* fn(const std::string& name) {
        std::lock_guard<std::mutex> lk(mu);
        if (offline) {
            auto it = offline_fns.find(name);
            if (it != offline_fns.end()) return &it->second;
            for (const SoxResource* r = sox_resources; r->name; r++)
                if (code_object_defines(r->start, (size_t)(r->end - r->start), name))
                    return &offline_fns.emplace(name, name).first->second;
            fail(SOX_E_NOT_FOUND, "HIP: kernel '" + name + "' not found in the embedded code objects");
        }
        auto it = fns.find(name);
        if (it != fns.end()) return it->second;
        for (void* m : modules) {
            void* f = nullptr;
            if (sox_module_function(&f, m, name.c_str()) == SOX_OK) {
                fns[name] = f;
                return f;
            }
        }
        fail(SOX_E_NOT_FOUND, "HIP: kernel '" + name + "' not found in the embedded code objects");
    }
};

namespace {
std::mutex g_default_mu;
sox_backend* g_default = nullptr;
}  // namespace

// ================================================================================================
// Graph model
// ================================================================================================
struct Patch {
    uint32_t off;
    sox_bind bind;
};

struct Dispatch {
    void* fn = nullptr;
    std::string name;    // the dispatch's label (the op it runs)
    std::string kernel;  // the code object function it launches
    int node = -1;
    uint32_t grid[3] = {1, 1, 1}, block[3] = {256, 1, 1}, lds = 0;
    std::vector<uint8_t> kernarg;
    std::vector<Patch> patches;
};

// Parts of the hidden width of the split MLP kernels (sox_mlpq_*), by K1.
int mlp_parts(int k1) { return k1 == 192 ? 3 : k1 == 128 ? 4 : 2; }

struct sox_graph {
    sox_backend* be = nullptr;
    sox_plan plan;  // private copy
    bool f16 = true;   // 16-bit activation / weight storage (fp16, or bf16 when bf16 is set)
    bool bf16 = false;
    int es = 2;
    void* consts = nullptr;
    uint64_t const_bytes = 0;
    uint64_t sync_bytes = 0;  // cross-workgroup counters per session (SOX_SLOT_SYNC)
    std::map<std::pair<int, int>, std::pair<uint64_t, uint64_t>> const_off;  // (value, kind) -> (offset, bytes)
    std::vector<Dispatch> disp;
    std::set<int> folded;  // nodes folded into another node at graph creation (emit nothing)
    std::map<int, std::pair<int, int>> residual_add;  // Gemm node -> (its Add node, the residual value)
    std::map<int, int> padded_ld;  // value -> row stride of its buffer when its rows are padded
    struct LnFold {
        int colsum;  // const value: column sums of the gamma-scaled weights (sox_igemm_args.ln_c)
        float eps;
    };
    std::map<int, LnFold> ln_fold;  // Gemm node -> the LayerNorm folded into it (its A is that LN's input)
    struct Mlp {
        int fc2, add, residual, out;  // the second Gemm, its fused Add (-1 none), the Add's residual, the output
        int proj = -1, proj_res = -1;  // the projection Gemm computing x with its residual Add (-1 none), that residual
        bool split = false;            // per (32 rows, part of the hidden width), then a sum of the parts
    };
    std::map<int, Mlp> mlp;  // first Gemm (LN-folded, GELU) -> the rest of a transformer MLP run as one kernel
    std::map<int, int> qkv_attn;  // qkv Gemm (LN-folded) -> the Attention node run with it as one kernel
    struct UpCat {
        int n = 0, c = 0;              // sources, channels each
        int src[4] = {-1, -1, -1, -1};  // the values concatenated (before their upsample)
        int shift[4] = {0, 0, 0, 0};    // log2 of each source's nearest upsample factor
    };
    std::map<int, UpCat> upcat;  // 3x3 conv -> its input as a concat of nearest upsamples, gathered by the conv
    // ResizeNearest + Add node -> (the 1x1 conv producing the addend, log2 of the factor): the conv runs in
    // the Add's place with the upsample as its residual, read at (y >> shift, x >> shift)
    std::map<int, std::pair<int, int>> upadd;
    std::set<int> moved;  // nodes that emit at another node's place (their reads still count there)
    // first ConvT (2x2 s2, run as a Gemm) -> the one-channel 2x2 s2 ConvT that alone reads its output:
    // both run as one kernel at the first one's place (plan_convt_chain)
    std::map<int, int> convt_chain;
    uint64_t scratch_off = 0, scratch_bytes = 0, tail_bytes = 0;
    int refs = 1;

    uint64_t arena_bytes() const {
        uint64_t a = std::max<uint64_t>(scratch_off + scratch_bytes, (tail_bytes + 255) & ~255ull);
        return std::max<uint64_t>(a, 256);
    }
    const PlanValue& V(int id) const {
        if (id < 0 || id >= (int)plan.values.size()) fail(SOX_E_INVALID, "value id out of range");
        return plan.values[id];
    }
    bool elem_fp32(int kind) const { return !f16 || kind == SOX_CK_F32 || kind == SOX_CK_F32T; }
    // n floats rounded to this graph's 16-bit storage type and back (what the kernels multiply)
    void round16(const float* x, float* y, int64_t n) const {
        if (!bf16) return round_f16_n(x, y, n);
        for (int64_t i = 0; i < n; i++) y[i] = bf16_bits_to_f32(f32_to_bf16_bits(x[i]));
    }
    void bits16(const float* x, uint16_t* y, int64_t n) const {
        if (!bf16) return f32_to_f16_n(x, y, n);
        for (int64_t i = 0; i < n; i++) y[i] = f32_to_bf16_bits(x[i]);
    }
    float from16(uint16_t b) const { return bf16 ? bf16_bits_to_f32(b) : f16_bits_to_f32(b); }
    // kernel name of the 16-bit family: "..._f16..." names the fp16 instance, "..._bf16..." the bf16 one
    std::string k16(const std::string& f16name) const {
        if (!bf16) return f16name;
        const size_t at = f16name.find("_f16");
        return at == std::string::npos ? f16name : f16name.substr(0, at) + "_bf16" + f16name.substr(at + 4);
    }
};

namespace {

enum { CK_GEMMNK_T = 6 };  // Gemm B already [N][K] (transB): k-padded copy
enum { CK_CONVT_NK = 9 };  // ConvTranspose weights [IC][OC][KH][KW] as a GEMM B: [tap*OC + o][pad8(IC)]
// Gemm B [K][N] (K % 16 == 0, N % 32 == 0) in v_mfma_f32_32x32x16 row-operand fragment order: block
// nb of 32 columns, k-step s, lane l -> 8 values W[16 s + 8 (l / 32) + e][32 nb + l % 32], e = 0..7, at
// ((nb * K / 16 + s) * 64 + l) * 8 + e, so a wave's fragment load is one contiguous KiB
enum { CK_FRAG32 = 10 };
// conv weights over channels padded with zeros to a multiple of 8 or 4 (16-byte chunks of 16-bit or fp32):
// [OC][tap * ICp + ic], ICp = ceil(IC / pad) pad
enum { CK_CONVWT_P8 = 11, CK_CONVWT_P4 = 12 };

int pad8(int k) { return (k + 7) & ~7; }
int round_up(int k, int to) { return (k + to - 1) / to * to; }

// Element count of a const in a packing (Extensions.cs:144-159; K rows padded to 8 for 16-byte loads).
int64_t packed_elems(const PlanValue& v, int kind) {
    const auto& s = v.shape;
    switch (kind) {
        case SOX_CK_CONVWT: return (int64_t)s[0] * pad8(s[1] * s[2] * s[3]);
        case CK_CONVWT_P8: case CK_CONVWT_P4:
            return (int64_t)s[0] * pad8(s[2] * s[3] * round_up(s[1], kind == CK_CONVWT_P8 ? 8 : 4));
        case SOX_CK_GEMMNK: return (int64_t)s[1] * pad8(s[0]);
        case CK_GEMMNK_T: return (int64_t)s[0] * pad8(s[1]);
        case CK_CONVT_NK: return (int64_t)s[1] * s[2] * s[3] * pad8(s[0]);
        case CK_FRAG32: return (int64_t)s[0] * s[1];
        // plain consts: padded with zeros to a multiple of 4 floats, so a float4 read of a bias
        // group that straddles the end stays inside the const
        default: return std::max<int64_t>((v.count() + 3) & ~3ll, 4);
    }
}

// GpuPack packings (Engine/Extensions.cs:169-245) into a pre-zeroed float buffer.
void pack_const(const PlanValue& v, int kind, float* d) {
    const auto& s = v.shape;
    const float* src = v.floats.data();
    switch (kind) {
        case SOX_CK_CONVWT: {  // [OC][IC][KH][KW] -> [OC][Kpad8], k = tap*IC + ic
            int oc = s[0], ic = s[1], taps = s[2] * s[3], kp = pad8(taps * ic);
            for (int o = 0; o < oc; o++)
                for (int c = 0; c < ic; c++)
                    for (int t = 0; t < taps; t++) d[(int64_t)o * kp + t * ic + c] = src[((int64_t)o * ic + c) * taps + t];
            break;
        }
        case CK_CONVWT_P8: case CK_CONVWT_P4: {
            const int oc = s[0], ic = s[1], taps = s[2] * s[3], icp = round_up(ic, kind == CK_CONVWT_P8 ? 8 : 4), kp = pad8(taps * icp);
            for (int o = 0; o < oc; o++)
                for (int c = 0; c < ic; c++)
                    for (int t = 0; t < taps; t++) d[(int64_t)o * kp + t * icp + c] = src[((int64_t)o * ic + c) * taps + t];
            break;
        }
        case CK_FRAG32: {  // [K][N] -> fragment order (see CK_FRAG32)
            const int K = s[0], N = s[1], KS = K / 16;
            for (int nb = 0; nb < N / 32; nb++)
                for (int st = 0; st < KS; st++)
                    for (int l = 0; l < 64; l++)
                        for (int e = 0; e < 8; e++)
                            d[(((int64_t)nb * KS + st) * 64 + l) * 8 + e] =
                                src[(int64_t)(16 * st + 8 * (l / 32) + e) * N + 32 * nb + l % 32];
            break;
        }
        case SOX_CK_GEMMNK: {  // [K][N] -> [N][Kpad8]
            int k = s[0], n = s[1], kp = pad8(k);
            for (int i = 0; i < k; i++)
                for (int j = 0; j < n; j++) d[(int64_t)j * kp + i] = src[(int64_t)i * n + j];
            break;
        }
        case CK_GEMMNK_T: {  // [N][K] -> [N][Kpad8]
            int n = s[0], k = s[1], kp = pad8(k);
            for (int j = 0; j < n; j++) memcpy(d + (int64_t)j * kp, src + (int64_t)j * k, sizeof(float) * k);
            break;
        }
        case CK_CONVT_NK: {  // [IC][OC][KH][KW] -> [tap*OC + o][pad8(IC)]
            int ic = s[0], oc = s[1], taps = s[2] * s[3], kp = pad8(ic);
            for (int c = 0; c < ic; c++)
                for (int o = 0; o < oc; o++)
                    for (int t = 0; t < taps; t++) d[((int64_t)t * oc + o) * kp + c] = src[((int64_t)c * oc + o) * taps + t];
            break;
        }
        case SOX_CK_DWW: {  // [C][1][KH][KW] -> [tap][C]
            int c = s[0], taps = s[2] * s[3];
            for (int ch = 0; ch < c; ch++)
                for (int t = 0; t < taps; t++) d[(int64_t)t * c + ch] = src[(int64_t)ch * taps + t];
            break;
        }
        case SOX_CK_F32T: {  // [A][B(...)] -> [B][A]
            int64_t a = s[0], bcount = v.count() / s[0];
            for (int64_t i = 0; i < a; i++)
                for (int64_t j = 0; j < bcount; j++) d[j * a + i] = src[i * bcount + j];
            break;
        }
        case SOX_CK_CONVTW: {  // [IC][OC][KH][KW] -> [tap][IC][OC]
            int ic = s[0], oc = s[1], taps = s[2] * s[3];
            for (int c = 0; c < ic; c++)
                for (int o = 0; o < oc; o++)
                    for (int t = 0; t < taps; t++) d[((int64_t)t * ic + c) * oc + o] = src[((int64_t)c * oc + o) * taps + t];
            break;
        }
        default: memcpy(d, src, sizeof(float) * v.floats.size());
    }
}

// fp16 ConvTranspose (stride == kernel) with ic % 8 == 0 runs as a GEMM over the input pixels on the
// LDS-DMA conv ring: [pixels][ic] x [ic][tap*oc], scattered to the output by the epilogue.
// A ConvTranspose to one output channel with at most 2x2 taps (the DB head's probability map) runs
// pixel-major, one input pixel per thread (sox_convt_one_*): as a Gemm its N would be 4.
bool convt_one_channel(const sox_graph& g, const PlanNode& n) {
    const PlanValue& wv = g.V(n.in[1]);
    const auto& p = n.p<sox_convt_p>();
    return wv.shape.size() == 4 && wv.shape[1] == 1 && p.kernel[0] * p.kernel[1] <= 4 && p.kernel[1] <= 2 &&
           wv.shape[0] % (g.f16 ? 8 : 4) == 0 && !getenv("SIMDONNX_HIP_CONVT_DIRECT");
}

bool convt_as_gemm(const sox_graph& g, const PlanNode& n) {
    const PlanValue& wv = g.V(n.in[1]);
    return g.f16 && wv.shape.size() == 4 && wv.shape[0] % 8 == 0 && !convt_one_channel(g, n) &&
           !getenv("SIMDONNX_HIP_CONVT_DIRECT");
}

int64_t axis_stride(const PlanValue& v, int axis);

// ---------------------------------------------------------------------------------------------
// Lowering of one ExecNode (the analogue of VkGraphModel.Emit, VkGraph.cs:472-1112).
// ---------------------------------------------------------------------------------------------
bool conv_pads_channels(const sox_graph& g, const PlanNode& n);
bool gemm_pads_k(const sox_graph& g, int64_t m, int n, int k);

struct Emitter {
    sox_graph& g;
    std::set<int> skip;  // nodes already lowered into a previous node's dispatch
    explicit Emitter(sox_graph& gg) : g(gg) { plan_concat_slices(); }

    // NHWC channel concats whose inputs are written straight into their slice of the output by
    // the producing node (row stride = the concat's channel total), instead of being copied there.
    struct Slice {
        int out, off, ctot;
    };
    std::map<int, Slice> concat_slice;  // concat input value -> its slice

    void plan_concat_slices() {
        const auto& nodes = g.plan.nodes;
        for (int ci = 0; ci < (int)nodes.size(); ci++) {
            const PlanNode& n = nodes[ci];
            if (n.op != SOX_OP_CONCAT || g.folded.count(ci)) continue;
            const PlanValue& ov = g.V(n.out[0]);
            const int axis0 = n.p<sox_concat_p>().axis;
            const int axis = axis0 < 0 ? axis0 + (int)ov.shape.size() : axis0;
            const int inner = ov.layout.empty() ? (int)ov.shape.size() - 1 : ov.layout.back();
            const int ctot = ov.phys().back();
            if (axis != inner || ctot % ld() != 0 || ov.buf < 0) continue;
            const auto orange = arena_range(n.out[0]);
            std::vector<std::pair<int, int>> cand;  // (input, channel offset)
            int off = 0;
            for (int in : n.in) {
                const int c = g.V(in).phys().back();
                if (c % ld() == 0 && off % ld() == 0 && g.V(in).buf >= 0) cand.push_back({in, off});
                off += c;
            }
            auto is_cand = [&](int v) {
                for (auto& cv : cand)
                    if (cv.first == v) return true;
                return false;
            };
            for (auto& cv : cand) {
                const int v = cv.first;
                if (v == g.plan.output || uses(v) != 1) continue;
                int pi = -1;
                for (int k = ci - 1; k >= 0 && pi < 0; k--)
                    if (!g.folded.count(k) && !nodes[k].out.empty() && nodes[k].out[0] == v) pi = k;
                if (pi < 0) continue;
                const PlanNode& pn = nodes[pi];
                // (a nearest-add that runs as its addend's conv writes with the residual's row stride)
                bool producer_ok = pn.op == SOX_OP_RESIZE_NEAREST && !g.upadd.count(pi);
                if (pn.op == SOX_OP_CONV) {
                    const auto& cp = pn.p<sox_conv_p>();
                    producer_ok = cp.group == 1 && !cp.has_pool && cp.add_value < 0;
                }
                if (!producer_ok) continue;
                // every value read or written from the producer up to the concat (other than this
                // concat's inputs, which never overlap its output) stays clear of the output
                bool ok = true;
                auto clear = [&](int u) {
                    if (u < 0 || is_cand(u) || g.V(u).buf < 0) return;
                    auto r = arena_range(u);
                    if (r.first < orange.second && orange.first < r.second) ok = false;
                };
                for (int k = pi; k < ci && ok; k++) {
                    if (g.folded.count(k)) continue;
                    for (int u : nodes[k].in) clear(u);
                    for (int u : nodes[k].out) clear(u);
                    if (nodes[k].op == SOX_OP_CONV) clear(nodes[k].p<sox_conv_p>().add_value);
                    auto uc = g.upcat.find(k);  // a conv that gathers its input from upsample sources
                    if (uc != g.upcat.end())
                        for (int i = 0; i < uc->second.n; i++) clear(uc->second.src[i]);
                    auto ua = g.upadd.find(k);  // a nearest-add run as its addend's conv reads that conv's input
                    if (ua != g.upadd.end()) clear(nodes[ua->second.first].in[0]);
                    // a conv fed by a gated product reads the gate's input instead
                    if (k >= 2 && nodes[k - 2].op == SOX_OP_CHANNEL_GATE && !nodes[k - 2].in.empty())
                        clear(nodes[k - 2].in[0]);
                }
                if (ok) concat_slice[v] = Slice{n.out[0], cv.second, ctot};
            }
        }
    }

    // Where node output v is written: its own buffer (row stride own_ld), or its concat slice.
    sox_bind out_bind(int v, int own_ld, int& ld_out, int& elem_off) {
        auto it = concat_slice.find(v);
        if (it == concat_slice.end()) {
            ld_out = own_ld;
            elem_off = 0;
            return bind(v);
        }
        ld_out = it->second.ctot;
        elem_off = it->second.off;
        sox_bind b = bind(it->second.out);
        b.offset += (uint64_t)it->second.off * g.es;
        b.size -= (uint64_t)it->second.off * g.es;
        return b;
    }

    // Reads of value v by any node (inputs and the value-id fields of the param records).
    int uses(int v) const {
        int u = 0;
        for (int ni = 0; ni < (int)g.plan.nodes.size(); ni++) {
            if (g.folded.count(ni)) continue;
            const PlanNode& n = g.plan.nodes[ni];
            for (int x : n.in) u += x == v;
            if (n.op == SOX_OP_CONV) {
                const auto& p = n.p<sox_conv_p>();
                u += (p.add_value == v) + (p.bias_value == v);
            }
        }
        return u + (v == g.plan.output);
    }

    // Arena byte range of an activation value (empty for consts).
    std::pair<uint64_t, uint64_t> arena_range(int v) {
        const PlanValue& pv = g.V(v);
        if (pv.buf < 0) return {0, 0};
        uint64_t off = (uint64_t)g.plan.buf_offset[pv.buf] * g.es;
        return {off, off + (uint64_t)std::max<int64_t>(pv.count(), 1) * g.es};
    }

    // The residual Add lowered into Gemm node ni's epilogue (decided at graph creation,
    // plan_residual_adds), or -1.
    int fusable_residual_add(int ni, const PlanNode&, int, int& residual) {
        auto it = g.residual_add.find(ni);
        residual = it == g.residual_add.end() ? -1 : it->second.second;
        return it == g.residual_add.end() ? -1 : it->second.first;
    }

    // SE gate folded into the consumer's weights: conv node -> (its input, gated weight copy)
    std::map<int, std::pair<int, sox_bind>> se_fold;
    // SE gate node -> the pixel-tile count of the depthwise conv that wrote its GAP partials
    std::map<int, int> gap_from_dw;
    std::set<int> se_with_dw;  // SE gate nodes emitted inside their depthwise conv's launch
    // a depthwise conv the LDS-tile kernels (sox_dwt_*) take
    bool dw_tiles_ok(const PlanNode& n) {
        if (n.op != SOX_OP_CONV || getenv("SIMDONNX_HIP_DW_DIRECT")) return false;
        const auto& p = n.p<sox_conv_p>();
        const PlanValue& wv = g.V(n.in[1]);
        if (!wv.is_const || wv.shape.size() != 4) return false;
        const int ic = nhwc(n.in[0])[3];
        return p.group > 1 && p.group == ic && wv.shape[0] == ic && ic % 8 == 0 && !p.has_pool &&
               p.kernel[0] == p.kernel[1] && (p.kernel[0] == 3 || p.kernel[0] == 5) && p.strides[0] == p.strides[1] &&
               (p.strides[0] == 1 || p.strides[0] == 2) && p.dilations[0] == 1 && p.dilations[1] == 1 &&
               (p.pad_mode == 1 || p.pad_value == 0.0f);
    }

    // ChannelGate node ni whose gate s feeds only "x * s" (the next node, x = the gate's own input)
    // and whose product feeds only a 1x1 / stride-1 / unpadded conv (the node after): the product is
    // never materialised; the gate scales that conv's weight columns instead (conv(x * s) =
    // conv'(x) with W'[n][c] = W[n][c] s[c]). One image only (the copy is per image), c % 8 == 0 (the
    // packed rows have no pad columns), and the conv's output must not overlap x in the arena (x is
    // read by the conv, which the arena plan did not expect). Returns the conv node or -1.
    int se_fold_target(int ni, const PlanNode& n, int nb, int c) {
        const int nn = (int)g.plan.nodes.size();
        if (nb != 1 || c % 8 != 0 || ni + 2 >= nn) return -1;
        const int x = n.in[0], s = n.out[0];
        const PlanNode& mul = g.plan.nodes[ni + 1];
        const PlanNode& cv = g.plan.nodes[ni + 2];
        if (mul.op != SOX_OP_ELEMENTWISE || mul.in.size() != 2 || mul.out.size() != 1) return -1;
        const auto& ep = mul.p<sox_ew_p>();
        if (ep.op != 2 || ep.act != 0) return -1;
        if (!((mul.in[0] == x && mul.in[1] == s) || (mul.in[0] == s && mul.in[1] == x))) return -1;
        const int y = mul.out[0];
        if (uses(s) != 1 || uses(y) != 1 || g.V(y).count() != g.V(x).count()) return -1;
        if (cv.op != SOX_OP_CONV || cv.in.empty() || cv.in[0] != y) return -1;
        const auto& cp = cv.p<sox_conv_p>();
        if (cp.group != 1 || cp.kernel[0] != 1 || cp.kernel[1] != 1 || cp.strides[0] != 1 || cp.strides[1] != 1 ||
            cp.dilations[0] != 1 || cp.dilations[1] != 1 || cp.has_pool || cp.pads[0] || cp.pads[1] || cp.pads[2] ||
            cp.pads[3])
            return -1;
        const PlanValue& wv = g.V(cv.in[1]);
        if (!wv.is_const || wv.shape.size() != 4 || wv.shape[1] != c) return -1;
        auto xr = arena_range(x), orr = arena_range(cv.out[0]);
        if (xr.first < orr.second && orr.first < xr.second) return -1;
        if (cp.add_value >= 0) {  // a residual read by the conv must not be x's product either
            if (cp.add_value == y) return -1;
        }
        return ni + 2;
    }

    const char* ty() const { return g.bf16 ? "bf16" : g.f16 ? "f16" : "f32"; }
    int ld() const { return g.f16 ? 8 : 4; }  // elements per 16-byte vector

    sox_bind bind(int v, int kind = SOX_CK_RAW) {
        const PlanValue& pv = g.V(v);
        sox_bind b{};
        if (pv.buf >= 0) {
            if (pv.buf >= (int)g.plan.buf_offset.size()) fail(SOX_E_INVALID, "value '" + pv.name + "' has no arena offset");
            b.slot = SOX_SLOT_ARENA;
            b.offset = (uint64_t)g.plan.buf_offset[pv.buf] * g.es;
            b.size = (uint64_t)std::max<int64_t>(pv.count(), 1) * g.es;
            auto pad = g.padded_ld.find(v);  // rows stored at a padded stride span more than count elements
            if (pad != g.padded_ld.end()) b.size = (uint64_t)(pv.count() / pv.shape.back()) * pad->second * g.es;
            return b;
        }
        auto it = g.const_off.find({v, kind});
        if (it == g.const_off.end()) fail(SOX_E_INVALID, "const '" + pv.name + "' not packed for this kind");
        b.slot = SOX_SLOT_CONSTS;
        b.offset = it->second.first;
        b.size = it->second.second;
        return b;
    }

    sox_bind none() { return sox_bind{SOX_SLOT_DUMMY, 0, 0, 256}; }
    // cross-workgroup counters of one dispatch, in the session's own zeroed block
    sox_bind sync_counters(uint64_t bytes) {
        sox_bind b{SOX_SLOT_SYNC, 0, g.sync_bytes, bytes};
        g.sync_bytes += (bytes + 63) & ~63ull;
        return b;
    }

    sox_bind scratch(uint64_t bytes) {
        g.scratch_bytes = std::max<uint64_t>(g.scratch_bytes, (bytes + 255) & ~255ull);
        return sox_bind{SOX_SLOT_ARENA, 0, g.scratch_off, bytes};
    }

    // rows x c elements of x copied to scratch with each row padded with zeros to cp
    sox_bind pad_channels(int node, sox_bind x, int64_t rows, int c, int cp) {
        const sox_bind y = scratch((uint64_t)rows * cp * g.es);
        sox_padc_args a{};
        a.rows = rows; a.c = c; a.cp = cp;
        add(node, std::string("sox_padc_") + (g.f16 ? "b16" : "b32"), a,
            {{offsetof(sox_padc_args, x), x}, {offsetof(sox_padc_args, y), y}}, blocks(rows * (cp / ld())), 1, 1, 256, 0, "pad_channels");
        return y;
    }

    template <class A>
    void add(int node, const std::string& kernel, const A& args, std::vector<std::pair<size_t, sox_bind>> ptrs,
             uint32_t gx, uint32_t gy = 1, uint32_t gz = 1, uint32_t block = 256, uint32_t lds = 0,
             const std::string& label = "") {
        Dispatch d;
        const std::string kname = g.k16(kernel);  // the bf16 instance on bf16 graphs
        d.fn = g.be->fn(kname);
        d.name = label.empty() ? kname : label;
        d.kernel = kname;
        d.node = node;
        d.grid[0] = std::max(gx, 1u);
        d.grid[1] = std::max(gy, 1u);
        d.grid[2] = std::max(gz, 1u);
        d.block[0] = block;
        d.lds = lds;
        d.kernarg.resize(sizeof(A));
        memcpy(d.kernarg.data(), &args, sizeof(A));
        for (auto& pr : ptrs) d.patches.push_back(Patch{(uint32_t)pr.first, pr.second});
        g.disp.push_back(std::move(d));
    }

    static uint32_t blocks(int64_t items, int per = 256) { return (uint32_t)((items + per - 1) / per); }

    // NHWC view [n, h, w, c] of a rank-4 value (its physical shape), or of a lower-rank one.
    std::vector<int> nhwc(int v) {
        std::vector<int> p = g.V(v).phys();
        while (p.size() < 4) p.insert(p.begin(), 1);
        if (p.size() > 4) fail(SOX_E_UNSUPPORTED, "rank > 4 activation");
        return p;
    }

    // ---- implicit-GEMM conv / Gemm: kernel choice ----
    std::string igemm_kernel(int64_t M, int N, int K, char amode, int& BM, int& BN) {
        if (g.f16) {
            if (N <= 32) { BM = 64; BN = 32; }
            else if (N <= 64) { BM = 64; BN = 64; }
            else {
                int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
                if (t128 >= 512) { BM = 128; BN = 128; }
                else { BM = 64; BN = 64; }
            }
        } else {
            // 64x64 tiles where they fill the GPU, except over at most 32 output channels: there a 64-wide
            // tile would multiply zero columns (a 3x3 conv to 24 channels at 240^2: 89 us on 64x64 tiles)
            int64_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
            const char* t32_env = getenv("SIMDONNX_HIP_F32_WIDE_N");  // the earlier choice, for comparison
            if (t64 >= 256 && (N > 32 || (t32_env && *t32_env))) { BM = 64; BN = 64; }
            else { BM = 32; BN = 32; }
        }
        char buf[64];
        snprintf(buf, sizeof buf, "sox_igemm_%s_%dx%d_%c", ty(), BM, BN, amode);
        std::string name = buf;
        // long K on the small fp16 tiles: 128-deep slices (one load round trip per 128 k)
        if (g.f16 && BM == 64 && amode != 's' && K >= 128) name += "k";
        return name;
    }

    void launch_igemm(int node, sox_igemm_args a, sox_bind x, sox_bind w, sox_bind bias, sox_bind add_b, sox_bind y,
                      char amode, const std::string& label) {
        int BM, BN;
        std::string k = igemm_kernel(a.m, a.n, a.k, amode, BM, BN);
        int64_t tm = (a.m + BM - 1) / BM, tn = (a.n + BN - 1) / BN;
        a.tiles_n = (int)tn;
        add(node, k, a,
            {{offsetof(sox_igemm_args, x), x}, {offsetof(sox_igemm_args, w), w}, {offsetof(sox_igemm_args, bias), bias},
             {offsetof(sox_igemm_args, add), add_b}, {offsetof(sox_igemm_args, y), y}},
            (uint32_t)(tm * tn), 1, 1, 256, 0, label);
    }

    static constexpr const char* kF32Split = "sox_conv_f32_split";
    // The fp32 32 x 32 tile with K split over its waves (conv_f32.hip)
    void launch_f32_split(int node, const sox_igemm_args& a, sox_bind x, sox_bind w, sox_bind bias, sox_bind add_b,
                          sox_bind y, const std::string& label) {
        add(node, kF32Split, a,
            {{offsetof(sox_igemm_args, x), x}, {offsetof(sox_igemm_args, w), w}, {offsetof(sox_igemm_args, bias), bias},
             {offsetof(sox_igemm_args, add), add_b}, {offsetof(sox_igemm_args, y), y}, {offsetof(sox_igemm_args, zeros), none()}},
            (uint32_t)((a.m + 31) / 32), (uint32_t)((a.n + 31) / 32), 1, 256, 0, label);
    }

    // A tiling of the LDS-DMA ring and what it takes on MI355X, in us: with q tiles on the busiest CU and nk
    // slices of bk, base + q tile + nk max(lat, q thr). lat is a slice's DMA and barrier round trip when the
    // CU has one tile, thr a slice's share when several workgroups overlap theirs. The constants are fits to
    // sweeps of every tiling over ~30 products (47 x 192 -> 768 to 8192 x 768 -> 3072) and ~20 convs; the
    // estimates fall within ~15% of the measured times, and the pick within ~8% of the fastest tiling. The
    // rule before, the largest tile that fills every resident slot, measured against the estimate's pick:
    // Gemm 6000 x 320 -> 1280 19.9 / 11.9 us, 3000 x 3072 -> 768 51.0 / 34, 3000 x 768 -> 768 17.5 / 10.7,
    // 1024 x 256 -> 3000 10.5 / 6.8, 786 x 768 -> 760 8.2 / 6.8; conv 8x64x64 128 -> 256 3x3 41.6 / 32.5,
    // 2x95x127 96 -> 168 32.0 / 25.0, 2x160x160 40 -> 80 24.3 / 16.5, 1x80x80 64 -> 24 5x5 19.0 / 14.9.
    struct RingCfg {
        const char* name;
        int bm, bn, bk, wgs_per_cu;
        float lat, thr, base, tile;
        int64_t tiles(int64_t m, int64_t n) const { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); }
        uint32_t threads() const { return strstr(name, "_w8") ? 512 : 256; }
    };
    uint32_t ring_grid(const RingCfg& c, int64_t m, int64_t n) const {
        const int64_t cus = std::max(1, g.be->info.compute_units);
        return (uint32_t)std::min<int64_t>(c.tiles(m, n), cus * c.wgs_per_cu);
    }
    // Rows that are not whole 4-element groups leave the ring as single elements, 32 rows an instruction, at a rate
    // that no tiling changes: 2.5 us per million (20000 x 8 -> 1142 fp16: 74 us, aligned 1440 25). The split tile's
    // lanes lie along a row: 0.7.
    static float ragged_us(const RingCfg& c, int64_t m, int64_t n) {
        return (c.name == kF32Split ? 0.7e-6f : 2.5e-6f) * (float)(m * n);
    }
    // The tiling of an m x n product over `taps` taps of k reduction elements each: the forced one where the table
    // holds it (where it does not: an error naming `what`, or without `what` no matter), else the one of [first, last)
    // with the smallest estimate (est)
    const RingCfg& ring_pick(const RingCfg* cfgs, size_t ncfg, int first, int last, int64_t m, int64_t n, int64_t k, int64_t taps,
                             bool ragged, const char* forced, const char* what, float* est) const {
        *est = 0.0f;
        if (forced && *forced) {
            for (size_t i = 0; i < ncfg; i++)
                if (!strcmp(cfgs[i].name, forced)) return cfgs[i];
            if (what) fail(SOX_E_INVALID, std::string(what) + ": unknown kernel " + forced);
        }
        const int64_t cus = std::max(1, g.be->info.compute_units);
        int pick = first;
        float best = 0.0f;
        for (int i = first; i < last; i++) {
            const RingCfg& c = cfgs[i];
            const float q = (float)((c.tiles(m, n) + cus - 1) / cus), nk = (float)(taps * ((k + c.bk - 1) / c.bk));
            const float t = c.base + q * c.tile + nk * std::max(c.lat, q * c.thr) + (ragged ? ragged_us(c, m, n) : 0.0f);
            if (i == first || t < best) {
                pick = i;
                best = t;
            }
        }
        *est = best;
        return cfgs[pick];
    }

    // Whether the implicit GEMM (igemm.hip) beats a ring estimate of ring_us over k reduction elements in all. It stores
    // single elements of 16 adjacent columns at 1.5 us per million whatever the row length, and it packs the taps of
    // few channels into one reduction where the ring multiplies a slice of mostly zeros for each. Its estimate has the
    // ring's form, fits over 5000 random products and fp32 convs, each timed on every kernel; it has to win by a
    // tenth. On those the pick is within 1% of the fastest kernel on average (ring only: 3 to 5%). Ring only / now:
    // fp16 20000 x 16 -> 1142 74 / 35 us, 8000 x 24 -> 301 10.1 / 6.7; fp32 8000 x 16 -> 1142 41.7 / 21.6,
    // conv 4x250x16 8 -> 344 3x3 39.4 / 25.6, 1x128x277 4 -> 366 5x5 3.1 times. 16-bit products only with ragged rows
    // and from 2^19 outputs on: below, its small tiles lose (22 x 8 -> 168 6.5 us, ring 2.9).
    bool igemm_wins(float ring_us, int64_t m, int n, int64_t k, char amode, bool ragged) {
        if (ring_us <= 0.0f || getenv("SIMDONNX_HIP_RING")) return false;  // (a forced tiling; tests of the ring)
        if (g.f16 && !(ragged && m * n >= 1 << 19)) return false;
        struct Cost { const char* tile; int bk; float lat, thr, base, tile_us, ragged; };
        static const Cost costs[] = {
            {"f32_32x32_d", 64, 0.92f, 0.52f, 2.3f, 0.11f, 0.7f},  {"f32_64x64_d", 32, 1.26f, 0.76f, 3.7f, 0.88f, 0.0f},
            {"f32_32x32_v", 64, 1.06f, 0.62f, 2.5f, 0.7f, 0.9f},  {"f32_64x64_v", 32, 1.36f, 0.85f, 4.9f, 0.76f, 0.0f},
            {"16_64x32_d", 32, 0.43f, 0.14f, 2.5f, 0.31f, 2.1f},   {"16_64x32_dk", 128, 0.69f, 0.53f, 3.1f, 0.0f, 1.2f},
            {"16_64x64_d", 32, 0.1f, 0.21f, 4.6f, 0.38f, 0.1f},    {"16_64x64_dk", 128, 0.93f, 0.79f, 3.3f, 1.4f, 0.7f},
            {"16_128x128_d", 32, 0.34f, 0.54f, 2.0f, 5.0f, 0.0f}};
        int bm, bn;
        const std::string kernel = igemm_kernel(m, n, (int)k, amode, bm, bn);
        const int64_t cus = std::max(1, g.be->info.compute_units);
        for (const Cost& c : costs) {
            const size_t at = kernel.rfind(c.tile);
            if (at == std::string::npos || at + strlen(c.tile) != kernel.size()) continue;
            const float q = (float)((((m + bm - 1) / bm) * ((n + bn - 1) / bn) + cus - 1) / cus), nk = (float)((k + c.bk - 1) / c.bk);
            const float t = c.base + q * c.tile_us + nk * std::max(c.lat, q * c.thr) + (ragged ? c.ragged * 1e-6f * (float)(m * n) : 0.0f);
            return 1.1f * t < ring_us;
        }
        return false;
    }

    // Dense product on the LDS-DMA ring (gemm_ring.h): a Gemm, or a 1x1 conv over its pixels. a holds m, n, k
    // (whole 16-byte chunks: a multiple of 8, fp32 of 4), ldy and the epilogue flags.
    // igemm: the implicit GEMM's mode for these operands where it may take the product instead, else 0.
    void launch_gemm_dma(int node, sox_igemm_args a, sox_bind x, sox_bind w, sox_bind bias, sox_bind add_b, sox_bind y,
                         const sox_graph::LnFold* ln, const std::string& label, char igemm) {
        static const RingCfg cfgs16[] = {
            {"sox_gemm_f16_256x192_w8k64s2", 256, 192, 64, 1, 1.6f, 1.6f, 4.0f, 2.0f},
            {"sox_gemm_f16_256x128_w8k64s2", 256, 128, 64, 1, 1.3f, 1.3f, 3.3f, 2.0f},
            {"sox_gemm_f16_128x128_k64s2", 128, 128, 64, 2, 0.72f, 0.67f, 4.0f, 1.6f},
            {"sox_gemm_f16_128x64_k64s2e", 128, 64, 64, 2, 0.46f, 0.345f, 3.9f, 0.4f},
            {"sox_gemm_f16_64x64_k64s2", 64, 64, 64, 4, 0.256f, 0.22f, 3.5f, 0.35f},
            {"sox_gemm_f16_128x32_k64s2", 128, 32, 64, 3, 0.32f, 0.25f, 3.2f, 0.7f},  // n <= 32
            // selectable with SIMDONNX_HIP_GEMM (tuning / tests)
            {"sox_gemm_f16_128x64_k64s2", 128, 64, 64, 3},     {"sox_gemm_f16_64x64_k64s4", 64, 64, 64, 2},
            {"sox_gemm_f16_128x64_k64s4", 128, 64, 64, 1},     {"sox_gemm_f16_256x192_k32s5", 256, 192, 32, 1},
            {"sox_gemm_f16_256x192_k32s4", 256, 192, 32, 1},   {"sox_gemm_f16_256x256_w8k32s4", 256, 256, 32, 1},
            {"sox_gemm_f16_256x256_w8k64s2", 256, 256, 64, 1}, {"sox_gemm_f16_256x128_k32s3", 256, 128, 32, 2},
            {"sox_gemm_f16_256x128_k32s5", 256, 128, 32, 1},   {"sox_gemm_f16_128x128_k32s4", 128, 128, 32, 2},
            {"sox_gemm_f16_128x192_k32s3", 128, 192, 32, 2}};
        // a K that is no multiple of 64 (a multiple of 8): 32-deep slices beside the 64-deep ones
        static const RingCfg cfgs_kt[] = {
            {"sox_gemm_kt_f16_256x128_w8k64s2", 256, 128, 64, 1, 1.3f, 1.3f, 3.3f, 2.0f},
            {"sox_gemm_kt_f16_128x128_k64s2", 128, 128, 64, 2, 0.72f, 0.67f, 4.0f, 1.6f},
            {"sox_gemm_kt_f16_128x64_k64s2", 128, 64, 64, 3, 0.5f, 0.42f, 3.9f, 0.5f},
            {"sox_gemm_kt_f16_64x64_k64s2", 64, 64, 64, 4, 0.3f, 0.25f, 3.5f, 0.35f},
            {"sox_gemm_kt_f16_128x96_k32s2", 128, 96, 32, 3, 0.3f, 0.26f, 4.0f, 0.7f},
            {"sox_gemm_kt_f16_64x64_k32s2", 64, 64, 32, 4, 0.19f, 0.16f, 3.4f, 0.35f},
            {"sox_gemm_kt_f16_128x32_k32s2", 128, 32, 32, 4, 0.4f, 0.16f, 3.2f, 0.5f}};  // n <= 32
        static const RingCfg cfgs32[] = {
            {"sox_gemm_f32_128x64_k32s2", 128, 64, 32, 3, 1.23f, 1.23f, 4.0f, 1.0f},
            {"sox_gemm_f32_64x64_k32s2", 64, 64, 32, 4, 0.62f, 0.62f, 3.5f, 0.6f},
            {"sox_gemm_f32_128x32_k32s2", 128, 32, 32, 4, 0.65f, 0.65f, 3.5f, 0.5f},
            {kF32Split, 32, 32, 16, 2, 0.105f, 0.1f, 3.0f, 0.8f}};
        const char* forced = getenv("SIMDONNX_HIP_GEMM");
        const RingCfg* pick;
        // a 32-wide 16-bit tile only where every wider one is at least half padding: over more columns it reads
        // A once more per 32 of them (57600 x 72 -> 40: 6.9 us against 64x64's 5.8). Its base puts it behind 64x64
        // for few rows (8 x 24 -> 24 3.3 us on 128x32, 2.7 on 64x64; 57600 x 96 -> 24 4.5 and 5.9)
        const int narrow = a.n <= 32 && !ln ? 1 : 0;
        const bool ragged = ((a.flags & SOX_F_PAD_ROWS) ? a.ldy : a.ldy | a.n) % 4 != 0;
        float est;
        if (!g.f16) pick = &ring_pick(cfgs32, 4, 0, 4, a.m, a.n, a.k, 1, ragged, forced, nullptr, &est);
        else if (a.k % 64 != 0) pick = &ring_pick(cfgs_kt, 7, 0, 6 + narrow, a.m, a.n, a.k, 1, ragged, forced, nullptr, &est);
        else pick = &ring_pick(cfgs16, sizeof(cfgs16) / sizeof(cfgs16[0]), ln ? 1 : 0, 5 + narrow, a.m, a.n, a.k, 1, ragged, forced, "SIMDONNX_HIP_GEMM", &est);
        if (igemm && igemm_wins(est, a.m, a.n, a.k, igemm, ragged)) {
            if (igemm == 'd') {
                a.kpad = pad8(a.k);
                a.lda = a.k;
                a.flags |= SOX_F_DENSE_A;
            }
            launch_igemm(node, a, x, w, bias, add_b, y, igemm, label);
            return;
        }
        a.kpad = pad8(a.k);
        a.lda = a.k;
        a.flags |= SOX_F_DENSE_A;
        if (pick->name == kF32Split) {  // a 1x1 conv over the rows
            a.ih = a.oh = 1;
            a.iw = a.ow = a.m;
            a.ic = a.k;
            a.kh = a.kw = a.sh = a.sw = 1;
            a.pt = a.pl = 0;
            launch_f32_split(node, a, x, w, bias, add_b, y, label);
            return;
        }
        a.tiles_n = (a.n + pick->bn - 1) / pick->bn;
        std::string kname = pick->name;
        std::vector<std::pair<size_t, sox_bind>> ptrs = {
            {offsetof(sox_igemm_args, x), x}, {offsetof(sox_igemm_args, w), w}, {offsetof(sox_igemm_args, bias), bias},
            {offsetof(sox_igemm_args, add), add_b}, {offsetof(sox_igemm_args, y), y}, {offsetof(sox_igemm_args, zeros), none()}};
        if (ln) {
            kname = "sox_gemm_ln_f16_" + kname.substr(strlen("sox_gemm_f16_"));
            if (kname.back() == 'e') kname.pop_back();  // (the folded 128x64 stores from registers)
            a.ln_eps = ln->eps;
            ptrs.push_back({offsetof(sox_igemm_args, ln_c), bind(ln->colsum, SOX_CK_F32)});
        }
        add(node, kname, a, ptrs, ring_grid(*pick, a.m, a.n), 1, 1, pick->threads(), 0, label);
    }

    // Every window coordinate of a reflect-padded conv lies in [-(dim-1), 2 dim - 2], so one fold
    // maps it into the image (ONNX reflect pads are < dim; this also rejects 1-pixel axes).
    static bool reflect_folds_once(const sox_igemm_args& a) {
        auto axis = [](int dim, int pad, int stride, int out, int k) {
            return dim >= 2 && pad <= dim - 1 && (int64_t)(out - 1) * stride - pad + k - 1 <= 2 * (int64_t)dim - 2;
        };
        return axis(a.ih, a.pt, a.sh, a.oh, a.kh) && axis(a.iw, a.pl, a.sw, a.ow, a.kw);
    }

    // Implicit-GEMM conv on the LDS-DMA ring (gemm_ring.h, CONV mode): the large-conv tiles by rule, else the
    // tiling with the smallest estimate.
    void launch_conv_dma(int node, sox_igemm_args a, sox_bind x, sox_bind w, sox_bind bias, sox_bind add_b,
                         sox_bind y) {
        static const RingCfg cfgs16[] = {
            {"sox_conv_f16_128x128_k64s2", 128, 128, 64, 2, 1.0f, 0.72f, 4.5f, 1.2f},
            {"sox_conv_f16_128x128_k32s4", 128, 128, 32, 2, 0.5f, 0.46f, 3.5f, 2.0f},
            {"sox_conv_f16_128x96_k64s2", 128, 96, 64, 2, 0.8f, 0.57f, 4.2f, 0.8f},
            {"sox_conv_f16_128x96_k32s2", 128, 96, 32, 3, 0.5f, 0.365f, 4.2f, 0.8f},
            {"sox_conv_f16_128x64_k64s2", 128, 64, 64, 3, 0.6f, 0.39f, 4.0f, 0.6f},
            {"sox_conv_f16_64x64_k64s4", 64, 64, 64, 2, 0.42f, 0.29f, 3.8f, 0.4f},
            {"sox_conv_f16_64x64_k32s4", 64, 64, 32, 2, 0.28f, 0.18f, 3.8f, 0.4f},
            {"sox_conv_f16_128x32_k32s2", 128, 32, 32, 4, 0.38f, 0.22f, 3.8f, 0.4f},  // n <= 32, as the dense one
            // by the rules for large convs below
            {"sox_conv_f16_256x128_w8k64s2", 256, 128, 64, 1}, {"sox_conv_f16_256x256_w8k64s2", 256, 256, 64, 1},
            {"sox_conv_f16_h256", 256, 256, 64, 1}};
        static const RingCfg cfgs32[] = {
            {"sox_conv_f32_128x64_k32s2", 128, 64, 32, 3, 1.4f, 1.2f, 4.0f, 1.0f},
            {"sox_conv_f32_64x64_k32s4", 64, 64, 32, 2, 0.73f, 0.7f, 3.5f, 0.6f},
            {"sox_conv_f32_128x32_k32s2", 128, 32, 32, 4, 0.88f, 0.7f, 3.5f, 0.6f},
            {kF32Split, 32, 32, 16, 2, 0.105f, 0.1f, 3.0f, 0.8f}};  // (zero padding only)
        // the ring keeps each row's receptive-field origin in 16 bits a coordinate and W offsets in 32
        if (a.ih > 30000 || a.iw > 30000) unsupported("conv: an image side over 30000 pixels");
        if ((int64_t)a.n * a.kpad >= (int64_t)1 << 31) unsupported("conv: weights of 2^31 elements or more");
        const int64_t cus = std::max(1, g.be->info.compute_units);
        auto tiles = [&](int bm, int bn) { return ((a.m + bm - 1) / bm) * (int64_t)((a.n + bn - 1) / bn); };
        // the input has fewer than 2^31 elements (the 256x256 tile's 32-bit DMA offsets); m = n * oh * ow
        // (a ConvTranspose's A side is its input pixels: oh, ow = ih, iw)
        const bool in32 = (int64_t)(a.m / ((int64_t)a.oh * a.ow)) * a.ih * a.iw * a.ic < ((int64_t)1 << 31);
        // 3x3 stride-1 zero-padded convs over ic % 64 == 0 and multiples of 256 output channels: 8 x 32-pixel
        // tiles from LDS input halos (sox_conv_*_h256; a row's last tile may be partial), at least two
        // rounds of them per CU; SIMDONNX_HIP_NO_H256 keeps such convs on the implicit-GEMM ring
        const int64_t h256_tiles = (a.m / ((int64_t)a.oh * a.ow)) * ((a.oh + 7) / 8) * ((a.ow + 31) / 32);
        const bool h256_ok = a.kh == 3 && a.kw == 3 && a.sh == 1 && a.sw == 1 && a.pt == 1 && a.pl == 1 &&
                             a.oh == a.ih && a.ow == a.iw && a.ic % 64 == 0 && a.n % 256 == 0 &&
                             !(a.flags & (SOX_F_REFLECT | SOX_F_CONVT | SOX_F_DENSE_A)) && a.res_shift == 0;
        const char* name = nullptr;
        const char* forced = getenv("SIMDONNX_HIP_CONV");  // tuning / tests
        if (forced && *forced) name = forced;
        else if (g.f16 && h256_ok && h256_tiles >= 2 * cus && !getenv("SIMDONNX_HIP_NO_H256"))
            name = "sox_conv_f16_h256";
        else if (g.f16 && a.ic % 64 == 0 && a.k >= 1024 && a.n % 256 == 0 && !(a.flags & SOX_F_CONVT) &&
                 tiles(256, 256) >= 2 * cus && in32)
            // large convs over a multiple of 256 output channels: at least two rounds of 256x256 tiles
            // (8 waves of 128x64; 0.67x the DMA and 0.75x the LDS fragment bytes per MFMA of 256x128);
            // its DMA rows hold 32-bit offsets into the input
            name = "sox_conv_f16_256x256_w8k64s2";
        else if (g.f16 && a.ic % 64 == 0 && a.k >= 1024 && a.n % 128 == 0 && !(a.flags & SOX_F_CONVT) &&
                 tiles(256, 128) >= 2 * cus)
            // large convs: at least two rounds of 256x128 tiles on every CU, 8 waves each
            name = "sox_conv_f16_256x128_w8k64s2";
        const int64_t taps = (int64_t)a.kh * a.kw;
        const bool ragged = !(a.flags & SOX_F_CONVT) && (a.ldy | a.n) % 4 != 0;
        const int ncfg32 = a.flags & SOX_F_REFLECT ? 3 : 4;
        float est = 0.0f;
        const RingCfg* c =
            g.f16 ? &ring_pick(cfgs16, sizeof(cfgs16) / sizeof(cfgs16[0]), 0, a.n <= 32 ? 8 : 7, a.m, a.n, a.ic, taps, ragged, name, "SIMDONNX_HIP_CONV", &est)
                  : &ring_pick(cfgs32, ncfg32, 0, ncfg32, a.m, a.n, a.ic, taps, ragged, name, nullptr, &est);
        if (!g.f16 && igemm_wins(est, a.m, a.n, a.k, 'v', ragged)) {
            launch_igemm(node, a, x, w, bias, add_b, y, 'v', "conv");
            return;
        }
        if (c->name == kF32Split) {
            launch_f32_split(node, a, x, w, bias, add_b, y, "conv");
            return;
        }
        if (!in32 && !strcmp(c->name, "sox_conv_f16_256x256_w8k64s2"))
            unsupported("conv: the 256x256 tile takes inputs of fewer than 2^31 elements");
        if (!strcmp(c->name, "sox_conv_f16_h256")) {
            if (!h256_ok) unsupported("conv: the halo tile takes 3x3 stride-1 zero-padded convs with ic % 64 == 0 "
                                      "and oc % 256 == 0");
            add(node, c->name, a,
                {{offsetof(sox_igemm_args, x), x}, {offsetof(sox_igemm_args, w), w}, {offsetof(sox_igemm_args, bias), bias},
                 {offsetof(sox_igemm_args, add), add_b}, {offsetof(sox_igemm_args, y), y},
                 {offsetof(sox_igemm_args, zeros), none()}},
                (uint32_t)std::min<int64_t>(h256_tiles, cus), (uint32_t)(a.n / 256), 1, 512, 0, "conv");
            return;
        }
        a.tiles_n = (a.n + c->bn - 1) / c->bn;
        add(node, c->name, a,
            {{offsetof(sox_igemm_args, x), x}, {offsetof(sox_igemm_args, w), w}, {offsetof(sox_igemm_args, bias), bias},
             {offsetof(sox_igemm_args, add), add_b}, {offsetof(sox_igemm_args, y), y},
             {offsetof(sox_igemm_args, zeros), none()}},
            ring_grid(*c, a.m, a.n), 1, 1, c->threads(), 0, "conv");
    }

    // a conv emitted in another node's place (plan_upsample_add): its output, and a residual read as the
    // nearest upsample by 2^shift of res
    struct ConvOverride {
        int out = -1, res = -1, shift = 0;
    } cov;

    void conv(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_conv_p>();
        if (p.dilations[0] != 1 || p.dilations[1] != 1) unsupported("conv: dilation");
        const int out_v = cov.out >= 0 ? cov.out : n.out[0];
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(out_v);
        const PlanValue& wv = g.V(n.in[1]);
        if (!wv.is_const || wv.shape.size() != 4) unsupported("conv: weights must be a rank-4 const");
        int oc = wv.shape[0], kh = p.kernel[0], kw = p.kernel[1];
        int ih = si[1], iw = si[2], ic = si[3], nb = si[0];
        int oh = so[1], ow = so[2];
        int act = p.act;
        int flags = (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (p.pad_mode == 1 ? SOX_F_REFLECT : 0) |
                    (p.add_value >= 0 || cov.res >= 0 ? SOX_F_RESIDUAL : 0) | (act << SOX_F_ACT_SHIFT);
        if (p.group > 1) {
            if (p.group != ic || oc != ic) unsupported("grouped non-depthwise conv");
            if (p.has_pool) unsupported("depthwise conv + pool");
            sox_dw_args a{};
            a.n = nb; a.c = ic; a.ih = ih; a.iw = iw; a.oh = oh; a.ow = ow;
            a.kh = kh; a.kw = kw; a.sh = p.strides[0]; a.sw = p.strides[1]; a.pt = p.pads[0]; a.pl = p.pads[1];
            a.flags = flags;
            a.pad_value = p.pad_mode == 0 ? p.pad_value : 0.0f;
            bool vec = ic % ld() == 0;
            const int k = kh, s = p.strides[0];
            if (dw_tiles_ok(n)) {
                // LDS tiles: 8 x 8 pixels x 64 channels per workgroup, or 4 x 8 when 8 x 8 tiles would
                // give the GPU fewer than two workgroups per CU (SIMDONNX_HIP_DWT_ROWS=8 / 4 forces either;
                // the opt-in gate inside the depthwise launch keeps 8 x 8)
                sox_dwt_args d{};
                d.n = nb; d.c = ic; d.ih = ih; d.iw = iw; d.oh = oh; d.ow = ow;
                d.kh = kh; d.kw = kw; d.sh = s; d.sw = s; d.pt = p.pads[0]; d.pl = p.pads[1];
                d.flags = flags;
                const int64_t cus = std::max(1, g.be->info.compute_units);
                const char* rows_env = getenv("SIMDONNX_HIP_DWT_ROWS");
                const char* se_env = getenv("SIMDONNX_HIP_SE_IN_DW");
                int th = (int64_t)((ow + 7) / 8) * ((oh + 7) / 8) * ((ic + 63) / 64) * nb < 2 * cus ? 4 : 8;
                if (rows_env && *rows_env) th = atoi(rows_env) == 4 ? 4 : 8;
                if (se_env && *se_env && strcmp(se_env, "0")) th = 8;
                d.tiles_x = (ow + 7) / 8;
                d.tiles_y = (oh + th - 1) / th;
                const int tiles = d.tiles_x * d.tiles_y;
                // an SE gate that reads this output next gets its GAP partials from the tiles
                sox_bind part = none();
                const int nn = (int)g.plan.nodes.size();
                // the gate's fc1 reduces the per-tile partials with up to 64 per thread: 4 phases per
                // channel for 64-channel groups, 8 / 16 for groups of <= 32 / <= 16 channels
                const int max_tiles = ic <= 16 ? 1024 : ic <= 32 ? 512 : 128;
                if (ni + 1 < nn && tiles <= max_tiles && !getenv("SIMDONNX_HIP_NO_DW_GAP")) {
                    const PlanNode& gate = g.plan.nodes[ni + 1];
                    if (gate.op == SOX_OP_CHANNEL_GATE && !gate.in.empty() && gate.in[0] == n.out[0]) {
                        part = scratch((uint64_t)nb * tiles * ic * 4);
                        d.gap = 1;
                        gap_from_dw[ni + 1] = tiles;
                        if (th == 8 && se_in_depthwise(ni + 1, ic)) {  // (the fused gate: 8 x 8 tiles only)
                            // the gate runs in this launch: its last tiles take fc1 and fc2
                            SeSetup st = se_setup(ni + 1, gate, tiles);
                            se_with_dw.insert(ni + 1);
                            sox_dwt_se_args da{};
                            da.dw = d;
                            da.se = st.a;
                            const size_t dw0 = offsetof(sox_dwt_se_args, dw), se0 = offsetof(sox_dwt_se_args, se);
                            std::vector<std::pair<size_t, sox_bind>> ptrs = {
                                {dw0 + offsetof(sox_dwt_args, x), bind(n.in[0])},
                                {dw0 + offsetof(sox_dwt_args, w), bind(n.in[1], SOX_CK_DWW)},
                                {dw0 + offsetof(sox_dwt_args, bias),
                                 p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                                {dw0 + offsetof(sox_dwt_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                                {dw0 + offsetof(sox_dwt_args, y), bind(n.out[0])},
                                {dw0 + offsetof(sox_dwt_args, part), st.part},
                                {offsetof(sox_dwt_se_args, sync),
                                 sync_counters((uint64_t)nb * (st.a.groups + 1) * 4)}};
                            for (auto& pr : st.ptrs) ptrs.push_back({se0 + pr.first, pr.second});
                            add(ni, std::string("sox_dwt_") + ty() + "_k" + std::to_string(k) + "s" + std::to_string(s) +
                                        "_se",
                                da, ptrs, (uint32_t)tiles, (uint32_t)((ic + 63) / 64), (uint32_t)nb, 256, 0,
                                "depthwise_se");
                            return;
                        }
                    }
                }
                add(ni, std::string("sox_dwt_") + ty() + "_k" + std::to_string(k) + "s" + std::to_string(s) +
                            (th == 4 ? "_h4" : ""),
                    d,
                    {{offsetof(sox_dwt_args, x), bind(n.in[0])}, {offsetof(sox_dwt_args, w), bind(n.in[1], SOX_CK_DWW)},
                     {offsetof(sox_dwt_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                     {offsetof(sox_dwt_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                     {offsetof(sox_dwt_args, y), bind(n.out[0])}, {offsetof(sox_dwt_args, part), part}},
                    (uint32_t)tiles, (uint32_t)((ic + 63) / 64), (uint32_t)nb, 256, 0, "depthwise");
                return;
            }
            int64_t items = (int64_t)nb * oh * ow * (vec ? ic / ld() : ic);
            // 3x3 / 5x5: taps unrolled with every load issued up front
            std::string kname = std::string("sox_dw_") + ty() + (vec ? "_v" : "_s");
            if (vec && kh == kw && (kh == 3 || kh == 5)) kname += std::to_string(kh);
            add(ni, kname, a,
                {{offsetof(sox_dw_args, x), bind(n.in[0])}, {offsetof(sox_dw_args, w), bind(n.in[1], SOX_CK_DWW)},
                 {offsetof(sox_dw_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_dw_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_dw_args, y), bind(n.out[0])}},
                blocks(items), 1, 1, 256, 0, "depthwise");
            return;
        }
        // an SE gate folded into this conv: read the gate's input with the gated weight copy
        sox_bind xb = bind(n.in[0]), wb = conv_pads_channels(g, n) ? none() : bind(n.in[1], SOX_CK_CONVWT);
        auto fold_it = se_fold.find(ni);
        if (fold_it != se_fold.end()) {
            xb = bind(fold_it->second.first);
            wb = fold_it->second.second;
        }
        int coh = oh, cow = ow;
        int ldy_out, yoff_unused;
        sox_bind ybind = out_bind(out_v, oc, ldy_out, yoff_unused);
        const int ocv = g.f16 ? 8 : 4;
        const bool direct = ic % ld() != 0 && oc % ocv == 0 && kh * kw * ic <= 64 && oc <= 128;
        if (p.has_pool) {
            coh = (ih + p.pads[0] + p.pads[2] - kh) / p.strides[0] + 1;
            cow = (iw + p.pads[1] + p.pads[3] - kw) / p.strides[1] + 1;
        }
        if (p.has_pool && direct && p.add_value < 0 && p.pool_kernel[0] == 2 && p.pool_kernel[1] == 2 &&
            p.pool_strides[0] == 2 && p.pool_strides[1] == 2 && !p.pool_pads[0] && !p.pool_pads[1] && !p.pool_pads[2] &&
            !p.pool_pads[3] && coh == 2 * oh && cow == 2 * ow) {
            // the reference's GPU ConvPool (small-ic stems, GraphCompiler.GpuSmallConv / VkGraph.cs:559-575):
            // each work item convolves its 2x2 quad and stores only the pooled pixel
            sox_igemm_args a{};
            a.m = nb * oh * ow;
            a.n = oc;
            a.k = kh * kw * ic;
            a.kpad = pad8(a.k);
            a.ih = ih; a.iw = iw; a.ic = ic; a.oh = coh; a.ow = cow;
            a.kh = kh; a.kw = kw; a.sh = p.strides[0]; a.sw = p.strides[1]; a.pt = p.pads[0]; a.pl = p.pads[1];
            a.flags = flags | SOX_F_POOL | (p.pool_relu ? SOX_F_POOL_RELU : 0);
            a.pad_value = p.pad_mode == 0 ? p.pad_value : 0.0f;
            a.ldy = ldy_out;
            const bool rgb33 = kh == 3 && kw == 3 && ic == 3 && (int64_t)a.m * (oc / ocv) < (1ll << 31) - 256;
            add(ni, std::string("sox_conv_direct_") + (rgb33 ? "333_" : "") + "pool_" + ty(), a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), none()}, {offsetof(sox_igemm_args, y), ybind}},
                blocks((int64_t)a.m * (oc / ocv)), 1, 1, 256, (uint32_t)(oc * a.k * 4), "convpool");
            return;
        }
        if (p.has_pool) {
            // conv into scratch at full resolution, then the 2x2/2 max pool pass
            // other convs with a pool (a CPU-plan fusion the reference GPU rejects): the conv into
            // scratch at full resolution, then the pool pass
            if (p.add_value >= 0) unsupported("conv + pool + residual");
            ybind = scratch((uint64_t)nb * coh * cow * oc * g.es);
        }
        sox_igemm_args a{};
        a.m = nb * coh * cow;
        a.n = oc;
        a.k = kh * kw * ic;
        a.kpad = pad8(a.k);
        a.ih = ih; a.iw = iw; a.ic = ic; a.oh = coh; a.ow = cow;
        a.kh = kh; a.kw = kw; a.sh = p.strides[0]; a.sw = p.strides[1]; a.pt = p.pads[0]; a.pl = p.pads[1];
        a.flags = flags;
        a.pad_value = p.pad_mode == 0 ? p.pad_value : 0.0f;
        a.ldy = p.has_pool ? oc : ldy_out;  // the pool pass writes the real output
        a.lda = 0;
        char amode = ic % ld() == 0 ? 'v' : 's';
        const int st = p.strides[0];
        if (fold_it == se_fold.end() && conv_pads_channels(g, n)) {
            const int icp = round_up(ic, ld());
            xb = pad_channels(ni, xb, (int64_t)nb * ih * iw, ic, icp);
            wb = bind(n.in[1], kh * kw == 1 ? SOX_CK_CONVWT : g.f16 ? CK_CONVWT_P8 : CK_CONVWT_P4);
            a.ic = ic = icp;
            a.k = kh * kw * ic;
            a.kpad = pad8(a.k);
            amode = 'v';
        }
        // fp32 with a short reduction (conv_f32.hip)
        const bool f32_short = !g.f16 && ic % 16 == 0 && a.k % 64 == 0 && a.k <= 576 && oc % 4 == 0 && a.ldy % 4 == 0 &&
                               p.pad_mode == 0 && p.pad_value == 0.0f && !getenv("SIMDONNX_HIP_IGEMM");
        // what the ring's packed origins and 32-bit offsets hold; larger fp32 convs stay on the implicit GEMM
        const bool ring_f32_ok = ih <= 30000 && iw <= 30000 && (int64_t)ih * iw * ic < ((int64_t)1 << 31) &&
                                 (int64_t)oc * a.kpad < ((int64_t)1 << 31) &&
                                 *std::max_element(p.pads, p.pads + 4) <= 2000;
        bool ring = false;  // took the LDS-DMA ring (the only route that reads an upsampled residual)
        if (direct && g.f16 && kh == 3 && kw == 3 && ic == 3 && st == p.strides[1] && (st == 1 || st == 2) &&
            oc <= 32 && a.ldy % 4 == 0 && !getenv("SIMDONNX_HIP_STEM_DIRECT")) {
            // 3x3 RGB stems, 16-bit: 16 x 16 output pixels per workgroup as a K = 27 matrix product from one
            // LDS copy of their input window
            const uint32_t tiles = (uint32_t)(((coh + 15) / 16) * ((cow + 15) / 16));  // the conv's own output
            add(ni, std::string("sox_conv_stem_s") + std::to_string(st) + "_" + ty(), a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_igemm_args, y), ybind}},
                tiles, (uint32_t)nb, 1, 256, 0, "conv_direct");
        } else if (direct) {
            // few input channels (stems): direct conv, weights staged in LDS (3x3 over RGB unrolled)
            const bool rgb33 = kh == 3 && kw == 3 && ic == 3 && (int64_t)a.m * (oc / ocv) < (1ll << 31) - 256;
            add(ni, std::string("sox_conv_direct_") + (rgb33 ? "333_" : "") + ty(), a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_igemm_args, y), ybind}},
                blocks((int64_t)a.m * (oc / ocv)), 1, 1, 256, (uint32_t)(oc * a.k * 4), "conv_direct");
        } else if (g.f16 && amode == 'v' && oc < 8 && a.k <= 1152 && !getenv("SIMDONNX_HIP_IGEMM") &&
                   !getenv("SIMDONNX_HIP_NONARROW")) {
            // few output channels: one pixel x all oc channels per work item, weights [K][8] in LDS
            add(ni, "sox_conv_narrow_f16_o" + std::to_string(oc), a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_igemm_args, y), ybind}},
                blocks(a.m), 1, 1, 256, (uint32_t)(a.k * 8 * 4), "conv_narrow");
        } else if (g.upcat.count(ni)) {
            // the input concat of nearest upsamples (plan_upsample_concat), gathered by the halo DMA
            const auto& uc = g.upcat.at(ni);
            a.up_n = uc.n;
            a.up_c = uc.c;
            std::vector<std::pair<size_t, sox_bind>> ptrs = {
                {offsetof(sox_igemm_args, w), wb},
                {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                {offsetof(sox_igemm_args, y), ybind}, {offsetof(sox_igemm_args, zeros), none()}};
            for (int i = 0; i < 4; i++) {
                a.up_shift[i] = uc.shift[i];
                ptrs.push_back({offsetof(sox_igemm_args, up) + i * sizeof(void*), i < uc.n ? bind(uc.src[i]) : none()});
            }
            const int tiles = ((cow + 15) / 16) * ((coh + 7) / 8) * nb;
            add(ni, "sox_conv_halo_f16_3x3s1_upcat", a, ptrs, (uint32_t)tiles, (uint32_t)((oc + 31) / 32), 1, 256, 0,
                "conv_halo");
        } else if (g.f16 && amode == 'v' && kh == 3 && kw == 3 && p.strides[0] == 1 && p.strides[1] == 1 &&
                   p.pad_mode == 0 && p.pad_value == 0.0f && oc <= 64 && !getenv("SIMDONNX_HIP_NOHALO") &&
                   !getenv("SIMDONNX_HIP_IGEMM")) {
            // 3x3 stride 1 with few output channels: every tap from one LDS copy of the input halo
            // (at stride 2 a pixel feeds ~2 outputs per tap row and the implicit-GEMM ring is faster)
            const int tiles = ((cow + 15) / 16) * ((coh + 7) / 8) * nb;
            // whole 16-byte output chunks and up to 32 input channels: persistent workgroups with the filter in
            // registers (1x544x960 32 -> 32 45.5 -> 22.0 us, 1x480x480 16 -> 16 19.3 -> 8.9, 1x60x60 32 -> 32
            // 5.8 -> 4.5). Up to 64: its 36 fragments take ~3 us to fetch, so from three tiles a CU on
            // (1x544x960 64 -> 64 109 -> 61 us, 8x128x128 48 -> 48 28.2 -> 16.7; at 1.8 a CU, 8x56x56 64 -> 64,
            // 12.6 against the LDS filter's 9.0). Three or two workgroups fit a CU; with two blocks of output
            // channels the grid is two high (32 -> 64 over 544x960: 36.6 us, 39.7 with three a CU and block).
            const int64_t cus = std::max(1, g.be->info.compute_units), nblk = (oc + 31) / 32;
            const bool reg = (ic <= 32 || (ic <= 64 && tiles * nblk >= 3 * cus)) && ((oc | a.ldy) & 7) == 0 && ybind.offset % 16 == 0;
            const uint32_t grid = reg ? (uint32_t)(std::min<int64_t>(tiles, cus * (ic <= 32 ? 3 : 2) / nblk) + 7) / 8 * 8 : (uint32_t)tiles;
            add(ni, !reg ? "sox_conv_halo_f16_3x3s1" : ic <= 32 ? "sox_conv_halo_f16_3x3s1_c32" : "sox_conv_halo_f16_3x3s1_c64", a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_igemm_args, y), ybind}, {offsetof(sox_igemm_args, zeros), none()}},
                grid, (uint32_t)nblk, 1, 256, 0, "conv_halo");
        } else if (amode == 'v' && !(p.pad_mode == 0 && p.pad_value != 0.0f) &&
                   (p.pad_mode != 1 || reflect_folds_once(a)) && !getenv("SIMDONNX_HIP_IGEMM") && !f32_short &&
                   (g.f16 || ring_f32_ok)) {
            // NHWC rows of whole 16-byte chunks and zero/reflect padding: the LDS-DMA implicit-GEMM ring
            a.res_shift = cov.shift;
            const char* forced = getenv("SIMDONNX_HIP_CONV");
            if (kh == 1 && kw == 1 && st == 1 && p.strides[1] == 1 && !p.pads[0] && !p.pads[1] && !p.pads[2] &&
                !p.pads[3] && cov.res < 0 && ih <= 30000 && iw <= 30000 && (int64_t)oc * a.kpad < ((int64_t)1 << 31) &&
                !(forced && *forced)) {
                // a 1x1 conv over its pixels is a dense product: no receptive fields to address
                launch_gemm_dma(ni, a, xb, wb, p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(),
                                p.add_value >= 0 ? bind(p.add_value) : none(), ybind, nullptr, "conv", g.f16 ? 0 : 'v');
            } else
            launch_conv_dma(ni, a, xb, wb,
                            p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(),
                            cov.res >= 0 ? bind(cov.res) : p.add_value >= 0 ? bind(p.add_value) : none(), ybind);
            ring = true;
        } else if (f32_short) {
            // fp32 with a short reduction: the whole 32x32 tile's operands in LDS, K split over the four
            // waves on the fp32 matrix cores, each wave loading its own quarter (conv_f32.hip)
            add(ni, "sox_conv_f32_short_k" + std::to_string(a.k), a,
                {{offsetof(sox_igemm_args, x), xb}, {offsetof(sox_igemm_args, w), wb},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, add), p.add_value >= 0 ? bind(p.add_value) : none()},
                 {offsetof(sox_igemm_args, y), ybind}, {offsetof(sox_igemm_args, zeros), none()}},
                (uint32_t)((a.m + 31) / 32), (uint32_t)((oc + 31) / 32), 1, 256, 0, "conv");
        } else {
            launch_igemm(ni, a, xb, wb,
                         p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(),
                         p.add_value >= 0 ? bind(p.add_value) : none(), ybind, amode, "conv");
        }
        if (cov.out >= 0 && !ring) fail(SOX_E_INVALID, "conv with an upsampled residual off the LDS-DMA ring");
        if (p.has_pool) {
            sox_pool_args q{};
            q.n = nb; q.ih = coh; q.iw = cow; q.c = oc; q.oh = oh; q.ow = ow;
            q.kh = p.pool_kernel[0]; q.kw = p.pool_kernel[1]; q.sh = p.pool_strides[0]; q.sw = p.pool_strides[1];
            q.pt = p.pool_pads[0]; q.pl = p.pool_pads[1];
            q.flags = p.pool_relu ? 1 : 0;
            add(ni, std::string("sox_pool_") + ty(), q,
                {{offsetof(sox_pool_args, x), ybind}, {offsetof(sox_pool_args, y), bind(n.out[0])}},
                blocks((int64_t)nb * oh * ow * oc), 1, 1, 256, 0, "convpool");
        }
    }

    // the fused transformer MLP (plan_fused_mlp): one workgroup per 32 rows, or per (32 rows, part of the
    // hidden width) and a sum of the parts
    void fused_mlp(int ni, const PlanNode& n, const sox_graph::Mlp& f) {
        const PlanNode& n2 = g.plan.nodes[f.fc2];
        const auto& p1 = n.p<sox_gemm_p>();
        const auto& p2 = n2.p<sox_gemm_p>();
        const auto& ln = g.ln_fold.at(ni);
        sox_mlp_args a{};
        a.k1 = g.V(n.in[0]).shape.back();
        a.h = g.V(n.out[0]).shape.back();
        a.n2 = g.V(f.out).shape.back();
        a.m = (int)(g.V(n.in[0]).count() / a.k1);
        a.ldw1 = pad8(a.k1);
        a.ldw2 = pad8(a.h);
        a.eps = ln.eps;
        const int act2 = f.add >= 0 ? g.plan.nodes[f.add].p<sox_ew_p>().act : 0;
        a.flags = (p2.bias_value >= 0 ? 1 : 0) | (f.residual >= 0 ? 2 : 0) | (act2 << 4);
        // split over the hidden width when one workgroup per 32 rows would leave CUs idle (the parts'
        // fc2 sums meet in sox_mlp_sum_*); SIMDONNX_HIP_MLP_SPLIT=0 / 1 forces either form
        const int rbs = (a.m + 31) / 32;
        const int parts = mlp_parts(a.k1);
        const bool split = f.split;
        char name[64];
        if (f.proj >= 0) snprintf(name, sizeof name, "sox_mlpqp_f16_k%d_h%d_q%d", a.k1, a.h, parts);
        else if (split) snprintf(name, sizeof name, "sox_mlpq_f16_k%d_h%d_q%d", a.k1, a.h, parts);
        else snprintf(name, sizeof name, "sox_mlp_f16_k%d_h%d", a.k1, a.h);
        sox_bind part = none();
        if (split) {
            a.parts = parts;
            part = scratch((uint64_t)parts * a.m * a.n2 * 4);
        }
        const sox_bind b2 = p2.bias_value >= 0 ? bind(p2.bias_value, SOX_CK_F32) : none();
        const sox_bind res = f.residual >= 0 ? bind(f.residual) : none();
        std::vector<std::pair<size_t, sox_bind>> binds = {
            {offsetof(sox_mlp_args, x), bind(n.in[0])}, {offsetof(sox_mlp_args, w1), bind(n.in[1], CK_FRAG32)},
            {offsetof(sox_mlp_args, b1), bind(p1.bias_value, SOX_CK_F32)},
            {offsetof(sox_mlp_args, c1), bind(ln.colsum, SOX_CK_F32)},
            {offsetof(sox_mlp_args, w2), bind(n2.in[1], CK_FRAG32)}, {offsetof(sox_mlp_args, b2), b2},
            {offsetof(sox_mlp_args, res), res}, {offsetof(sox_mlp_args, y), bind(f.out)},
            {offsetof(sox_mlp_args, part), part}};
        if (f.proj >= 0) {  // x = the projection Gemm's output with its residual Add, computed in the part kernel
            const PlanNode& np = g.plan.nodes[f.proj];
            const auto& pp = np.p<sox_gemm_p>();
            a.pflags = pp.bias_value >= 0 ? 1 : 0;
            binds.push_back({offsetof(sox_mlp_args, po), bind(np.in[0])});
            binds.push_back({offsetof(sox_mlp_args, pw), bind(np.in[1], pp.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK)});
            binds.push_back({offsetof(sox_mlp_args, pb), pp.bias_value >= 0 ? bind(pp.bias_value, SOX_CK_F32) : none()});
            binds.push_back({offsetof(sox_mlp_args, px), bind(f.proj_res)});
            binds.push_back({offsetof(sox_mlp_args, xout), bind(n.in[0])});
        }
        add(ni, name, a, binds, (uint32_t)(rbs * (split ? parts : 1)), 1, 1, 512, 0, "mlp");
        if (split)
            add(ni, "sox_mlp_sum_f16", a,
                {{offsetof(sox_mlp_args, b2), b2}, {offsetof(sox_mlp_args, res), res},
                 {offsetof(sox_mlp_args, y), bind(f.out)}, {offsetof(sox_mlp_args, part), part}},
                blocks((int64_t)a.m * a.n2 / 4), 1, 1, 256, 0, "mlp_sum");
    }

    // LayerNorm -> qkv Gemm -> attention (plan_fused_attention): one workgroup per (image, head)
    void qkv_attention(int ni, const PlanNode& n, int ai) {
        const PlanNode& na = g.plan.nodes[ai];
        const auto& pq = n.p<sox_gemm_p>();
        const auto& pa = na.p<sox_attention_p>();
        const auto& ln = g.ln_fold.at(ni);
        const PlanValue& xv = g.V(n.in[0]);
        const int dim = xv.shape.back();
        sox_qkvattn_args a{};
        a.t = g.V(na.in[0]).shape[pa.dims[0][2]];
        a.n = (int)(xv.count() / dim / a.t);
        a.kpad = pad8(dim);
        a.eps = ln.eps;
        a.scale = pa.scale;
        a.flags = pq.bias_value >= 0 ? 2 : 0;
        char name[64];
        snprintf(name, sizeof name, "sox_qkvattn_f16_d%d", dim);
        add(ni, name, a,
            {{offsetof(sox_qkvattn_args, x), bind(n.in[0])},
             {offsetof(sox_qkvattn_args, wqkv), bind(n.in[1], pq.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK)},
             {offsetof(sox_qkvattn_args, bqkv), pq.bias_value >= 0 ? bind(pq.bias_value, SOX_CK_F32) : none()},
             {offsetof(sox_qkvattn_args, cqkv), bind(ln.colsum, SOX_CK_F32)},
             {offsetof(sox_qkvattn_args, o), bind(na.out[0])}},
            (uint32_t)(a.n * (dim / 32)), 1, 1, 576, 0, "qkv_attn");
    }

    void gemm(int ni, const PlanNode& n) {
        auto mf = g.mlp.find(ni);
        if (mf != g.mlp.end()) {
            fused_mlp(ni, n, mf->second);
            return;
        }
        auto qa = g.qkv_attn.find(ni);
        if (qa != g.qkv_attn.end()) {
            qkv_attention(ni, n, qa->second);
            return;
        }
        const auto& p = n.p<sox_gemm_p>();
        const PlanValue& av = g.V(n.in[0]);
        const PlanValue& bv = g.V(n.in[1]);
        if (!bv.is_const || bv.shape.size() != 2) unsupported("Gemm: B must be a rank-2 const");
        int k = av.shape.back();
        if (av.phys().back() != k) unsupported("Gemm: K not innermost");
        int64_t m = av.count() / k;
        int nn = g.V(n.out[0]).shape.back();
        sox_igemm_args a{};
        a.m = (int)m;
        a.n = nn;
        a.k = k;
        a.kpad = pad8(k);
        // a directly following residual Add runs in the epilogue (its ReLU, if any, too)
        int residual = -1;
        const int fused_add = fusable_residual_add(ni, n, p.act, residual);
        int act = p.act, out_value = n.out[0];
        if (fused_add >= 0) {
            act = g.plan.nodes[fused_add].p<sox_ew_p>().act;
            out_value = g.plan.nodes[fused_add].out[0];
            skip.insert(fused_add);
        }
        const sox_bind res_b = residual >= 0 ? bind(residual) : none();
        a.flags = (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (act << SOX_F_ACT_SHIFT) | (residual >= 0 ? SOX_F_RESIDUAL : 0);
        a.ldy = nn;
        // rows of whole 16-byte chunks: the LDS-DMA pipelined persistent kernel (any N: rows that are not
        // whole 4-element groups are stored element by element)
        auto pad_it = g.padded_ld.find(out_value);
        const bool pad_rows = pad_it != g.padded_ld.end();
        auto ln_it = g.ln_fold.find(ni);
        const bool ln = ln_it != g.ln_fold.end();  // A is a folded LayerNorm's input
        const bool pad_k = gemm_pads_k(g, m, nn, k);
        const bool dma = pad_k || (k % ld() == 0 && (g.f16 || !getenv("SIMDONNX_HIP_IGEMM")));
        if (ln && !dma) fail(SOX_E_INVALID, "Gemm: LayerNorm folded into a Gemm off the LDS-DMA route");
        // opt-in (SIMDONNX_HIP_GEMMPP), 16-bit graphs: whole 256 x 128 tiles, K = 768, bias + none / relu / GELU, at
        // least a tile per CU, on the kernel that runs each tile's epilogue under the next tile's
        // matrix-core work (gemm_pp.h; measured slower than the ring on the 8192 x 768 x 3072 Gemm)
        const char* forced_gemm = getenv("SIMDONNX_HIP_GEMM");
        const char* want_pp = getenv("SIMDONNX_HIP_GEMMPP");
        const int cus_pp = std::max(1, g.be->info.compute_units);
        if (g.f16 && dma && !ln && residual < 0 && !pad_rows && !(forced_gemm && *forced_gemm) &&
            want_pp && *want_pp && strcmp(want_pp, "0") != 0 && m % 256 == 0 && nn % 128 == 0 && k == 768 &&
            (act == SOX_ACT_NONE || act == SOX_ACT_RELU || act == SOX_ACT_GELU) &&
            (m / 256) * (int64_t)(nn / 128) >= cus_pp) {
            sox_igemm_args a{};
            a.m = (int)m; a.n = nn; a.k = k; a.kpad = pad8(k);
            a.flags = (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (act << SOX_F_ACT_SHIFT) | SOX_F_DENSE_A;
            a.ldy = nn; a.lda = k;
            a.tiles_n = nn / 128;
            const int64_t tiles = (m / 256) * (int64_t)a.tiles_n;
            const char* an = act == SOX_ACT_GELU ? "gelu" : act == SOX_ACT_RELU ? "relu" : "none";
            add(ni, std::string("sox_gemmpp_f16_256x128_k768_") + an, a,
                {{offsetof(sox_igemm_args, x), bind(n.in[0])},
                 {offsetof(sox_igemm_args, w), bind(n.in[1], p.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK)},
                 {offsetof(sox_igemm_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_igemm_args, zeros), none()},
                 {offsetof(sox_igemm_args, y), bind(out_value)}},
                (uint32_t)std::min<int64_t>(tiles, cus_pp), 1, 1, 256, 0, "gemm");
            return;
        }
        if (dma) {
            sox_igemm_args a{};
            a.m = (int)m; a.n = nn; a.k = pad_k ? round_up(k, ld()) : k;
            a.flags = (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (act << SOX_F_ACT_SHIFT) |
                      (residual >= 0 ? SOX_F_RESIDUAL : 0) | (pad_rows ? SOX_F_PAD_ROWS : 0);
            a.ldy = pad_rows ? pad_it->second : nn;
            const sox_bind xb = pad_k ? pad_channels(ni, bind(n.in[0]), m, k, a.k) : bind(n.in[0]);
            launch_gemm_dma(ni, a, xb, bind(n.in[1], p.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK),
                            p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(), res_b, bind(out_value),
                            ln ? &ln_it->second : nullptr, ln ? "gemm_ln" : "gemm", ln || pad_rows || pad_k ? 0 : 'd');
            return;
        }
        char amode;
        if (k % ld() == 0) {
            amode = 'd';
            a.flags |= SOX_F_DENSE_A;
            a.lda = k;
        } else {
            // any K: the rows as a 1 x M "image" of K channels through the scalar gather (a 1x1 conv)
            amode = 's';
            a.ih = 1; a.iw = (int)m; a.ic = k; a.oh = 1; a.ow = (int)m;
            a.kh = 1; a.kw = 1; a.sh = 1; a.sw = 1;
        }
        launch_igemm(ni, a, bind(n.in[0]), bind(n.in[1], p.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK),
                     p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(), res_b, bind(out_value), amode,
                     "gemm");
    }

    void conv_transpose(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_convt_p>();
        std::vector<int> si = nhwc(n.in[0]);
        const PlanValue& wv = g.V(n.in[1]);
        int oc = wv.shape[1];
        auto chain = g.convt_chain.find(ni);
        if (chain != g.convt_chain.end()) {  // this ConvT and the one-channel ConvT after it (plan_convt_chain)
            const PlanNode& n2 = g.plan.nodes[chain->second];
            const auto& p2 = n2.p<sox_convt_p>();
            if (g.padded_ld.count(n2.out[0])) fail(SOX_E_INVALID, "convt2: the output's rows are padded");
            sox_convt2_args a{};
            a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.ic = si[3]; a.oc1 = oc; a.kpad = pad8(si[3]);
            a.act1 = p.act; a.act2 = p2.act;
            add(ni, std::string("sox_convt2_") + ty() + "_n" + std::to_string(oc / 8), a,
                {{offsetof(sox_convt2_args, x), bind(n.in[0])}, {offsetof(sox_convt2_args, w1), bind(n.in[1], CK_CONVT_NK)},
                 {offsetof(sox_convt2_args, b1), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_convt2_args, w2), bind(n2.in[1], SOX_CK_CONVTW)},
                 {offsetof(sox_convt2_args, b2), p2.bias_value >= 0 ? bind(p2.bias_value, SOX_CK_F32) : none()},
                 {offsetof(sox_convt2_args, y), bind(n2.out[0])}},
                (uint32_t)(((int64_t)a.n * a.ih * a.iw + 127) / 128), 1, 1, 256, 0, "convt2");
            return;
        }
        if (convt_as_gemm(g, n)) {
            const int kh = p.kernel[0], kw = p.kernel[1];
            sox_igemm_args a{};
            a.m = si[0] * si[1] * si[2];
            a.n = kh * kw * oc;
            a.k = si[3];
            a.kpad = pad8(si[3]);
            a.ih = si[1]; a.iw = si[2]; a.ic = si[3]; a.oh = si[1]; a.ow = si[2];
            a.kh = 1; a.kw = 1; a.sh = 1; a.sw = 1;  // the A side is a 1x1 conv over the input pixels
            a.flags = SOX_F_CONVT | (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (p.act << SOX_F_ACT_SHIFT);
            a.ldy = a.n;
            a.ct_kh = kh; a.ct_kw = kw; a.ct_oc = oc;
            launch_conv_dma(ni, a, bind(n.in[0]), bind(n.in[1], CK_CONVT_NK),
                            p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none(), none(), bind(n.out[0]));
            return;
        }
        sox_convt_args a{};
        a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.ic = si[3]; a.oc = oc; a.kh = p.kernel[0]; a.kw = p.kernel[1];
        a.flags = (p.bias_value >= 0 ? SOX_F_BIAS : 0) | (p.act << SOX_F_ACT_SHIFT);
        std::vector<std::pair<size_t, sox_bind>> ptrs = {
            {offsetof(sox_convt_args, x), bind(n.in[0])}, {offsetof(sox_convt_args, w), bind(n.in[1], SOX_CK_CONVTW)},
            {offsetof(sox_convt_args, bias), p.bias_value >= 0 ? bind(p.bias_value, SOX_CK_F32) : none()},
            {offsetof(sox_convt_args, y), bind(n.out[0])}};
        const int64_t taps = (int64_t)a.kh * a.kw, nw = taps * a.ic * oc;
        if (convt_one_channel(g, n)) {
            add(ni, std::string("sox_convt_one_") + ty(), a, ptrs, blocks((int64_t)a.n * a.ih * a.iw), 1, 1, 256,
                (uint32_t)(nw * 4), "convt");
            return;
        }
        if (taps <= 4 && nw <= 16384) {  // pixel-major: weights in LDS, every tap from one read of x
            int64_t items = (int64_t)a.n * a.ih * a.iw * ((oc + 7) / 8);
            add(ni, std::string("sox_convt_pix_") + ty(), a, ptrs, blocks(items), 1, 1, 256, (uint32_t)(nw * 4), "convt");
            return;
        }
        int64_t items = (int64_t)a.n * a.ih * a.iw * a.kh * a.kw * oc;
        add(ni, std::string("sox_convt_") + ty(), a, ptrs, blocks(items), 1, 1, 256, 0, "convt");
    }

    // The SE gate's arguments and bindings (one scratch block: GAP partials over `chunks` pixel chunks,
    // fc1's per-group sums, and the gated weight copy when the gate folds into its consumer conv, whose
    // fold it registers).
    struct SeSetup {
        sox_se_args a{};
        std::vector<std::pair<size_t, sox_bind>> ptrs;
        sox_bind part;
    };
    SeSetup se_setup(int ni, const PlanNode& n, int chunks) {
        const auto& p = n.p<sox_channel_gate_p>();
        std::vector<int> si = nhwc(n.in[0]);
        const PlanValue& w1 = g.V(n.in[1]);  // [R, C, 1, 1]
        int nb = si[0], hw = si[1] * si[2], c = si[3], r = w1.shape[0];
        const int groups = (c + 63) / 64;
        const int fold = se_fold_target(ni, n, nb, c);
        const uint64_t part_bytes = ((uint64_t)nb * chunks * c * 4 + 255) & ~255ull;
        const uint64_t hid_bytes = ((uint64_t)nb * groups * r * 4 + 255) & ~255ull;
        uint64_t wbytes = 0;
        int wn = 0;
        if (fold >= 0) {
            wn = g.V(g.plan.nodes[fold].in[1]).shape[0];
            wbytes = (uint64_t)wn * c * g.es;
        }
        SeSetup st;
        sox_bind part = scratch(part_bytes + hid_bytes + wbytes);
        sox_bind hid = part, wdst = part;
        hid.offset += part_bytes;
        hid.size = hid_bytes;
        wdst.offset += part_bytes + hid_bytes;
        wdst.size = wbytes;
        part.size = part_bytes;
        st.part = part;
        sox_se_args& sa = st.a;
        sa.c = c; sa.r = r; sa.chunks = chunks; sa.hw = hw; sa.groups = groups;
        sa.flags = (p.b1 >= 0 ? 1 : 0) | (p.b2 >= 0 ? 2 : 0) | (p.act1 == SOX_ACT_RELU ? 4 : 0) | (p.hard ? 8 : 0);
        sa.alpha = p.alpha; sa.beta = p.beta; sa.offset = p.offset;
        st.ptrs = {
            {offsetof(sox_se_args, part), part}, {offsetof(sox_se_args, w1), bind(n.in[1], SOX_CK_F32)},
            {offsetof(sox_se_args, b1), p.b1 >= 0 ? bind(p.b1, SOX_CK_F32) : none()},
            {offsetof(sox_se_args, w2), bind(n.in[2], SOX_CK_F32)},
            {offsetof(sox_se_args, b2), p.b2 >= 0 ? bind(p.b2, SOX_CK_F32) : none()},
            {offsetof(sox_se_args, hid), hid}};
        if (fold >= 0) {
            const PlanNode& cv = g.plan.nodes[fold];
            sa.flags |= SOX_SE_FOLD;
            sa.wn = wn;
            sa.wk = c;  // pad8(c) == c
            st.ptrs.push_back({offsetof(sox_se_args, s), none()});
            st.ptrs.push_back({offsetof(sox_se_args, wsrc), bind(cv.in[1], SOX_CK_CONVWT)});
            st.ptrs.push_back({offsetof(sox_se_args, wdst), wdst});
            se_fold[fold] = {n.in[0], wdst};
            skip.insert(ni + 1);
        } else {
            st.ptrs.push_back({offsetof(sox_se_args, s), bind(n.out[0])});
            st.ptrs.push_back({offsetof(sox_se_args, wsrc), none()});
            st.ptrs.push_back({offsetof(sox_se_args, wdst), none()});
        }
        return st;
    }

    // Whether the SE gate node gi runs inside the depthwise launch before it (sox_dwt_*_se): asked for
    // with SIMDONNX_HIP_SE_IN_DW, the gate reads only that conv's output, r <= 256 (four W2 values per
    // lane) and fc2's LDS (h and the gates) fits the smallest depthwise tile's. Not the default: fc2 of
    // a whole image in one workgroup is a chain of dependent memory round trips (28-96 us per
    // MobileNetV3-small block on MI355X against 22-24 us for the depthwise + fc1 + fc2 launches).
    bool se_in_depthwise(int gi, int ic) {
        const char* want = getenv("SIMDONNX_HIP_SE_IN_DW");
        if (!want || !*want || !strcmp(want, "0")) return false;
        const PlanNode& gate = g.plan.nodes[gi];
        const int r = g.V(gate.in[1]).shape[0];
        return r <= 256 && ((r + 63) / 64 * 64 + ic) * 4 <= 14 * 1024;
    }

    void channel_gate(int ni, const PlanNode& n) {
        if (se_with_dw.count(ni)) return;  // ran in the depthwise launch that produced its input
        std::vector<int> si = nhwc(n.in[0]);
        int nb = si[0], hw = si[1] * si[2], c = si[3];
        // GAP partials: (c / cv) channel vectors x P pixel phases per 256-thread block, ~4 pixels
        // per thread per chunk and at most 64 chunks; fc1 then reduces them once per 64-channel group
        bool vec = c % ld() == 0;
        int cg = vec ? c / ld() : c;
        int P = std::max(1, 256 / cg);
        int chunks = (int)std::min<int64_t>(64, std::max<int64_t>(1, ((int64_t)hw + 4 * P - 1) / (4 * P)));
        auto dw_gap = gap_from_dw.find(ni);
        if (dw_gap != gap_from_dw.end()) chunks = dw_gap->second;  // partials written by the depthwise conv
        SeSetup st = se_setup(ni, n, chunks);
        if (dw_gap == gap_from_dw.end()) {
            sox_gap_args ga{};
            ga.n = nb; ga.hw = hw; ga.c = c; ga.chunks = chunks;
            add(ni, std::string("sox_gap_") + ty() + (vec ? "_v" : "_s"), ga,
                {{offsetof(sox_gap_args, x), bind(n.in[0])}, {offsetof(sox_gap_args, part), st.part}},
                (uint32_t)chunks, (uint32_t)nb, 1, 256, 0, "gap_part");
        }
        add(ni, "sox_se_fc1", st.a, st.ptrs, (uint32_t)st.a.groups, (uint32_t)nb, 1, 256, 0, "se_gate");
        add(ni, std::string("sox_se_fc2_") + ty(), st.a, st.ptrs, (uint32_t)((c + 3) / 4), (uint32_t)nb, 1, 256,
            (uint32_t)(st.a.r * 4), "se_gate");
    }

    void elementwise(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_ew_p>();
        const PlanValue& a = g.V(n.in[0]);
        const PlanValue& b = g.V(n.in[1]);
        const PlanValue& o = g.V(n.out[0]);
        int64_t cnt = o.count();
        // x op scalar const: one affine pass
        for (int k = 0; k < 2; k++) {
            const PlanValue& s = k == 0 ? b : a;
            const PlanValue& x = k == 0 ? a : b;
            if (!(s.is_const && s.floats.size() == 1 && !x.is_const && x.count() == cnt)) continue;
            float c = s.floats[0], al = 0, be = 0;
            bool ok = true;
            switch (p.op) {
                case 0: al = 1; be = c; break;
                case 1: if (k == 0) { al = 1; be = -c; } else { al = -1; be = c; } break;
                case 2: al = c; be = 0; break;
                default: if (k == 0) { al = 1.0f / c; be = 0; } else ok = false;
            }
            if (!ok || p.act != 0) break;
            sox_unary_args u{};
            u.count = cnt; u.mode = 1; u.alpha = al; u.beta = be;
            add(ni, std::string("sox_unary_") + ty(), u,
                {{offsetof(sox_unary_args, x), bind(n.in[k == 0 ? 0 : 1])}, {offsetof(sox_unary_args, y), bind(n.out[0])}},
                blocks((cnt + ld() - 1) / ld()), 1, 1, 256, 0, "unary2");
            return;
        }
        if (!a.is_const && !b.is_const && a.count() == cnt && b.count() == cnt) {
            sox_ew_args e{};
            e.count = cnt; e.op = p.op; e.flags = p.act << SOX_F_ACT_SHIFT;
            add(ni, std::string("sox_ew_") + ty(), e,
                {{offsetof(sox_ew_args, a), bind(n.in[0])}, {offsetof(sox_ew_args, b), bind(n.in[1])},
                 {offsetof(sox_ew_args, y), bind(n.out[0])}},
                blocks((cnt + ld() - 1) / ld()), 1, 1, 256, 0, "ew2v");
            return;
        }
        // NHWC per-channel broadcast: full [N,H,W,C] op vec [N,C,1,1] (SE scale, ChannelBroadcast), or op a
        // per-channel const [C,1,1] / [1,C,1,1] / [C] (an unfolded BatchNormalization, GraphCompiler.cs:1898-1923)
        for (int k = 0; k < 2; k++) {
            const PlanValue& full = k == 0 ? a : b;
            const PlanValue& vec = k == 0 ? b : a;
            if (full.is_const || full.count() != cnt || full.shape.size() != 4) continue;
            std::vector<int> fs = nhwc(n.in[k]);
            int nb = fs[0], c = fs[3];
            bool per_img = vec.shape.size() == 4 && vec.shape[0] == nb && vec.shape[1] == c && vec.shape[2] == 1 &&
                           vec.shape[3] == 1 && !vec.is_const;
            bool per_chan_const = vec.is_const && vec.count() == c &&
                                  (vec.shape.size() == 1 || (vec.shape.size() >= 3 && vec.shape[vec.shape.size() - 3] == c));
            if (!per_img && !per_chan_const) continue;
            sox_chan_args ca{};
            ca.rows = (int64_t)nb * fs[1] * fs[2];
            ca.c = c;
            ca.hw = fs[1] * fs[2];
            ca.op = p.op;
            ca.flags = (k == 1 ? 1 : 0) | (per_chan_const ? 2 : 0) | (p.act << SOX_F_ACT_SHIFT);
            bool vecw = c % ld() == 0;
            add(ni, std::string("sox_chan_") + ty() + (vecw ? "_v" : "_s"), ca,
                {{offsetof(sox_chan_args, x), bind(n.in[k])}, {offsetof(sox_chan_args, v), bind(n.in[1 - k])},
                 {offsetof(sox_chan_args, y), bind(n.out[0])}},
                blocks(ca.rows * (vecw ? c / ld() : c)), 1, 1, 256, 0, "ew2");
            return;
        }
        unsupported("elementwise broadcast pattern");
    }

    void unary_act(int ni, const PlanNode& n, int act, int mode = 0, float al = 1, float be = 0) {
        int64_t cnt = g.V(n.out[0]).count();
        sox_unary_args u{};
        u.count = cnt; u.mode = mode; u.act = act; u.alpha = al; u.beta = be;
        add(ni, std::string("sox_unary_") + ty(), u,
            {{offsetof(sox_unary_args, x), bind(n.in[0])}, {offsetof(sox_unary_args, y), bind(n.out[0])}},
            blocks((cnt + ld() - 1) / ld()), 1, 1, 256, 0, "unary");
    }

    void resize_nearest(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_resize_nearest_p>();
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]);
        sox_nearest_args a{};
        a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.c = si[3]; a.oh = so[1]; a.ow = so[2];
        const PlanValue& v = g.V(n.in[0]);
        int r = (int)v.shape.size();
        a.sy = p.scales[r - 2];
        a.sx = p.scales[r - 1];
        bool has_add = n.in.size() > 1;
        a.flags = (has_add ? 1 : 0) | (p.add_relu ? 2 : 0);
        int ldy, yoff;
        sox_bind yb = out_bind(n.out[0], a.c, ldy, yoff);
        a.ldy = ldy; a.y_off = 0;  // the bind already points at the slice
        bool vec = a.c % ld() == 0;
        add(ni, std::string("sox_nearest_") + ty() + (vec ? "_v" : "_s"), a,
            {{offsetof(sox_nearest_args, x), bind(n.in[0])},
             {offsetof(sox_nearest_args, add), has_add ? bind(n.in[1]) : none()},
             {offsetof(sox_nearest_args, y), yb}},
            blocks((int64_t)a.n * a.oh * a.ow * (vec ? a.c / ld() : a.c)), 1, 1, 256, 0, "nearest");
    }

    void concat(int ni, const PlanNode& n) {
        std::vector<int> so = g.V(n.out[0]).phys();
        const auto& p = n.p<sox_concat_p>();
        // NHWC channel concat: the concat axis must be the innermost physical dim
        const PlanValue& ov = g.V(n.out[0]);
        int axis = p.axis < 0 ? p.axis + (int)ov.shape.size() : p.axis;
        int inner_logical = ov.layout.empty() ? (int)ov.shape.size() - 1 : ov.layout.back();
        if (axis != inner_logical) unsupported("concat over a non-innermost physical axis");
        int ctot = so.back();
        int64_t rows = ov.count() / ctot;
        int off = 0;
        for (int in : n.in) {
            int c = g.V(in).phys().back();
            if (concat_slice.count(in)) {  // already written into its slice by its producer
                off += c;
                continue;
            }
            sox_slice_copy_args a{};
            a.rows = rows; a.c = c; a.ldy = ctot; a.y_off = off;
            bool vec = c % ld() == 0 && ctot % ld() == 0 && off % ld() == 0;
            add(ni, std::string("sox_slice_") + ty() + (vec ? "_v" : "_s"), a,
                {{offsetof(sox_slice_copy_args, x), bind(in)}, {offsetof(sox_slice_copy_args, y), bind(n.out[0])}},
                blocks(rows * (vec ? c / ld() : c)), 1, 1, 256, 0, "concat");
            off += c;
        }
    }

    void layer_norm(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_ln_p>();
        const PlanValue& v = g.V(n.in[0]);
        int len = v.shape.back();
        if (v.phys().back() != len) unsupported("LayerNorm: last dim not innermost");
        sox_ln_args a{};
        a.rows = v.count() / len; a.len = len; a.eps = p.eps;
        add(ni, std::string("sox_ln_") + ty(), a,
            {{offsetof(sox_ln_args, x), bind(n.in[0])}, {offsetof(sox_ln_args, gamma), bind(n.in[1], SOX_CK_F32)},
             {offsetof(sox_ln_args, beta), bind(n.in[2], SOX_CK_F32)}, {offsetof(sox_ln_args, y), bind(n.out[0])}},
            (uint32_t)((a.rows + 3) / 4), 1, 1, 256, 0, "layernorm");
    }

    void softmax(int ni, const PlanNode& n) {
        const PlanValue& v = g.V(n.in[0]);
        int len = v.shape.back();
        if (v.phys().back() != len) unsupported("Softmax: last dim not innermost");
        sox_softmax_args a{};
        a.rows = v.count() / len; a.len = len;
        auto pad_it = g.padded_ld.find(n.in[0]);
        a.ldx = pad_it != g.padded_ld.end() ? pad_it->second : len;
        a.staged = len <= 16384;  // the row fits a 64 KiB LDS window: read it from memory once
        add(ni, std::string("sox_softmax_") + ty(), a,
            {{offsetof(sox_softmax_args, x), bind(n.in[0])}, {offsetof(sox_softmax_args, y), bind(n.out[0])}},
            (uint32_t)a.rows, 1, 1, 256, a.staged ? (uint32_t)len * 4 : 0, "softmax");
    }

    // Element stride of logical axis `axis` in value v's storage (VkGraph.LogicalStride).
    int64_t logical_stride(const PlanValue& v, int axis) {
        const int64_t s = axis_stride(v, axis);
        if (s < 0) fail(SOX_E_INVALID, "attention: axis not found");
        return s;
    }

    void attention(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_attention_p>();
        int64_t sb[4], sh[4], st[4], base[4];
        int dims_n = 1, dims_h = 1, dims_t = 1, dims_s = 1, dims_d = 1;
        for (int i = 0; i < 3; i++) {
            const PlanValue& v = g.V(n.in[i]);
            const int* d = p.dims[i];
            sb[i] = d[0] >= 0 ? logical_stride(v, d[0]) : 0;
            sh[i] = d[1] >= 0 ? logical_stride(v, d[1]) : 0;
            st[i] = d[2] >= 0 ? logical_stride(v, d[2]) : 0;
            if (logical_stride(v, d[3]) != 1) unsupported("attention: head dim not contiguous");
            base[i] = p.fix_axis[i] >= 0 ? p.fix_index[i] * logical_stride(v, p.fix_axis[i]) : 0;
            if (i == 0) {
                dims_n = d[0] >= 0 ? v.shape[d[0]] : 1;
                dims_h = d[1] >= 0 ? v.shape[d[1]] : 1;
                dims_t = d[2] >= 0 ? v.shape[d[2]] : 1;
                dims_d = v.shape[d[3]];
            }
            if (i == 1) dims_s = d[2] >= 0 ? v.shape[d[2]] : 1;
        }
        // output: logical [n, h, t, d] stored in out_layout order
        const PlanValue& ov = g.V(n.out[0]);
        int ol[4] = {0, 1, 2, 3};
        if (p.out_layout[0] >= 0) for (int i = 0; i < 4; i++) ol[i] = p.out_layout[i];
        int ls[4] = {dims_n, dims_h, dims_t, dims_d};
        int64_t ostr[4];
        {
            int64_t s = 1;
            for (int j = 3; j >= 0; j--) { ostr[ol[j]] = s; s *= ls[ol[j]]; }
        }
        if (ostr[3] != 1) unsupported("attention: output head dim not contiguous");
        if (ov.count() != (int64_t)dims_n * dims_h * dims_t * dims_d) fail(SOX_E_INVALID, "attention: output size");
        if (dims_d > 64) unsupported("attention: head size > 64");
        sox_attn_args a{};
        a.batch = dims_n; a.heads = dims_h; a.t = dims_t; a.s = dims_s; a.d = dims_d; a.scale = p.scale;
        a.q_sb = sb[0]; a.q_sh = sh[0]; a.q_st = st[0];
        a.k_sb = sb[1]; a.k_sh = sh[1]; a.k_st = st[1];
        a.v_sb = sb[2]; a.v_sh = sh[2]; a.v_st = st[2];
        a.o_sb = ostr[0]; a.o_sh = ostr[1]; a.o_st = ostr[2];
        sox_bind bq = bind(n.in[0]), bk = bind(n.in[1]), bv = bind(n.in[2]);
        bq.offset += base[0] * g.es; bk.offset += base[1] * g.es; bv.offset += base[2] * g.es;
        bool aligned = true;
        for (int i = 0; i < 3; i++)
            aligned &= sb[i] % 8 == 0 && sh[i] % 8 == 0 && st[i] % 8 == 0 && base[i] % 8 == 0;
        aligned &= ostr[0] % 8 == 0 && ostr[1] % 8 == 0 && ostr[2] % 8 == 0;
        if (g.f16 && (dims_d == 32 || dims_d == 64) && dims_s <= 128 && aligned) {
            // matrix-core attention: one workgroup per (batch, head), one wave per 16 queries (<= 8 waves)
            int sk = dims_s <= 32 ? 32 : dims_s <= 64 ? 64 : dims_s <= 80 ? 80 : 128;
            char kn[64];
            snprintf(kn, sizeof kn, "sox_attn_f16_mfma_s%d_d%d", sk, dims_d);
            const int waves = std::max(1, std::min(8, (dims_t + 15) / 16));
            add(ni, kn, a,
                {{offsetof(sox_attn_args, q), bq}, {offsetof(sox_attn_args, k), bk}, {offsetof(sox_attn_args, v), bv},
                 {offsetof(sox_attn_args, o), bind(n.out[0])}},
                (uint32_t)(dims_n * dims_h), 1, 1, (uint32_t)(64 * waves), 0, "attn");
            return;
        }
        int D = dims_d <= 32 ? 32 : 64;
        uint32_t lds = (uint32_t)(2 * dims_s * D * 4);
        uint32_t gy = (uint32_t)((dims_t + 127) / 128);
        add(ni, std::string("sox_attn_") + ty() + (D == 32 ? "_d32" : "_d64"), a,
            {{offsetof(sox_attn_args, q), bq}, {offsetof(sox_attn_args, k), bk}, {offsetof(sox_attn_args, v), bv},
             {offsetof(sox_attn_args, o), bind(n.out[0])}},
            (uint32_t)(dims_n * dims_h), gy, 1, 128, lds, "attn");
    }

    void maxpool(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_pool_p>();
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]);
        sox_pool_args q{};
        q.n = si[0]; q.ih = si[1]; q.iw = si[2]; q.c = si[3]; q.oh = so[1]; q.ow = so[2];
        q.kh = p.kernel[0]; q.kw = p.kernel[1]; q.sh = p.strides[0]; q.sw = p.strides[1]; q.pt = p.pads[0]; q.pl = p.pads[1];
        q.flags = p.fuse_relu ? 1 : 0;
        add(ni, std::string("sox_pool_") + ty(), q,
            {{offsetof(sox_pool_args, x), bind(n.in[0])}, {offsetof(sox_pool_args, y), bind(n.out[0])}},
            blocks((int64_t)q.n * q.oh * q.ow * q.c), 1, 1, 256, 0, "maxpool");
    }

    // ---- the rest of the ExecOp surface (VkGraph.cs:795-1068) ----
    static void need_i32(int64_t count, const char* what) {
        if (count >= ((int64_t)1 << 31)) fail(SOX_E_UNSUPPORTED, std::string("HIP: ") + what + ": more than 2^31 elements");
    }

    // ResizeBilinear (VkGraph.cs:795-810; Kernels/Nhwc.cs:818-870)
    void resize_bilinear(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_resize_p>();
        if (g.V(n.in[0]).shape.size() != 4) unsupported("ResizeBilinear: rank != 4");
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]);
        const bool has_add = n.in.size() > 1;
        if (has_add && g.V(n.in[1]).count() != g.V(n.out[0]).count()) fail(SOX_E_INVALID, "ResizeBilinear: addend shape");
        if (si[0] != so[0] || si[3] != so[3]) fail(SOX_E_INVALID, "ResizeBilinear: batch / channel mismatch");
        sox_bilinear_args a{};
        a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.c = si[3]; a.oh = so[1]; a.ow = so[2];
        a.sy = p.scales[2]; a.sx = p.scales[3];
        a.flags = (p.fuse_relu ? 1 : 0) | (has_add ? 2 : 0) | (p.add_relu ? 4 : 0);
        need_i32((int64_t)a.n * a.oh * a.ow, "ResizeBilinear");
        const bool vec = a.c % ld() == 0;
        add(ni, std::string("sox_bilinear_") + ty() + (vec ? "_v" : "_s"), a,
            {{offsetof(sox_bilinear_args, x), bind(n.in[0])},
             {offsetof(sox_bilinear_args, add), has_add ? bind(n.in[1]) : none()},
             {offsetof(sox_bilinear_args, y), bind(n.out[0])}},
            blocks((int64_t)a.n * a.oh * a.ow * (vec ? a.c / ld() : a.c)), 1, 1, 256, 0, "bilinear");
    }

    // Pad, generic rank-4 in storage order: begin pads permuted to physical dims (VkGraph.cs:812-828)
    void pad(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_pad_p>();
        const PlanValue& x = g.V(n.in[0]);
        if (x.shape.size() != 4 || p.rank != 4) unsupported("Pad: rank != 4");
        std::vector<int> id = x.phys(), od = g.V(n.out[0]).phys();
        sox_pad_args a{};
        for (int d = 0; d < 4; d++) {
            const int l = x.layout.empty() ? d : x.layout[d];
            a.id[d] = id[d]; a.od[d] = od[d]; a.pb[d] = p.pads[l];
            if (p.mode == 1 && id[d] < 1) fail(SOX_E_INVALID, "Pad: reflect of an empty axis");
        }
        a.reflect = p.mode == 1;
        a.value = p.value;
        need_i32(g.V(n.out[0]).count(), "Pad");
        const bool vec = a.pb[3] == 0 && id[3] == od[3] && od[3] % ld() == 0;
        add(ni, std::string("sox_pad_") + ty() + (vec ? "_v" : "_s"), a,
            {{offsetof(sox_pad_args, x), bind(n.in[0])}, {offsetof(sox_pad_args, y), bind(n.out[0])}},
            blocks(g.V(n.out[0]).count() / (vec ? ld() : 1)), 1, 1, 256, 0, "pad");
    }

    // Transpose (physical perm, VkGraph.cs:830-844) and Slice (physical axes, VkGraph.cs:846-865) as one
    // strided gather. Every source offset is checked against the input here, so the kernel cannot
    // read outside it.
    void gather(int ni, const PlanNode& n, const std::vector<int>& od, const std::vector<int64_t>& str, int64_t base,
                const char* label) {
        const std::vector<int> is = g.V(n.in[0]).phys();
        const int64_t cnt = g.V(n.out[0]).count(), icnt = g.V(n.in[0]).count();
        need_i32(cnt, label);
        int64_t lo = base, hi = base;
        for (size_t k = 0; k < od.size(); k++) {
            if (od[k] <= 0) { lo = hi = 0; break; }
            const int64_t span = (int64_t)(od[k] - 1) * str[k];
            (span < 0 ? lo : hi) += span;
        }
        if (cnt > 0 && (lo < 0 || hi >= icnt)) fail(SOX_E_INVALID, std::string(label) + ": source outside the input");
        sox_gather_args a{};
        a.count = cnt; a.base = base;
        const int r = (int)od.size();
        if (r > 6) unsupported(std::string(label) + ": rank > 6");
        for (int k = 0; k < 6; k++) {
            const int kk = k - (6 - r);
            a.od[k] = kk < 0 ? 1 : od[kk];
            a.str[k] = kk < 0 ? 0 : str[kk];
        }
        add(ni, std::string("sox_gather_") + ty(), a,
            {{offsetof(sox_gather_args, x), bind(n.in[0])}, {offsetof(sox_gather_args, y), bind(n.out[0])}},
            blocks(cnt), 1, 1, 256, 0, label);
    }

    static std::vector<int64_t> strides_of(const std::vector<int>& s) {
        std::vector<int64_t> st(s.size(), 1);
        for (int d = (int)s.size() - 2; d >= 0; d--) st[d] = st[d + 1] * s[d + 1];
        return st;
    }

    void transpose(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_transpose_p>();
        const std::vector<int> is = g.V(n.in[0]).phys(), os = g.V(n.out[0]).phys();
        const int r = (int)is.size();
        if (p.rank != r || (int)os.size() != r || r > 6) fail(SOX_E_INVALID, "Transpose: rank");
        const std::vector<int64_t> ist = strides_of(is);
        std::vector<int64_t> str(r);
        for (int k = 0; k < r; k++) {
            const int pk = p.perm[k];
            if (pk < 0 || pk >= r || os[k] != is[pk]) fail(SOX_E_INVALID, "Transpose: perm / shape mismatch");
            str[k] = ist[pk];
        }
        // perm = identity prefix, then two contiguous groups of dims swapped: a batched 2D transpose
        // [batch][R][C] -> [batch][C][R] through LDS tiles (coalesced on both sides)
        int k0 = 0;
        while (k0 < r && p.perm[k0] == k0) k0++;
        if (k0 < r) {
            const int j = p.perm[k0];  // the first input dim of the group that moves to the front
            bool two = j > k0;
            for (int k = k0; two && k < r; k++) {
                const int want = k < k0 + (r - j) ? j + (k - k0) : k0 + (k - k0 - (r - j));
                two = p.perm[k] == want;
            }
            if (two) {
                int64_t batch = 1, rows = 1, cols = 1;
                for (int d = 0; d < k0; d++) batch *= is[d];
                for (int d = k0; d < j; d++) rows *= is[d];
                for (int d = j; d < r; d++) cols *= is[d];
                need_i32(g.V(n.out[0]).count(), "transpose");
                if (rows > 1 && cols > 1 && batch <= 65535 && (rows + 63) / 64 <= 65535) {
                    sox_transpose2d_args a{};
                    a.rows = (int)rows; a.cols = (int)cols;
                    add(ni, std::string("sox_transpose2d_") + ty(), a,
                        {{offsetof(sox_transpose2d_args, x), bind(n.in[0])}, {offsetof(sox_transpose2d_args, y), bind(n.out[0])}},
                        (uint32_t)((cols + 63) / 64), (uint32_t)((rows + 63) / 64), (uint32_t)batch, 256, 0, "transpose");
                    return;
                }
            }
        }
        gather(ni, n, os, str, 0, "transpose");
    }

    void slice(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_slice_p>();
        const std::vector<int> is = g.V(n.in[0]).phys(), os = g.V(n.out[0]).phys();
        const int r = (int)is.size();
        if ((int)os.size() != r || p.naxes < 0 || p.naxes > 6) fail(SOX_E_INVALID, "Slice: rank");
        const std::vector<int64_t> ist = strides_of(is);
        std::vector<int64_t> start(r, 0), step(r, 1);
        for (int i = 0; i < p.naxes; i++) {
            const int ax = p.axes[i] < 0 ? p.axes[i] + r : p.axes[i];
            if (ax < 0 || ax >= r || p.steps[i] == 0) fail(SOX_E_INVALID, "Slice: axis / step");
            start[ax] = p.starts[i];
            step[ax] = p.steps[i];
        }
        int64_t base = 0;
        std::vector<int64_t> str(r);
        for (int d = 0; d < r; d++) {
            base += start[d] * ist[d];
            str[d] = step[d] * ist[d];
        }
        gather(ni, n, os, str, base, "slice");
    }

    // LeakyRelu / Tanh / Clip / Erf (unary2.comp, VkGraph.cs:493-502, 994-1006)
    void unary2(int ni, const PlanNode& n, int mode, float a, float b) {
        const int64_t cnt = g.V(n.out[0]).count();
        sox_unary2_args u{};
        u.count = cnt; u.mode = mode; u.a = a; u.b = b;
        add(ni, std::string("sox_unary2_") + ty(), u,
            {{offsetof(sox_unary2_args, x), bind(n.in[0])}, {offsetof(sox_unary2_args, y), bind(n.out[0])}},
            blocks((cnt + ld() - 1) / ld()), 1, 1, 256, 0, "unary2");
    }

    // DepthToSpace / SpaceToDepth, NHWC (VkGraph.cs:1008-1019)
    void depth_space(int ni, const PlanNode& n, bool s2d) {
        const auto& p = n.p<sox_depth_to_space_p>();
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]);
        const int b = p.block;
        if (b < 1) fail(SOX_E_INVALID, "DepthToSpace: block");
        const bool ok = s2d ? (si[1] == so[1] * b && si[2] == so[2] * b && so[3] == si[3] * b * b)
                            : (so[1] == si[1] * b && so[2] == si[2] * b && si[3] == so[3] * b * b);
        if (!ok || si[0] != so[0]) fail(SOX_E_INVALID, "DepthToSpace: shapes");
        sox_d2s_args a{};
        a.count = g.V(n.out[0]).count();
        a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.ic = si[3]; a.oh = so[1]; a.ow = so[2]; a.oc = so[3];
        a.block = b; a.crd = p.crd ? 1 : 0; a.s2d = s2d ? 1 : 0;
        need_i32(std::max(a.count, g.V(n.in[0]).count()), "DepthToSpace");
        if (!p.crd && (s2d ? a.ic : a.oc) % ld() == 0) {  // DCR, whole 16-byte channel vectors
            add(ni, std::string("sox_d2s_dcr_") + ty(), a,
                {{offsetof(sox_d2s_args, x), bind(n.in[0])}, {offsetof(sox_d2s_args, y), bind(n.out[0])}},
                blocks(a.count / ld()), 1, 1, 256, 0, s2d ? "s2d" : "d2s");
            return;
        }
        add(ni, std::string("sox_d2s_") + ty(), a,
            {{offsetof(sox_d2s_args, x), bind(n.in[0])}, {offsetof(sox_d2s_args, y), bind(n.out[0])}},
            blocks(a.count), 1, 1, 256, 0, s2d ? "s2d" : "d2s");
    }

    // AvgPool, NHWC (VkGraph.cs:1038-1049)
    void avgpool(int ni, const PlanNode& n) {
        const auto& p = n.p<sox_pool_p>();
        std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]);
        sox_avgpool_args q{};
        q.n = si[0]; q.ih = si[1]; q.iw = si[2]; q.c = si[3]; q.oh = so[1]; q.ow = so[2];
        q.kh = p.kernel[0]; q.kw = p.kernel[1]; q.sh = p.strides[0]; q.sw = p.strides[1]; q.pt = p.pads[0]; q.pl = p.pads[1];
        q.count_include_pad = p.count_include_pad ? 1 : 0;
        need_i32(std::max(g.V(n.out[0]).count(), g.V(n.in[0]).count()), "AvgPool");
        const bool vec = q.c % ld() == 0;
        add(ni, std::string("sox_avgpool_") + ty() + (vec ? "_v" : "_s"), q,
            {{offsetof(sox_avgpool_args, x), bind(n.in[0])}, {offsetof(sox_avgpool_args, y), bind(n.out[0])}},
            blocks((int64_t)q.n * q.oh * q.ow * (vec ? q.c / ld() : q.c)), 1, 1, 256, 0, "avgpool");
    }

    // GlobalAvgPool (VkGraph.cs:899-916): the SE path's GAP partials, then the chunk sums in order
    void global_avg_pool(int ni, const PlanNode& n) {
        std::vector<int> si = nhwc(n.in[0]);
        const int nb = si[0], hw = si[1] * si[2], c = si[3];
        const bool vec = c % ld() == 0;
        const int cg = vec ? c / ld() : c;
        const int P = std::max(1, 256 / cg);
        // ~4 pixels per thread per chunk, up to 256 chunks per image (the SE path stops at 64, where
        // its fc1 reduces the partials; here the chunk sums are the whole second pass)
        const int chunks = (int)std::min<int64_t>(256, std::max<int64_t>(1, ((int64_t)hw + 4 * P - 1) / (4 * P)));
        sox_bind part = scratch((uint64_t)nb * chunks * c * 4);
        sox_gap_args ga{};
        ga.n = nb; ga.hw = hw; ga.c = c; ga.chunks = chunks;
        add(ni, std::string("sox_gap_") + ty() + (vec ? "_v" : "_s"), ga,
            {{offsetof(sox_gap_args, x), bind(n.in[0])}, {offsetof(sox_gap_args, part), part}},
            (uint32_t)chunks, (uint32_t)nb, 1, 256, 0, "gap_part");
        sox_gap_mean_args m{};
        m.n = nb; m.c = c; m.chunks = chunks; m.inv_hw = 1.0f / (float)hw;
        add(ni, std::string("sox_gap_mean_") + ty(), m,
            {{offsetof(sox_gap_mean_args, part), part}, {offsetof(sox_gap_mean_args, y), bind(n.out[0])}},
            (uint32_t)((c + 63) / 64), (uint32_t)nb, 1, 256, 0, "gap_mean");
    }

    // MatMul, batched, identity layouts, B may broadcast over the batch (VkGraph.cs:1051-1068)
    void matmul(int ni, const PlanNode& n) {
        const PlanValue &a = g.V(n.in[0]), &b = g.V(n.in[1]), &o = g.V(n.out[0]);
        auto identity = [](const PlanValue& v) {
            for (size_t i = 0; i < v.layout.size(); i++)
                if (v.layout[i] != (int)i) return false;
            return true;
        };
        if (!identity(a) || !identity(b) || !identity(o)) unsupported("MatMul: permuted layout");
        if (a.shape.size() < 2 || b.shape.size() < 2) fail(SOX_E_INVALID, "MatMul: rank < 2");
        const int m = a.shape[a.shape.size() - 2], k = a.shape.back(), nn = b.shape.back();
        if (b.shape[b.shape.size() - 2] != k) fail(SOX_E_INVALID, "MatMul: inner dims");
        const int64_t batch = o.count() / ((int64_t)m * nn);
        const int64_t ab = a.count() / ((int64_t)m * k), bb = b.count() / ((int64_t)k * nn);
        if (ab != batch || (bb != batch && bb != 1)) unsupported("MatMul: batch broadcast");
        if (batch > 65535) unsupported("MatMul: batch > 65535");
        need_i32(std::max({a.count(), b.count(), o.count()}), "MatMul");
        sox_matmul_args q{};
        q.batch = (int)batch; q.m = m; q.n = nn; q.k = k;
        q.a_stride = (int64_t)m * k; q.b_stride = bb == 1 ? 0 : (int64_t)k * nn; q.y_stride = (int64_t)m * nn;
        add(ni, std::string("sox_matmul_") + ty(), q,
            {{offsetof(sox_matmul_args, a), bind(n.in[0])}, {offsetof(sox_matmul_args, b), bind(n.in[1])},
             {offsetof(sox_matmul_args, y), bind(n.out[0])}},
            (uint32_t)((nn + 63) / 64), (uint32_t)((m + 63) / 64), (uint32_t)batch, 256, 0, "matmul");
    }

    // ---- built-in extension ops (Engine/Fusions/*.cs EmitVulkan twins) ----
    bool builtin_ext(int ni, const PlanNode& n) {
        if (n.ext == "SafeDiv") {  // SafeDivOp.cs:26-33
            const auto& p = n.p<sox_safediv_p>();
            const int64_t cnt = g.V(n.out[0]).count();
            if (g.V(n.in[0]).count() < cnt || g.V(n.in[1]).count() < cnt) fail(SOX_E_INVALID, "SafeDiv: operand shorter than the output");
            sox_safediv_args a{};
            a.count = cnt; a.eps = p.eps; a.lo = p.lo; a.hi = p.hi;
            add(ni, std::string("sox_safediv_") + ty(), a,
                {{offsetof(sox_safediv_args, a), bind(n.in[0])}, {offsetof(sox_safediv_args, b), bind(n.in[1])},
                 {offsetof(sox_safediv_args, y), bind(n.out[0])}},
                blocks((cnt + ld() - 1) / ld()), 1, 1, 256, 0, "safediv");
            return true;
        }
        if (n.ext == "ChannelShift") {  // ChannelShiftOp.cs:33-52
            const auto& p = n.p<sox_shift_p>();
            if (g.V(n.in[0]).shape.size() != 4) unsupported("ChannelShift: rank != 4");
            std::vector<int> si = nhwc(n.in[0]);
            if (p.ngroups < 1 || p.ngroups > 5) unsupported("ChannelShift: > 5 groups");
            if (p.axis != 2 && p.axis != 3) fail(SOX_E_INVALID, "ChannelShift: axis");
            sox_shift_args a{};
            a.n = si[0]; a.h = si[1]; a.w = si[2]; a.c = si[3]; a.axis = p.axis; a.ngroups = p.ngroups;
            bool vec = a.c % ld() == 0;
            for (int i = 0; i < 5; i++) {
                a.ends[i] = i < p.ngroups ? std::min(p.group_ends[i], a.c) : a.c;
                a.offs[i] = i < p.ngroups ? p.offsets[i] : 0;
                vec = vec && a.ends[i] % ld() == 0;
            }
            add(ni, std::string("sox_shift_") + ty() + (vec ? "_v" : "_s"), a,
                {{offsetof(sox_shift_args, x), bind(n.in[0])}, {offsetof(sox_shift_args, y), bind(n.out[0])}},
                blocks((int64_t)a.n * a.h * a.w * (vec ? a.c / ld() : a.c)), 1, 1, 256, 0, "shift");
            return true;
        }
        if (n.ext == "UpHead") {  // UpHeadOp.cs:88-150
            const auto& p = n.p<sox_uphead_p>();
            std::vector<int> si = nhwc(n.in[0]), so = nhwc(n.out[0]), sk = nhwc(n.in[1]);
            const PlanValue& wv = g.V(n.in[2]);
            const int c = si[3], oc = so[3];
            if (oc > 8 || c > 128 || c % 4 != 0) unsupported("UpHead: c=" + std::to_string(c) + " oc=" + std::to_string(oc));
            if (wv.count() != (int64_t)oc * c) fail(SOX_E_INVALID, "UpHead: weights are not [oc, c]");
            if (p.act != SOX_ACT_NONE && p.act != SOX_ACT_RELU && p.act != SOX_ACT_SIGMOID) unsupported("UpHead: activation");
            if (sk[0] != so[0] || sk[1] != so[1] || sk[2] != so[2] || si[0] != so[0]) fail(SOX_E_INVALID, "UpHead: shapes");
            sox_uphead_args a{};
            a.n = si[0]; a.ih = si[1]; a.iw = si[2]; a.c = c; a.oh = so[1]; a.ow = so[2]; a.oc = oc;
            a.sy = p.scales[2]; a.sx = p.scales[3];
            const bool has_bias = n.in.size() > 3;
            a.flags = (p.resize_relu ? 1 : 0) | (p.skip_relu ? 2 : 0) | (has_bias ? 4 : 0) | (p.has_skip_conv ? 8 : 0) |
                      (p.act << 4);
            sox_bind wsc = none(), bsc = none();
            if (p.has_skip_conv) {
                // GraphCompiler.GpuSmallConv + UpHeadOp.SkipPc: group 1, stride 1, ic < 8, oc == c <= 32,
                // oc * ic * kh * kw <= 4096, output the skip's own size
                const auto& sc = p.skip_conv;
                const PlanValue& cw = g.V(p.skip_w);
                if (cw.shape.size() != 4 || cw.shape[0] != c || c > 32 || cw.shape[1] != sk[3] || sk[3] >= 8 ||
                    cw.count() > 4096 || sc.group != 1 || sc.strides[0] != 1 || sc.strides[1] != 1 ||
                    sc.dilations[0] != 1 || sc.dilations[1] != 1 || (sc.act != SOX_ACT_NONE && sc.act != SOX_ACT_RELU) ||
                    sc.pads[0] + sc.pads[2] != cw.shape[2] - 1 || sc.pads[1] + sc.pads[3] != cw.shape[3] - 1)
                    unsupported("UpHead: unsupported skip conv");
                if (sc.pad_mode == 1 && (sc.pads[0] >= so[1] || sc.pads[2] >= so[1] || sc.pads[1] >= so[2] || sc.pads[3] >= so[2]))
                    unsupported("UpHead: reflect pad wider than the image");
                a.skc = sk[3]; a.kh = cw.shape[2]; a.kw = cw.shape[3]; a.pt = sc.pads[0]; a.pl = sc.pads[1];
                a.sc_flags = (p.skip_b >= 0 ? 1 : 0) | (sc.pad_mode == 1 ? 2 : 0) | (sc.act == SOX_ACT_RELU ? 4 : 0);
                a.sc_pad_value = sc.pad_mode == 0 ? sc.pad_value : 0.0f;
                wsc = bind(p.skip_w);
                if (p.skip_b >= 0) bsc = bind(p.skip_b, SOX_CK_F32);
            } else if (sk[3] != c) {
                fail(SOX_E_INVALID, "UpHead: skip channels");
            }
            need_i32(std::max(g.V(n.out[0]).count(), g.V(n.in[0]).count()), "UpHead");
            add(ni, std::string("sox_uphead_") + ty() + (!g.f16 || c % 8 == 0 ? "_v" : "_s"), a,
                {{offsetof(sox_uphead_args, x), bind(n.in[0])}, {offsetof(sox_uphead_args, skip), bind(n.in[1])},
                 {offsetof(sox_uphead_args, w), bind(n.in[2])},
                 {offsetof(sox_uphead_args, bias), has_bias ? bind(n.in[3], SOX_CK_F32) : none()},
                 {offsetof(sox_uphead_args, y), bind(n.out[0])}, {offsetof(sox_uphead_args, w_sc), wsc},
                 {offsetof(sox_uphead_args, b_sc), bsc}},
                blocks((int64_t)a.n * a.oh * a.ow), 1, 1, 256, 0, "uphead");
            return true;
        }
        return false;
    }

    void emit(int ni) {
        const PlanNode& n = g.plan.nodes[ni];
        if (skip.count(ni) || g.folded.count(ni) || g.moved.count(ni)) return;
        auto ua = g.upadd.find(ni);
        if (ua != g.upadd.end()) {  // the addend's conv, writing this node's output, the upsample as residual
            cov = {n.out[0], n.in[0], ua->second.second};
            conv(ua->second.first, g.plan.nodes[ua->second.first]);
            cov = {};
            return;
        }
        switch (n.op) {
            case SOX_OP_CONV: conv(ni, n); break;
            case SOX_OP_GEMM: gemm(ni, n); break;
            case SOX_OP_CONV_TRANSPOSE: conv_transpose(ni, n); break;
            case SOX_OP_CHANNEL_GATE: channel_gate(ni, n); break;
            case SOX_OP_ELEMENTWISE: elementwise(ni, n); break;
            case SOX_OP_RELU: unary_act(ni, n, SOX_ACT_RELU); break;
            case SOX_OP_SIGMOID: unary_act(ni, n, SOX_ACT_SIGMOID); break;
            case SOX_OP_GELU: unary_act(ni, n, SOX_ACT_GELU); break;
            case SOX_OP_HARDSWISH: unary_act(ni, n, SOX_ACT_HARDSWISH); break;
            case SOX_OP_SWISH: unary_act(ni, n, SOX_ACT_SWISH); break;
            case SOX_OP_COPY: unary_act(ni, n, 0, 3); break;
            case SOX_OP_HARD_SIGMOID: {
                const auto& p = n.p<sox_hard_sigmoid_p>();
                unary_act(ni, n, 0, 2, p.alpha, p.beta);
                break;
            }
            case SOX_OP_RESIZE_NEAREST: resize_nearest(ni, n); break;
            case SOX_OP_CONCAT: concat(ni, n); break;
            case SOX_OP_LAYERNORM: layer_norm(ni, n); break;
            case SOX_OP_SOFTMAX: softmax(ni, n); break;
            case SOX_OP_ATTENTION: attention(ni, n); break;
            case SOX_OP_MAXPOOL: maxpool(ni, n); break;
            case SOX_OP_RESIZE_BILINEAR: resize_bilinear(ni, n); break;
            case SOX_OP_PAD: pad(ni, n); break;
            case SOX_OP_TRANSPOSE: transpose(ni, n); break;
            case SOX_OP_SLICE: slice(ni, n); break;
            case SOX_OP_ERF: unary2(ni, n, 3, 0.0f, 0.0f); break;
            case SOX_OP_LEAKY_RELU: unary2(ni, n, 0, n.p<sox_leaky_relu_p>().alpha, 0.0f); break;
            case SOX_OP_TANH: {  // a missing record means TanhP's defaults (1, 1)
                const bool has = n.params.size() >= sizeof(sox_tanh_p);
                unary2(ni, n, 1, has ? n.p<sox_tanh_p>().in_scale : 1.0f, has ? n.p<sox_tanh_p>().out_scale : 1.0f);
                break;
            }
            case SOX_OP_CLIP: unary2(ni, n, 2, n.p<sox_clip_p>().min, n.p<sox_clip_p>().max); break;
            case SOX_OP_DEPTH_TO_SPACE: depth_space(ni, n, false); break;
            case SOX_OP_SPACE_TO_DEPTH: depth_space(ni, n, true); break;
            case SOX_OP_AVGPOOL: avgpool(ni, n); break;
            case SOX_OP_GLOBAL_AVG_POOL: global_avg_pool(ni, n); break;
            case SOX_OP_MATMUL: matmul(ni, n); break;
            case SOX_OP_EXT: {
                auto it = g.be->exts.find(n.ext);
                if (it == g.be->exts.end()) {  // a consumer registration wins over a built-in of the same name
                    if (builtin_ext(ni, n)) break;
                    unsupported("extension op " + n.ext + " not implemented");
                }
                int rc = it->second.emit(it->second.user, &g, ni);
                if (rc != SOX_OK) fail(rc, "extension op " + n.ext + " emit failed");
                break;
            }
            default: {
                char b[64];
                snprintf(b, sizeof b, "ExecOp %d not implemented", n.op);
                unsupported(b);
            }
        }
    }
};

// Element stride of logical axis `axis` in value v's storage (VkGraph.LogicalStride), -1 if absent.
int64_t axis_stride(const PlanValue& v, int axis) {
    std::vector<int> ps = v.phys();
    int64_t s = 1;
    for (int j = (int)ps.size() - 1; j >= 0; j--) {
        if ((v.layout.empty() ? j : v.layout[j]) == axis) return s;
        s *= ps[j];
    }
    return -1;
}

// Reads of value v's buffer, through v or any alias of it, by the nodes not folded away other than
// node `except`, plus the plan output when it lives there.
int buffer_reads(const sox_graph& g, int v, int except) {
    const auto& P = g.plan;
    const int buf = P.values[v].buf;
    if (buf < 0) return 1;
    int u = P.values[P.output].buf == buf;
    for (int ni = 0; ni < (int)P.nodes.size(); ni++) {
        if (ni == except || g.folded.count(ni)) continue;
        for (int x : P.nodes[ni].in) u += P.values[x].buf == buf;
        if (P.nodes[ni].op == SOX_OP_CONV) {
            const auto& cp = P.nodes[ni].p<sox_conv_p>();
            for (int x : {cp.add_value, cp.bias_value}) u += x >= 0 && P.values[x].buf == buf;
        }
    }
    return u;
}

// Reads of value v by the nodes not folded away (inputs and the value-id fields of conv params) plus
// the plan output.
int value_reads(const sox_graph& g, int v) {
    const auto& P = g.plan;
    int u = v == P.output;
    for (int ni = 0; ni < (int)P.nodes.size(); ni++) {
        if (g.folded.count(ni)) continue;
        for (int x : P.nodes[ni].in) u += x == v;
        if (P.nodes[ni].op == SOX_OP_CONV) {
            const auto& cp = P.nodes[ni].p<sox_conv_p>();
            u += (cp.add_value == v) + (cp.bias_value == v);
        }
    }
    return u;
}

// Element range of an activation value in the arena plan (empty for consts).
std::pair<int64_t, int64_t> value_range(const sox_plan& P, int v) {
    const PlanValue& pv = P.values[v];
    if (pv.buf < 0) return {0, 0};
    const int64_t off = P.buf_offset[pv.buf];
    return {off, off + std::max<int64_t>(pv.count(), 1)};
}

// The activations node k's dispatches write at its place in the dispatch order: its outputs, and the
// outputs of the nodes folded into it (a Gemm's residual Add, the rest of a fused transformer MLP and
// the projection output its part kernel stores, the Attention run with a qkv Gemm). None for a node
// folded into another or moved to another node's place (those writes count there).
std::vector<int> emitted_writes(const sox_graph& g, int k) {
    std::vector<int> w;
    if (g.folded.count(k) || g.moved.count(k)) return w;
    const sox_plan& P = g.plan;
    w = P.nodes[k].out;
    auto ra = g.residual_add.find(k);
    if (ra != g.residual_add.end())
        for (int o : P.nodes[ra->second.first].out) w.push_back(o);
    auto m = g.mlp.find(k);
    if (m != g.mlp.end()) {
        w.push_back(m->second.out);
        if (m->second.proj >= 0) w.push_back(P.nodes[k].in[0]);
    }
    auto q = g.qkv_attn.find(k);
    if (q != g.qkv_attn.end())
        for (int o : P.nodes[q->second].out) w.push_back(o);
    auto ct = g.convt_chain.find(k);
    if (ct != g.convt_chain.end())
        for (int o : P.nodes[ct->second].out) w.push_back(o);
    return w;
}

// Moves value v's buffer to a place of its own past the activations (the arena grows by its size).
// Every value on that buffer moves with it: the zero-copy views of v (Reshape, Squeeze, Unsqueeze,
// Identity; AliasOf, Engine/ExecPlan.cs:207, 211) share its buffer id and are bound through that
// buffer's offset (Backends/Vulkan/VkGraph.cs:365-367), so a view left behind would read the old place.
void relocate_value(sox_plan& P, int v) {
    const int old = P.values[v].buf;
    if (old < 0) fail(SOX_E_INVALID, "relocate_value: not an activation");
    int64_t n = 1;
    for (const PlanValue& pv : P.values)
        if (pv.buf == old) n = std::max<int64_t>(n, pv.count());
    const int64_t at = (P.arena_floats + 63) & ~63ll;
    P.buf_offset.push_back(at);
    const int nb = (int)P.buf_offset.size() - 1;
    for (PlanValue& pv : P.values)
        if (pv.buf == old) pv.buf = nb;
    P.arena_floats = at + n;
}

// Gemm node followed directly by an Add of its output and a same-shape activation (+ ReLU): the Add
// is lowered into the Gemm epilogue (v = acc + bias + residual -> act) when the Gemm has no
// activation of its own, nothing else reads the Gemm output and the residual was produced before the
// Gemm. The epilogue writes the Add's output while other workgroups still read the Gemm's input A and
// the residual, so when the arena plan put that output over A, or over the residual at another
// offset, the output gets a buffer of its own.
void plan_residual_adds(sox_graph& g) {
    if (getenv("SIMDONNX_HIP_NO_RES_FUSE")) return;
    auto& P = g.plan;
    for (int ni = 0; ni + 1 < (int)P.nodes.size(); ni++) {
        const PlanNode& n = P.nodes[ni];
        if (n.op != SOX_OP_GEMM || g.folded.count(ni) || g.folded.count(ni + 1)) continue;
        if (n.p<sox_gemm_p>().act != 0 || g.padded_ld.count(n.out[0])) continue;
        const PlanNode& nx = P.nodes[ni + 1];
        if (nx.op != SOX_OP_ELEMENTWISE || nx.in.size() != 2 || nx.out.size() != 1) continue;
        const auto& ep = nx.p<sox_ew_p>();
        if (ep.op != 0 || (ep.act != 0 && ep.act != SOX_ACT_RELU)) continue;
        const int y = n.out[0];
        const int other = nx.in[0] == y ? nx.in[1] : nx.in[1] == y ? nx.in[0] : -1;
        if (other < 0 || other == y || value_reads(g, y) != 1) continue;
        const PlanValue &yv = P.values[y], &rv = P.values[other], &ov = P.values[nx.out[0]];
        if (rv.is_const || rv.buf < 0 || ov.buf < 0 || rv.count() != yv.count() || ov.count() != yv.count()) continue;
        if (rv.phys() != yv.phys() || ov.phys() != yv.phys()) continue;
        bool later = false;  // residual produced before the Gemm
        for (int k = ni + 1; k < (int)P.nodes.size() && !later; k++)
            for (int o : P.nodes[k].out) later |= o == other;
        if (later) continue;
        const int out = nx.out[0];
        auto a = value_range(P, n.in[0]), o = value_range(P, out), r = value_range(P, other);
        const bool over_a = a.first < o.second && o.first < a.second;
        const bool over_r = r.first < o.second && o.first < r.second && r.first != o.first;
        if (over_a || over_r) relocate_value(P, out);
        g.residual_add[ni] = {ni + 1, other};
    }
}

// An SE gate whose product x·s only a 1x1 conv reads folds into that conv's weights at emit time (fc2
// writes W'[n][c] = W[n][c]·s[c], the conv reads x; Emitter::se_fold_target). The folded conv reads x
// while it writes its output, and the arena plan of the unfused graph may have put that output over x
// (dead after the Mul there): the output then gets a buffer of its own, so the fold, and with it the
// removal of the full-tensor multiply's dispatch, does not depend on where the planner put it.
void plan_se_fold_space(sox_graph& g) {
    auto& P = g.plan;
    for (int ni = 0; ni + 2 < (int)P.nodes.size(); ni++) {
        const PlanNode& n = P.nodes[ni];
        if (n.op != SOX_OP_CHANNEL_GATE || n.in.empty() || n.out.size() != 1) continue;
        const int x = n.in[0], s = n.out[0];
        const PlanValue& xv = P.values[x];
        if (xv.buf < 0 || xv.shape.size() != 4 || xv.shape[0] != 1 || xv.shape[1] % 8 != 0) continue;
        const int c = xv.shape[1];
        const PlanNode& mul = P.nodes[ni + 1];
        const PlanNode& cv = P.nodes[ni + 2];
        if (mul.op != SOX_OP_ELEMENTWISE || mul.in.size() != 2 || mul.out.size() != 1) continue;
        const auto& ep = mul.p<sox_ew_p>();
        if (ep.op != 2 || ep.act != 0) continue;
        if (!((mul.in[0] == x && mul.in[1] == s) || (mul.in[0] == s && mul.in[1] == x))) continue;
        const int y = mul.out[0];
        if (value_reads(g, s) != 1 || value_reads(g, y) != 1 || P.values[y].count() != xv.count()) continue;
        if (cv.op != SOX_OP_CONV || cv.in.empty() || cv.in[0] != y || cv.out.size() != 1) continue;
        const auto& cp = cv.p<sox_conv_p>();
        if (cp.group != 1 || cp.kernel[0] != 1 || cp.kernel[1] != 1 || cp.strides[0] != 1 || cp.strides[1] != 1 ||
            cp.dilations[0] != 1 || cp.dilations[1] != 1 || cp.has_pool || cp.pads[0] || cp.pads[1] || cp.pads[2] ||
            cp.pads[3] || cp.add_value == y)
            continue;
        const PlanValue& wv = P.values[cv.in[1]];
        if (!wv.is_const || wv.shape.size() != 4 || wv.shape[1] != c) continue;
        const int out = cv.out[0];
        if (P.values[out].buf < 0) continue;
        const auto xr = value_range(P, x), orr = value_range(P, out);
        if (xr.first < orr.second && orr.first < xr.second) relocate_value(P, out);
    }
}

// An fp16 Gemm whose N is not a multiple of 4 (the SVTR class head, N = 6625) and whose output only
// a Softmax over its rows reads: the output gets a buffer of its own with rows padded to a multiple
// of 8, so the LDS-DMA Gemm stores whole 8-byte groups (SOX_F_PAD_ROWS) and the Softmax reads
// 16-byte-aligned rows (sox_softmax_args.ldx); the pad columns are never read.
void plan_padded_rows(sox_graph& g) {
    if (!g.f16) return;
    auto& P = g.plan;
    for (int ni = 0; ni < (int)P.nodes.size(); ni++) {
        const PlanNode& n = P.nodes[ni];
        if (n.op != SOX_OP_GEMM || g.folded.count(ni)) continue;
        const int y = n.out[0];
        const PlanValue& yv = P.values[y];
        const PlanValue& av = P.values[n.in[0]];
        const int N = yv.shape.back(), K = av.shape.back();
        if (N % 4 == 0 || K % 64 != 0 || yv.buf < 0 || y == P.output || yv.phys().back() != N) continue;
        if (value_reads(g, y) != 1) continue;
        bool viewed = false;  // a view of y would read the unpadded layout
        for (int v = 0; v < (int)P.values.size() && !viewed; v++) viewed = v != y && P.values[v].buf == yv.buf;
        if (viewed) continue;
        int consumer = -1;
        for (int k = ni + 1; k < (int)P.nodes.size(); k++)
            if (!g.folded.count(k))
                for (int x : P.nodes[k].in)
                    if (x == y) consumer = k;
        if (consumer < 0 || P.nodes[consumer].op != SOX_OP_SOFTMAX) continue;
        const int ldp = (N + 7) & ~7;
        const int64_t rows = yv.count() / N;
        const int64_t at = (P.arena_floats + 63) & ~63ll;
        P.buf_offset.push_back(at);
        P.values[y].buf = (int)P.buf_offset.size() - 1;
        P.arena_floats = at + rows * ldp;
        g.padded_ld[y] = ldp;
    }
}

// A ConvTranspose (no activation) whose output feeds only "* s[c]" with a per-channel const, whose
// product feeds only "+ t[c]" (+ ReLU): an unfolded BatchNormalization (the reference lowers it to
// per-channel Mul + Add, GraphCompiler.cs:1898-1923). The pair folds into the ConvTranspose's
// weights and bias, (sum x w + b) s + t = sum x (w s) + (b s + t), as two new consts; the Mul and
// Add emit nothing and the ConvTranspose writes the Add's output (moved to a buffer of its own when
// the arena plan put it over the ConvTranspose's input, dead by then).
void fold_affine_after_convt(sox_graph& g) {
    if (getenv("SIMDONNX_HIP_NO_CONVT_FOLD")) return;
    auto& P = g.plan;
    auto reads = [&](int v) { return value_reads(g, v); };
    auto range = [&](int v) { return value_range(P, v); };
    for (int ni = 0; ni + 2 < (int)P.nodes.size(); ni++) {
        PlanNode& ct = P.nodes[ni];
        if (ct.op != SOX_OP_CONV_TRANSPOSE || g.folded.count(ni) || ct.in.size() < 2) continue;
        const sox_convt_p cp = ct.p<sox_convt_p>();
        const PlanValue& wv = P.values[ct.in[1]];
        if (cp.act != 0 || !wv.is_const || wv.shape.size() != 4) continue;
        const int ic = wv.shape[0], oc = wv.shape[1], taps = wv.shape[2] * wv.shape[3];
        const PlanNode& mul = P.nodes[ni + 1];
        const PlanNode& add = P.nodes[ni + 2];
        if (mul.op != SOX_OP_ELEMENTWISE || add.op != SOX_OP_ELEMENTWISE || mul.in.size() != 2 || add.in.size() != 2)
            continue;
        const auto &mp = mul.p<sox_ew_p>(), &ap = add.p<sox_ew_p>();
        if (mp.op != 2 || mp.act != 0 || ap.op != 0 || (ap.act != 0 && ap.act != SOX_ACT_RELU)) continue;
        const int y = ct.out[0];
        auto other = [](const PlanNode& n, int v) { return n.in[0] == v ? n.in[1] : n.in[1] == v ? n.in[0] : -1; };
        const int sv = other(mul, y);
        if (sv < 0) continue;
        const int m = mul.out[0], tv = other(add, m);
        if (tv < 0) continue;
        const PlanValue &S = P.values[sv], &T = P.values[tv];
        if (!S.is_const || !T.is_const || (int)S.floats.size() != oc || (int)T.floats.size() != oc) continue;
        // per-channel consts only ([C], or C on the channel axis of a rank >= 3 shape such as [C,1,1] /
        // [1,C,1,1]), the shapes the unfused broadcast reads per channel: [1,1,1,C] would broadcast
        // along W instead
        auto per_chan = [&](const PlanValue& v) {
            return v.shape.size() == 1 || (v.shape.size() >= 3 && v.shape[v.shape.size() - 3] == oc);
        };
        if (!per_chan(S) || !per_chan(T)) continue;
        if (reads(y) != 1 || reads(m) != 1) continue;
        const int out = add.out[0];
        if (P.values[out].count() != P.values[y].count()) continue;
        auto a = range(ct.in[0]), o = range(out);
        if (a.first < o.second && o.first < a.second)
            relocate_value(P, out);  // planned over the input (dead by the Add)
        PlanValue w2 = wv, b2;
        w2.name = wv.name + ".affine";
        for (int c = 0; c < ic; c++)
            for (int k = 0; k < oc; k++)
                for (int t = 0; t < taps; t++) w2.floats[((size_t)c * oc + k) * taps + t] *= S.floats[k];
        b2.is_const = true;
        b2.shape = {oc};
        b2.name = wv.name + ".affine_bias";
        b2.floats.resize(oc);
        for (int k = 0; k < oc; k++)
            b2.floats[k] = (cp.bias_value >= 0 ? P.values[cp.bias_value].floats[k] : 0.0f) * S.floats[k] + T.floats[k];
        P.values.push_back(std::move(w2));
        ct.in[1] = (int)P.values.size() - 1;
        P.values.push_back(std::move(b2));
        sox_convt_p np = cp;
        np.bias_value = (int)P.values.size() - 1;
        np.act = ap.act;
        memcpy(ct.params.data(), &np, sizeof(np));
        ct.out[0] = out;
        g.folded.insert(ni + 1);
        g.folded.insert(ni + 2);
    }
}

// Two stride-2 2x2 ConvTransposes in a row, the first run as a Gemm (16-bit storage, ic <= 32 and
// ic % 8 == 0, oc1 % 8 == 0 and oc1 <= 32) and the second to one channel (sox_convt_one_*), where only
// the second reads the first one's output and every node between them is folded away (the DB head's
// ConvT + BatchNorm + ReLU -> ConvT + Sigmoid, after fold_affine_after_convt): one sox_convt2_* kernel
// at the first one's place writes the second one's output, and the first one's output map is never
// stored. The second output gets a buffer of its own when the arena plan put it over the first one's
// input (read by the same kernel).
void plan_convt_chain(sox_graph& g) {
    if (getenv("SIMDONNX_HIP_NO_CONVT_CHAIN") || !g.f16) return;
    auto& P = g.plan;
    for (int n1 = 0; n1 < (int)P.nodes.size(); n1++) {
        const PlanNode& a = P.nodes[n1];
        if (a.op != SOX_OP_CONV_TRANSPOSE || g.folded.count(n1) || !convt_as_gemm(g, a)) continue;
        const auto& pa = a.p<sox_convt_p>();
        const PlanValue& wa = P.values[a.in[1]];
        const int ic = wa.shape[0], oc1 = wa.shape[1];
        if (pa.kernel[0] != 2 || pa.kernel[1] != 2 || ic > 32 || ic % 8 || oc1 % 8 || oc1 > 32) continue;
        const int y1 = a.out[0];
        if (value_reads(g, y1) != 1 || buffer_reads(g, y1, -1) != 1 || y1 == P.output) continue;
        int n2 = n1 + 1;
        while (n2 < (int)P.nodes.size() && g.folded.count(n2)) n2++;
        if (n2 >= (int)P.nodes.size()) continue;
        const PlanNode& b = P.nodes[n2];
        if (b.op != SOX_OP_CONV_TRANSPOSE || b.in.size() < 2 || b.in[0] != y1 || !convt_one_channel(g, b)) continue;
        const auto& pb = b.p<sox_convt_p>();
        if (pb.kernel[0] != 2 || pb.kernel[1] != 2 || P.values[b.in[1]].shape[0] != oc1) continue;
        auto r = value_range(P, a.in[0]), o = value_range(P, b.out[0]);
        if (r.first < o.second && o.first < r.second) relocate_value(P, b.out[0]);
        g.convt_chain[n1] = n2;
        g.folded.insert(n2);
    }
}

int fusable_attention(sox_graph& g, int qi, int x);
bool fusable_mlp(sox_graph& g, int f1, int x, sox_graph::Mlp& f);

// A LayerNorm over the innermost dim whose output only an fp16 Gemm reads, as its A (the recognizer
// blocks' ln1 -> qkv and ln2 -> fc1, the final norm -> head): the LayerNorm folds into the Gemm,
// which then reads the LayerNorm's input and normalises its rows itself (sox_gemm_ln_* kernels):
//   LN(x) W + b = rstd (x (gamma W) - mean colsum(gamma W)) + (b + beta W)
// with gamma W as the Gemm's weights, b + beta W as its bias and the column sums of gamma W as
// rounded to fp16 (the values the kernel multiplies) as ln_c. The mean and variance come from one
// pass of sums and sums of squares, as the reference's GPU LayerNorm takes them
// (Backends/Vulkan/Shaders/layernorm.comp:24-38). Taken only where the Gemm runs on the LDS-DMA
// ring (K % 64 == 0, N % 4 == 0 or padded rows; at least 64 rows, or fewer where the Gemm then runs in
// a fused attention or MLP), gamma W keeps the storage type's precision and no node in between writes over
// the LayerNorm's input; the Gemm's output moves to a buffer of its own when the arena plan put it
// over that input (dead after the LayerNorm, read by the Gemm now).
void fold_layernorm_into_gemm(sox_graph& g) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_LN_FOLD")) return;
    auto& P = g.plan;
    auto overlap = [](std::pair<int64_t, int64_t> a, std::pair<int64_t, int64_t> b) {
        return a.first < b.second && b.first < a.second;
    };
    for (int li = 0; li < (int)P.nodes.size(); li++) {
        const PlanNode& ln = P.nodes[li];
        if (ln.op != SOX_OP_LAYERNORM || g.folded.count(li) || ln.in.size() < 3 || ln.out.size() != 1) continue;
        const int x = ln.in[0], y = ln.out[0];
        const float eps = ln.p<sox_ln_p>().eps;
        const PlanValue &xv = P.values[x], &gv = P.values[ln.in[1]], &bv = P.values[ln.in[2]];
        const int K = xv.shape.back();
        if (xv.buf < 0 || xv.phys().back() != K || K % 64 != 0) continue;
        if (!gv.is_const || !bv.is_const || (int)gv.floats.size() != K || (int)bv.floats.size() != K) continue;
        if (y == P.output || value_reads(g, y) != 1) continue;
        int gi = -1;
        for (int k = li + 1; k < (int)P.nodes.size() && gi < 0; k++)
            if (!g.folded.count(k))
                for (int v : P.nodes[k].in)
                    if (v == y) gi = k;
        if (gi < 0) continue;
        PlanNode& gm = P.nodes[gi];
        if (gm.op != SOX_OP_GEMM || gm.in.size() < 2 || gm.in[0] != y || gm.in[1] == y) continue;
        const sox_gemm_p gp = gm.p<sox_gemm_p>();
        const PlanValue& wv = P.values[gm.in[1]];
        if (!wv.is_const || wv.shape.size() != 2 || (gp.trans_b ? wv.shape[1] : wv.shape[0]) != K) continue;
        const int N = gp.trans_b ? wv.shape[0] : wv.shape[1];
        const int out = gm.out[0];
        if (N % 4 != 0 && !g.padded_ld.count(out)) continue;
        if (gp.bias_value >= 0 && (int)P.values[gp.bias_value].floats.size() != N) continue;
        const auto xr = value_range(P, x);
        bool clobbered = false;
        for (int k = li + 1; k < gi && !clobbered; k++)
            if (!g.folded.count(k))
                for (int o : P.nodes[k].out) clobbered |= overlap(value_range(P, o), xr);
        if (clobbered) continue;
        // below 64 rows only for a fused block: the fold takes the attention's or the MLP's dispatches with it
        // (one line of 47 tokens through the recognizer: 62 -> 30 dispatches, 327 -> 234 us)
        sox_graph::Mlp probe;
        if (xv.count() / K < 64 && fusable_attention(g, gi, x) < 0 && !fusable_mlp(g, gi, x, probe)) continue;
        PlanValue w2 = wv, b2, c2;
        w2.name = wv.name + ".ln";
        std::vector<double> bsum(N, 0.0), csum(N, 0.0);
        for (int k = 0; k < K; k++)
            for (int n = 0; n < N; n++) {
                const size_t at = gp.trans_b ? (size_t)n * K + k : (size_t)k * N + n;
                const float w = wv.floats[at];
                w2.floats[at] = w * gv.floats[k];
                bsum[n] += (double)bv.floats[k] * w;
            }
        std::vector<float> w16(w2.floats.size()), wsq(N, 0.0f), esq(N, 0.0f);
        g.round16(w2.floats.data(), w16.data(), (int64_t)w16.size());
        const float normal = g.bf16 ? 0.0f : 0x1p-14f;
        for (int i = 0; i < (gp.trans_b ? N : K); i++) {
            const int len = gp.trans_b ? K : N;
            const float *v = &w2.floats[(size_t)i * len], *r = &w16[(size_t)i * len];
            for (int j = 0; j < len; j++) {
                const int n = gp.trans_b ? i : j;
                const float lost = std::fabs(v[j]) < normal ? r[j] - v[j] : 0.0f;
                csum[n] += r[j];
                wsq[n] += v[j] * v[j];
                esq[n] += lost * lost;
            }
        }
        // gamma W has to fit fp16 as W does: finite, and what a column's values below the normal range lose stays
        // under what rounding takes from the others (0.15 of half a unit in the last place, squared). Weights of
        // 0.02 under gamma 1e-3, 16 rows of 192: 9.3e-4 from 64 bits folded, 3.7e-4 as two nodes (gamma 3e-3 4.3e-4 and
        // 3.6e-4, gamma 1e-2 3.6e-4 both, gamma 1 3.0e-4 and 3.7e-4).
        bool keeps = true;
        for (int n = 0; n < N; n++) keeps = keeps && std::isfinite(csum[n]) && esq[n] <= 0.15f * 0x1p-22f * wsq[n];
        if (!keeps) continue;
        b2.is_const = c2.is_const = true;
        b2.shape = c2.shape = {N};
        b2.name = wv.name + ".ln_bias";
        c2.name = wv.name + ".ln_colsum";
        b2.floats.resize(N);
        c2.floats.resize(N);
        for (int n = 0; n < N; n++) {
            b2.floats[n] = (float)((gp.bias_value >= 0 ? P.values[gp.bias_value].floats[n] : 0.0f) + bsum[n]);
            c2.floats[n] = (float)csum[n];
        }
        P.values.push_back(std::move(w2));  // (references into P.values are stale from here)
        gm.in[1] = (int)P.values.size() - 1;
        P.values.push_back(std::move(b2));
        sox_gemm_p np = gp;
        np.bias_value = (int)P.values.size() - 1;
        memcpy(gm.params.data(), &np, sizeof(np));
        P.values.push_back(std::move(c2));
        g.ln_fold[gi] = {(int)P.values.size() - 1, eps};
        gm.in[0] = x;
        g.folded.insert(li);
        if (!g.padded_ld.count(out) && overlap(value_range(P, out), xr)) relocate_value(P, out);
    }
}

// A transformer MLP: Gemm f1 with a LayerNorm folded in and GELU, whose output only the next Gemm f2
// (no activation; its residual Add, if any, already lowered into its epilogue) reads. Both run as one
// kernel (mlp.hip) when the shapes have an instance (K1 x H in {192 x 768, 128 x 512, 64 x 256},
// N2 a multiple of 32 up to 256); the hidden activation is never stored. Every workgroup reads its
// own rows of x and of the residual before it writes the same rows of the output, so the output may
// share x's or the residual's buffer only at the same offset with the same row length; otherwise it
// moves to a buffer of its own.
// Whether f1, the Gemm that folds a LayerNorm of x, and the Gemm after it are such an MLP (f: its parts).
bool fusable_mlp(sox_graph& g, int f1, int x, sox_graph::Mlp& f) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_MLP_FUSE") || g.folded.count(f1)) return false;
    auto& P = g.plan;
    const PlanNode& n1 = P.nodes[f1];
    const sox_gemm_p p1 = n1.p<sox_gemm_p>();
    if (p1.act != SOX_ACT_GELU || p1.trans_b) return false;
    const int h = n1.out[0];
    const int K1 = P.values[x].shape.back(), H = P.values[h].shape.back();
    if (!((K1 == 192 && H == 768) || (K1 == 128 && H == 512) || (K1 == 64 && H == 256))) return false;
    if (h == P.output || value_reads(g, h) != 1 || g.padded_ld.count(h)) return false;
    int f2 = -1;
    for (int k = f1 + 1; k < (int)P.nodes.size() && f2 < 0; k++)
        if (!g.folded.count(k))
            for (int v : P.nodes[k].in)
                if (v == h) f2 = k;
    if (f2 < 0 || g.ln_fold.count(f2)) return false;
    // the kernel runs at f1's place: nothing may run between the two Gemms (it would see the output
    // early), and the residual must exist by then
    for (int k = f1 + 1; k < f2; k++)
        if (!g.folded.count(k)) return false;
    const PlanNode& n2 = P.nodes[f2];
    if (n2.op != SOX_OP_GEMM || n2.in[0] != h || n2.in[1] == h) return false;
    const sox_gemm_p p2 = n2.p<sox_gemm_p>();
    const PlanValue& w2 = P.values[n2.in[1]];
    if (p2.trans_b || p2.act != 0 || !w2.is_const || w2.shape.size() != 2 || w2.shape[0] != H) return false;
    const int N2 = w2.shape[1];
    if (N2 % 32 != 0 || N2 > 256) return false;
    auto ra = g.residual_add.find(f2);
    const int add = ra == g.residual_add.end() ? -1 : ra->second.first;
    const int res = ra == g.residual_add.end() ? -1 : ra->second.second;
    for (int k = f2 + 1; k < add; k++)  // the Add follows f2 directly (plan_residual_adds), nothing else
        if (!g.folded.count(k)) return false;
    const int out = add >= 0 ? P.nodes[add].out[0] : n2.out[0];
    if (g.padded_ld.count(out) || P.values[out].shape.back() != N2) return false;
    f = {f2, add, res, out};
    return true;
}

void plan_fused_mlp(sox_graph& g) {
    auto& P = g.plan;
    for (auto& kv : g.ln_fold) {
        const int f1 = kv.first, x = P.nodes[f1].in[0];
        sox_graph::Mlp f;
        if (!fusable_mlp(g, f1, x, f) || P.nodes[f1].p<sox_gemm_p>().bias_value < 0) continue;
        const int out = f.out, res = f.residual, K1 = P.values[x].shape.back(), N2 = P.values[out].shape.back();
        auto same_rows = [&](int v, int row_len) {
            return value_range(P, v).first == value_range(P, out).first && row_len == N2;
        };
        auto clash = [&](int v, int row_len) {
            const auto a = value_range(P, v), o = value_range(P, out);
            return a.first < o.second && o.first < a.second && !same_rows(v, row_len);
        };
        if (clash(x, K1) || (res >= 0 && clash(res, N2))) relocate_value(P, out);
        // split over the hidden width when one workgroup per 32 rows would leave CUs idle (the parts'
        // fc2 sums meet in sox_mlp_sum_*); SIMDONNX_HIP_MLP_SPLIT=0 / 1 forces either form
        const int64_t rbs = (P.values[x].count() / K1 + 31) / 32;
        const char* mode = getenv("SIMDONNX_HIP_MLP_SPLIT");
        f.split = mode && *mode ? mode[0] == '1' : rbs < std::max(1, g.be->info.compute_units);
        g.mlp[f1] = f;
        g.folded.insert(f.fc2);
        if (f.add >= 0) g.folded.insert(f.add);
    }
}

// LayerNorm -> qkv Gemm -> Attention of an SVTR / ViT block (Backends/Vulkan/VkGraph.cs:719-793 for the
// attention, the LN-folded Gemm as lowered above): the Gemm and the Attention over its packed
// [n][t][3][heads][32] output run as one kernel per (image, head) (qkv_attn.hip) when dim = heads * 32 = 192,
// t <= 96, the attention output is stored [n][t][heads][32] and nothing else reads the qkv rows (they
// then stay in LDS). A workgroup reads its image's x rows while the image's other heads write their
// output columns, so the output must not overlap x.
// fusable_attention: the Attention node that Gemm qi, which folds a LayerNorm of x, runs with, or -1.
int fusable_attention(sox_graph& g, int qi, int x) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_ATTN_FUSE")) return -1;
    auto& P = g.plan;
    const int ai = qi + 1;
    if (ai >= (int)P.nodes.size() || g.folded.count(qi) || g.mlp.count(qi) || g.folded.count(ai)) return -1;
    const PlanNode &nq = P.nodes[qi], &na = P.nodes[ai];
    if (na.op != SOX_OP_ATTENTION) return -1;
    const sox_gemm_p pq = nq.p<sox_gemm_p>();
    if (pq.act != 0 || g.residual_add.count(qi)) return -1;
    const int qkv = nq.out[0], att = na.out[0];
    const PlanValue &xv = P.values[x], &qv = P.values[qkv], &ov = P.values[att];
    constexpr int DIM = 192;
    if (xv.buf < 0 || !xv.layout.empty() || xv.shape.back() != DIM || g.padded_ld.count(x)) return -1;
    if (qv.buf < 0 || !qv.layout.empty() || qv.shape.back() != 3 * DIM || g.padded_ld.count(qkv)) return -1;
    const int64_t rows = xv.count() / DIM;
    // the attention reads q, k, v as [n][t][3][heads][32] views of the qkv rows, one image per n
    const auto& pa = na.p<sox_attention_p>();
    int64_t nb = -1, t = -1;
    for (int i = 0; i < 3; i++) {
        const PlanValue& v = P.values[na.in[i]];
        const int* d = pa.dims[i];
        if (v.buf != qv.buf || v.count() != qv.count() || d[0] < 0 || d[1] < 0 || d[2] < 0 || pa.fix_axis[i] < 0 ||
            pa.fix_index[i] != i)
            return -1;
        if (i == 0) {
            nb = v.shape[d[0]];
            t = v.shape[d[2]];
        }
        if (v.shape[d[0]] != nb || v.shape[d[1]] * 32 != DIM || v.shape[d[2]] != t || v.shape[d[3]] != 32 ||
            axis_stride(v, d[0]) != t * 3 * DIM || axis_stride(v, d[1]) != 32 || axis_stride(v, d[2]) != 3 * DIM ||
            axis_stride(v, d[3]) != 1 || axis_stride(v, pa.fix_axis[i]) != DIM)
            return -1;
    }
    if (nb * t != rows || t < 1 || t > 96) return -1;
    // output [n, h, t, d] stored as [n][t][h][d]
    int ol[4] = {0, 1, 2, 3};
    if (pa.out_layout[0] >= 0)
        for (int i = 0; i < 4; i++) ol[i] = pa.out_layout[i];
    if (!(ol[0] == 0 && ol[1] == 2 && ol[2] == 1 && ol[3] == 3) || ov.buf < 0 || ov.count() != rows * DIM) return -1;
    if (buffer_reads(g, qkv, ai) != 0) return -1;
    const auto xr = value_range(P, x), o = value_range(P, att);
    return xr.first < o.second && o.first < xr.second ? -1 : ai;  // (views of the output share its buffer)
}

void plan_fused_attention(sox_graph& g) {
    for (auto& kv : g.ln_fold) {
        const int qi = kv.first, ai = fusable_attention(g, qi, g.plan.nodes[qi].in[0]);
        if (ai < 0) continue;
        g.qkv_attn[qi] = ai;
        g.folded.insert(ai);
    }
}

// The projection Gemm of a transformer block with its residual Add, x = o . Wp^T + bp + r (the SVTR
// mixer's proj and Add, Backends/Vulkan/VkGraph.cs:1029-1049 with the Add lowered as above), when x is
// the input of a split fused MLP (plan_fused_mlp): the MLP's part kernel computes x's 32 rows itself
// from o and Wp before its LayerNorm phase (sox_mlpqp_*), and part 0 of each row block stores them
// (they are the MLP's residual and may have other readers). Wp is K1 x K1, nothing runs between the
// Add and the MLP, and x must not overlap o or r: part 0 writes x's rows while the other parts of
// the same rows still read o and r (otherwise x moves to a buffer of its own when no view shares its
// buffer, else the Gemm stays).
void plan_fused_proj(sox_graph& g) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_PROJ_FUSE")) return;
    auto& P = g.plan;
    for (auto& kv : g.mlp) {
        const int f1 = kv.first;
        sox_graph::Mlp& f = kv.second;
        if (!f.split) continue;
        const int x = P.nodes[f1].in[0];
        const PlanValue& xv = P.values[x];
        const int K1 = xv.shape.back();
        int pi = -1;
        for (auto& ra : g.residual_add)
            if (P.nodes[ra.second.first].out[0] == x) pi = ra.first;
        if (pi < 0 || g.folded.count(pi) || g.mlp.count(pi) || g.qkv_attn.count(pi) || g.ln_fold.count(pi)) continue;
        const int add = g.residual_add.at(pi).first, r = g.residual_add.at(pi).second;
        if (g.folded.count(add) || P.nodes[add].p<sox_ew_p>().act != 0) continue;
        bool between = false;  // the fused kernel runs at f1's place
        for (int k = pi + 1; k < f1; k++) between |= k != add && !g.folded.count(k);
        if (between) continue;
        const PlanNode& np = P.nodes[pi];
        const sox_gemm_p pp = np.p<sox_gemm_p>();
        const int o = np.in[0];
        const PlanValue &ov = P.values[o], &wv = P.values[np.in[1]], &rv = P.values[r];
        if (pp.act != 0 || !wv.is_const || wv.shape.size() != 2 || wv.shape[0] != K1 || wv.shape[1] != K1) continue;
        if (ov.buf < 0 || !ov.layout.empty() || ov.shape.back() != K1 || ov.count() != xv.count() || g.padded_ld.count(o))
            continue;
        if (rv.buf < 0 || !rv.layout.empty() || rv.count() != xv.count() || g.padded_ld.count(r)) continue;
        if (!xv.layout.empty() || g.padded_ld.count(x) || x == P.output) continue;
        auto overlaps = [&](int a, int b) {
            const auto ra = value_range(P, a), rb = value_range(P, b);
            return ra.first < rb.second && rb.first < ra.second;
        };
        if (overlaps(x, o) || overlaps(x, r)) {
            // the MLP's output may have shared x's rows (same offset, another buffer): it keeps its
            // place, x and its views move
            relocate_value(P, x);
        }
        f.proj = pi;
        f.proj_res = r;
        g.folded.insert(pi);
        g.folded.insert(add);
    }
}

// A 16-bit 3x3 stride-1 conv on the halo route whose input is a channel concat of nearest upsamples by
// powers of two (and activations at full size): the DB FPN's fuse = concat(up8(p5), up4(p4), up2(p3),
// p2) before its 3x3 conv (VkGraph.cs:486-510, 555-703). The conv gathers each channel chunk from its
// source at (y >> s, x >> s) (sox_conv_halo_*_upcat), so neither the upsampled maps nor the concat are
// stored. Needs: 2 to 4 sources of equal channels (a multiple of 8), each upsample and the concat read
// only there, no Add on an upsample, and the sources still intact when the conv runs (no node left
// between their last reader and the conv writes over them; the conv's own output moves to a buffer of
// its own when it overlaps one, or the fusion is skipped when a view shares that buffer).
void plan_upsample_concat(sox_graph& g) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_UPCAT") || getenv("SIMDONNX_HIP_NOHALO") || getenv("SIMDONNX_HIP_IGEMM"))
        return;
    auto& P = g.plan;
    const int nn = (int)P.nodes.size();
    auto producer = [&](int v, int before) {
        for (int k = before - 1; k >= 0; k--)
            if (!g.folded.count(k))
                for (int o : P.nodes[k].out)
                    if (o == v) return k;
        return -1;
    };
    auto overlaps = [&](int a, int b) {
        const auto ra = value_range(P, a), rb = value_range(P, b);
        return ra.first < rb.second && rb.first < ra.second;
    };
    for (int ci = 0; ci < nn; ci++) {
        const PlanNode& n = P.nodes[ci];
        if (n.op != SOX_OP_CONV || g.folded.count(ci)) continue;
        const sox_conv_p cp = n.p<sox_conv_p>();
        if (cp.group != 1 || cp.kernel[0] != 3 || cp.kernel[1] != 3 || cp.strides[0] != 1 || cp.strides[1] != 1 ||
            cp.dilations[0] != 1 || cp.dilations[1] != 1 || cp.pad_mode != 0 || cp.pad_value != 0.0f || cp.has_pool ||
            cp.add_value >= 0)
            continue;
        const PlanValue& wv = P.values[n.in[1]];
        // (oc >= 8: fewer output channels take the narrow route, which reads x itself)
        if (!wv.is_const || wv.shape.size() != 4 || wv.shape[0] > 64 || wv.shape[0] < 8) continue;
        const int x = n.in[0];
        const PlanValue& xv = P.values[x];
        if (x == P.output || xv.buf < 0 || value_reads(g, x) != 1) continue;
        const std::vector<int> xs = xv.phys();
        if (xs.size() != 4 || xs[3] % 8 != 0) continue;
        const int cat = producer(x, ci);
        if (cat < 0 || P.nodes[cat].op != SOX_OP_CONCAT) continue;
        const PlanNode& cn = P.nodes[cat];
        const int axis0 = cn.p<sox_concat_p>().axis;
        const int axis = axis0 < 0 ? axis0 + (int)xv.shape.size() : axis0;
        const int inner = xv.layout.empty() ? (int)xv.shape.size() - 1 : xv.layout.back();
        if (axis != inner || cn.in.size() < 2 || cn.in.size() > 4) continue;
        sox_graph::UpCat uc;
        std::vector<int> fold = {cat}, readers = {cat};
        bool ok = true;
        for (int v : cn.in) {
            const PlanValue& vv = P.values[v];
            const std::vector<int> vs = vv.phys();
            if (vv.buf < 0 || vs.size() != 4 || vs[0] != xs[0] || vs[1] != xs[1] || vs[2] != xs[2]) { ok = false; break; }
            if (uc.n == 0) uc.c = vs[3];
            if (vs[3] != uc.c || uc.c % 8 != 0) { ok = false; break; }
            int src = v, sh = 0;
            const int pv = producer(v, cat);
            if (pv >= 0 && P.nodes[pv].op == SOX_OP_RESIZE_NEAREST && P.nodes[pv].in.size() == 1 && v != P.output &&
                value_reads(g, v) == 1) {
                const auto& rp = P.nodes[pv].p<sox_resize_nearest_p>();
                const int r = (int)vv.shape.size();
                const float f = rp.scales[r - 1];
                int k = 0;
                while (k < 5 && (float)(1 << k) != f) k++;
                const PlanValue& uv = P.values[P.nodes[pv].in[0]];
                const std::vector<int> us = uv.phys();
                if (k < 5 && rp.scales[r - 2] == f && uv.buf >= 0 && us.size() == 4 && us[3] == uc.c &&
                    (us[1] << k) == xs[1] && (us[2] << k) == xs[2] && us[0] == xs[0]) {
                    src = P.nodes[pv].in[0];
                    sh = k;
                    fold.push_back(pv);
                    readers.push_back(pv);
                }
            }
            uc.src[uc.n] = src;
            uc.shift[uc.n] = sh;
            uc.n++;
        }
        if (!ok || uc.n * uc.c != xs[3]) continue;
        // the sources stay intact from their last reader up to the conv
        const int first = *std::min_element(readers.begin(), readers.end());
        for (int k = first; k < ci && ok; k++) {
            if (std::find(fold.begin(), fold.end(), k) != fold.end()) continue;
            for (int o : emitted_writes(g, k))
                for (int i = 0; i < uc.n; i++) ok &= P.values[o].buf < 0 || !overlaps(o, uc.src[i]) || o == uc.src[i];
        }
        if (!ok) continue;
        const int y = n.out[0];
        bool clash = false;
        for (int i = 0; i < uc.n; i++) clash |= overlaps(y, uc.src[i]);
        if (clash) relocate_value(P, y);
        g.upcat[ci] = uc;
        for (int k : fold) g.folded.insert(k);
    }
}

// The FPN's top-down Add, out = up(u) + a (ResizeNearest by a power of two with an addend,
// Backends/Vulkan/VkGraph.cs:486-510), where a is the output of a 16-bit 1x1 conv (no activation, no
// residual of its own) that nothing else reads: the conv runs in the Add's place on the LDS-DMA ring with
// u as its residual, read at (y >> s, x >> s), and writes out directly (v = acc + bias + u, rounded
// once; the unfused path rounds a first). a is never stored and the upsample pass disappears. The conv's
// input must survive until the Add's place: an output written over it in between moves to a buffer of
// its own (or the fusion is skipped when a view shares that buffer), and out must not overlap the conv's
// input or u (same rule).
void plan_upsample_add(sox_graph& g) {
    if (!g.f16 || getenv("SIMDONNX_HIP_NO_UPADD") || getenv("SIMDONNX_HIP_IGEMM")) return;
    auto& P = g.plan;
    const int nn = (int)P.nodes.size();
    auto overlaps = [&](int a, int b) {
        const auto ra = value_range(P, a), rb = value_range(P, b);
        return ra.first < rb.second && rb.first < ra.second;
    };
    for (int ri = 0; ri < nn; ri++) {
        const PlanNode& r = P.nodes[ri];
        if (r.op != SOX_OP_RESIZE_NEAREST || g.folded.count(ri) || r.in.size() != 2 || r.out.size() != 1) continue;
        const auto& rp = r.p<sox_resize_nearest_p>();
        if (rp.add_relu) continue;
        const int u = r.in[0], a = r.in[1], o = r.out[0];
        const PlanValue &uv = P.values[u], &av = P.values[a], &ov = P.values[o];
        if (uv.buf < 0 || av.buf < 0 || ov.buf < 0 || a == P.output || a == u || value_reads(g, a) != 1) continue;
        if (g.padded_ld.count(u) || g.padded_ld.count(a) || g.padded_ld.count(o)) continue;
        const std::vector<int> us = uv.phys(), as = av.phys(), os = ov.phys();
        if (us.size() != 4 || as != os || us[0] != os[0] || us[3] != os[3]) continue;
        const int rank = (int)ov.shape.size();
        const float f = rp.scales[rank - 1];
        int k = 1;
        while (k < 5 && (float)(1 << k) != f) k++;
        if (k >= 5 || rp.scales[rank - 2] != f || (us[1] << k) != os[1] || (us[2] << k) != os[2]) continue;
        int li = -1;
        for (int j = ri - 1; j >= 0 && li < 0; j--)
            if (!g.folded.count(j) && !P.nodes[j].out.empty() && P.nodes[j].out[0] == a) li = j;
        if (li < 0 || g.moved.count(li) || g.upcat.count(li)) continue;
        const PlanNode& L = P.nodes[li];
        if (L.op != SOX_OP_CONV || L.out.size() != 1) continue;
        const sox_conv_p lp = L.p<sox_conv_p>();
        if (lp.group != 1 || lp.kernel[0] != 1 || lp.kernel[1] != 1 || lp.strides[0] != 1 || lp.strides[1] != 1 ||
            lp.dilations[0] != 1 || lp.dilations[1] != 1 || lp.pads[0] || lp.pads[1] || lp.pads[2] || lp.pads[3] ||
            lp.has_pool || lp.act != 0 || lp.add_value >= 0)
            continue;
        const PlanValue& wv = P.values[L.in[1]];
        const std::vector<int> xs = P.values[L.in[0]].phys();
        // the LDS-DMA ring route of the conv emitter: ic % 8 == 0, at least 8 output channels
        if (!wv.is_const || wv.shape.size() != 4 || wv.shape[0] < 8 || xs.size() != 4 || xs[3] % 8 != 0) continue;
        const int x = L.in[0];
        std::vector<int> move;
        for (int j = li + 1; j < ri; j++)
            for (int w : emitted_writes(g, j))
                if (P.values[w].buf >= 0 && overlaps(w, x)) move.push_back(w);
        for (int w : move)
            if (overlaps(w, x)) relocate_value(P, w);  // (a view of an earlier w has moved with it)
        if (overlaps(o, x) || overlaps(o, u)) relocate_value(P, o);
        g.upadd[ri] = {li, k};
        g.moved.insert(li);
    }
}

// Rows that are not whole 16-byte chunks (channels, or a Gemm's K, no multiple of 8; fp32: of 4) cannot take the
// LDS-DMA kernels: padded with zeros into scratch first, they can, for one pass over the input. Against the
// implicit GEMM's element gather, fp16 / fp32: Gemm 4096 x 1023 -> 2000 172 -> 37 / 350 -> 218 us, 256 x 1001 -> 97
// 73 -> 13.6 / 41 -> 12.2, 64 x 65 -> 64 10.2 -> 5.3 / 6.6 -> 5.7; conv 4x128x128 65 -> 129 3x3 190 -> 90 / 309 -> 245,
// 1x20x20 250 -> 250 3x3 (fp32 251) 156 -> 22 / 89 -> 21, 1x32x32 33 -> 64 3x3 27 -> 8.9 / 15 -> 8.2. Not where few
// channels are mostly padding (the ring multiplies whole 32- or 16-channel slices of every tap: 1x224x224 3 -> 64
// 7x7 16.4 us, 20.5 padded; fp32 1x480x480 5 -> 9 3x3 50 / 67), nor a short fp32 K (5000 x 30 -> 90 7.2 / 7.6),
// nor where the copy would grow the arena by more than kPadBytes. SIMDONNX_HIP_NO_PAD_ROWS leaves every such row
// to the implicit GEMM, for an arena without the copies.
constexpr int64_t kPadBytes = 1ll << 30;
bool pads_rows(const sox_graph& g, int64_t rows, int c, int64_t n, int taps) {
    const int ld = g.f16 ? 8 : 4;
    return c % ld != 0 && c >= (taps > 1 ? 9 : g.f16 ? 16 : 32) && !getenv("SIMDONNX_HIP_IGEMM") &&
           !getenv("SIMDONNX_HIP_NO_PAD_ROWS") &&
           rows * round_up(c, ld) * (g.f16 ? 2 : 4) <= kPadBytes && n * pad8(taps * round_up(c, ld)) < ((int64_t)1 << 31);
}
bool gemm_pads_k(const sox_graph& g, int64_t m, int n, int k) { return pads_rows(g, m, k, n, 1); }
bool conv_pads_channels(const sox_graph& g, const PlanNode& n) {
    const auto& p = n.p<sox_conv_p>();
    const int ld = g.f16 ? 8 : 4;
    const PlanValue& wv = g.V(n.in[1]);
    const std::vector<int> xs = g.V(n.in[0]).phys(), ys = g.V(n.out[0]).phys();
    if (p.group != 1 || p.has_pool || xs.size() != 4 || ys.size() != 4 || wv.shape.size() != 4) return false;
    sox_igemm_args a{};
    a.kh = p.kernel[0]; a.kw = p.kernel[1]; a.sh = p.strides[0]; a.sw = p.strides[1]; a.pt = p.pads[0]; a.pl = p.pads[1];
    a.ih = xs[1]; a.iw = xs[2]; a.oh = ys[1]; a.ow = ys[2];
    const int oc = wv.shape[0], ic = xs[3], taps = a.kh * a.kw;
    if (oc % ld == 0 && taps * ic <= 64 && oc <= 128) return false;  // the direct convs read such rows themselves
    if (p.pad_mode == 0 ? p.pad_value != 0.0f : !Emitter::reflect_folds_once(a)) return false;
    // what the ring's packed origins hold
    if (a.ih > 30000 || a.iw > 30000 || *std::max_element(p.pads, p.pads + 4) > 2000) return false;
    return pads_rows(g, (int64_t)xs[0] * a.ih * a.iw, ic, oc, taps);
}

// Const kinds each node's dispatches bind (the per-consumer packing, VkGraph.cs:81-143).
void collect_consts(sox_graph& g, std::vector<std::pair<int, int>>& need) {
    auto want = [&](int v, int k) {
        if (v < 0 || !g.V(v).is_const) return;
        if (std::find(need.begin(), need.end(), std::make_pair(v, k)) == need.end()) need.emplace_back(v, k);
    };
    for (int ni = 0; ni < (int)g.plan.nodes.size(); ni++) {
        if (g.folded.count(ni)) continue;
        const PlanNode& n = g.plan.nodes[ni];
        switch (n.op) {
            case SOX_OP_CONV: {
                const auto& p = n.p<sox_conv_p>();
                want(n.in[0], SOX_CK_RAW);
                want(n.in[1], p.group > 1 ? SOX_CK_DWW
                              : p.kernel[0] * p.kernel[1] > 1 && conv_pads_channels(g, n) ? (g.f16 ? CK_CONVWT_P8 : CK_CONVWT_P4)
                                                                                          : SOX_CK_CONVWT);
                want(p.bias_value, SOX_CK_F32);
                want(p.add_value, SOX_CK_RAW);
                break;
            }
            case SOX_OP_GEMM: {
                const auto& p = n.p<sox_gemm_p>();
                want(n.in[0], SOX_CK_RAW);
                want(n.in[1], p.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK);
                want(p.bias_value, SOX_CK_F32);
                auto lf = g.ln_fold.find(ni);
                if (lf != g.ln_fold.end()) want(lf->second.colsum, SOX_CK_F32);
                auto mf = g.mlp.find(ni);
                if (mf != g.mlp.end()) {  // both weights in fragment order, the second Gemm's bias
                    const PlanNode& n2 = g.plan.nodes[mf->second.fc2];
                    want(n.in[1], CK_FRAG32);
                    want(n2.in[1], CK_FRAG32);
                    want(n2.p<sox_gemm_p>().bias_value, SOX_CK_F32);
                    if (mf->second.proj >= 0) {  // the projection Gemm folded into it
                        const PlanNode& np = g.plan.nodes[mf->second.proj];
                        const auto& pp = np.p<sox_gemm_p>();
                        want(np.in[1], pp.trans_b ? CK_GEMMNK_T : SOX_CK_GEMMNK);
                        want(pp.bias_value, SOX_CK_F32);
                    }
                }
                break;
            }
            case SOX_OP_LAYERNORM:
                want(n.in[0], SOX_CK_RAW);
                want(n.in[1], SOX_CK_F32);
                want(n.in[2], SOX_CK_F32);
                break;
            case SOX_OP_CONV_TRANSPOSE: {
                const auto& p = n.p<sox_convt_p>();
                want(n.in[1], convt_as_gemm(g, n) ? CK_CONVT_NK : SOX_CK_CONVTW);
                want(p.bias_value, SOX_CK_F32);
                auto ch = g.convt_chain.find(ni);
                if (ch != g.convt_chain.end()) {  // the second ConvT run in the same kernel
                    const PlanNode& n2 = g.plan.nodes[ch->second];
                    want(n2.in[1], SOX_CK_CONVTW);
                    want(n2.p<sox_convt_p>().bias_value, SOX_CK_F32);
                }
                break;
            }
            case SOX_OP_CHANNEL_GATE: {
                const auto& p = n.p<sox_channel_gate_p>();
                want(n.in[1], SOX_CK_F32);
                want(n.in[2], SOX_CK_F32);
                want(p.b1, SOX_CK_F32);
                want(p.b2, SOX_CK_F32);
                break;
            }
            case SOX_OP_ELEMENTWISE: {
                // scalar consts fold into the affine pass; other consts bind raw
                for (int v : n.in)
                    if (g.V(v).is_const && g.V(v).floats.size() != 1) want(v, SOX_CK_RAW);
                break;
            }
            case SOX_OP_EXT: {
                auto it = g.be->exts.find(n.ext);
                if (it == g.be->exts.end()) {  // built-ins: their GpuConsts (UpHeadOp.cs:67-77)
                    if (n.ext == "UpHead" && n.params.size() >= sizeof(sox_uphead_p)) {
                        const auto& p = n.p<sox_uphead_p>();
                        want(n.in[2], SOX_CK_RAW);
                        if (n.in.size() > 3) want(n.in[3], SOX_CK_F32);
                        if (p.has_skip_conv) {
                            want(p.skip_w, SOX_CK_RAW);
                            want(p.skip_b, SOX_CK_F32);
                        }
                    } else {
                        for (int v : n.in) want(v, SOX_CK_RAW);
                    }
                    break;
                }
                if (it->second.consts) {
                    int32_t vals[64], kinds[64];
                    int cnt = it->second.consts(it->second.user, &g.plan, ni, vals, kinds, 64);
                    for (int i = 0; i < cnt; i++) want(vals[i], kinds[i]);
                }
                break;
            }
            default:
                for (int v : n.in) want(v, SOX_CK_RAW);
        }
    }
}

void upload_consts(sox_graph& g) {
    std::vector<std::pair<int, int>> need;
    collect_consts(g, need);
    uint64_t total = 0;
    std::vector<uint64_t> offs(need.size()), bytes(need.size());
    for (size_t i = 0; i < need.size(); i++) {
        const PlanValue& v = g.V(need[i].first);
        int64_t n = packed_elems(v, need[i].second);
        total = (total + 63) & ~63ull;
        offs[i] = total;
        bytes[i] = (uint64_t)n * (g.elem_fp32(need[i].second) ? 4 : 2);
        total += bytes[i];
        g.const_off[need[i]] = {offs[i], bytes[i]};
    }
    total = std::max<uint64_t>((total + 255) & ~255ull, 256);
    std::vector<uint8_t> host(total, 0);
    std::vector<float> tmp;
    for (size_t i = 0; i < need.size(); i++) {
        const PlanValue& v = g.V(need[i].first);
        int64_t n = packed_elems(v, need[i].second);
        tmp.assign((size_t)n, 0.0f);
        pack_const(v, need[i].second, tmp.data());
        if (g.elem_fp32(need[i].second)) {
            memcpy(host.data() + offs[i], tmp.data(), (size_t)n * 4);
        } else {
            uint16_t* d = reinterpret_cast<uint16_t*>(host.data() + offs[i]);
            g.bits16(tmp.data(), d, n);
        }
    }
    g.const_bytes = total;
    if (g.be->offline) return;  // packed and checked; nothing to upload to
    check(sox_malloc(&g.consts, total), "const store");
    check(sox_memcpy_h2d(g.consts, host.data(), total, nullptr), "const upload");
    check(sox_stream_sync(nullptr), "const upload");
}

}  // namespace

// ================================================================================================
// Session
// ================================================================================================
namespace {

// True when a rocprofiler-sdk tool (rocprofv3) is loaded into this process. Replaying a captured HIP
// graph under its kernel tracer has ended in a host segmentation fault inside hipGraphLaunch, for a
// cause not yet shown, so sessions launch their dispatches directly while such a tool is present.
// (The SDK is loaded only for a registered tool; the HIP runtime itself maps rocprofiler-register.)
bool profiler_tool_loaded() {
    static const bool loaded = [] {
        FILE* f = fopen("/proc/self/maps", "r");
        if (!f) return false;
        char line[4096];
        bool found = false;
        while (!found && fgets(line, sizeof line, f)) found = strstr(line, "librocprofiler-sdk") != nullptr;
        fclose(f);
        return found;
    }();
    return loaded;
}

// The kernels that move a graph's fp32 host windows (pinned and mapped: the device reads and writes them in
// place) to and from the arena in its storage type (staging.hip).
struct Staging {
    void *in = nullptr, *out = nullptr;  // sox_stage_in_*, sox_stage_out_*
    void* cvt = nullptr;                 // 16-bit -> fp32 on the device, in front of a copy-engine download

    // Downloads above this go through the copy engine: 30 MB take 556 us from the kernel and 557 with the
    // conversion and the copy, 70 MB 1288 and ~1265.
    static constexpr int64_t kEngineBytes = 32ll << 20;
    static bool engine(int64_t out_count) { return out_count * 4 > kEngineBytes; }
    // fp32 device staging a graph needs: only the 16-bit outputs that the copy engine fetches
    static int64_t stage_floats(const sox_graph& g, int64_t out_count) { return g.f16 && engine(out_count) ? out_count : 0; }

    void bind(const sox_graph& g) {
        const std::string ty = g.bf16 ? "bf16" : g.f16 ? "f16" : "f32";
        in = g.be->fn("sox_stage_in_" + ty);
        out = g.be->fn("sox_stage_out_" + ty);
        if (g.f16) cvt = g.be->fn("sox_" + ty + "_to_f32");
    }
    static void launch(void* fn, const void* x, void* y, int64_t count, int64_t blocks, void* stream) {
        if (count <= 0) return;
        sox_cvt_args a{x, y, count};
        const uint32_t grid[3] = {(uint32_t)blocks, 1, 1}, block[3] = {256, 1, 1};
        check(sox_launch(fn, grid, block, 0, stream, &a, sizeof a), "staging");
    }
    void upload(const float* host, void* dst, int64_t count, void* stream) const {
        launch(in, host, dst, count, std::min<int64_t>(64, (count + 2047) / 2048), stream);
    }
    void download(const void* src, float* host, int64_t count, void* stage, bool f16, void* stream) const {
        if (!engine(count)) {
            launch(out, src, host, count, std::min<int64_t>(256, (count + 4095) / 4096), stream);
            return;
        }
        if (f16) {
            launch(cvt, src, stage, count, count / 1024 + 1, stream);
            src = stage;
        }
        check(sox_memcpy_d2h(host, src, (size_t)count * 4, stream), "output download");
    }
};

}  // namespace

// Device buffers shared by the sessions of one owner that run one at a time (VkBufferPool /
// VkSessionBuffers, Backends/Vulkan/VkBatch.cs:6-25, VkSession.cs:10-55): the arena slab, the device
// fp32 staging of large 16-bit outputs and the pinned fp32 input / output staging. They grow to the
// largest session (by half again each time, as Ensure); growing replaces a buffer and bumps the
// generation, which makes the sessions created before it stale. The borrowing sessions enqueue on the
// pool's one stream, so their runs never overlap on the device.
struct sox_buffer_pool {
    sox_backend* be = nullptr;
    void* stream = nullptr;
    void* arena = nullptr;
    void* stage = nullptr;
    float* in_host = nullptr;
    float* out_host = nullptr;
    uint64_t arena_bytes = 0, stage_bytes = 0, in_bytes = 0, out_bytes = 0;
    int generation = 0;
    int borrowers = 0;      // sessions created on the pool and not yet destroyed
    bool released = false;  // sox_buffer_pool_destroy was called: freed with its last borrower

    static uint64_t grown(uint64_t need, uint64_t have) { return std::max(need, have + have / 2); }

    void ensure(uint64_t arena_need, uint64_t stage_need, uint64_t in_need, uint64_t out_need) {
        const bool grow = arena_need > arena_bytes || stage_need > stage_bytes || in_need > in_bytes ||
                          out_need > out_bytes;
        if (!grow) return;
        check(sox_stream_sync(stream), "buffer pool");  // earlier sessions' work is done with the old buffers
        if (arena_need > arena_bytes) {
            check(sox_free(arena), "buffer pool");
            arena = nullptr;
            arena_bytes = grown(arena_need, arena_bytes);
            check(sox_malloc(&arena, arena_bytes), "buffer pool arena");
        }
        if (stage_need > stage_bytes) {
            check(sox_free(stage), "buffer pool");
            stage = nullptr;
            stage_bytes = grown(stage_need, stage_bytes);
            check(sox_malloc(&stage, stage_bytes), "buffer pool device staging");
        }
        if (in_need > in_bytes) {
            check(sox_host_free(in_host), "buffer pool");
            in_host = nullptr;
            in_bytes = grown(in_need, in_bytes);
            check(sox_host_alloc((void**)&in_host, in_bytes), "buffer pool input staging");
            memset(in_host, 0, in_bytes);
        }
        if (out_need > out_bytes) {
            check(sox_host_free(out_host), "buffer pool");
            out_host = nullptr;
            out_bytes = grown(out_need, out_bytes);
            check(sox_host_alloc((void**)&out_host, out_bytes), "buffer pool output staging");
        }
        generation++;
    }

    void free_all() {
        if (stream) sox_stream_sync(stream);
        sox_free(arena);
        sox_free(stage);
        sox_host_free(in_host);
        sox_host_free(out_host);
        if (stream) sox_stream_destroy(stream);
        arena = stage = stream = nullptr;
        in_host = out_host = nullptr;
    }
};

struct sox_session {
    sox_graph* g = nullptr;
    void* stream = nullptr;
    void* arena = nullptr;
    sox_buffer_pool* pool = nullptr;  // the borrowed buffers (stream included), or null: its own
    int pool_gen = 0;

    bool stale() const { return pool && pool->generation != pool_gen; }
    // VkInferenceSession.Run on a session whose pool grew after it was made (VkSession.cs:178-180)
    void current() const {
        if (stale())
            fail(SOX_E_INVALID, "session is stale: a larger session on its buffer pool regrew the shared "
                                "buffers; create it again");
    }
    std::vector<float*> in_host;
    std::vector<int64_t> in_count;
    float* out_host = nullptr;
    int64_t out_count = 0;
    void* stage = nullptr;  // device fp32 staging of a 16-bit output that the copy engine fetches, or null
    void* sync = nullptr;   // the graph's cross-workgroup counters: this session's own, also on a pool
    std::vector<std::vector<uint8_t>> kernargs;
    Staging staging;
    bool replay = false;
    void* exec_full = nullptr;
    void* exec_disp = nullptr;

    void* resolve(const sox_bind& b) const {
        switch (b.slot) {
            case SOX_SLOT_ARENA: return (uint8_t*)arena + b.offset;
            case SOX_SLOT_CONSTS: return (uint8_t*)g->consts + b.offset;
            case SOX_SLOT_SYNC: return (uint8_t*)sync + b.offset;
            default: return g->be->dummy;
        }
    }

    void* value_ptr(int v) const {
        current();
        const PlanValue& pv = g->V(v);
        if (pv.buf < 0) fail(SOX_E_INVALID, "value is not an activation");
        return (uint8_t*)arena + (uint64_t)g->plan.buf_offset[pv.buf] * g->es;
    }

    void stage_in() {
        for (size_t i = 0; i < g->plan.inputs.size(); i++)
            staging.upload(in_host[i], value_ptr(g->plan.inputs[i]), in_count[i], stream);
    }

    void stage_out() { staging.download(value_ptr(g->plan.output), out_host, out_count, stage, g->f16, stream); }

    void dispatch(size_t i) {
        current();
        const Dispatch& d = g->disp[i];
        check(sox_launch(d.fn, d.grid, d.block, d.lds, stream, kernargs[i].data(), kernargs[i].size()), d.name.c_str());
    }

    void enqueue_direct(int flags) {
        if (flags & SOX_RUN_STAGING) stage_in();
        if (flags & SOX_RUN_DISPATCHES)
            for (size_t i = 0; i < g->disp.size(); i++) dispatch(i);
        if (flags & SOX_RUN_STAGING) stage_out();
    }

    void enqueue(int flags) {
        current();
        if (!replay) {
            enqueue_direct(flags);
            return;
        }
        bool full = (flags & SOX_RUN_STAGING) != 0;
        void*& ex = full ? exec_full : exec_disp;
        if (!ex) {
            check(sox_graph_begin(stream), "capture begin");
            try {
                enqueue_direct(full ? (SOX_RUN_STAGING | SOX_RUN_DISPATCHES) : SOX_RUN_DISPATCHES);
            } catch (...) {
                void* dummy = nullptr;
                sox_graph_end(stream, &dummy);
                sox_graph_destroy(dummy);
                throw;
            }
            check(sox_graph_end(stream, &ex), "capture end");
        }
        check(sox_graph_launch(ex, stream), "graph launch");
    }
};

// ================================================================================================
// C ABI
// ================================================================================================
extern "C" {

const char* sox_last_error(void) { return g_err.c_str(); }

int sox_plan_create(sox_plan** plan) {
    if (!plan) return SOX_E_INVALID;
    *plan = new sox_plan();
    return SOX_OK;
}

void sox_plan_destroy(sox_plan* plan) { delete plan; }

int sox_plan_add_value(sox_plan* plan, const int32_t* shape, int32_t rank, const int32_t* layout, int32_t buf,
                       const float* floats, int64_t nfloats, const char* name, int32_t* id) {
    return guarded([&] {
        if (!plan || rank < 0 || rank > 8) fail(SOX_E_INVALID, "bad value");
        PlanValue v;
        v.shape.assign(shape, shape + rank);
        if (layout) {
            v.layout.assign(layout, layout + rank);
            bool ident = true;
            for (int i = 0; i < rank; i++) ident &= layout[i] == i;
            if (ident) v.layout.clear();
        }
        v.buf = buf;
        if (buf < 0) {
            v.is_const = true;
            if (!floats || nfloats != v.count()) fail(SOX_E_INVALID, "const value needs its data");
            v.floats.assign(floats, floats + nfloats);
        }
        v.name = name ? name : "";
        plan->values.push_back(std::move(v));
        if (id) *id = (int32_t)plan->values.size() - 1;
    });
}

int sox_plan_add_node(sox_plan* plan, int32_t op, const int32_t* in, int32_t nin, const int32_t* out, int32_t nout,
                      const void* params, size_t params_bytes, const char* ext_name, int32_t* id) {
    return guarded([&] {
        if (!plan || nin < 0 || nout < 1) fail(SOX_E_INVALID, "bad node");
        PlanNode n;
        n.op = op;
        n.in.assign(in, in + nin);
        n.out.assign(out, out + nout);
        if (params && params_bytes) n.params.assign((const uint8_t*)params, (const uint8_t*)params + params_bytes);
        n.ext = ext_name ? ext_name : "";
        plan->nodes.push_back(std::move(n));
        if (id) *id = (int32_t)plan->nodes.size() - 1;
    });
}

int sox_plan_set_arena(sox_plan* plan, const int64_t* buf_offset, int32_t nbuf, int64_t arena_floats) {
    if (!plan || nbuf < 0) return SOX_E_INVALID;
    plan->buf_offset.assign(buf_offset, buf_offset + nbuf);
    plan->arena_floats = arena_floats;
    return SOX_OK;
}

int sox_plan_set_io(sox_plan* plan, const int32_t* inputs, int32_t ninputs, int32_t output) {
    if (!plan || ninputs < 1) return SOX_E_INVALID;
    plan->inputs.assign(inputs, inputs + ninputs);
    plan->output = output;
    return SOX_OK;
}

int sox_backend_default(sox_backend** backend) {
    return guarded([&] {
        std::lock_guard<std::mutex> lk(g_default_mu);
        if (g_default && !g_default->lost && !sox_device_lost()) {
            *backend = g_default;
            return;
        }
        if (g_default) {
            // abandon the lost device's objects (VkBackend.cs:21-47) and start over
            g_default->lost = true;
            g_default = nullptr;
            sox_device_reset_lost();
        }
        auto be = std::make_unique<sox_backend>();
        check(sox_init(0, &be->info), "device init");
        for (const SoxResource* r = sox_resources; r->name; r++) {
            void* m = nullptr;
            check(sox_module_load(&m, r->start, (size_t)(r->end - r->start)), r->name);
            be->modules.push_back(m);
        }
        check(sox_scratch(be->info.device, &be->scratch, &be->scratch_bytes), "device scratch");
        check(sox_event_create(&be->scratch_ev), "device scratch event");
        check(sox_malloc(&be->dummy, 256), "dummy buffer");
        std::vector<uint8_t> zero(256, 0);
        check(sox_memcpy_h2d(be->dummy, zero.data(), 256, nullptr), "dummy buffer");
        check(sox_stream_sync(nullptr), "dummy buffer");
        g_default = be.release();
        *backend = g_default;
    });
}

int sox_backend_create_offline(const sox_device_info* info, sox_backend** backend) {
    return guarded([&] {
        if (!backend) fail(SOX_E_INVALID, "no output");
        auto be = std::make_unique<sox_backend>();
        be->offline = true;
        if (info) {
            be->info = *info;
        } else {  // an MI355X: 256 CUs in 8 XCDs, 160 KiB LDS per CU, 288 GB HBM3E
            snprintf(be->info.name, sizeof be->info.name, "%s", "offline (no device)");
            snprintf(be->info.arch, sizeof be->info.arch, "%s", "gfx950");
            be->info.compute_units = 256;
            be->info.lds_per_cu = 160 * 1024;
            be->info.clock_khz = 2400000;
            be->info.warp_size = 64;
            be->info.vendor_id = 0x1002;
            be->info.hbm_bytes = 288ull << 30;
            be->info.xcds = 8;
        }
        be->info.device = -1;
        *backend = be.release();
    });
}

void sox_backend_destroy(sox_backend* backend) {
    if (backend && backend->offline) delete backend;  // (the device backend lives for the process)
}

int sox_backend_info(sox_backend* backend, sox_device_info* info) {
    if (!backend || !info) return SOX_E_INVALID;
    *info = backend->info;
    return SOX_OK;
}

int sox_backend_is_lost(sox_backend* backend) { return backend && (backend->lost || sox_device_lost()) ? 1 : 0; }

int sox_backend_load_module(sox_backend* backend, const void* image, size_t bytes, void** module) {
    return guarded([&] {
        if (!backend) fail(SOX_E_INVALID, "no backend");
        backend->need_device("extension code object");
        check(sox_module_load(module, image, bytes), "extension code object");
        std::lock_guard<std::mutex> lk(backend->mu);
        backend->modules.push_back(*module);
    });
}

int sox_backend_register_ext(sox_backend* backend, const char* name, sox_ext_emit_fn emit, sox_ext_consts_fn consts,
                             void* user) {
    if (!backend || !name || !emit) return SOX_E_INVALID;
    std::lock_guard<std::mutex> lk(backend->mu);
    backend->exts[name] = ExtEntry{emit, consts, user};
    return SOX_OK;
}

int sox_graph_bind(sox_graph* graph, int32_t value, int32_t const_kind, sox_bind* out) {
    return guarded([&] {
        Emitter e(*graph);
        *out = e.bind(value, const_kind);
    });
}

int sox_graph_scratch(sox_graph* graph, uint64_t bytes, sox_bind* out) {
    return guarded([&] {
        Emitter e(*graph);
        *out = e.scratch(bytes);
    });
}

int sox_graph_dispatch(sox_graph* graph, int32_t node, void* module, const char* kernel, const sox_bind* binds,
                       int32_t nbinds, const void* params, size_t params_bytes, const uint32_t grid[3],
                       const uint32_t block[3], uint32_t lds_bytes) {
    return guarded([&] {
        Dispatch d;
        if (module) {
            if (sox_module_function(&d.fn, module, kernel) != SOX_OK)
                fail(SOX_E_NOT_FOUND, std::string("extension kernel ") + kernel + " not found");
        } else {
            d.fn = graph->be->fn(kernel);
        }
        d.name = kernel;
        d.kernel = kernel;
        d.node = node;
        for (int i = 0; i < 3; i++) {
            d.grid[i] = grid[i];
            d.block[i] = block[i];
        }
        d.lds = lds_bytes;
        d.kernarg.assign((size_t)nbinds * 8 + params_bytes, 0);
        for (int i = 0; i < nbinds; i++) d.patches.push_back(Patch{(uint32_t)(i * 8), binds[i]});
        if (params_bytes) memcpy(d.kernarg.data() + nbinds * 8, params, params_bytes);
        graph->disp.push_back(std::move(d));
    });
}

int sox_graph_node_info(sox_graph* graph, int32_t node, int32_t* op, const void** params, size_t* params_bytes) {
    if (!graph || node < 0 || node >= (int)graph->plan.nodes.size()) return SOX_E_INVALID;
    const PlanNode& n = graph->plan.nodes[node];
    if (op) *op = n.op;
    if (params) *params = n.params.data();
    if (params_bytes) *params_bytes = n.params.size();
    return SOX_OK;
}

int sox_graph_node_values(sox_graph* graph, int32_t node, int32_t* in, int32_t in_cap, int32_t* nin, int32_t* out,
                          int32_t out_cap, int32_t* nout) {
    if (!graph || node < 0 || node >= (int)graph->plan.nodes.size()) return SOX_E_INVALID;
    const PlanNode& n = graph->plan.nodes[node];
    for (int i = 0; i < (int)n.in.size() && i < in_cap; i++) in[i] = n.in[i];
    for (int i = 0; i < (int)n.out.size() && i < out_cap; i++) out[i] = n.out[i];
    if (nin) *nin = (int32_t)n.in.size();
    if (nout) *nout = (int32_t)n.out.size();
    return SOX_OK;
}

int sox_graph_value_shape(sox_graph* graph, int32_t value, int32_t* phys_shape, int32_t cap, int32_t* rank) {
    if (!graph || value < 0 || value >= (int)graph->plan.values.size()) return SOX_E_INVALID;
    std::vector<int> p = graph->plan.values[value].phys();
    if (rank) *rank = (int32_t)p.size();
    for (int i = 0; i < (int)p.size() && i < cap; i++) phys_shape[i] = p[i];
    return SOX_OK;
}

int sox_graph_is_f16(sox_graph* graph) {
    return !graph ? 0 : graph->bf16 ? SOX_STORAGE_BF16 : graph->f16 ? SOX_STORAGE_F16 : SOX_STORAGE_F32;
}

int sox_graph_create(sox_backend* backend, const sox_plan* plan, int32_t f16, sox_graph** graph) {
    sox_graph* g = new sox_graph();
    int rc = guarded([&] {
        if (!backend || !plan) fail(SOX_E_INVALID, "no backend / plan");
        if (backend->lost || sox_device_lost()) fail(SOX_E_LOST, "device lost");
        g->be = backend;
        g->plan = *plan;
        if (f16 < SOX_STORAGE_F32 || f16 > SOX_STORAGE_BF16) fail(SOX_E_INVALID, "storage mode");
        g->f16 = f16 != SOX_STORAGE_F32;
        g->bf16 = f16 == SOX_STORAGE_BF16;
        g->es = g->f16 ? 2 : 4;
        if (g->plan.inputs.empty() || g->plan.output < 0) fail(SOX_E_INVALID, "plan has no inputs/output");
        for (int v : g->plan.inputs)
            if (g->V(v).buf < 0) fail(SOX_E_INVALID, "graph input is not an activation");
        if (g->V(g->plan.output).buf < 0) fail(SOX_E_INVALID, "graph output is not an activation");
        fold_affine_after_convt(*g);
        plan_convt_chain(*g);
        plan_padded_rows(*g);
        fold_layernorm_into_gemm(*g);
        plan_residual_adds(*g);
        plan_fused_mlp(*g);
        plan_fused_attention(*g);
        plan_fused_proj(*g);
        plan_upsample_concat(*g);
        plan_upsample_add(*g);
        plan_se_fold_space(*g);
        // activations occupy [0, arena_floats*es); scratch follows, 256-byte aligned (VkGraph.cs:145)
        g->scratch_off = ((uint64_t)g->plan.arena_floats * g->es + 255) & ~255ull;
        for (const PlanValue& v : g->plan.values)
            if (v.buf >= 0)
                g->tail_bytes = std::max<uint64_t>(g->tail_bytes, ((uint64_t)g->plan.buf_offset.at(v.buf) + v.count()) * g->es);
        upload_consts(*g);
        Emitter e(*g);
        for (int i = 0; i < (int)g->plan.nodes.size(); i++) e.emit(i);
    });
    if (rc != SOX_OK) {
        if (g->consts) sox_free(g->consts);
        delete g;
        *graph = nullptr;
        return rc;
    }
    *graph = g;
    return SOX_OK;
}

void sox_graph_release(sox_graph* graph) {
    if (!graph) return;
    if (--graph->refs > 0) return;
    if (graph->consts) sox_free(graph->consts);
    delete graph;
}

int sox_graph_dispatch_count(sox_graph* graph) { return graph ? (int)graph->disp.size() : 0; }

int sox_graph_dispatch_info(sox_graph* graph, int32_t index, char* name, size_t name_cap, uint32_t grid[3], int32_t* node) {
    if (!graph || index < 0 || index >= (int)graph->disp.size()) return SOX_E_INVALID;
    const Dispatch& d = graph->disp[index];
    if (name && name_cap) snprintf(name, name_cap, "%s", d.name.c_str());
    if (grid)
        for (int i = 0; i < 3; i++) grid[i] = d.grid[i];
    if (node) *node = d.node;
    return SOX_OK;
}

int sox_graph_dispatch_kernel(sox_graph* graph, int32_t index, char* kernel, size_t kernel_cap) {
    if (!graph || index < 0 || index >= (int)graph->disp.size() || !kernel || !kernel_cap) return SOX_E_INVALID;
    snprintf(kernel, kernel_cap, "%s", graph->disp[index].kernel.c_str());
    return SOX_OK;
}

int sox_graph_dispatch_binds(sox_graph* graph, int32_t index, sox_bind* binds, int32_t cap, int32_t* n) {
    if (!graph || index < 0 || index >= (int)graph->disp.size() || (cap > 0 && !binds)) return SOX_E_INVALID;
    const Dispatch& d = graph->disp[index];
    for (int i = 0; i < (int)d.patches.size() && i < cap; i++) binds[i] = d.patches[i].bind;
    if (n) *n = (int32_t)d.patches.size();
    return SOX_OK;
}

int sox_graph_value_place(sox_graph* graph, int32_t value, uint64_t* offset, uint64_t* bytes) {
    return guarded([&] {
        if (!graph) fail(SOX_E_INVALID, "no graph");
        const PlanValue& pv = graph->V(value);
        if (pv.buf < 0) fail(SOX_E_INVALID, "value '" + pv.name + "' is not an activation");
        if (offset) *offset = (uint64_t)graph->plan.buf_offset.at(pv.buf) * graph->es;
        if (bytes) *bytes = (uint64_t)std::max<int64_t>(pv.count(), 1) * graph->es;
    });
}

uint64_t sox_graph_arena_bytes(sox_graph* graph) { return graph ? graph->arena_bytes() : 0; }
uint64_t sox_graph_const_bytes(sox_graph* graph) { return graph ? graph->const_bytes : 0; }
uint64_t sox_graph_sync_bytes(sox_graph* graph) { return graph ? graph->sync_bytes : 0; }

}  // extern "C"

namespace {

// NewSession (VkSession.cs:83-115): with a pool the session borrows its buffers (Ensure grows them to
// this graph's needs), else it allocates its own slab, staging and stream.
int session_create(sox_graph* graph, sox_buffer_pool* pool, sox_session** session) {
    if (!session) return SOX_E_INVALID;
    sox_session* s = new sox_session();
    int rc = guarded([&] {
        if (!graph) fail(SOX_E_INVALID, "no graph");
        graph->be->need_device("session");
        if (pool && pool->released) fail(SOX_E_INVALID, "buffer pool was destroyed");
        if (pool && pool->be != graph->be) fail(SOX_E_INVALID, "buffer pool of another backend");
        s->g = graph;
        graph->refs++;
        int64_t in_total = 0;
        std::vector<int64_t> in_off;
        for (int v : graph->plan.inputs) {
            const int64_t n = graph->V(v).count();
            in_off.push_back(in_total);
            in_total += (n + 15) & ~15ll;  // each input 64-byte aligned in the shared staging
            s->in_count.push_back(n);
        }
        s->out_count = graph->V(graph->plan.output).count();
        const int64_t stage = Staging::stage_floats(*graph, s->out_count);
        if (pool) {
            pool->ensure(graph->arena_bytes(), (uint64_t)stage * 4, (uint64_t)in_total * 4, (uint64_t)s->out_count * 4);
            s->pool = pool;
            pool->borrowers++;
            s->pool_gen = pool->generation;
            s->stream = pool->stream;
            s->arena = pool->arena;
            s->stage = pool->stage;
            for (int64_t off : in_off) s->in_host.push_back(pool->in_host + off);
            s->out_host = pool->out_host;
        } else {
            check(sox_stream_create(&s->stream), "stream");
            check(sox_malloc(&s->arena, graph->arena_bytes()), "arena slab");
            for (int64_t n : s->in_count) {
                float* h = nullptr;
                check(sox_host_alloc((void**)&h, (size_t)n * 4), "input staging");
                memset(h, 0, (size_t)n * 4);
                s->in_host.push_back(h);
            }
            check(sox_host_alloc((void**)&s->out_host, (size_t)s->out_count * 4), "output staging");
            if (stage) check(sox_malloc(&s->stage, (size_t)stage * 4), "device staging");
        }
        if (graph->sync_bytes) {  // zero once: every launch leaves its counters at 0
            check(sox_malloc(&s->sync, graph->sync_bytes), "counters");
            std::vector<uint8_t> zeros(graph->sync_bytes, 0);
            check(sox_memcpy_h2d(s->sync, zeros.data(), zeros.size(), s->stream), "counters");
            check(sox_stream_sync(s->stream), "counters");
        }
        s->staging.bind(*graph);
        for (const Dispatch& d : graph->disp) {
            std::vector<uint8_t> ka = d.kernarg;
            for (const Patch& p : d.patches) {
                void* ptr = s->resolve(p.bind);
                memcpy(ka.data() + p.off, &ptr, sizeof ptr);
            }
            s->kernargs.push_back(std::move(ka));
        }
    });
    if (rc != SOX_OK) {
        sox_session_destroy(s);
        *session = nullptr;
        return rc;
    }
    *session = s;
    return SOX_OK;
}

}  // namespace

extern "C" {

int sox_session_create(sox_graph* graph, sox_session** session) { return session_create(graph, nullptr, session); }

int sox_session_create_pooled(sox_graph* graph, sox_buffer_pool* pool, sox_session** session) {
    if (!pool) return SOX_E_INVALID;
    return session_create(graph, pool, session);
}

int sox_session_is_stale(sox_session* s) { return s && s->stale() ? 1 : 0; }

int sox_buffer_pool_create(sox_backend* backend, sox_buffer_pool** pool) {
    if (!pool) return SOX_E_INVALID;
    auto p = std::make_unique<sox_buffer_pool>();
    int rc = guarded([&] {
        if (!backend) fail(SOX_E_INVALID, "no backend");
        backend->need_device("buffer pool");
        p->be = backend;
        check(sox_stream_create(&p->stream), "buffer pool stream");
    });
    if (rc != SOX_OK) {
        p->free_all();
        *pool = nullptr;
        return rc;
    }
    *pool = p.release();
    return SOX_OK;
}

void sox_buffer_pool_destroy(sox_buffer_pool* pool) {
    if (!pool || pool->released) return;
    pool->released = true;
    if (pool->borrowers == 0) {
        pool->free_all();
        delete pool;
    }
}

int sox_buffer_pool_info(sox_buffer_pool* pool, uint64_t* arena_bytes, int32_t* generation) {
    if (!pool) return SOX_E_INVALID;
    if (arena_bytes) *arena_bytes = pool->arena_bytes;
    if (generation) *generation = pool->generation;
    return SOX_OK;
}

void sox_session_destroy(sox_session* s) {
    if (!s) return;
    if (s->stream) sox_stream_sync(s->stream);
    sox_graph_destroy(s->exec_full);
    sox_graph_destroy(s->exec_disp);
    if (s->sync) sox_free(s->sync);
    if (s->pool) {  // borrowed buffers stay with the pool
        sox_buffer_pool* p = s->pool;
        if (--p->borrowers == 0 && p->released) {
            p->free_all();
            delete p;
        }
    } else {
        for (float* h : s->in_host) sox_host_free(h);
        sox_host_free(s->out_host);
        sox_free(s->stage);
        sox_free(s->arena);
        if (s->stream) sox_stream_destroy(s->stream);
    }
    if (s->g) sox_graph_release(s->g);
    delete s;
}

int sox_session_input(sox_session* s, int32_t index, float** host, int64_t* count) {
    if (!s || index < 0 || index >= (int)s->in_host.size()) return SOX_E_INVALID;
    if (s->stale()) return guarded([&] { s->current(); });
    *host = s->in_host[index];
    if (count) *count = s->in_count[index];
    return SOX_OK;
}

int sox_session_output(sox_session* s, float** host, int64_t* count) {
    if (!s) return SOX_E_INVALID;
    if (s->stale()) return guarded([&] { s->current(); });
    *host = s->out_host;
    if (count) *count = s->out_count;
    return SOX_OK;
}

int sox_session_submit(sox_session* s) {
    return guarded([&] {
        if (s->g->be->lost || sox_device_lost()) fail(SOX_E_LOST, "device lost");
        s->enqueue(SOX_RUN_STAGING | SOX_RUN_DISPATCHES);
    });
}

int sox_session_wait(sox_session* s) { return guarded([&] { check(sox_stream_sync(s->stream), "wait"); }); }

int sox_session_run(sox_session* s) {
    int rc = sox_session_submit(s);
    return rc != SOX_OK ? rc : sox_session_wait(s);
}

int sox_session_set_replay(sox_session* s, int32_t on) {
    if (!s) return SOX_E_INVALID;
    if (on && profiler_tool_loaded()) {
        static std::once_flag note;
        std::call_once(note, [] {
            fprintf(stderr, "simdonnx_amd: a rocprofiler-sdk tool is loaded; sessions launch their dispatches "
                            "directly instead of replaying a captured HIP graph\n");
        });
        on = 0;
    }
    s->replay = on != 0;
    return SOX_OK;
}

int sox_session_is_replaying(sox_session* s) { return s && s->replay ? 1 : 0; }

int sox_session_time(sox_session* s, int32_t iters, int32_t flags, float* total_ms) {
    return guarded([&] {
        void *e0 = nullptr, *e1 = nullptr;
        check(sox_event_create(&e0), "event");
        check(sox_event_create(&e1), "event");
        try {
            check(sox_event_record(e0, s->stream), "event");
            for (int i = 0; i < iters; i++) s->enqueue(flags);
            check(sox_event_record(e1, s->stream), "event");
            check(sox_event_sync(e1), "event");
            check(sox_event_elapsed_ms(total_ms, e0, e1), "event");
        } catch (...) {
            sox_event_destroy(e0);
            sox_event_destroy(e1);
            throw;
        }
        sox_event_destroy(e0);
        sox_event_destroy(e1);
    });
}

int sox_session_profile(sox_session* s, int32_t reps, float* ms, int32_t cap) {
    return guarded([&] {
        size_t n = s->g->disp.size();
        std::vector<void*> ev(n + 1, nullptr);
        for (auto& e : ev) check(sox_event_create(&e), "event");
        std::vector<float> best(n, 1e30f);
        for (int r = 0; r < std::max(reps, 1); r++) {
            check(sox_event_record(ev[0], s->stream), "event");
            for (size_t i = 0; i < n; i++) {
                s->dispatch(i);
                check(sox_event_record(ev[i + 1], s->stream), "event");
            }
            check(sox_event_sync(ev[n]), "event");
            for (size_t i = 0; i < n; i++) {
                float t = 0;
                check(sox_event_elapsed_ms(&t, ev[i], ev[i + 1]), "event");
                best[i] = std::min(best[i], t);
            }
        }
        for (auto e : ev) sox_event_destroy(e);
        for (size_t i = 0; i < n && (int)i < cap; i++) ms[i] = best[i];
    });
}

int sox_session_read_value(sox_session* s, int32_t value, float* host, int64_t count) {
    return guarded([&] {
        const PlanValue& v = s->g->V(value);
        if (count != v.count()) fail(SOX_E_INVALID, "count mismatch");
        void* src = s->value_ptr(value);
        check(sox_stream_sync(s->stream), "sync");
        if (s->g->f16) {
            std::vector<uint16_t> tmp((size_t)count);
            check(sox_memcpy_d2h(tmp.data(), src, (size_t)count * 2, s->stream), "read");
            check(sox_stream_sync(s->stream), "sync");
            for (int64_t i = 0; i < count; i++) host[i] = s->g->from16(tmp[i]);
        } else {
            check(sox_memcpy_d2h(host, src, (size_t)count * 4, s->stream), "read");
            check(sox_stream_sync(s->stream), "sync");
        }
    });
}

int sox_session_value_ptr(sox_session* s, int32_t value, void** dev) {
    return guarded([&] { *dev = s->value_ptr(value); });
}

void* sox_session_stream(sox_session* s) { return s ? s->stream : nullptr; }

}  // extern "C"

// ---- CTC head (CtcProjection, Decoding/CtcProjection.cs:12-75; kernels in ctc.hip) ----
struct sox_ctc {
    sox_backend* be = nullptr;
    int inner = 0, columns = 0, ldw = 0;
    bool has_bias = false;
    void* w = nullptr;     // fp16 [columns][ldw]
    void* bias = nullptr;  // fp32 [columns]
    std::mutex mu;         // the workspace below is shared by the calls on this object
    void* work = nullptr;  // the column ranges' partials
    uint64_t work_bytes = 0;
    void* host = nullptr;  // pinned and mapped: indices, probs, status
    uint64_t host_bytes = 0;

    bool finite = true;    // weights and bias: a non-finite one makes every row's logits non-finite
    void* part_fn = nullptr;   // the two passes, resolved at creation (fused heads)
    void* merge_fn = nullptr;

    // W range + bias of one column range fit 128 KiB of LDS; at most 64 ranges (one merge wave per row)
    int lds_tiles() const { return 131072 / (32 * (inner * 2 + 4)); }
    bool fused() const {
        return inner >= 64 && columns >= 1024 && inner % 16 == 0 && inner <= 256 &&
               ((columns + 31) / 32 + lds_tiles() - 1) / lds_tiles() <= 64;
    }
    ~sox_ctc() {
        if (w) sox_free(w);
        if (bias) sox_free(bias);
        if (work) sox_free(work);
        if (host) sox_host_free(host);
    }
};

namespace {

// The launch geometry of one ArgMax over R rows of a session's features, after the checks both
// entry points share: the feature value must be the whole [R, inner] activation, still intact after
// the run (no later node's output overlaps it in the arena) and stored with dense rows.
struct CtcLaunch {
    int64_t R = 0;
    int splits = 0, cps = 0;
    const void* x = nullptr;
};

CtcLaunch ctc_prepare(sox_ctc* c, sox_session* s, int32_t feature_value, int32_t batch, int32_t rows) {
    if (!c || !s || batch <= 0 || rows <= 0) fail(SOX_E_INVALID, "CtcProjection.ArgMax: arguments");
    if (!c->fused()) fail(SOX_E_UNSUPPORTED, "CtcProjection.ArgMax: head not fused (inner / columns)");
    if (!s->g->f16 || s->g->bf16) fail(SOX_E_INVALID, "CtcProjection.ArgMax: fp16 graphs only");
    if (!c->finite) fail(SOX_E_INVALID, "Recognizer output is invalid.");
    const sox_plan& P = s->g->plan;
    CtcLaunch L;
    L.R = (int64_t)batch * rows;
    if (L.R >= ((int64_t)1 << 31) / 3) fail(SOX_E_INVALID, "CtcProjection.ArgMax: too many rows");
    if (s->g->V(feature_value).buf < 0 || s->g->V(feature_value).count() != L.R * c->inner)
        fail(SOX_E_INVALID, "CtcProjection.ArgMax: features must be an activation of batch x rows x inner values");
    if (s->g->padded_ld.count(feature_value)) fail(SOX_E_INVALID, "CtcProjection.ArgMax: features rows are padded");
    int producer = -1;
    for (int ni = 0; ni < (int)P.nodes.size(); ni++)
        for (int o : P.nodes[ni].out)
            if (o == feature_value) producer = ni;
    const auto fr = value_range(P, feature_value);
    for (int ni = producer + 1; ni < (int)P.nodes.size(); ni++) {
        if (s->g->folded.count(ni)) continue;
        for (int o : P.nodes[ni].out) {
            if (o == feature_value || P.values[o].buf < 0) continue;
            const auto r = value_range(P, o);
            if (r.first < fr.second && fr.first < r.second)
                fail(SOX_E_INVALID, "CtcProjection.ArgMax: a later node overwrites the features in the arena");
        }
    }
    L.x = s->value_ptr(feature_value);
    // column ranges: as many as fill one round of the CUs, at least as many as the LDS bound needs,
    // at most 64 and at most one per 32-column tile
    const int64_t row_blocks = (L.R + 255) / 256;
    const int cus = std::max(1, c->be->info.compute_units);
    const int tiles = (c->columns + 31) / 32;
    int splits = (int)std::max<int64_t>((tiles + c->lds_tiles() - 1) / c->lds_tiles(), cus / row_blocks);
    splits = std::min(std::min(splits, tiles), 64);
    L.cps = ((tiles + splits - 1) / splits) * 32;
    L.splits = (c->columns + L.cps - 1) / L.cps;
    return L;
}

// The two passes on the session's stream: partials into `part` (splits x R triples), then per row the
// winner's column, its probability and the status word (cleared by pass 1, set by pass 2).
void ctc_enqueue(sox_ctc* c, sox_session* s, const CtcLaunch& L, float* part, int32_t* d_idx, float* d_prob,
                 int32_t* d_status) {
    sox_ctc_args a{};
    a.x = L.x; a.w = c->w; a.bias = c->has_bias ? (const float*)c->bias : (const float*)c->be->dummy; a.part = part;
    a.status = d_status;
    a.rows = (int)L.R; a.inner = c->inner; a.columns = c->columns; a.ldw = c->ldw; a.cols_per_split = L.cps;
    a.has_bias = c->has_bias ? 1 : 0;
    const uint32_t g1[3] = {(uint32_t)((L.R + 255) / 256), (uint32_t)L.splits, 1}, blk1[3] = {512, 1, 1},
                   blk[3] = {256, 1, 1};
    check(sox_launch(c->part_fn, g1, blk1, 0, s->stream, &a, sizeof a), "CtcProjection pass 1");
    sox_ctc_merge_args mg{part, d_idx, d_prob, d_status, (int)L.R, L.splits};
    const uint32_t g2[3] = {(uint32_t)((L.R + 3) / 4), 1, 1};
    check(sox_launch(c->merge_fn, g2, blk, 0, s->stream, &mg, sizeof mg), "CtcProjection pass 2");
}

}  // namespace

extern "C" {

int sox_ctc_create(sox_backend* be, const float* weights, const float* bias, int32_t inner, int32_t columns,
                   sox_ctc** out) {
    return guarded([&] {
        if (!be || !weights || !out || inner <= 0 || columns <= 0) fail(SOX_E_INVALID, "CtcProjection: arguments");
        be->need_device("CtcProjection");
        auto c = std::make_unique<sox_ctc>();
        c->be = be;
        c->inner = inner;
        c->columns = columns;
        c->ldw = (inner + 7) & ~7;
        c->has_bias = bias != nullptr;
        // [inner][columns] row-major -> fp16 [columns][ldw] (a column's inner values contiguous)
        for (size_t i = 0; i < (size_t)inner * columns; i++) c->finite = c->finite && std::isfinite(weights[i]);
        for (int i = 0; bias && i < columns; i++) c->finite = c->finite && std::isfinite(bias[i]);
        std::vector<uint16_t> wh((size_t)columns * c->ldw, 0), wk(columns);
        for (int k = 0; k < inner; k++) {
            f32_to_f16_n(weights + (size_t)k * columns, wk.data(), columns);
            for (int n = 0; n < columns; n++) wh[(size_t)n * c->ldw + k] = wk[n];
        }
        check(sox_malloc(&c->w, wh.size() * 2), "CtcProjection weights");
        check(sox_memcpy_h2d(c->w, wh.data(), wh.size() * 2, nullptr), "CtcProjection weights upload");
        if (bias) {
            check(sox_malloc(&c->bias, (size_t)columns * 4), "CtcProjection bias");
            check(sox_memcpy_h2d(c->bias, bias, (size_t)columns * 4, nullptr), "CtcProjection bias upload");
        }
        check(sox_device_sync(), "CtcProjection upload");
        if (c->fused()) {
            c->part_fn = be->fn("sox_ctc_part_k" + std::to_string(inner / 16));
            c->merge_fn = be->fn("sox_ctc_merge");
        }
        *out = c.release();
    });
}

void sox_ctc_destroy(sox_ctc* c) { delete c; }

int sox_ctc_is_fused(sox_ctc* c) { return c && c->fused() ? 1 : 0; }

int sox_ctc_argmax_noalloc(sox_ctc* c, sox_session* s, int32_t feature_value, int32_t batch, int32_t rows,
                           int32_t* d_indices, float* d_probabilities, int32_t* d_status) {
    return guarded([&] {
        if (!d_indices || !d_probabilities || !d_status) fail(SOX_E_INVALID, "CtcProjection.ArgMax: arguments");
        const CtcLaunch L = ctc_prepare(c, s, feature_value, batch, rows);
        const uint64_t part_b = (uint64_t)L.splits * L.R * 12;
        if (!c->be->scratch) fail(SOX_E_INVALID, "CtcProjection.ArgMax: no device scratch on this backend");
        if (part_b > c->be->scratch_bytes)
            fail(SOX_E_INVALID, "CtcProjection.ArgMax (no allocation): " + std::to_string(L.splits) + " column ranges x " +
                                    std::to_string(L.R) + " rows need " + std::to_string(part_b) +
                                    " bytes of partials, more than the " + std::to_string(c->be->scratch_bytes) +
                                    "-byte device scratch");
        sox_backend* be = c->be;
        std::lock_guard<std::mutex> lk_scratch(be->scratch_mu);
        std::lock_guard<std::mutex> lk(c->mu);
        int capturing = 0;
        check(sox_stream_is_capturing(s->stream, &capturing), "CtcProjection.ArgMax: capture state");
        if (!capturing && be->scratch_used)
            check(sox_stream_wait_event(s->stream, be->scratch_ev), "CtcProjection.ArgMax: scratch order");
        ctc_enqueue(c, s, L, (float*)be->scratch, d_indices, d_probabilities, d_status);
        if (!capturing) {
            check(sox_event_record(be->scratch_ev, s->stream), "CtcProjection.ArgMax: scratch order");
            be->scratch_used = true;
        }
    });
}

int sox_ctc_argmax(sox_ctc* c, sox_session* s, int32_t feature_value, int32_t batch, int32_t rows, int32_t* indices,
                   float* probabilities) {
    return guarded([&] {
        if (!indices || !probabilities) fail(SOX_E_INVALID, "CtcProjection.ArgMax: arguments");
        const CtcLaunch L = ctc_prepare(c, s, feature_value, batch, rows);
        const int64_t R = L.R;
        std::lock_guard<std::mutex> lk(c->mu);
        const uint64_t part_b = ((uint64_t)L.splits * R * 12 + 255) & ~255ull, out_b = ((uint64_t)R * 4 + 255) & ~255ull;
        if (part_b > c->work_bytes) {
            if (c->work) sox_free(c->work);
            c->work = nullptr;
            c->work_bytes = 0;
            check(sox_malloc(&c->work, part_b), "CtcProjection workspace");
            c->work_bytes = part_b;
        }
        const uint64_t host_need = 2 * out_b + 256;
        if (host_need > c->host_bytes) {
            if (c->host) sox_host_free(c->host);
            c->host = nullptr;
            c->host_bytes = 0;
            check(sox_host_alloc(&c->host, host_need), "CtcProjection staging");
            c->host_bytes = host_need;
        }
        // the merge pass writes its rows' results and the status into the mapped host block itself: three
        // copy-engine downloads behind it took ~25 us of a call
        uint8_t* h = (uint8_t*)c->host;
        int32_t* h_status = (int32_t*)(h + 2 * out_b);
        ctc_enqueue(c, s, L, (float*)c->work, (int32_t*)h, (float*)(h + out_b), h_status);
        check(sox_stream_sync(s->stream), "CtcProjection sync");
        if (*h_status) fail(SOX_E_INVALID, "Recognizer output is invalid.");
        memcpy(indices, h, (size_t)R * 4);
        memcpy(probabilities, h + out_b, (size_t)R * 4);
    });
}

}  // extern "C"

// ---- image session (VkImageSession, Backends/Vulkan/VkImageSession.cs; kernels in tensor.hip) ----
constexpr uint64_t kImageChunk = 768 << 10;  // bytes: ~14 us of PCIe

struct sox_image_session {
    sox_backend* be = nullptr;
    void* lut = nullptr;  // device [3][256] fp32
    bool rgb_order = false, top_left = false;
    float scale = 255.0f;
    int pad_multiple = 1;
    sox_graph* g = nullptr;  // the graph of the bound tensor size (reference held by its session)
    sox_session* s = nullptr;
    void* d_src = nullptr;    // packed u8 pixels
    uint64_t d_bytes = 0;
    void* h_stage = nullptr;  // pinned and mapped: the pixels on their way up, then the output words
    std::vector<void*> ev;    // one per output chunk
    uint64_t h_bytes = 0;

    ~sox_image_session() {
        if (s) sox_session_destroy(s);
        if (lut) sox_free(lut);
        if (d_src) sox_free(d_src);
        if (h_stage) sox_host_free(h_stage);
        for (void* e : ev) sox_event_destroy(e);
    }
    void pads(int height, int width, int& pt, int& pl, int& h, int& w) const {  // ImageSessionOptions.Pads
        const int ph = (pad_multiple - height % pad_multiple) % pad_multiple;
        const int pw = (pad_multiple - width % pad_multiple) % pad_multiple;
        pt = top_left ? ph : 0;
        pl = top_left ? pw : 0;
        h = height + ph;
        w = width + pw;
    }
};

extern "C" {

int sox_image_session_create(sox_backend* be, const float* lut, int32_t rgb_order, float output_scale,
                             int32_t pad_multiple, int32_t pad_top_left, sox_image_session** out) {
    return guarded([&] {
        if (!be || !lut || !out) fail(SOX_E_INVALID, "ImageSession: arguments");
        if (pad_multiple < 1) fail(SOX_E_INVALID, "ImageSession: PadMultiple < 1");
        be->need_device("ImageSession");
        auto is = std::make_unique<sox_image_session>();
        is->be = be;
        is->rgb_order = rgb_order != 0;
        is->top_left = pad_top_left != 0;
        is->scale = output_scale;
        is->pad_multiple = pad_multiple;
        check(sox_malloc(&is->lut, 768 * 4), "ImageSession table");
        check(sox_memcpy_h2d(is->lut, lut, 768 * 4, nullptr), "ImageSession table upload");
        check(sox_device_sync(), "ImageSession table upload");
        *out = is.release();
    });
}

void sox_image_session_destroy(sox_image_session* is) { delete is; }

int sox_image_session_tensor_size(sox_image_session* is, int32_t width, int32_t height, int32_t* th, int32_t* tw) {
    return guarded([&] {
        if (!is || !th || !tw || width < 1 || height < 1) fail(SOX_E_INVALID, "ImageSession: size");
        int pt, pl, h, w;
        is->pads(height, width, pt, pl, h, w);
        *th = h;
        *tw = w;
    });
}

int sox_image_session_run(sox_image_session* is, sox_graph* graph, const uint8_t* src, int32_t width, int32_t height,
                          int32_t src_stride, uint8_t* dst, int32_t dst_stride, int32_t format) {
    return guarded([&] {
        if (!is || !graph || !src || !dst) fail(SOX_E_INVALID, "ImageSession.Run: arguments");
        if (format < SOX_PIX_BGR24 || format > SOX_PIX_RGBA32) fail(SOX_E_INVALID, "ImageSession.Run: pixel format");
        const int bpp = format >= SOX_PIX_BGRA32 ? 4 : 3;
        if (width < 1 || height < 1) fail(SOX_E_INVALID, "ImageSession.Run: image size");
        if (src_stride < width * bpp || dst_stride < width * bpp) fail(SOX_E_INVALID, "ImageSession.Run: row stride");
        int pt, pl, h, w;
        is->pads(height, width, pt, pl, h, w);
        const sox_plan& P = graph->plan;
        auto is_img = [&](int v) {
            const PlanValue& pv = graph->V(v);
            const std::vector<int> ph = pv.phys();
            return pv.shape.size() == 4 && pv.shape[0] == 1 && pv.shape[1] == 3 && pv.shape[2] == h && pv.shape[3] == w &&
                   ph.size() == 4 && ph[3] == 3 && ph[1] == h && ph[2] == w;
        };
        if (P.inputs.size() != 1 || !is_img(P.inputs[0]) || !is_img(P.output))
            fail(SOX_E_UNSUPPORTED, "An image session needs a single-input model with NHWC [1, 3, " + std::to_string(h) +
                                        ", " + std::to_string(w) + "] input and output");
        if (graph != is->g) {  // bind the graph of this tensor size
            if (is->s) sox_session_destroy(is->s);
            is->s = nullptr;
            is->g = nullptr;
            check(sox_session_create(graph, &is->s), "ImageSession session");
            is->g = graph;
        }
        sox_session* s = is->s;
        const uint64_t row = (uint64_t)width * bpp, bytes = row * height;
        const uint64_t need = (bytes + 4 + 255) & ~255ull;
        if (need > is->d_bytes) {  // grow-only pixel buffers (a quarter of headroom, VkImageSession.Staging)
            if (is->d_src) sox_free(is->d_src);
            is->d_src = nullptr;
            is->d_bytes = 0;
            const uint64_t size = need + need / 4;
            check(sox_malloc(&is->d_src, size), "ImageSession pixels");
            is->d_bytes = size;
        }
        if (need > is->h_bytes) {
            if (is->h_stage) sox_host_free(is->h_stage);
            is->h_stage = nullptr;
            is->h_bytes = 0;
            const uint64_t size = need + need / 4;
            check(sox_host_alloc(&is->h_stage, size), "ImageSession staging");
            is->h_bytes = size;
        }
        uint8_t* hs = (uint8_t*)is->h_stage;
        // The frame goes up and comes home in chunks: while one chunk crosses PCIe the host copies the next
        // between the caller's rows and the staging (a 1920x1080 Bgr24 frame through a six-layer model:
        // 835 -> 660 us, with the copy up, the copy home and both row copies one after the other before).
        const int chunks = (int)std::clamp<uint64_t>(bytes / kImageChunk, 1, 8);
        void* up = graph->be->fn("sox_stage_in_f32");
        uint64_t sent = 0;  // whole 64-byte lines, the last chunk to the end (the buffers have slack for its last word)
        for (int c = 0, y = 0; c < chunks; c++) {
            const int y1 = c + 1 == chunks ? height : (int)((int64_t)height * (c + 1) / chunks);
            for (; y < y1; y++) memcpy(hs + (uint64_t)y * row, src + (uint64_t)y * src_stride, row);
            const uint64_t end = c + 1 == chunks ? (bytes + 3) & ~3ull : (uint64_t)y1 * row & ~63ull;
            const int64_t words = (int64_t)(end - sent) / 4;
            Staging::launch(up, hs + sent, (uint8_t*)is->d_src + sent, words, std::min<int64_t>(64, (words + 2047) / 2048),
                            s->stream);
            sent = end;
        }
        const bool rgb_bytes = format == SOX_PIX_RGB24 || format == SOX_PIX_RGBA32;
        const int swap = rgb_bytes != is->rgb_order ? 1 : 0;  // ImageSessionOptions.Swap
        const char* ty = graph->bf16 ? "bf16" : graph->f16 ? "f16" : "f32";
        sox_img2nhwc_args a{};
        a.src = (const uint8_t*)is->d_src; a.y = s->value_ptr(P.inputs[0]); a.lut = (const float*)is->lut;
        a.oh = h; a.ow = w; a.ih = height; a.iw = width; a.pt = pt; a.pl = pl; a.stride = (int)row; a.bpp = bpp; a.swap = swap;
        const int64_t pairs = ((int64_t)h * w + 1) / 2;  // two tensor pixels per thread
        const uint32_t blk[3] = {256, 1, 1}, g1[3] = {(uint32_t)((pairs + 255) / 256), 1, 1};
        check(sox_launch(graph->be->fn(std::string("sox_img2nhwc_") + ty), g1, blk, 0, s->stream, &a, sizeof a), "img2nhwc");
        s->enqueue(SOX_RUN_DISPATCHES);
        sox_nhwc2img_args b{};
        const int64_t nwords = bpp == 4 ? (int64_t)height * width : ((int64_t)height * width * 3 + 3) / 4;
        if (nwords >= ((int64_t)1 << 31)) fail(SOX_E_UNSUPPORTED, "ImageSession.Run: image too large");
        b.x = s->value_ptr(P.output); b.dst = (uint32_t*)hs; b.alpha = (const uint32_t*)is->d_src;
        b.h = h; b.w = w; b.ih = height; b.iw = width; b.pt = pt; b.pl = pl; b.bpp = bpp;
        b.swap = swap; b.scale = is->scale;
        void* down = graph->be->fn(std::string("sox_nhwc2img_") + ty);
        while ((int)is->ev.size() < chunks) {
            void* e = nullptr;
            check(sox_event_create(&e), "ImageSession event");
            is->ev.push_back(e);
        }
        auto chunk_end = [&](int c) { return c + 1 == chunks ? nwords : nwords * (c + 1) / chunks & ~255ll; };
        for (int c = 0; c < chunks; c++) {  // straight into the mapped staging
            b.first = c ? (int)chunk_end(c - 1) : 0;
            b.nwords = (int)chunk_end(c);
            const uint32_t g2[3] = {(uint32_t)((b.nwords - b.first + 255) / 256), 1, 1};
            check(sox_launch(down, g2, blk, 0, s->stream, &b, sizeof b), "nhwc2img");
            check(sox_event_record(is->ev[c], s->stream), "ImageSession event");
        }
        for (int c = 0, y = 0; c < chunks; c++) {
            check(sox_event_sync(is->ev[c]), "ImageSession wait");
            const int y1 = c + 1 == chunks ? height : (int)((uint64_t)chunk_end(c) * 4 / row);
            for (; y < y1; y++) memcpy(dst + (uint64_t)y * dst_stride, hs + (uint64_t)y * row, row);
        }
    });
}

}  // extern "C"

// ---- unit runner (VkUnitRunner, Backends/Vulkan/VkUnitRunner.cs) ----
constexpr size_t kPairLaunches = 24;  // a submit's launches from which a second thread pays (its start is ~20 us)
constexpr int kQueueFill = 4;  // streams that even out the hardware queues before a runner creates its own

struct sox_unit_runner {
    struct Unit {
        sox_graph* g = nullptr;
        uint64_t arena_off = 0, stage_off = 0;  // bytes into the shared device arena / download staging
        uint64_t sync_off = 0;                   // bytes into the shared counter block
        int64_t in_off = 0, out_off = 0;         // floats into the pinned host staging
        int64_t in_count = 0, out_count = 0;
        std::vector<std::vector<uint8_t>> kernargs;
        Staging staging;
    };
    sox_backend* be = nullptr;
    std::vector<void*> streams;
    std::vector<Unit> units;
    std::vector<int> wave_end;           // exclusive unit index ending each wave
    std::vector<std::vector<void*>> ev;  // per wave: one event per stream
    void *arena = nullptr, *dstage = nullptr, *sync = nullptr;
    uint64_t arena_bytes = 0, dstage_bytes = 0, sync_bytes = 0;
    float *h_in = nullptr, *h_out = nullptr;
    int64_t h_in_count = 0, h_out_count = 0;
    bool laid_out = false, in_flight = false, submitted = false;  // submitted: since the last Clear
    int waited = -1;

    ~sox_unit_runner() {
        for (auto& w : ev)
            for (void* e : w) sox_event_destroy(e);
        for (Unit& u : units) sox_graph_release(u.g);
        for (void* st : streams) sox_stream_destroy(st);
        if (arena) sox_free(arena);
        if (dstage) sox_free(dstage);
        if (sync) sox_free(sync);
        if (h_in) sox_host_free(h_in);
        if (h_out) sox_host_free(h_out);
    }
    void cut() {
        const int last = wave_end.empty() ? 0 : wave_end.back();
        if ((int)units.size() > last) wave_end.push_back((int)units.size());
    }
    // one region per unit in each shared buffer (all grow-only), kernargs patched to the unit's arena
    void layout() {
        if (laid_out) return;
        cut();
        uint64_t a = 0, d = 0, sy = 0;
        int64_t hi = 0, ho = 0;
        for (Unit& u : units) {
            u.arena_off = a;
            a += (u.g->arena_bytes() + 255) & ~255ull;
            u.sync_off = sy;
            sy += (u.g->sync_bytes + 255) & ~255ull;
            u.in_count = u.g->V(u.g->plan.inputs[0]).count();
            u.out_count = u.g->V(u.g->plan.output).count();
            u.stage_off = d;
            d += ((uint64_t)Staging::stage_floats(*u.g, u.out_count) * 4 + 255) & ~255ull;
            u.staging.bind(*u.g);
            u.in_off = hi;
            hi += (u.in_count + 63) & ~63ll;
            u.out_off = ho;
            ho += (u.out_count + 63) & ~63ll;
        }
        auto grow_dev = [](void*& p, uint64_t& have, uint64_t need, const char* what) {
            if (need <= have) return;
            if (p) sox_free(p);
            p = nullptr;
            have = 0;
            check(sox_malloc(&p, need + need / 4), what);
            have = need + need / 4;
        };
        auto grow_host = [](float*& p, int64_t& have, int64_t need, const char* what) {
            if (need <= have) return;
            if (p) sox_host_free(p);
            p = nullptr;
            have = 0;
            check(sox_host_alloc((void**)&p, (size_t)(need + need / 4) * 4), what);
            have = need + need / 4;
        };
        grow_dev(arena, arena_bytes, std::max<uint64_t>(a, 256), "UnitRunner arena");
        grow_dev(dstage, dstage_bytes, d, "UnitRunner staging");
        if (sy > sync_bytes) {  // counters: zeroed when (re)allocated, back at 0 after every launch
            grow_dev(sync, sync_bytes, sy, "UnitRunner counters");
            std::vector<uint8_t> zeros(sync_bytes, 0);
            check(sox_memcpy_h2d(sync, zeros.data(), zeros.size(), streams[0]), "UnitRunner counters");
            check(sox_stream_sync(streams[0]), "UnitRunner counters");
        }
        grow_host(h_in, h_in_count, std::max<int64_t>(hi, 64), "UnitRunner input staging");
        grow_host(h_out, h_out_count, std::max<int64_t>(ho, 64), "UnitRunner output staging");
        for (Unit& u : units) {
            u.kernargs.clear();
            for (const Dispatch& dd : u.g->disp) {
                std::vector<uint8_t> ka = dd.kernarg;
                for (const Patch& p : dd.patches) {
                    void* ptr = p.bind.slot == SOX_SLOT_ARENA ? (uint8_t*)arena + u.arena_off + p.bind.offset
                                : p.bind.slot == SOX_SLOT_CONSTS ? (uint8_t*)u.g->consts + p.bind.offset
                                : p.bind.slot == SOX_SLOT_SYNC   ? (uint8_t*)sync + u.sync_off + p.bind.offset
                                                                 : be->dummy;
                    memcpy(ka.data() + p.off, &ptr, sizeof ptr);
                }
                u.kernargs.push_back(std::move(ka));
            }
        }
        laid_out = true;
    }
    void* value_ptr(const Unit& u, int v) const {
        const PlanValue& pv = u.g->V(v);
        return (uint8_t*)arena + u.arena_off + (uint64_t)u.g->plan.buf_offset[pv.buf] * u.g->es;
    }
    void run_unit(Unit& u, void* st) {
        u.staging.upload(h_in + u.in_off, value_ptr(u, u.g->plan.inputs[0]), u.in_count, st);
        for (size_t i = 0; i < u.g->disp.size(); i++) {
            const Dispatch& d = u.g->disp[i];
            check(sox_launch(d.fn, d.grid, d.block, d.lds, st, u.kernargs[i].data(), u.kernargs[i].size()), d.name.c_str());
        }
        u.staging.download(value_ptr(u, u.g->plan.output), h_out + u.out_off, u.out_count, dstage ? (uint8_t*)dstage + u.stage_off : nullptr,
                           u.g->f16, st);
    }
};

extern "C" {

int sox_unit_runner_create(sox_backend* be, int32_t nstreams, sox_unit_runner** out) {
    return guarded([&] {
        if (!be || !out || nstreams < 1 || nstreams > 16) fail(SOX_E_INVALID, "UnitRunner: arguments");
        be->need_device("UnitRunner");
        auto r = std::make_unique<sox_unit_runner>();
        r->be = be;
        // HIP puts a new stream on the hardware queue with the fewest streams, and queues hold one stream more or
        // less than others (the null stream's, a closed session's): two of four streams could then share a queue
        // while another idled. Placeholders fill the gaps first, so that the runner's streams, created one after
        // the other, take the queues in turn (12 text lines on 4 streams: 478 us with a shared queue, 370 without)
        struct Placeholders {
            std::vector<void*> st;
            ~Placeholders() {
                for (void* p : st) sox_stream_destroy(p);
            }
        } fill;
        for (int i = 0; i < nstreams + kQueueFill; i++) {
            void* st = nullptr;
            check(sox_stream_create(&st), "UnitRunner stream");
            (i < kQueueFill ? fill.st : r->streams).push_back(st);
        }
        *out = r.release();
    });
}

void sox_unit_runner_destroy(sox_unit_runner* r) {
    if (!r) return;
    for (void* st : r->streams) sox_stream_sync(st);
    delete r;
}

int sox_unit_runner_clear(sox_unit_runner* r) {
    return guarded([&] {
        if (!r) fail(SOX_E_INVALID, "UnitRunner: null");
        if (r->in_flight) fail(SOX_E_INVALID, "UnitRunner: previous run still in flight");
        for (auto& u : r->units) sox_graph_release(u.g);
        r->units.clear();
        r->wave_end.clear();
        r->laid_out = false;
        r->submitted = false;
    });
}

int sox_unit_runner_add(sox_unit_runner* r, sox_graph* g, int32_t* unit) {
    return guarded([&] {
        if (!r || !g || !unit) fail(SOX_E_INVALID, "UnitRunner.Add: arguments");
        if (r->laid_out) fail(SOX_E_INVALID, "UnitRunner.Add: add units before writing inputs");
        if (g->plan.inputs.size() != 1) fail(SOX_E_UNSUPPORTED, "UnitRunner.Add: single-input graphs only");
        g->refs++;
        sox_unit_runner::Unit u;
        u.g = g;
        r->units.push_back(std::move(u));
        *unit = (int32_t)r->units.size() - 1;
    });
}

int sox_unit_runner_cut(sox_unit_runner* r) {
    return guarded([&] {
        if (!r) fail(SOX_E_INVALID, "UnitRunner: null");
        if (r->laid_out) fail(SOX_E_INVALID, "UnitRunner.Cut: after the layout");
        r->cut();
    });
}

int sox_unit_runner_waves(sox_unit_runner* r) { return r ? (int)r->wave_end.size() : 0; }

int sox_unit_runner_wave_end(sox_unit_runner* r, int32_t wave) {
    return r && wave >= 0 && wave < (int)r->wave_end.size() ? r->wave_end[wave] : SOX_E_INVALID;
}

int sox_unit_runner_input(sox_unit_runner* r, int32_t unit, float** host, int64_t* count) {
    return guarded([&] {
        if (!r || !host || !count || unit < 0 || unit >= (int)r->units.size()) fail(SOX_E_INVALID, "UnitRunner.Input: unit");
        if (r->in_flight) fail(SOX_E_INVALID, "UnitRunner.Input: run in flight");
        r->layout();
        *host = r->h_in + r->units[unit].in_off;
        *count = r->units[unit].in_count;
    });
}

int sox_unit_runner_output(sox_unit_runner* r, int32_t unit, float** host, int64_t* count) {
    return guarded([&] {
        if (!r || !host || !count || unit < 0 || unit >= (int)r->units.size()) fail(SOX_E_INVALID, "UnitRunner.Output: unit");
        r->layout();
        *host = r->h_out + r->units[unit].out_off;
        *count = r->units[unit].out_count;
    });
}

int sox_unit_runner_submit(sox_unit_runner* r) {
    return guarded([&] {
        if (!r) fail(SOX_E_INVALID, "UnitRunner: null");
        if (r->in_flight) fail(SOX_E_INVALID, "UnitRunner.Submit: previous run still in flight");
        if (r->be->lost || sox_device_lost()) fail(SOX_E_LOST, "device lost");
        r->layout();
        const int S = (int)r->streams.size();
        while (r->ev.size() < r->wave_end.size()) {
            std::vector<void*> w(S, nullptr);
            for (int i = 0; i < S; i++) check(sox_event_create(&w[i]), "UnitRunner event");
            r->ev.push_back(std::move(w));
        }
        r->in_flight = true;
        r->submitted = true;
        r->waited = -1;
        // enqueues every `step`-th stream from `first`; a stream's work stays in one thread, in order
        auto enqueue = [&](int first, int step) {
            int u0 = 0;
            for (size_t w = 0; w < r->wave_end.size(); w++) {
                for (int u = u0; u < r->wave_end[w]; u++)
                    if ((u - u0) % S % step == first) r->run_unit(r->units[u], r->streams[(u - u0) % S]);
                for (int i = first; i < S; i += step) check(sox_event_record(r->ev[w][i], r->streams[i]), "UnitRunner event");
                u0 = r->wave_end[w];
            }
        };
        // A launch is ~2 us of host work and the units' kernels are short, so the host bounds the run: from
        // kPairLaunches on a second thread enqueues half of the streams while this one does the other half, and
        // both are done before the call returns (text lines on 4 streams, 12 launches each: 12 lines 436 -> 339 us,
        // 4 lines 170 -> 124, 2 lines 106 -> 99)
        size_t launches = 0;
        for (const auto& u : r->units) launches += u.g->disp.size() + 2;
        std::thread helper;
        std::exception_ptr err;
        if (S > 1 && r->units.size() > 1 && launches >= kPairLaunches) {
            try {
                helper = std::thread([&] {
                    try {
                        check(sox_init(r->be->info.device, nullptr), "UnitRunner device");  // this thread's current device
                        enqueue(1, 2);
                    } catch (...) {
                        err = std::current_exception();
                    }
                });
            } catch (const std::system_error&) {  // no thread to be had
            }
        }
        if (!helper.joinable()) {
            enqueue(0, 1);
            return;
        }
        try {
            enqueue(0, 2);
        } catch (...) {
            helper.join();
            throw;
        }
        helper.join();
        if (err) std::rethrow_exception(err);
    });
}

int sox_unit_runner_wait(sox_unit_runner* r, int32_t wave) {
    return guarded([&] {
        if (!r || !r->submitted) fail(SOX_E_INVALID, "UnitRunner.Wait: nothing submitted");
        if (wave < 0 || wave >= (int)r->wave_end.size()) fail(SOX_E_INVALID, "UnitRunner.Wait: wave");
        for (int w = r->waited + 1; w <= wave; w++)
            for (void* e : r->ev[w]) check(sox_event_sync(e), "UnitRunner wait");
        r->waited = std::max(r->waited, (int)wave);
        if (r->waited == (int)r->wave_end.size() - 1) r->in_flight = false;
    });
}

}  // extern "C"
