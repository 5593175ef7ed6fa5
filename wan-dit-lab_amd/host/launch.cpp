// The launchers of the hot path's calls: outputs allocated by torch, raw pointers, sizes and the caller's stream handed
// to one wdl_* entry point of libwdl.so (include/wdl.h). The Python functions of the same names in wdl/ops.py, fp8.py,
// rope.py check their arguments and call these; through ctypes a launch's two dozen arguments and its outputs'
// allocations took 8 - 15 us of host time, here 3 - 5.
//
// Nothing is kept between calls but the entry points' addresses (bind). The library's status becomes the RuntimeError
// that wdl._lib.call raises.
#include <dlfcn.h>
#include <torch/extension.h>

#include <optional>
#include <stdexcept>
#include <string>

#include "wdl.h"

namespace {

using at::Tensor;
using Opt = std::optional<Tensor>;

#define WDL_ENTRIES(X)                                                                                              \
    X(wdl_last_error) X(wdl_abi_version) X(wdl_kv_append_fp8) X(wdl_act_quant_workspace_floats) X(wdl_act_quant_w4) \
    X(wdl_w4a4_gemm)                                                                                                \
    X(wdl_w4a4_gemm_gelu_quant_workspace_floats) X(wdl_w4a4_gemm_gelu_quant) X(wdl_fp8_quantize_workspace_floats)   \
    X(wdl_fp8_quantize) X(wdl_fp8_gemm) X(wdl_fp8wo_gemm) X(wdl_qk_norm_rope) X(wdl_sage_prep_workspace_floats)     \
    X(wdl_sage_prep) X(wdl_sage_prep_cached) X(wdl_sage_prep_cached_append) X(wdl_sage_attn_q16)                    \
    X(wdl_sage_attn_q16_framed) X(wdl_attn_bf16) X(wdl_rope3d_rotate)

struct Entries {
#define X(name) decltype(&::name) name = nullptr;
    WDL_ENTRIES(X)
#undef X
} lib;

void bind(const std::string& path) {
    void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (!h) throw std::runtime_error(std::string("dlopen: ") + dlerror());
    Entries e;
#define X(name)                                                                              \
    e.name = reinterpret_cast<decltype(e.name)>(dlsym(h, #name));                            \
    if (!e.name) throw std::runtime_error(path + " has no entry point " #name);
    WDL_ENTRIES(X)
#undef X
    if (e.wdl_abi_version() != WDL_ABI_VERSION)
        throw std::runtime_error(path + " has ABI version " + std::to_string(e.wdl_abi_version()) +
                                 ", the launchers are compiled for " + std::to_string(WDL_ABI_VERSION) +
                                 ": build both again (python -m wdl.build)");
    lib = e;
}

void ok(const char* name, int status) {
    if (status)
        throw std::runtime_error(std::string(name) + " failed (" + std::to_string(status) + "): " + lib.wdl_last_error());
}
#define CALL(name, ...) ok(#name, lib.name(__VA_ARGS__))

void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const Opt& t) { return t ? t->data_ptr() : nullptr; }
float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
float* f32(const Opt& t) { return t ? static_cast<float*>(t->data_ptr()) : nullptr; }
wdl_stream_t str(uintptr_t s) { return reinterpret_cast<wdl_stream_t>(s); }
Tensor buf(const Tensor& like, at::IntArrayRef shape, at::ScalarType type) {
    return at::empty(shape, like.options().dtype(type).memory_format(at::MemoryFormat::Contiguous));
}
int code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return 0;
        case at::kHalf: return 1;
        case at::kBFloat16: return 2;
        case at::kDouble: return 3;
        default: throw std::invalid_argument("not a floating type of the library");
    }
}

// sizes and strides below are read by position
void dims(const char* what, const Tensor& t, int64_t least, int64_t most) {
    if (t.dim() < least || t.dim() > most)
        throw std::invalid_argument(std::string(what) + ": a tensor of " + std::to_string(t.dim()) + " dimensions, not " +
                                    std::to_string(least));
}

constexpr int64_t PAD = 128, ROW6 = 48, RANK = 32, D = 128;

std::tuple<Tensor, Tensor, Opt> act_quant(const Tensor& x, const Tensor& smooth, const Opt& pdt, double qshift,
                                          bool is_unsigned, bool ln, const Opt& shift, const Opt& scale,
                                          const Opt& weight, const Opt& bias, double eps, const Opt& partials,
                                          const Opt& v_out, uintptr_t stream) {
    dims("act_quant x", x, 2, 2);
    const int64_t M = x.size(0), K = x.size(1), Mp = (M + PAD - 1) / PAD * PAD;
    Tensor q = buf(x, {Mp / PAD, K / 64, PAD, ROW6}, at::kByte), asc = buf(x, {K / 64, Mp}, at::kBFloat16);
    Opt lora;
    if (pdt) lora = buf(x, {Mp, RANK}, at::kFloat);
    Tensor ws = buf(x, {lib.wdl_act_quant_workspace_floats(Mp, K)}, at::kFloat);
    CALL(wdl_act_quant_w4, ptr(x), x.stride(0), M, K, ptr(smooth), float(qshift), is_unsigned, ptr(pdt), RANK, ptr(q),
         ptr(asc), f32(lora), Mp, f32(shift), f32(scale), f32(weight), f32(bias), ln, float(eps), f32(partials),
         ptr(v_out), f32(ws), str(stream));
    return {q, asc, lora};
}

void gemm(const Tensor& q, const Tensor& asc, const Opt& lora, const Tensor& wc, const Tensor& ws, const Opt& pu,
          const Opt& bias, int64_t M, const Tensor& out, int epilogue, const Opt& gate, const Opt& ln_out,
          const Opt& workspace, uintptr_t stream) {
    CALL(wdl_w4a4_gemm, ptr(q), ptr(asc), ptr(wc), ptr(ws), f32(lora), ptr(pu), ptr(bias), M, q.size(0) * PAD,
         wc.size(0) * PAD, q.size(1) * 64, RANK, ptr(out), out.stride(0), epilogue, f32(gate), f32(ln_out),
         ptr(workspace), str(stream));
}

std::tuple<Tensor, Tensor, Tensor> gelu_quant(const Tensor& q, const Tensor& asc, const Opt& lora, const Tensor& wc,
                                              const Tensor& ws, const Opt& pu, const Opt& bias, int64_t M,
                                              const Tensor& smooth2, const Tensor& pd2, uintptr_t stream) {
    const int64_t Mp = q.size(0) * PAD, K = q.size(1) * 64, N = wc.size(0) * PAD;
    Tensor q2 = buf(q, {Mp / PAD, N / 64, PAD, ROW6}, at::kByte), asc2 = buf(q, {N / 64, Mp}, at::kBFloat16);
    Tensor lora2 = buf(q, {Mp, RANK}, at::kFloat);
    Tensor work = buf(q, {lib.wdl_w4a4_gemm_gelu_quant_workspace_floats(Mp, N)}, at::kFloat);
    CALL(wdl_w4a4_gemm_gelu_quant, ptr(q), ptr(asc), ptr(wc), ptr(ws), f32(lora), ptr(pu), ptr(bias), M, Mp, N, K, RANK,
         ptr(smooth2), ptr(pd2), ptr(q2), ptr(asc2), f32(lora2), f32(work), str(stream));
    return {q2, asc2, lora2};
}

std::tuple<Tensor, Opt> qk_norm_rope(const Tensor& q, const Opt& k, const Opt& wq, const Opt& wk, const Tensor& freq,
                                     int f, int h, int w, int64_t start, double eps, const Opt& q_into,
                                     const Opt& k_into, uintptr_t stream) {
    dims("qk_norm_rope q", q, 2, 2);
    const int64_t M = q.size(0), C = q.size(1);
    Tensor qo = q_into ? *q_into : buf(q, {M, C}, at::kBFloat16);
    Opt ko = k_into;
    if (k && !ko) ko = buf(q, {M, C}, at::kBFloat16);
    CALL(wdl_qk_norm_rope, ptr(q), q.stride(0), ptr(k), k ? k->stride(0) : 0, ptr(wq), ptr(wk), ptr(freq),
         code(freq.scalar_type()), freq.size(1), M, int(C / D), f, h, w, int(start), float(eps), ptr(qo), ptr(ko),
         qo.stride(0), str(stream));
    return {qo, ko};
}

// k_int8, k_scale, v_fp8, v_scale, k_mean of the cache's rows [0, at) and the chunk
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> sage_prep(const Tensor& ck, const Tensor& cks, const Tensor& cv,
                                                             const Tensor& cvs, const Tensor& k, const Tensor& v,
                                                             int64_t at, int splits, const Opt& stats, bool append,
                                                             uintptr_t stream) {
    const int64_t n = k.size(0), H = k.size(1) / D, Lp = (at + n + 63) / 64 * 64, cap = ck.size(1);
    Tensor ws = buf(k, {lib.wdl_sage_prep_workspace_floats(H, splits)}, at::kFloat);
    Tensor k8 = buf(k, {H, Lp, D}, at::kChar), ks = buf(k, {H, Lp / 16}, at::kFloat), v8 = buf(k, {H, D, Lp}, at::kByte);
    Tensor mean = buf(k, {H, D}, at::kFloat), vs = buf(k, {H, D}, at::kFloat);
    if (!stats)
        CALL(wdl_sage_prep, ptr(ck), f32(cks), ptr(cv), f32(cvs), cap, ptr(k), k.stride(0), ptr(v), v.stride(0), H, at, n,
             splits, f32(ws), ptr(k8), f32(ks), ptr(v8), f32(mean), f32(vs), str(stream));
    else if (append)
        CALL(wdl_sage_prep_cached_append, ptr(ck), f32(cks), ptr(cv), f32(cvs), cap, ptr(k), k.stride(0), ptr(v),
             v.stride(0), H, at, n, f32(stats), splits, f32(ws), ptr(k8), f32(ks), ptr(v8), f32(mean), f32(vs),
             str(stream));
    else
        CALL(wdl_sage_prep_cached, ptr(ck), f32(cks), ptr(cv), f32(cvs), cap, ptr(k), k.stride(0), ptr(v), v.stride(0), H,
             at, n, f32(stats), splits, f32(ws), ptr(k8), f32(ks), ptr(v8), f32(mean), f32(vs), str(stream));
    return {k8, ks, v8, vs, mean};
}

Tensor sage_attn_q16(const Tensor& q, const Tensor& k, const Tensor& ks, const Tensor& v, const Tensor& vs, int64_t L,
                     double sm, const Opt& into, int64_t frame, const Opt& workspace, uintptr_t stream) {
    const int64_t n = q.size(0), H = q.size(1) / D;
    Tensor out = into ? *into : buf(q, {n, H * D}, at::kBFloat16);
    if (frame)
        CALL(wdl_sage_attn_q16_framed, ptr(q), q.stride(0), ptr(k), f32(ks), ptr(v), f32(vs), n, L, H, float(sm), frame,
             ptr(out), out.stride(0), nullptr, str(stream));
    else
        CALL(wdl_sage_attn_q16, ptr(q), q.stride(0), ptr(k), f32(ks), ptr(v), f32(vs), n, L, H, float(sm), ptr(out),
             out.stride(0), ptr(workspace), str(stream));
    return out;
}

Tensor attn_bf16(const Tensor& q, const Tensor& kp, const Tensor& vp, int64_t L, double sm, const Opt& into,
                 uintptr_t stream) {
    Tensor out = into ? *into : buf(q, q.sizes(), at::kBFloat16);
    CALL(wdl_attn_bf16, ptr(q), q.stride(0), ptr(kp), ptr(vp), q.size(0), L, q.size(1) / D, float(sm), ptr(out),
         out.stride(0), str(stream));
    return out;
}

void kv_append(const Tensor& k, const Tensor& v, const Tensor& ck, const Tensor& cks, const Tensor& cv,
               const Tensor& cvs, int64_t at, uintptr_t stream) {
    dims("kv_append k", k, 4, 4);
    dims("kv_append v", v, 4, 64);
    CALL(wdl_kv_append_fp8, ptr(k), code(k.scalar_type()), k.strides().data(), ptr(v), code(v.scalar_type()),
         v.strides().data(), k.size(0), k.size(1), k.size(2), k.size(3), ptr(ck), f32(cks), ptr(cv), f32(cvs), ck.size(1),
         at, str(stream));
}

std::tuple<Tensor, Tensor> fp8_quantize(const Tensor& x, bool rows, int64_t pad, uintptr_t stream) {
    const int64_t M = x.size(0), K = x.size(1), Mp = (M + pad - 1) / pad * pad;
    Tensor q = buf(x, {Mp, K}, at::kByte), scale = buf(x, {rows ? Mp : 1}, at::kFloat);
    Opt ws;
    if (!rows) ws = buf(x, {lib.wdl_fp8_quantize_workspace_floats(M, K)}, at::kFloat);
    CALL(wdl_fp8_quantize, ptr(x), code(x.scalar_type()), x.stride(0), M, K, Mp, rows, ptr(q), f32(scale), f32(ws),
         str(stream));
    return {q, scale};
}

Tensor fp8_gemm(const Tensor& q, const Tensor& xs, int64_t M, const Tensor& w, const Tensor& ws, const Opt& bias,
                bool rows, const Opt& workspace, uintptr_t stream) {
    const int64_t N = w.size(0);
    Tensor out = buf(q, {M, N}, at::kBFloat16);
    CALL(wdl_fp8_gemm, ptr(q), f32(xs), ptr(w), f32(ws), ptr(bias), M, q.size(0), N, q.size(1), rows, ptr(out),
         out.stride(0), ptr(workspace), str(stream));
    return out;
}

void fp8wo_gemm(const Tensor& x, const Tensor& w, const Tensor& ws, const Opt& bias, const Tensor& out, const Opt& gate,
                uintptr_t stream) {
    const int64_t N = w.size(0);
    CALL(wdl_fp8wo_gemm, ptr(x), x.stride(0), ptr(w), f32(ws), ws.numel() == N && N > 1, ptr(bias), x.size(0), N, x.size(1),
         ptr(out), out.stride(0), gate ? 2 : 0, f32(gate), str(stream));
}

Tensor rope3d(const Tensor& x, const Tensor& freq, const std::vector<int32_t>& grids, int64_t start, bool inverse,
              at::ScalarType type, uintptr_t stream) {
    dims("rope3d x", x, 4, 4);
    dims("rope3d freq", freq, 3, 64);
    if (int64_t(grids.size()) < 3 * x.size(0)) throw std::invalid_argument("rope3d: one grid of 3 sizes per sample");
    Tensor out = buf(x, x.sizes(), type);
    CALL(wdl_rope3d_rotate, ptr(x), code(x.scalar_type()), x.strides().data(), ptr(freq), code(freq.scalar_type()),
         freq.strides().data(), freq.size(1), x.size(0), x.size(1), x.size(2), x.size(3), grids.data(), start, inverse,
         ptr(out), code(type), str(stream));
    return out;
}

// Whether every requirement of cache_fp8.py's _refusal holds (a refusal and its message stay that function's)
bool kv_valid(const Tensor& k, const Tensor& v, const Tensor& ck, const Tensor& cks, const Tensor& cv,
              const Tensor& cvs, int64_t at) {
    if (k.dim() != 4 || v.sizes() != k.sizes() || k.size(3) < 1 || k.size(3) > 1024 || !k.is_cuda()) return false;
    for (const Tensor* t : {&k, &v, &ck, &cks, &cv, &cvs})
        if (t->device() != k.device() || t->requires_grad()) return false;
    for (const Tensor* t : {&k, &v}) {
        const auto d = t->scalar_type();
        if (d != at::kHalf && d != at::kBFloat16 && d != at::kFloat) return false;
    }
    for (const Tensor* t : {&ck, &cv})
        if (t->scalar_type() != at::kFloat8_e4m3fn || t->dim() != 4 || t->size(0) != k.size(0) || t->size(2) != k.size(2) ||
            t->size(3) != k.size(3) || t->size(1) != ck.size(1) || !t->is_contiguous())
            return false;
    for (const Tensor* t : {&cks, &cvs})
        if (t->scalar_type() != at::kFloat || t->dim() != 4 || t->size(0) != ck.size(0) || t->size(1) != ck.size(1) ||
            t->size(2) != ck.size(2) || t->size(3) != 1 || !t->is_contiguous())
            return false;
    return at >= 0 && k.size(1) <= ck.size(1) && at <= ck.size(1) - k.size(1);  // (at + n may not fit 64 bits)
}

// Whether every requirement of sage_kv.py's _check holds for a call without head and token maps
bool attend_valid(const Tensor& q, const Tensor& ck, const Tensor& cks, const Tensor& cv, const Tensor& cvs, int64_t at,
                  const Tensor& k, const Tensor& v) {
    if (q.dim() != 4 || k.dim() != 4 || v.sizes() != k.sizes() || q.size(0) != 1 || k.size(3) != D || q.size(3) != D ||
        q.size(2) != k.size(2))
        return false;
    for (const Tensor* t : {&q, &k, &v})
        if (t->scalar_type() != at::kBFloat16 || t->stride(3) != 1 || t->stride(2) != D) return false;
    for (const Tensor* t : {&ck, &cv})
        if (t->scalar_type() != at::kFloat8_e4m3fn || t->dim() != 4 || t->size(0) != 1 || t->size(1) != ck.size(1) ||
            t->size(2) != k.size(2) || t->size(3) != D || !t->is_contiguous())
            return false;
    for (const Tensor* t : {&cks, &cvs})
        if (t->scalar_type() != at::kFloat || t->dim() != 4 || t->size(0) != 1 || t->size(1) != ck.size(1) ||
            t->size(2) != ck.size(2) || t->size(3) != 1 || !t->is_contiguous())
            return false;
    return at >= 0 && at <= ck.size(1);
}

}  // namespace

PYBIND11_MODULE(wdl_host, m) {
    py::register_exception_translator([](std::exception_ptr p) {  // torch's own type for a failed allocation
        try {
            if (p) std::rethrow_exception(p);
        } catch (const c10::OutOfMemoryError& e) {
            PyErr_SetString(py::module_::import("torch").attr("OutOfMemoryError").ptr(), e.what_without_backtrace());
        }
    });
    m.def("bind", &bind);
    // an allocation or a launch may wait (allocator retry, first module load, full queue): other Python threads run on
    const py::call_guard<py::gil_scoped_release> nogil;
    m.def("act_quant", &act_quant, nogil);
    m.def("gemm", &gemm, nogil);
    m.def("gelu_quant", &gelu_quant, nogil);
    m.def("qk_norm_rope", &qk_norm_rope, nogil);
    m.def("sage_prep", &sage_prep, nogil);
    m.def("sage_attn_q16", &sage_attn_q16, nogil);
    m.def("attn_bf16", &attn_bf16, nogil);
    m.def("kv_append", &kv_append, nogil);
    m.def("fp8_quantize", &fp8_quantize, nogil);
    m.def("fp8_gemm", &fp8_gemm, nogil);
    m.def("fp8wo_gemm", &fp8wo_gemm, nogil);
    m.def("rope3d", &rope3d, nogil);
    m.def("kv_valid", &kv_valid);
    m.def("attend_valid", &attend_valid);
}
