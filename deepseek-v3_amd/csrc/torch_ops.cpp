// Device implementations of the torch.ops.dsv3fp8 operators of the linear, cast and attention layers: allocate the results,
// pass raw pointers and the current stream of the tensors' device to libdsv3fp8.so.
//
// Why native: at a few tokens the launches of a layer are shorter than the host's way to them.  The same bodies in Python
// behind torch.library cost 10 to 14 us an operator (argument boxing, device and stream contexts, two or three ctypes
// calls); one sequence's decode step of the attention layer (five operators, kernels 72 us) was bound by that at 118 us and
// takes 71 with these.
// Scratch memory comes from the caching allocator on each call: it belongs to the current stream, and under stream capture
// to the graph's pool.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <initializer_list>
#include <tuple>

#include "../../include/dsv3_fp8.h"

namespace {

using at::Tensor;
using std::tuple;
typedef c10::optional<Tensor> OptTensor;

constexpr auto kFp8 = at::kFloat8_e4m3fn;

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return DSV3_BF16;
        case at::kHalf: return DSV3_F16;
        case at::kFloat: return DSV3_F32;
        default: TORCH_CHECK_TYPE(false, "dsv3fp8: unsupported dtype ", t, " (bf16, fp16 and fp32 are implemented)");
    }
}
at::ScalarType dtype_of(int64_t code) {
    switch (code) {
        case DSV3_BF16: return at::kBFloat16;
        case DSV3_F16: return at::kHalf;
        case DSV3_F32: return at::kFloat;
        default: TORCH_CHECK_VALUE(false, "dsv3fp8: unknown dtype code ", code);
    }
}
void check(int rc, const char* what) {
    TORCH_CHECK(rc == DSV3_OK, what, " failed: ", dsv3_status_string(rc), " (dsv3_status ", rc, ")");
}

// A block size as the library takes it: one that is cut to 32 bits would not be the one the results are laid out for.
int checked_block(int64_t block, const char* what) {
    TORCH_CHECK(block > 0 && block <= 0x7fffffff, what, ": block_size must be positive and fit 32 bits, got ", block);
    return (int)block;
}

// The device of an operator's tensors made current, and its stream.
struct On {
    c10::DeviceGuard guard;
    void* stream;
    explicit On(const Tensor& t) : guard(t.device()), stream((void*)c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

// The kernels get raw pointers: a tensor of another device or of the host would fault the GPU.  (The dispatcher comes here as
// soon as one argument is on the GPU.)
void on_one_device(const char* what, const Tensor& x, std::initializer_list<const Tensor*> others) {
    for (const Tensor* t : others)
        TORCH_CHECK(t->device() == x.device(), what, ": all tensors must be on one device, got ", x.device(), " and ", t->device());
}
void on_one_gpu(const char* what, const Tensor& x, std::initializer_list<const Tensor*> others) {
    on_one_device(what, x, others);
    TORCH_CHECK(x.is_cuda(), what, ": tensors must be on the GPU, got ", x.device());
}

// The library sees no sizes of its operands: what it will read has to be there (nothing, where the result is empty).
void check_weight(const char* what, const Tensor& b, const Tensor& b_s, int64_t n, int64_t k, int64_t block) {
    if (n == 0 || k == 0) return;
    TORCH_CHECK(b.element_size() == 1 && b.is_contiguous() && b.numel() >= n * k, what, ": the weight must be contiguous, one byte an element, [", n, ", ", k, "]");
    TORCH_CHECK(b_s.scalar_type() == at::kFloat && b_s.is_contiguous() && b_s.numel() >= ((n + block - 1) / block) * ((k + block - 1) / block),
                what, ": the weight's scales must be contiguous fp32, one per block");
}

Tensor scratch(const Tensor& like, size_t bytes) {
    return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
}
Tensor with_last(const Tensor& x, int64_t last, at::ScalarType dtype) {
    auto size = x.sizes().vec();
    size.back() = last;
    return at::empty(size, x.options().dtype(dtype));
}

tuple<Tensor, Tensor> act_quant(const Tensor& x, int64_t block, int64_t fmt) {
    const int bs = checked_block(block, "act_quant");
    const int64_t last = x.size(-1);
    const int code = dtype_code(x.scalar_type());
    Tensor y = at::empty_like(x, x.options().dtype(kFp8)), s = with_last(x, last / bs, at::kFloat);
    On on(x);
    check(dsv3_act_quant(x.data_ptr(), code, y.data_ptr(), (float*)s.data_ptr(), x.numel(), last, bs, (int)fmt, on.stream),
          "dsv3_act_quant");
    return {y, s};
}

Tensor weight_dequant(const Tensor& x, const Tensor& s, int64_t block, int64_t out) {
    TORCH_CHECK_VALUE(x.dim() == 2, "weight_dequant: a matrix is needed");
    const int bs = checked_block(block, "weight_dequant");
    check_weight("weight_dequant", x, s, x.size(0), x.size(1), bs);
    on_one_gpu("weight_dequant", x, { &s });
    Tensor y = at::empty_like(x, x.options().dtype(dtype_of(out)));
    On on(x);
    check(dsv3_weight_dequant(x.data_ptr(), (const float*)s.data_ptr(), y.data_ptr(), (int)out, x.size(0), x.size(1), bs,
                              on.stream), "dsv3_weight_dequant");
    return y;
}

tuple<Tensor, Tensor> weight_quant(const Tensor& w, int64_t block, int64_t fmt) {
    TORCH_CHECK_VALUE(w.dim() == 2, "weight_quant: a matrix is needed");
    const int bs = checked_block(block, "weight_quant");
    const int code = dtype_code(w.scalar_type());
    const int64_t m = w.size(0), n = w.size(1);
    Tensor y = at::empty_like(w, w.options().dtype(kFp8));
    Tensor s = at::empty({(m + bs - 1) / bs, (n + bs - 1) / bs}, w.options().dtype(at::kFloat));
    On on(w);
    check(dsv3_weight_quant(w.data_ptr(), code, y.data_ptr(), (float*)s.data_ptr(), m, n, bs, (int)fmt, on.stream),
          "dsv3_weight_quant");
    return {y, s};
}

// Scratch of the GEMMs.  Taken before the quantised input and the result: cut out of a free block before those, it lies where
// it lay in the call before, and they do not lie in what was scratch there (MLP at 193 rows: 152.9 us; 153.6 with the scratch
// behind the quantised input, 152.8 with a buffer kept for good).
Tensor gemm_scratch(const Tensor& like, int64_t m, int64_t n, int64_t k) {
    const size_t need = dsv3_fp8_gemm_workspace_bytes(m, n, k);
    return need ? scratch(like, need) : Tensor();
}
Tensor gemm(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, int64_t out, const Tensor& ws, int64_t m,
            decltype(dsv3_fp8_gemm)* entry, const char* what, void* stream) {
    const int64_t k = a.size(-1), n = b.size(0);
    Tensor c = with_last(a, n, dtype_of(out));
    check(entry(a.data_ptr(), (const float*)a_s.data_ptr(), b.data_ptr(), (const float*)b_s.data_ptr(), c.data_ptr(), (int)out,
                m, n, k, ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? (size_t)ws.numel() : 0, stream), what);
    return c;
}
Tensor gemm(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, int64_t out, decltype(dsv3_fp8_gemm)* entry,
            const char* what) {
    const int64_t k = a.size(-1), m = k ? a.numel() / k : 0;
    TORCH_CHECK(m == 0 || b.size(0) == 0 || (a.element_size() == 1 && a.is_contiguous() && a_s.scalar_type() == at::kFloat && a_s.is_contiguous() &&
                a_s.numel() >= m * ((k + 127) / 128)), what, ": activations must be contiguous, one byte an element, with fp32 scales per block of 128");
    check_weight(what, b, b_s, m ? b.size(0) : 0, k, 128);
    on_one_gpu(what, a, { &a_s, &b, &b_s });
    On on(a);
    const Tensor ws = gemm_scratch(a, m, b.size(0), k);
    return gemm(a, a_s, b, b_s, out, ws, m, entry, what, on.stream);
}
Tensor fp8_gemm(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, int64_t out) {
    return gemm(a, a_s, b, b_s, out, dsv3_fp8_gemm, "dsv3_fp8_gemm");
}
Tensor fp8_gemm_pow2(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, int64_t out) {
    return gemm(a, a_s, b, b_s, out, dsv3_fp8_gemm_pow2, "dsv3_fp8_gemm_pow2");
}

// act_quant(x, 128, fmt) followed by fp8_gemm, one launch where the library implements it, else two calls
Tensor linear_fp8(const Tensor& x, const Tensor& b, const Tensor& b_s, int64_t fmt, int64_t out) {
    const int64_t k = x.size(-1), m = k ? x.numel() / k : 0, n = b.size(0);
    TORCH_CHECK(x.is_contiguous(), "linear_fp8: x must be contiguous");
    check_weight("linear_fp8", b, b_s, m ? n : 0, k, 128);
    on_one_gpu("linear_fp8", x, { &b, &b_s });
    On on(x);
    const Tensor ws = gemm_scratch(x, m, n, k);
    if (x.scalar_type() != at::kBFloat16 || !dsv3_linear_fp8_fused(m, n, k)) {
        auto [a, a_s] = act_quant(x, 128, fmt);
        return gemm(a, a_s, b, b_s, out, ws, m, dsv3_fp8_gemm, "dsv3_fp8_gemm", on.stream);
    }
    Tensor c = with_last(x, n, dtype_of(out));
    check(dsv3_linear_fp8(x.data_ptr(), DSV3_BF16, b.data_ptr(), (const float*)b_s.data_ptr(), c.data_ptr(), (int)out, m, n, k, 128,
                          (int)fmt, ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? (size_t)ws.numel() : 0, on.stream),
          "dsv3_linear_fp8");
    return c;
}

tuple<Tensor, Tensor> swiglu_quant(const Tensor& h, int64_t block, int64_t fmt) {
    TORCH_CHECK(h.dim() == 2 && h.is_contiguous() && h.size(1) % 2 == 0, "swiglu_quant: a contiguous matrix of even width is needed");
    const int bs = checked_block(block, "swiglu_quant");
    const int code = dtype_code(h.scalar_type());
    const int64_t rows = h.size(0), inter = h.size(1) / 2;
    Tensor y = at::empty({rows, inter}, h.options().dtype(kFp8)), s = at::empty({rows, inter / bs}, h.options().dtype(at::kFloat));
    On on(h);
    check(dsv3_swiglu_quant(h.data_ptr(), code, y.data_ptr(), (float*)s.data_ptr(), rows, inter, bs, (int)fmt, on.stream),
          "dsv3_swiglu_quant");
    return {y, s};
}

void check_caches(const Tensor& kv, const Tensor& pe, int64_t batch, int64_t positions) {
    for (const Tensor* c : {&kv, &pe})
        TORCH_CHECK(c->dim() == 3 && c->scalar_type() == at::kBFloat16 && c->stride(2) == 1 && c->stride(1) == c->size(2) &&
                    c->size(0) >= batch && c->size(1) >= positions, "mla: caches must be bf16 [batch, positions, width] with dense rows");
}
void check_freqs(const Tensor& f, int64_t rows, int64_t rope) {
    TORCH_CHECK(f.scalar_type() == at::kComplexFloat && f.is_contiguous() && f.dim() == 2 && f.size(0) == rows && f.size(1) == rope / 2 &&
                !f.is_conj() && !f.is_neg(), "mla: freqs must be a contiguous complex64 [rows, rope / 2], not lazily conjugated");
}

// What the two attention operators check and pass on alike; `call` gets the shape and the workspace.
template <class Bytes, class Call>
void attention(const Tensor& q, const Tensor& freqs, const Tensor& kv, const Tensor& pe, const Tensor& w, const Tensor& ws,
               const OptTensor& mask, int64_t positions, Bytes bytes, Call call) {
    TORCH_CHECK(q.dim() == 4 && q.is_contiguous() && q.scalar_type() == at::kBFloat16, "mla: q must be a contiguous bf16 [b, s, h, d]");
    const int64_t b = q.size(0), s = q.size(1), h = q.size(2);
    check_caches(kv, pe, b, positions);
    check_freqs(freqs, s, pe.size(2));
    TORCH_CHECK(w.dim() == 2 && w.is_contiguous() && ws.is_contiguous() && w.element_size() == 1 && w.size(1) == kv.size(2) &&
                h > 0 && w.size(0) % h == 0, "mla: wkv_b must be a contiguous fp8 [h * (nope + v), kv_rank]");
    TORCH_CHECK(ws.scalar_type() == at::kFloat && ws.dim() == 2 && ws.size(0) >= (w.size(0) + 127) / 128 && ws.size(1) == (w.size(1) + 127) / 128,
                "mla: wkv_b's scales must be fp32, one per block of 128 x 128");
    if (mask)
        TORCH_CHECK(mask->dim() == 2 && mask->size(0) == s && mask->size(1) == positions && mask->is_contiguous() &&
                    (mask->scalar_type() == at::kBFloat16 || mask->scalar_type() == at::kFloat),
                    "mla: mask must be a contiguous bf16 or fp32 [s, positions]");
    on_one_gpu("mla", q, { &freqs, &kv, &pe, &w, &ws, mask ? &*mask : &q });
    On on(q);
    const size_t need = bytes(b, s, positions, (int)h);
    Tensor buf = scratch(q, need);
    const int rope = (int)pe.size(2), nope = (int)q.size(3) - rope, v = (int)(w.size(0) / h) - nope;
    call(b, s, (int)h, nope, rope, v, mask ? mask->data_ptr() : nullptr, mask ? dtype_code(mask->scalar_type()) : 0, buf.data_ptr(),
         need, on.stream);
}

tuple<Tensor, Tensor> mla_prefill(const Tensor& q, const Tensor& freqs, const Tensor& kv, const Tensor& pe, const Tensor& w,
                                  const Tensor& ws, const OptTensor& mask, int64_t positions, double scale) {
    Tensor y, ys;
    attention(q, freqs, kv, pe, w, ws, mask, positions, dsv3_mla_prefill_workspace_bytes,
              [&](int64_t b, int64_t s, int h, int nope, int rope, int v, void* m, int md, void* buf, size_t need, void* stream) {
        y = at::empty({b, s, (int64_t)h * v}, q.options().dtype(kFp8));
        ys = at::empty({b, s, h}, q.options().dtype(at::kFloat));
        check(dsv3_mla_prefill(q.data_ptr(), (const float*)freqs.data_ptr(), kv.data_ptr(), kv.stride(0), pe.data_ptr(), pe.stride(0),
                               w.data_ptr(), (const float*)ws.data_ptr(), m, md, y.data_ptr(), (float*)ys.data_ptr(), b, s, positions,
                               h, nope, rope, v, kv.size(2), (float)scale, buf, need, stream), "dsv3_mla_prefill");
    });
    return {y, ys};
}

Tensor mla_decode(const Tensor& q, const Tensor& freqs, const Tensor& kv, const Tensor& pe, const Tensor& w, const Tensor& ws,
                  const OptTensor& mask, int64_t positions, double scale) {
    Tensor y;
    attention(q, freqs, kv, pe, w, ws, mask, positions, dsv3_mla_decode_workspace_bytes,
              [&](int64_t b, int64_t s, int h, int nope, int rope, int v, void* m, int md, void* buf, size_t need, void* stream) {
        y = at::empty({b, s, (int64_t)h * v}, q.options());
        check(dsv3_mla_decode(q.data_ptr(), (const float*)freqs.data_ptr(), kv.data_ptr(), kv.stride(0), pe.data_ptr(), pe.stride(0),
                              w.data_ptr(), (const float*)ws.data_ptr(), m, md, y.data_ptr(), b, s, positions, h, nope, rope, v,
                              kv.size(2), (float)scale, buf, need, stream), "dsv3_mla_decode");
    });
    return y;
}
// the same, rounded to bf16 and quantised per (token, head): the output projection's input
tuple<Tensor, Tensor> mla_decode_quant(const Tensor& q, const Tensor& freqs, const Tensor& kv, const Tensor& pe, const Tensor& w,
                                       const Tensor& ws, const OptTensor& mask, int64_t positions, double scale) {
    Tensor y, ys;
    attention(q, freqs, kv, pe, w, ws, mask, positions, dsv3_mla_decode_workspace_bytes,
              [&](int64_t b, int64_t s, int h, int nope, int rope, int v, void* m, int md, void* buf, size_t need, void* stream) {
        y = at::empty({b, s, (int64_t)h * v}, q.options().dtype(kFp8));
        ys = at::empty({b, s, h}, q.options().dtype(at::kFloat));
        check(dsv3_mla_decode_quant(q.data_ptr(), (const float*)freqs.data_ptr(), kv.data_ptr(), kv.stride(0), pe.data_ptr(), pe.stride(0),
                                    w.data_ptr(), (const float*)ws.data_ptr(), m, md, y.data_ptr(), (float*)ys.data_ptr(), b, s, positions,
                                    h, nope, rope, v, kv.size(2), (float)scale, buf, need, stream), "dsv3_mla_decode_quant");
    });
    return {y, ys};
}

// What mla_latent and mla_query need of everything but the projected rows
void check_latent(const Tensor& x, const Tensor& qn, const Tensor& kn, const Tensor& freqs, const Tensor& kv, const Tensor& pe, int64_t start) {
    const int64_t b = x.size(0), s = x.size(1);
    TORCH_CHECK(start >= 0 && kv.dim() == 3 && start <= kv.size(1), "mla_latent: start lies behind the caches' end");     // start + s cannot overflow
    check_caches(kv, pe, b, start + s);
    check_freqs(freqs, s, pe.size(2));
    TORCH_CHECK(kn.numel() == kv.size(2) && qn.scalar_type() == at::kBFloat16 && kn.scalar_type() == at::kBFloat16 &&
                qn.is_contiguous() && kn.is_contiguous(), "mla_latent: norm weights do not fit the row");
    on_one_gpu("mla_latent", x, { &qn, &kn, &freqs, &kv, &pe });
}

// a [b, s, q_rank + kv_rank + rope] -> the normalised query latent, quantised, and the caches' rows start .. start + s - 1
tuple<Tensor, Tensor> mla_latent(const Tensor& a, const Tensor& qn, const Tensor& kn, const Tensor& freqs, Tensor kv, Tensor pe,
                                 int64_t start, double q_eps, double kv_eps) {
    TORCH_CHECK(a.dim() == 3 && a.is_contiguous() && a.scalar_type() == at::kBFloat16 && start >= 0, "mla_latent: a must be a contiguous bf16 [b, s, width]");
    const int64_t b = a.size(0), s = a.size(1), qr = qn.numel();
    check_latent(a, qn, kn, freqs, kv, pe, start);
    const int64_t c = kv.size(2), r = pe.size(2);
    TORCH_CHECK(a.size(2) == qr + c + r, "mla_latent: norm weights do not fit the row");
    Tensor y = at::empty({b, s, qr}, a.options().dtype(kFp8)), ys = at::empty({b, s, qr / 128}, a.options().dtype(at::kFloat));
    On on(a);
    check(dsv3_mla_latent(a.data_ptr(), a.size(2), qn.data_ptr(), kn.data_ptr(), (const float*)freqs.data_ptr(),
                          (char*)kv.data_ptr() + start * c * 2, kv.stride(0), (char*)pe.data_ptr() + start * r * 2, pe.stride(0),
                          y.data_ptr(), (float*)ys.data_ptr(), b, s, qr, c, (int)r, (float)q_eps, (float)kv_eps, on.stream),
          "dsv3_mla_latent");
    return {y, ys};
}

// The operators above as MLA.forward strings them together, in one call each: a decode step of a few sequences is bound by the
// host, and an operator's way through Python and the dispatcher takes 3 to 5 us.
// x [b, s, dim] -> per-head queries [b, s, heads, d]; the caches get the new rows
Tensor mla_query(const Tensor& x, const Tensor& wa, const Tensor& wa_s, const Tensor& qn, const Tensor& kn, const Tensor& freqs,
                 Tensor kv, Tensor pe, int64_t start, double q_eps, double kv_eps, const Tensor& wq, const Tensor& wq_s, int64_t heads) {
    TORCH_CHECK(x.dim() == 3 && heads > 0 && wq.dim() == 2 && wq.size(0) % heads == 0, "mla_query: x must be [b, s, dim], the query's weight [heads * d, q_rank]");
    const int64_t b = x.size(0), s = x.size(1), k = x.size(2), qr = qn.numel(), m = b * s;
    const int64_t n = wa.dim() == 2 ? wa.size(0) : 0;
    on_one_device("mla_query", x, { &wa, &wa_s, &wq, &wq_s });          // before the caches are written
    Tensor y, ys;
    if (m == 0 || k == 0 || x.scalar_type() != at::kBFloat16 || dsv3_linear_fp8_fused(m, n, k)) {
        std::tie(y, ys) = mla_latent(linear_fp8(x, wa, wa_s, DSV3_SCALE_FMT_NONE, DSV3_BF16), qn, kn, freqs, kv, pe, start, q_eps, kv_eps);
    } else {            // the projection's K slices, if it has any, are added by the kernel behind it
        TORCH_CHECK(x.is_contiguous() && kv.dim() == 3 && pe.dim() == 3 && n == qr + kv.size(2) + pe.size(2),
                    "mla_query: x must be contiguous, the projections' weight [q_rank + kv_rank + rope, dim]");
        check_weight("mla_query", wa, wa_s, n, k, 128);
        check_latent(x, qn, kn, freqs, kv, pe, start);
        const int64_t c = kv.size(2), r = pe.size(2);
        On on(x);
        const Tensor scr = gemm_scratch(x, m, n, k);
        const auto [xq, xs] = act_quant(x, 128, DSV3_SCALE_FMT_NONE);
        const Tensor a = at::empty({m, n}, x.options());
        y = at::empty({b, s, qr}, x.options().dtype(kFp8));
        ys = at::empty({b, s, qr / 128}, x.options().dtype(at::kFloat));
        check(dsv3_mla_latent_gemm(xq.data_ptr(), (const float*)xs.data_ptr(), wa.data_ptr(), (const float*)wa_s.data_ptr(), k, a.data_ptr(),
                                   qn.data_ptr(), kn.data_ptr(), (const float*)freqs.data_ptr(), (char*)kv.data_ptr() + start * c * 2,
                                   kv.stride(0), (char*)pe.data_ptr() + start * r * 2, pe.stride(0), y.data_ptr(), (float*)ys.data_ptr(),
                                   b, s, qr, c, (int)r, (float)q_eps, (float)kv_eps, scr.defined() ? scr.data_ptr() : nullptr,
                                   scr.defined() ? (size_t)scr.numel() : 0, on.stream), "dsv3_mla_latent_gemm");
    }
    return fp8_gemm(y, ys, wq, wq_s, DSV3_BF16).view({b, s, heads, wq.size(0) / heads});
}
// queries and caches -> the layer's output [b, s, dim]
Tensor mla_output(const Tensor& q, const Tensor& freqs, const Tensor& kv, const Tensor& pe, const Tensor& w, const Tensor& ws,
                  const OptTensor& mask, int64_t positions, double scale, bool explicit_form, const Tensor& wo, const Tensor& wo_s) {
    on_one_device("mla_output", q, { &wo, &wo_s });
    const auto [y, ys] = (explicit_form ? mla_prefill : mla_decode_quant)(q, freqs, kv, pe, w, ws, mask, positions, scale);
    return fp8_gemm(y, ys, wo, wo_s, DSV3_BF16);
}

}  // namespace

TORCH_LIBRARY_IMPL(dsv3fp8, CUDA, m) {
    m.impl("act_quant", act_quant);
    m.impl("weight_dequant", weight_dequant);
    m.impl("weight_quant", weight_quant);
    m.impl("fp8_gemm", fp8_gemm);
    m.impl("fp8_gemm_pow2", fp8_gemm_pow2);
    m.impl("linear_fp8", linear_fp8);
    m.impl("swiglu_quant", swiglu_quant);
    m.impl("mla_prefill", mla_prefill);
    m.impl("mla_decode", mla_decode);
    m.impl("mla_decode_quant", mla_decode_quant);
    m.impl("mla_latent", mla_latent);
    m.impl("mla_query", mla_query);
    m.impl("mla_output", mla_output);
}
