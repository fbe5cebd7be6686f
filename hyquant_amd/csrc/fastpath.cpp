// Eager fast paths of a decode step: fused_d_stage_decode
// (src/ops/decode_d_stage.py:470-1005 is the reference's call), the same over
// a layer cache's own buffers, and its staging append
// (src/ops/d_stage_kv_cache.py:195-207).  A Python extension that reads the
// tensors' metadata natively, fills one hyq_decode_params, allocates the
// output and calls hyq_decode_hybrid through the pointer the Python side
// hands over at set-up (the library ctypes loaded, whichever file that is).
//
// decode takes exactly the calls the Python fast path takes (bf16 / fp16 q
// with unit channel stride, kv_repeat dividing the query heads, CUDA tensors,
// the three bf16 segments with unit channel strides, equal K / V lengths and
// one dtype, the quantised prefix with unit innermost strides); decode_cache
// the same over a cache's buffers, with q's heads one stride apart; append
// plain CUDA rows of the buffers' type and device that autograd does not
// record.  Anything else returns status -1 and the caller takes its other
// paths (the checked call, two tensor copies).  The library
// validates every field (alignment, 32-bit strides, sizes) before it
// launches, as for every other caller.  Host code only: no kernel here.

#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <torch/extension.h>

#include <cmath>
#include <cstddef>
#include <cstdint>

#include "../../include/hyq.h"

namespace {

using HybridFn = int (*)(const hyq_decode_params*, void*, size_t, void*);
HybridFn g_hybrid = nullptr;
using AppendFn = decltype(&hyq_append_rows);
AppendFn g_append = nullptr;

// The first n rows (all of them: n < 0) of one bf16 / fp16 segment: 0 empty,
// 1 bf16, 2 fp16, -1 not taken
int segment(const at::Tensor& k, const at::Tensor& v, hyq_decode_params& p, int s, int64_t n = -1) {
    if (k.dim() != 3 || v.dim() != 3) return -1;
    if (v.size(1) != k.size(1) || n > k.size(1)) return k.size(1) == 0 && n <= 0 ? 0 : -1;
    if (n < 0) n = k.size(1);
    if (n == 0) return 0;
    const auto dt = k.scalar_type();
    if (k.stride(2) != 1 || v.stride(2) != 1 || v.scalar_type() != dt) return -1;
    if (dt != at::kBFloat16 && dt != at::kHalf) return -1;
    p.seg_k[s] = static_cast<const uint16_t*>(k.data_ptr());
    p.seg_k_stride_bh[s] = k.stride(0);
    p.seg_k_stride_n[s] = k.stride(1);
    p.seg_v[s] = static_cast<const uint16_t*>(v.data_ptr());
    p.seg_v_stride_bh[s] = v.stride(0);
    p.seg_v_stride_n[s] = v.stride(1);
    p.seg_n[s] = n;
    return dt == at::kBFloat16 ? 1 : 2;
}

using Result = std::tuple<int64_t, at::Tensor>;

// q: query rows of d channels, q_stride apart; nq and ns: the tokens of the
// prefix and of the staging segment (-1: the tensors' own); out_shape: the
// shape of the returned tensor (contiguous, bh_q * d values)
Result run(const at::Tensor& q, int64_t bh_q, int64_t d, int64_t q_stride, at::IntArrayRef out_shape,
           const at::Tensor& kp, const at::Tensor& vp, const at::Tensor& ks, const at::Tensor& vs, int64_t nq,
           const at::Tensor& kt, const at::Tensor& vt, const at::Tensor& kst, const at::Tensor& vst, int64_t ns,
           const at::Tensor& kw, const at::Tensor& vw, int64_t k_bits, int64_t v_bits, int64_t kv_repeat,
           double sm_scale, int64_t split_tokens, int64_t stream, int64_t ws, int64_t ws_bytes) {
    const Result skip{-1, at::Tensor()};
    hyq_decode_params p{};
    const auto qdt = q.scalar_type();
    if (qdt == at::kBFloat16) p.dtype_flags = 0;
    else if (qdt == at::kHalf) p.dtype_flags = HYQ_DT_Q_FP16 | HYQ_DT_OUT_FP16;
    else return skip;
    if (kv_repeat < 1 || bh_q % kv_repeat) return skip;
    int dts = 0;
    const at::Tensor* segs[3][2] = {{&kt, &vt}, {&kst, &vst}, {&kw, &vw}};
    for (int s = 0; s < 3; ++s) {
        const int dt = segment(*segs[s][0], *segs[s][1], p, s, s == 1 ? ns : -1);
        if (dt < 0) return skip;
        if (dt > 0) {
            if (dts && dts != dt) return skip;
            dts = dt;
        }
    }
    if (dts == 2) p.dtype_flags |= HYQ_DT_SEG_FP16;
    if (kp.dim() != 3 || vp.dim() != 3 || ks.dim() != 2 || vs.dim() != 2) return skip;
    if (nq < 0) nq = kp.size(1);
    if (nq > kp.size(1)) return skip;
    if (nq > 0) {
        if (kp.stride(2) != 1 || vp.stride(2) != 1 || ks.stride(1) != 1 || vs.stride(1) != 1) return skip;
        p.k_packed = static_cast<const int8_t*>(kp.data_ptr());
        p.kp_stride_bh = kp.stride(0);
        p.kp_stride_n = kp.stride(1);
        p.v_packed = static_cast<const int8_t*>(vp.data_ptr());
        p.vp_stride_bh = vp.stride(0);
        p.vp_stride_n = vp.stride(1);
        p.k_scale = static_cast<const uint16_t*>(ks.data_ptr());
        p.ks_stride_bh = ks.stride(0);
        p.v_scale = static_cast<const uint16_t*>(vs.data_ptr());
        p.vs_stride_bh = vs.stride(0);
    }
    p.n_quant = nq;
    at::Tensor out = at::empty(out_shape, q.options());
    p.q = static_cast<const uint16_t*>(q.data_ptr());
    p.q_stride = q_stride;
    p.out = static_cast<uint16_t*>(out.data_ptr());
    p.out_stride = d;
    p.bh_kv = static_cast<int32_t>(bh_q / kv_repeat);
    p.kv_repeat = static_cast<int32_t>(kv_repeat);
    p.head_dim = static_cast<int32_t>(d);
    p.k_bits = static_cast<int32_t>(k_bits);
    p.v_bits = static_cast<int32_t>(v_bits);
    // (head_dim ** -0.5 as Python computes it, then rounded to float)
    p.sm_scale = std::isnan(sm_scale) ? static_cast<float>(std::pow(static_cast<double>(d), -0.5))
                                      : static_cast<float>(sm_scale);
    p.split_tokens = static_cast<int32_t>(split_tokens);
    const int st = g_hybrid(&p, reinterpret_cast<void*>(ws), static_cast<size_t>(ws_bytes),
                            reinterpret_cast<void*>(stream));
    return {st, out};
}

}  // namespace

// the library entry points (addresses from ctypes)
void set_entry(int64_t hybrid, int64_t append) {
    g_hybrid = reinterpret_cast<HybridFn>(hybrid);
    g_append = reinterpret_cast<AppendFn>(append);
}

// (status, out): status 0 launched; -1 not taken (nothing launched); any
// other value is the library's status for this call (nothing launched)
Result decode(const at::Tensor& q, const at::Tensor& kp, const at::Tensor& vp, const at::Tensor& ks,
              const at::Tensor& vs, const at::Tensor& kt, const at::Tensor& vt, const at::Tensor& kst,
              const at::Tensor& vst, const at::Tensor& kw, const at::Tensor& vw, int64_t k_bits, int64_t v_bits,
              int64_t kv_repeat, double sm_scale, int64_t split_tokens, int64_t stream, int64_t ws, int64_t ws_bytes) {
    if (!g_hybrid || q.dim() != 2 || !q.is_cuda() || q.stride(1) != 1) return {-1, at::Tensor()};
    return run(q, q.size(0), q.size(1), q.stride(0), {q.size(0), q.size(1)}, kp, vp, ks, vs, -1, kt, vt, kst, vst, -1,
               kw, vw, k_bits, v_bits, kv_repeat, sm_scale, split_tokens, stream, ws, ws_bytes);
}

// One layer's decode step over its cache's own buffers: q [b, hq, 1, d] of the
// cache's batch, the first nq tokens of the prefix store, the first ns rows of
// the staging buffers.  Returns [b, hq, 1, d].
Result decode_cache(const at::Tensor& q, int64_t batch, const at::Tensor& kp, const at::Tensor& vp, const at::Tensor& ks,
                    const at::Tensor& vs, int64_t nq, const at::Tensor& kt, const at::Tensor& vt, const at::Tensor& kst,
                    const at::Tensor& vst, int64_t ns, const at::Tensor& kw, const at::Tensor& vw, int64_t k_bits,
                    int64_t v_bits, int64_t kv_repeat, int64_t stream, int64_t ws, int64_t ws_bytes) {
    const Result skip{-1, at::Tensor()};
    if (!g_hybrid || q.dim() != 4 || !q.is_cuda() || nq < 0 || ns < 0) return skip;
    const int64_t b = q.size(0), h = q.size(1), d = q.size(3);
    // the rows of all heads have to be one stride apart
    if (q.size(2) != 1 || q.stride(3) != 1 || b * h * d == 0 || (h > 1 && b > 1 && q.stride(0) != h * q.stride(1)))
        return skip;
    if (b != batch || kt.size(0) * kv_repeat != b * h) return skip;
    const int64_t row = h > 1 ? q.stride(1) : b > 1 ? q.stride(0) : d;
    return run(q, b * h, d, row, {b, h, 1, d}, kp, vp, ks, vs, nq, kt, vt, kst, vst, ns, kw, vw, k_bits, v_bits,
               kv_repeat, std::nan(""), 0, stream, ws, ws_bytes);
}

// Rows of k and v [b, h, n, d] into staging buffers [b * h, cap, d] at `row`.
// Status 0 launched, -1 not taken (nothing written), else the library's.
int64_t append(const at::Tensor& k, const at::Tensor& v, const at::Tensor& dk, const at::Tensor& dv, int64_t row,
               int64_t stream) {
    if (!g_append || k.dim() != 4 || dk.dim() != 3 || !k.is_cuda() || !v.is_cuda()) return -1;
    if (k.sizes() != v.sizes() || dk.sizes() != dv.sizes() || dk.strides() != dv.strides()) return -1;
    if (k.scalar_type() != dk.scalar_type() || v.scalar_type() != dk.scalar_type() || dv.scalar_type() != dk.scalar_type())
        return -1;
    if (k.device() != dk.device() || v.device() != dk.device() || dk.element_size() != 2) return -1;
    // a copy that autograd records, or a tensor that is not plain memory, goes to copy_
    if (at::GradMode::is_enabled() && (k.requires_grad() || v.requires_grad())) return -1;
    if (k.is_conj() || v.is_conj() || k.is_neg() || v.is_neg()) return -1;
    if (at::isTensorSubclassLike(k) || at::isTensorSubclassLike(v)) return -1;
    const int64_t n = k.size(2), d = k.size(3);
    if (k.size(0) * k.size(1) != dk.size(0) || d != dk.size(2) || row < 0 || row + n > dk.size(1)) return -1;
    if (k.stride(3) != 1 || v.stride(3) != 1 || dk.stride(2) != 1 || dk.stride(1) != d) return -1;
    const c10::DeviceGuard guard(k.device());             // as copy_ does
    return g_append(static_cast<const uint16_t*>(k.data_ptr()), k.stride(0), k.stride(1), k.stride(2),
                    static_cast<const uint16_t*>(v.data_ptr()), v.stride(0), v.stride(1), v.stride(2),
                    static_cast<int32_t>(k.size(0)), static_cast<int32_t>(k.size(1)), n, static_cast<int32_t>(d),
                    static_cast<uint16_t*>(dk.data_ptr()), static_cast<uint16_t*>(dv.data_ptr()), dk.stride(0), row,
                    reinterpret_cast<void*>(stream));
}

// the parameter block's size and the offsets of its first and last fields,
// which the caller compares with its own view of include/hyq.h before it
// uses this module
std::tuple<int64_t, int64_t, int64_t> layout() {
    return {static_cast<int64_t>(sizeof(hyq_decode_params)),
            static_cast<int64_t>(offsetof(hyq_decode_params, seg_n)),
            static_cast<int64_t>(offsetof(hyq_decode_params, dtype_flags))};
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("signatures", [] { return 2; }, "counts up when a function of this module takes other arguments");
    m.def("layout", &layout, "sizeof(hyq_decode_params), offsetof(seg_n), offsetof(dtype_flags)");
    m.def("set_entry", &set_entry, "the addresses of hyq_decode_hybrid and hyq_append_rows");
    m.def("decode", &decode, "fused_d_stage_decode eager fast path");
    m.def("decode_cache", &decode_cache, "a layer cache's decode step");
    m.def("append", &append, "a layer cache's staging append");
}
