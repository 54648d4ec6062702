// Python module exl3_amd_torch: the at::Tensor operators of exl3_amd_adapter.cpp, called
// exactly as amp_torch.cpp's bindings call them.  c10::Error raised by an operator reaches
// Python as RuntimeError.
//
// gemm_call / linear_call / mgemm_call are the launch path of ampstein_amd.ops and LinearEXL3:
// the argument checks, the outputs and the C-ABI call of one operator in one native call.  They
// launch only what passes every check; anything else they decline, and the Python statement of
// the operator raises its error (or takes the rarer route).  A 4096 -> 4096 row spent 13 us per
// call in Python checks and ctypes marshalling around a 7 us kernel.
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>

#include "exl3_amd.h"
#include "exl3_amd_adapter.h"

using OptT = c10::optional<at::Tensor>;

namespace
{

constexpr int DECLINED = -1000000;      // below every C-ABI return code

bool given(const OptT& t) { return t.has_value() && t->defined(); }

bool plain(const at::Tensor& t) { return t.is_cuda() && t.is_contiguous(); }

// an absent operand, or a contiguous GPU tensor of the type and at least n elements
bool operand(const OptT& t, at::ScalarType dt, int64_t n)
{
    return !given(t) || (t->scalar_type() == dt && plain(*t) && t->numel() >= n);
}

bool trellis(const at::Tensor& B, bool mcg, bool mul1)
{
    return B.dim() == 3 && (B.scalar_type() == at::kShort || B.scalar_type() == at::kUInt16) && plain(B) && !(mcg && mul1) &&
           (B.size(2) % 16 == 0 || (B.size(2) % 16 == 8 && mul1));
}

float rate(const at::Tensor& B) { return (float) (B.size(2) / 16) + (B.size(2) % 16 ? 0.5f : 0.0f); }

template <class T>
T* ptr(const OptT& t) { return given(t) ? (T*) t->data_ptr() : nullptr; }

void* stream_of(const at::Tensor& t) { return (void*) c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ops.exl3_gemm
int gemm_call(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, const OptT& suh, const OptT& A_had,
              const OptT& svh, int force_shape_idx, bool mcg, bool mul1)
{
    if (!trellis(B, mcg, mul1) || A.dim() < 1 || C.dim() < 1 || A.scalar_type() != at::kHalf) return DECLINED;
    const int64_t k = B.size(0) * 16, n = B.size(1) * 16;
    const bool fp32 = C.scalar_type() == at::kFloat;
    if (k == 0 || A.size(-1) != k || C.size(-1) != n || (!fp32 && C.scalar_type() != at::kHalf)) return DECLINED;
    const int64_t m = A.numel() / k;
    if (C.numel() != m * n || !plain(A) || !plain(C) || !operand(suh, at::kHalf, k) || !operand(svh, at::kHalf, n)) return DECLINED;
    const c10::OptionalDeviceGuard guard(A.device());
    return exl3_amd_gemm((const uint16_t*) A.data_ptr(), (const uint16_t*) B.data_ptr(), C.data_ptr(), fp32,
                         ptr<const uint16_t>(suh), ptr<uint16_t>(A_had), ptr<const uint16_t>(svh), (int) m, (int) k, (int) n,
                         rate(B), mcg, mul1, force_shape_idx, stream_of(A));
}

// LinearEXL3.forward's exl3_gemm route for contiguous 2-D x of at most max_rows rows: y = x @ W
// (+ bias), or None
OptT linear_call(const at::Tensor& x, const at::Tensor& B, const at::Tensor& suh, const at::Tensor& svh, const OptT& bias,
                 bool mcg, bool mul1, int64_t max_rows)
{
    if (x.dim() != 2 || x.size(0) < 1 || x.size(0) > max_rows || x.scalar_type() != at::kHalf || B.dim() != 3) return c10::nullopt;
    const int64_t m = x.size(0), k = B.size(0) * 16, n = B.size(1) * 16;
    if (x.size(1) != k || suh.numel() != k || svh.numel() != n || !x.is_cuda()) return c10::nullopt;
    const c10::OptionalDeviceGuard guard(x.device());
    at::Tensor y = at::empty({ m, n }, x.options());
    OptT A_had;                                   // the kernels of up to 8 rows rotate their input themselves
    if (m > 8) A_had = at::empty_like(x);
    if (gemm_call(x, B, y, suh, A_had, svh, 0, mcg, mul1) < 0) return c10::nullopt;
    return given(bias) ? y.add(*bias) : y;
}

// ops.mgemm without the split norm: stacked (no lists) or sliced (all four)
int mgemm_call(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, const at::Tensor& suh, const OptT& A_had,
               const at::Tensor& svh, double K, bool mcg, bool mul1, const OptT& size_n_list, const OptT& c_ptrs,
               const OptT& n_stride_list, const OptT& had_src_list, int num_had_src)
{
    const bool sliced = given(size_n_list);
    if (given(c_ptrs) != sliced || given(n_stride_list) != sliced || given(had_src_list) != sliced) return DECLINED;
    if (A.dim() != 3 || C.dim() != 3 || A.size(1) != C.size(1) || A.scalar_type() != at::kHalf || !plain(A) || !plain(C))
        return DECLINED;
    const bool fp32 = C.scalar_type() == at::kFloat;
    if (!fp32 && C.scalar_type() != at::kHalf) return DECLINED;
    for (const at::Tensor* t : { &B, &suh, &svh })
        if (t->scalar_type() != at::kLong || t->dim() != 1 || !plain(*t)) return DECLINED;
    if (given(A_had) && !plain(*A_had)) return DECLINED;
    if (!operand(size_n_list, at::kInt, 0) || !operand(c_ptrs, at::kLong, 0) || !operand(n_stride_list, at::kInt, 0) ||
        !operand(had_src_list, at::kInt, 0))
        return DECLINED;
    for (const OptT* t : { &c_ptrs, &n_stride_list, &had_src_list })
        if (given(*t) && (*t)->dim() < 1) return DECLINED;
    const c10::OptionalDeviceGuard guard(A.device());
    return exl3_amd_mgemm((const uint16_t*) A.data_ptr(), (int) A.size(0), (int) A.size(1), (int) A.size(2),
                          (const uint64_t*) B.data_ptr(), (int) B.size(0), C.data_ptr(), (int) C.size(0), (int) C.size(2), fp32,
                          (const uint64_t*) suh.data_ptr(), (int) suh.size(0), ptr<uint16_t>(A_had),
                          given(A_had) ? A_had->numel() : 0, (const uint64_t*) svh.data_ptr(), (int) svh.size(0), nullptr, 0,
                          nullptr, (float) K, -1, mcg, mul1, -1, -1, 0, 1, ptr<const int>(size_n_list),
                          ptr<const uint64_t>(c_ptrs), sliced ? (int) c_ptrs->size(0) : 0, ptr<const int>(n_stride_list),
                          sliced ? (int) n_stride_list->size(0) : 0, ptr<const int>(had_src_list),
                          sliced ? (int) had_src_list->size(0) : 0, num_had_src, stream_of(A));
}

}  // namespace

PYBIND11_MODULE(exl3_amd_torch, m)
{
    m.attr("DECLINED") = DECLINED;
    // without the GIL, as the ctypes calls they stand for: a call can wait (the first one on a device
    // allocates and synchronises, a launch waits on a full queue) while other Python threads run
    const auto nogil = py::call_guard<py::gil_scoped_release>();
    m.def("gemm_call", &gemm_call, nogil);
    m.def("linear_call", &linear_call, nogil);
    m.def("mgemm_call", &mgemm_call, nogil);
    m.def("exl3_gemm", [](const at::Tensor& A, const at::Tensor& B, at::Tensor C, const OptT& suh, const OptT& A_had,
                          const OptT& svh, int force_shape_idx, bool mcg, bool mul1, int force_num_sms) {
        return exl3_gemm(A, B, C, suh, A_had, svh, force_shape_idx, mcg, mul1, force_num_sms);
    });
    m.def("reconstruct", &reconstruct);
    m.def("reconstruct_had_slice", &reconstruct_had_slice);
    m.def("had_r_128", &had_r_128);
    m.def("exl3_mgemm",
          [](const at::Tensor& A, const at::Tensor& B, at::Tensor C, const at::Tensor& suh, const at::Tensor& A_had,
             const at::Tensor& svh, const OptT& indices, const OptT& weights, float K, int force_shape_idx,
             uint32_t mcg_mult, uint32_t mul1_mult, int min_index, int max_index, int force_num_sms, int num_tokens,
             const OptT& size_n_list, const OptT& c_ptrs, const OptT& n_stride_list, const OptT& had_src_list,
             int num_had_src) {
              return exl3_mgemm(A, B, C, suh, A_had, svh, indices, weights, K, force_shape_idx, mcg_mult, mul1_mult,
                                min_index, max_index, force_num_sms, num_tokens, size_n_list, c_ptrs, n_stride_list,
                                had_src_list, num_had_src);
          });
    m.def("exl3_moe_coop",
          [](const at::Tensor& x, const at::Tensor& sel, const at::Tensor& rw, int min_expert, int max_expert, int Hi,
             const at::Tensor& g_trellis, const at::Tensor& g_suh, const at::Tensor& g_svh,
             const at::Tensor& u_trellis, const at::Tensor& u_suh, const at::Tensor& u_svh,
             const at::Tensor& d_trellis, const at::Tensor& d_suh, const at::Tensor& d_svh, const OptT& g_bias,
             const OptT& u_bias, const OptT& d_bias, float Kg, float Ku, float Kd, bool mcg, bool mul1, int act,
             float act_limit, bool gated, at::Tensor had_g, at::Tensor had_u, at::Tensor gu_g, at::Tensor gu_u,
             at::Tensor act_out, at::Tensor d_out, at::Tensor ctr, at::Tensor out, const OptT& sh_out,
             const OptT& sh_gate_w, const OptT& bits_g, const OptT& bits_u, const OptT& bits_d) {
              exl3_moe_coop(x, sel, rw, min_expert, max_expert, Hi, g_trellis, g_suh, g_svh, u_trellis, u_suh, u_svh,
                            d_trellis, d_suh, d_svh, g_bias, u_bias, d_bias, Kg, Ku, Kd, mcg, mul1, act, act_limit,
                            gated, had_g, had_u, gu_g, gu_u, act_out, d_out, ctr, out, sh_out, sh_gate_w, bits_g,
                            bits_u, bits_d);
          });
    m.def("exl3_moe_max_concurrency", &exl3_moe_max_concurrency);
    m.def("exl3_moe_gather", &exl3_moe_gather);
    m.def("exl3_moe", &exl3_moe);
    m.def("rms_norm_res", [](const at::Tensor& x, const at::Tensor& r, const at::Tensor& w, at::Tensor y,
                             at::Tensor n, double eps) {
        const long dim = w.numel();
        const int rc = amp_rms_norm_res_fp16(x.data_ptr(), r.data_ptr(), w.data_ptr(), y.data_ptr(), n.data_ptr(),
                                             x.numel() / std::max(dim, 1L), (int) dim, eps,
                                             (void*) c10::hip::getCurrentHIPStream(x.device().index()).stream());
        TORCH_CHECK(rc == 0, "rms_norm_res: launch failed");
    });
    m.def("silu_mul", [](const at::Tensor& g, const at::Tensor& u, at::Tensor out) {
        const int rc = amp_silu_mul_fp16(g.data_ptr(), u.data_ptr(), out.data_ptr(), g.numel(),
                                         (void*) c10::hip::getCurrentHIPStream(g.device().index()).stream());
        TORCH_CHECK(rc == 0, "silu_mul: launch failed");
    });
}
