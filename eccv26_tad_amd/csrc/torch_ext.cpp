// `opentad_sparse_ops`: the PyTorch-ROCm extension module. Thin layer over the
// C ABI in include/svtad_sparse.h: argument checks, output allocation through
// the caching allocator, and the current HIP stream of the input's device.
//
// The five reference functions keep their names, argument order and meaning
// (opentad/models/bricks/2d_sparse_v3_bind.cpp:8-14); the rest are additions
// the autograd wrapper and the table utilities use.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <tuple>

#include "../../include/svtad_sparse.h"

namespace {

int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return SVTAD_F32;
        case at::kHalf: return SVTAD_F16;
        case at::kBFloat16: return SVTAD_BF16;
        case at::kDouble: return SVTAD_F64;
        default: TORCH_CHECK(false, "opentad_sparse_ops: unsupported dtype ", t.scalar_type());
    }
    return -1;
}

void* stream_of(const at::Tensor& t) {
    return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

void check_status(int st, const char* who) {
    TORCH_CHECK(st == SVTAD_OK, "opentad_sparse_ops.", who, ": ", svtad_last_error(), " (status ",
                st, ")");
}

void check_gpu(const at::Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda(), "opentad_sparse_ops: ", name, " must be a GPU tensor");
}

at::Tensor rows_view(const at::Tensor& t) {
    TORCH_CHECK(t.dim() >= 1, "expected at least 1 dimension");
    return t.contiguous();
}

int64_t n_rows(const at::Tensor& t) { return t.size(-1) == 0 ? 0 : t.numel() / t.size(-1); }

at::Tensor table_i32(const at::Tensor& nbr, int64_t n) {
    check_gpu(nbr, "neighbor_indices");
    TORCH_CHECK(nbr.scalar_type() == at::kInt, "neighbor_indices must be int32, got ",
                nbr.scalar_type());
    TORCH_CHECK(nbr.numel() == n * 9, "neighbor_indices has ", nbr.numel(), " entries, expected ",
                n, " x 9");
    return nbr.contiguous();
}

bool bias_present(const c10::optional<at::Tensor>& b) { return b.has_value() && b->defined() && b->numel() > 0; }

at::Tensor conv_fwd(const at::Tensor& x_in, const at::Tensor& nbr_in, const at::Tensor& w_in,
                    const c10::optional<at::Tensor>& bias_in, int64_t tpb, int bias_mode,
                    int64_t c_out_arg) {
    check_gpu(x_in, "x");
    check_gpu(w_in, "weight");
    at::Tensor x = rows_view(x_in);
    const int64_t c_in = x.size(-1);
    const int64_t n = n_rows(x);
    TORCH_CHECK(w_in.dim() == 3 && w_in.size(0) == 9 && w_in.size(1) == c_in,
                "weight must be (9, C_in, C_out) with C_in = ", c_in, ", got ", w_in.sizes());
    const int64_t c_out = w_in.size(2);
    TORCH_CHECK(c_out_arg < 0 || c_out_arg == c_out, "C_out argument ", c_out_arg,
                " does not match weight.size(2) = ", c_out);
    TORCH_CHECK(w_in.scalar_type() == x.scalar_type(), "x and weight dtypes differ: ",
                x.scalar_type(), " vs ", w_in.scalar_type());
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    at::Tensor bias;
    if (bias_mode != SVTAD_BIAS_NONE && bias_present(bias_in)) {
        TORCH_CHECK(bias_in->numel() == c_out, "bias must have C_out = ", c_out, " elements");
        if (bias_mode == SVTAD_BIAS_FP32 && bias_in->scalar_type() == x.scalar_type()) {
            // widened exactly inside the kernel: no conversion launch
            bias_mode = SVTAD_BIAS_PRE;
            bias = bias_in->contiguous();
        } else {
            const at::ScalarType bt =
                bias_mode == SVTAD_BIAS_FP32
                    ? (x.scalar_type() == at::kDouble ? at::kDouble : at::kFloat)
                    : x.scalar_type();
            bias = bias_in->to(x.device(), bt).contiguous();
        }
        TORCH_CHECK(bias.device() == x.device(), "bias must be on x's device");
    } else {
        bias_mode = SVTAD_BIAS_NONE;
    }
    at::Tensor out = at::empty({n, c_out}, x.options());
    const int dt = dtype_code(x);
    const size_t ws_bytes = svtad_fwd_workspace_bytes((int)c_in, (int)c_out, dt);
    at::Tensor ws;
    if (ws_bytes && n > 0) ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    const int st = svtad_fwd(x.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(),
                             bias.defined() ? bias.data_ptr() : nullptr, bias_mode, out.data_ptr(),
                             ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, n, (int)c_in,
                             (int)c_out, tpb, dt, stream_of(x));
    check_status(st, "fwd");
    return out;
}

}  // namespace

// fwd(x, neighbor_indices, weight, C_out, tokens_per_batch) -> [N, C_out], no bias
// (2d_sparse_v3.cu:751-822)
at::Tensor op_fwd(const at::Tensor& x, const at::Tensor& nbr, const at::Tensor& w, int64_t c_out,
                  int64_t tpb) {
    return conv_fwd(x, nbr, w, c10::nullopt, tpb, SVTAD_BIAS_NONE, c_out);
}

// implicit_gemm_fwd_v2(x, neighbor_indices, weight, bias, tokens_per_batch); an empty
// bias means no bias, bias is added in fp32 (implicit_gemm_v2.cu:197-300)
at::Tensor op_implicit_gemm_fwd_v2(const at::Tensor& x, const at::Tensor& nbr, const at::Tensor& w,
                                   const c10::optional<at::Tensor>& bias, int64_t tpb) {
    return conv_fwd(x, nbr, w, bias, tpb, SVTAD_BIAS_FP32, -1);
}

// implicit_gemm_fwd_v2_chunked(..., chunk_size): same result; chunk_size was a
// memory knob of the reference's host chunk loop (implicit_gemm_v2.cu:306-417),
// which this implementation does not need.
at::Tensor op_implicit_gemm_fwd_v2_chunked(const at::Tensor& x, const at::Tensor& nbr,
                                           const at::Tensor& w,
                                           const c10::optional<at::Tensor>& bias, int64_t tpb,
                                           int64_t chunk_size) {
    TORCH_CHECK(chunk_size > 0, "chunk_size must be positive, got ", chunk_size);
    return conv_fwd(x, nbr, w, bias, tpb, SVTAD_BIAS_FP32, -1);
}

// fwd_bias(x, neighbor_indices, weight, bias, tokens_per_batch, bias_mode)
at::Tensor op_fwd_bias(const at::Tensor& x, const at::Tensor& nbr, const at::Tensor& w,
                       const c10::optional<at::Tensor>& bias, int64_t tpb, int64_t bias_mode) {
    TORCH_CHECK(bias_mode >= 0 && bias_mode <= 2, "bias_mode must be 0, 1 or 2");
    return conv_fwd(x, nbr, w, bias, tpb, (int)bias_mode, -1);
}

// pack_weight(weight, fwd, bwd) -> (packed_fwd, packed_bwd): the weight in the
// fragment order of the matrix-core kernels; an empty tensor for a layout not
// requested or not available for this shape / dtype.
std::tuple<at::Tensor, at::Tensor> op_pack_weight(const at::Tensor& w_in, bool fwd, bool bwd) {
    check_gpu(w_in, "weight");
    TORCH_CHECK(w_in.dim() == 3 && w_in.size(0) == 9, "weight must be (9, C_in, C_out)");
    at::Tensor w = w_in.contiguous();
    const int c_in = (int)w.size(1), c_out = (int)w.size(2);
    const int dt = dtype_code(w);
    const size_t bf = fwd ? svtad_fwd_workspace_bytes(c_in, c_out, dt) : 0;
    const size_t bb = bwd ? svtad_bwd_in_workspace_bytes(c_in, c_out, dt) : 0;
    c10::DeviceGuard g(w.device());
    at::Tensor pf = at::empty({(int64_t)bf}, w.options().dtype(at::kByte));
    at::Tensor pb = at::empty({(int64_t)bb}, w.options().dtype(at::kByte));
    if (bf || bb)
        check_status(svtad_pack_weight(w.data_ptr(), bf ? pf.data_ptr() : nullptr,
                                       bb ? pb.data_ptr() : nullptr, c_in, c_out, dt, stream_of(w)),
                     "pack_weight");
    return {pf, pb};
}

// fwd_packed(x, neighbor_indices, weight, packed_fwd, bias, tokens_per_batch,
// bias_mode): fwd_bias with a weight packed by pack_weight (falls back to
// fwd_bias when packed_fwd is empty or the shape has no packed path).
at::Tensor op_fwd_packed(const at::Tensor& x_in, const at::Tensor& nbr_in, const at::Tensor& w,
                         const at::Tensor& packed, const c10::optional<at::Tensor>& bias_in,
                         int64_t tpb, int64_t bias_mode) {
    TORCH_CHECK(bias_mode >= 0 && bias_mode <= 2, "bias_mode must be 0, 1 or 2");
    if (packed.numel() == 0) return conv_fwd(x_in, nbr_in, w, bias_in, tpb, (int)bias_mode, -1);
    check_gpu(x_in, "x");
    at::Tensor x = rows_view(x_in);
    const int64_t c_in = x.size(-1), n = n_rows(x);
    TORCH_CHECK(w.dim() == 3 && w.size(0) == 9 && w.size(1) == c_in, "weight must be (9, C_in, C_out)");
    TORCH_CHECK(w.scalar_type() == x.scalar_type(), "x and weight dtypes differ");
    const int64_t c_out = w.size(2);
    const int dt = dtype_code(x);
    TORCH_CHECK((size_t)packed.numel() == svtad_fwd_workspace_bytes((int)c_in, (int)c_out, dt),
                "packed_fwd does not match the weight");
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    int mode = (int)bias_mode;
    at::Tensor bias;
    if (mode != SVTAD_BIAS_NONE && bias_present(bias_in)) {
        TORCH_CHECK(bias_in->numel() == c_out, "bias must have C_out = ", c_out, " elements");
        if (mode == SVTAD_BIAS_FP32 && bias_in->scalar_type() == x.scalar_type()) {
            mode = SVTAD_BIAS_PRE;
            bias = bias_in->contiguous();
        } else {
            bias = bias_in->to(x.device(), mode == SVTAD_BIAS_FP32 ? at::kFloat : x.scalar_type()).contiguous();
        }
    } else {
        mode = SVTAD_BIAS_NONE;
    }
    at::Tensor out = at::empty({n, c_out}, x.options());
    const int st = svtad_fwd_packed(x.data_ptr(), nbr.data_ptr<int32_t>(), packed.data_ptr(),
                                    bias.defined() ? bias.data_ptr() : nullptr, mode, out.data_ptr(),
                                    n, (int)c_in, (int)c_out, tpb, dt, stream_of(x));
    if (st == SVTAD_ERR_UNSUPPORTED) return conv_fwd(x_in, nbr_in, w, bias_in, tpb, (int)bias_mode, -1);
    check_status(st, "fwd_packed");
    return out;
}

// table_flags from the `symmetric` keyword of the backward ops: the caller's
// promise that every table entry has its partner (SVTAD_TABLE_SYMMETRIC)
static unsigned table_flags(bool symmetric) { return symmetric ? (unsigned)SVTAD_TABLE_SYMMETRIC : 0u; }

static at::Tensor bwd_in_raw(const at::Tensor& go_in, const at::Tensor& nbr_in, const at::Tensor& w_in,
                             int64_t n_kept, int64_t c_in, int64_t tpb, bool symmetric) {
    check_gpu(go_in, "grad_output");
    check_gpu(w_in, "weight");
    at::Tensor go = rows_view(go_in);
    const int64_t c_out = go.size(-1);
    TORCH_CHECK(n_rows(go) == n_kept, "grad_output has ", n_rows(go), " rows, n_kept = ", n_kept);
    TORCH_CHECK(w_in.dim() == 3 && w_in.size(0) == 9 && w_in.size(1) == c_in && w_in.size(2) == c_out,
                "weight must be (9, ", c_in, ", ", c_out, "), got ", w_in.sizes());
    TORCH_CHECK(w_in.scalar_type() == go.scalar_type(), "grad_output and weight dtypes differ");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n_kept);
    c10::DeviceGuard g(go.device());
    at::Tensor gi = at::empty({n_kept, c_in}, go.options());
    const int dt = dtype_code(go);
    const size_t ws_bytes = symmetric ? svtad_bwd_in_workspace_bytes((int)c_in, (int)c_out, dt)
                                      : svtad_bwd_in_ex_workspace_bytes(n_kept, (int)c_in, (int)c_out, dt);
    at::Tensor ws;
    if (ws_bytes && n_kept > 0) ws = at::empty({(int64_t)ws_bytes}, go.options().dtype(at::kByte));
    const int st = svtad_bwd_in_ex(go.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(), gi.data_ptr(),
                                   ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, n_kept, (int)c_in,
                                   (int)c_out, tpb, dt, table_flags(symmetric), stream_of(go));
    check_status(st, "bwd_in");
    return gi;
}

// bwd_in(grad_output, neighbor_indices, weight, n_kept, C_in, tokens_per_batch)
// -> [n_kept, C_in] in grad_output's dtype (2d_sparse_v3.cu:824-835)
at::Tensor op_bwd_in(const at::Tensor& go, const at::Tensor& nbr, const at::Tensor& w, int64_t n_kept,
                     int64_t c_in, int64_t tpb) {
    return bwd_in_raw(go, nbr, w, n_kept, c_in, tpb, false);
}

// bwd_in_packed(grad_output, neighbor_indices, weight, packed_bwd, n_kept, C_in,
// tokens_per_batch, symmetric=False): bwd_in with a weight packed by
// pack_weight (falls back to bwd_in when packed_bwd is empty or the shape has
// no packed path).
at::Tensor op_bwd_in_packed(const at::Tensor& go_in, const at::Tensor& nbr_in, const at::Tensor& w_in,
                            const at::Tensor& packed, int64_t n_kept, int64_t c_in, int64_t tpb,
                            bool symmetric) {
    if (packed.numel() == 0) return bwd_in_raw(go_in, nbr_in, w_in, n_kept, c_in, tpb, symmetric);
    check_gpu(go_in, "grad_output");
    at::Tensor go = rows_view(go_in);
    const int64_t c_out = go.size(-1);
    TORCH_CHECK(n_rows(go) == n_kept, "grad_output has ", n_rows(go), " rows, n_kept = ", n_kept);
    TORCH_CHECK(w_in.dim() == 3 && w_in.size(0) == 9 && w_in.size(1) == c_in && w_in.size(2) == c_out,
                "weight must be (9, ", c_in, ", ", c_out, ")");
    TORCH_CHECK(w_in.scalar_type() == go.scalar_type(), "grad_output and weight dtypes differ");
    const int dt = dtype_code(go);
    TORCH_CHECK((size_t)packed.numel() == svtad_bwd_in_workspace_bytes((int)c_in, (int)c_out, dt),
                "packed_bwd does not match the weight");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n_kept);
    c10::DeviceGuard g(go.device());
    at::Tensor gi = at::empty({n_kept, c_in}, go.options());
    const int st = svtad_bwd_in_packed_ex(go.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(),
                                          packed.data_ptr(), gi.data_ptr(), n_kept, (int)c_in,
                                          (int)c_out, tpb, dt, table_flags(symmetric), stream_of(go));
    if (st == SVTAD_ERR_UNSUPPORTED) return bwd_in_raw(go_in, nbr_in, w_in, n_kept, c_in, tpb, symmetric);
    check_status(st, "bwd_in_packed");
    return gi;
}

// bwd_in_gemm(grad_output, neighbor_indices, packed_bwd, C_in, tokens_per_batch) -> [n, C_in]:
// backward-input's gathered GEMM alone (timing; equals bwd_in_packed for
// tables whose entries all have their symmetric partner)
at::Tensor op_bwd_in_gemm(const at::Tensor& go_in, const at::Tensor& nbr_in, const at::Tensor& packed,
                          int64_t c_in, int64_t tpb, bool symmetric) {
    check_gpu(go_in, "grad_output");
    at::Tensor go = rows_view(go_in);
    const int64_t n = n_rows(go), c_out = go.size(-1);
    const int dt = dtype_code(go);
    TORCH_CHECK(packed.numel() > 0 &&
                    (size_t)packed.numel() == svtad_bwd_in_workspace_bytes((int)c_in, (int)c_out, dt),
                "packed_bwd does not match C_in x C_out in grad_output's dtype");
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(go.device());
    at::Tensor gi = at::empty({n, c_in}, go.options());
    check_status(svtad_bwd_in_gemm(go.data_ptr(), nbr.data_ptr<int32_t>(), packed.data_ptr(), gi.data_ptr(), n,
                                   (int)c_in, (int)c_out, tpb, dt, table_flags(symmetric), stream_of(go)),
                 "bwd_in_gemm");
    return gi;
}

// bwd_w_bias(grad_output, x, neighbor_indices, C_in, tokens_per_batch, with_bias)
// -> (grad_weight [9, C_in, C_out] in x's dtype, grad_bias [C_out] or empty)
std::tuple<at::Tensor, at::Tensor> op_bwd_w_bias(const at::Tensor& go_in, const at::Tensor& x_in,
                                                 const at::Tensor& nbr_in, int64_t c_in,
                                                 int64_t tpb, bool with_bias) {
    check_gpu(go_in, "grad_output");
    check_gpu(x_in, "x");
    at::Tensor go = rows_view(go_in);
    at::Tensor x = rows_view(x_in);
    TORCH_CHECK(x.size(-1) == c_in, "x has ", x.size(-1), " channels, C_in = ", c_in);
    const int64_t n = n_rows(x);
    TORCH_CHECK(n_rows(go) == n, "grad_output has ", n_rows(go), " rows, x has ", n);
    TORCH_CHECK(go.scalar_type() == x.scalar_type(), "grad_output and x dtypes differ");
    const int64_t c_out = go.size(-1);
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    const int dt = dtype_code(x);
    const size_t ws_bytes = svtad_bwd_w_workspace_bytes(n, (int)c_in, (int)c_out, dt);
    TORCH_CHECK(ws_bytes > 0, "bwd_w: ", svtad_last_error());
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    at::Tensor gw = at::empty({9, c_in, c_out}, x.options());
    at::Tensor gb = with_bias ? at::empty({c_out}, x.options()) : at::Tensor();
    const int st = svtad_bwd_w(go.data_ptr(), x.data_ptr(), nbr.data_ptr<int32_t>(), gw.data_ptr(),
                               with_bias ? gb.data_ptr() : nullptr, ws.data_ptr(), ws_bytes, n,
                               (int)c_in, (int)c_out, tpb, dt, stream_of(x));
    check_status(st, "bwd_w");
    return {gw, with_bias ? gb : at::empty({0}, x.options())};
}

// bwd_packed(grad_output, x, neighbor_indices, weight, packed_bwd, C_in,
// tokens_per_batch, with_bias) -> (grad_input [n, C_in], grad_weight, grad_bias
// or empty): the autograd backward in one call (what bwd_in_packed and
// bwd_w_bias give, with one launch less); falls back to those two when
// packed_bwd is empty or the shape has no packed path.
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_bwd_packed(const at::Tensor& go_in, const at::Tensor& x_in,
                                                             const at::Tensor& nbr_in, const at::Tensor& w_in,
                                                             const at::Tensor& packed, int64_t c_in,
                                                             int64_t tpb, bool with_bias, bool symmetric) {
    check_gpu(go_in, "grad_output");
    check_gpu(x_in, "x");
    at::Tensor go = rows_view(go_in);
    at::Tensor x = rows_view(x_in);
    TORCH_CHECK(x.size(-1) == c_in, "x has ", x.size(-1), " channels, C_in = ", c_in);
    const int64_t n = n_rows(x), c_out = go.size(-1);
    auto separate = [&]() {
        at::Tensor gi = op_bwd_in_packed(go_in, nbr_in, w_in, packed, n, c_in, tpb, symmetric);
        auto gwb = op_bwd_w_bias(go_in, x_in, nbr_in, c_in, tpb, with_bias);
        return std::make_tuple(gi, std::get<0>(gwb), std::get<1>(gwb));
    };
    if (packed.numel() == 0) return separate();
    TORCH_CHECK(n_rows(go) == n, "grad_output has ", n_rows(go), " rows, x has ", n);
    TORCH_CHECK(go.scalar_type() == x.scalar_type() && w_in.scalar_type() == x.scalar_type(),
                "grad_output, x and weight dtypes differ");
    TORCH_CHECK(w_in.dim() == 3 && w_in.size(0) == 9 && w_in.size(1) == c_in && w_in.size(2) == c_out,
                "weight must be (9, ", c_in, ", ", c_out, ")");
    const int dt = dtype_code(x);
    TORCH_CHECK((size_t)packed.numel() == svtad_bwd_in_workspace_bytes((int)c_in, (int)c_out, dt),
                "packed_bwd does not match the weight");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    const size_t ws_bytes = svtad_bwd_w_workspace_bytes(n, (int)c_in, (int)c_out, dt);
    TORCH_CHECK(ws_bytes > 0, "bwd_packed: ", svtad_last_error());
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    at::Tensor gi = at::empty({n, c_in}, x.options());
    at::Tensor gw = at::empty({9, c_in, c_out}, x.options());
    at::Tensor gb = with_bias ? at::empty({c_out}, x.options()) : at::Tensor();
    const int st = svtad_bwd_packed_ex(go.data_ptr(), x.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(),
                                       packed.data_ptr(), gi.data_ptr(), gw.data_ptr(),
                                       with_bias ? gb.data_ptr() : nullptr, ws.data_ptr(), ws_bytes, n,
                                       (int)c_in, (int)c_out, tpb, dt, table_flags(symmetric), stream_of(x));
    if (st == SVTAD_ERR_UNSUPPORTED) return separate();
    check_status(st, "bwd_packed");
    return {gi, gw, with_bias ? gb : at::empty({0}, x.options())};
}

// bwd_w_partials(grad_output, x, neighbor_indices, C_in, tokens_per_batch, with_bias)
// -> workspace bytes holding the row-split partial sums only (no reduction).
// For timing the partial-sum kernel of backward-weight on its own.
at::Tensor op_bwd_w_partials(const at::Tensor& go_in, const at::Tensor& x_in, const at::Tensor& nbr_in,
                             int64_t c_in, int64_t tpb, bool with_bias) {
    check_gpu(go_in, "grad_output");
    check_gpu(x_in, "x");
    at::Tensor go = rows_view(go_in);
    at::Tensor x = rows_view(x_in);
    TORCH_CHECK(x.size(-1) == c_in, "x has ", x.size(-1), " channels, C_in = ", c_in);
    const int64_t n = n_rows(x), c_out = go.size(-1);
    TORCH_CHECK(n_rows(go) == n && go.scalar_type() == x.scalar_type(), "grad_output must match x");
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    const int dt = dtype_code(x);
    const size_t ws_bytes = svtad_bwd_w_workspace_bytes(n, (int)c_in, (int)c_out, dt);
    TORCH_CHECK(ws_bytes > 0, "bwd_w_partials: ", svtad_last_error());
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    at::Tensor gb = with_bias ? at::empty({c_out}, x.options()) : at::Tensor();
    check_status(svtad_bwd_w(go.data_ptr(), x.data_ptr(), nbr.data_ptr<int32_t>(), nullptr,
                             with_bias ? gb.data_ptr() : nullptr, ws.data_ptr(), ws_bytes, n,
                             (int)c_in, (int)c_out, tpb, dt, stream_of(x)),
                 "bwd_w_partials");
    return ws;
}

// bwd_w(grad_output, x, neighbor_indices, C_in, tokens_per_batch) -> [9, C_in, C_out]
// (2d_sparse_v3.cu:837-850)
at::Tensor op_bwd_w(const at::Tensor& go, const at::Tensor& x, const at::Tensor& nbr, int64_t c_in,
                    int64_t tpb) {
    return std::get<0>(op_bwd_w_bias(go, x, nbr, c_in, tpb, false));
}

// ---------------------------------------------------------------------------
// depthwise (groups = C), weight (9, C)
// ---------------------------------------------------------------------------

at::Tensor op_dw_fwd(const at::Tensor& x_in, const at::Tensor& nbr_in, const at::Tensor& w_in,
                     const c10::optional<at::Tensor>& bias_in, int64_t tpb) {
    check_gpu(x_in, "x");
    at::Tensor x = rows_view(x_in);
    const int64_t c = x.size(-1), n = n_rows(x);
    TORCH_CHECK(w_in.dim() == 2 && w_in.size(0) == 9 && w_in.size(1) == c,
                "depthwise weight must be (9, ", c, "), got ", w_in.sizes());
    TORCH_CHECK(w_in.scalar_type() == x.scalar_type(), "x and weight dtypes differ");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    at::Tensor bias;
    if (bias_present(bias_in)) bias = bias_in->to(x.device(), x.scalar_type()).contiguous();
    at::Tensor out = at::empty({n, c}, x.options());
    const int st = svtad_dw_fwd(x.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(),
                                bias.defined() ? bias.data_ptr() : nullptr, out.data_ptr(), n, (int)c,
                                tpb, dtype_code(x), stream_of(x));
    check_status(st, "dw_fwd");
    return out;
}

at::Tensor op_dw_bwd_in(const at::Tensor& go_in, const at::Tensor& nbr_in, const at::Tensor& w_in,
                        int64_t tpb, bool symmetric) {
    check_gpu(go_in, "grad_output");
    at::Tensor go = rows_view(go_in);
    const int64_t c = go.size(-1), n = n_rows(go);
    TORCH_CHECK(w_in.dim() == 2 && w_in.size(0) == 9 && w_in.size(1) == c,
                "depthwise weight must be (9, ", c, ")");
    TORCH_CHECK(w_in.scalar_type() == go.scalar_type(), "grad_output and weight dtypes differ");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(go.device());
    at::Tensor gi = at::empty({n, c}, go.options());
    const int st = svtad_dw_bwd_in_ex(go.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(), gi.data_ptr(), n,
                                      (int)c, tpb, dtype_code(go), table_flags(symmetric), stream_of(go));
    check_status(st, "dw_bwd_in");
    return gi;
}

std::tuple<at::Tensor, at::Tensor> op_dw_bwd_w(const at::Tensor& go_in, const at::Tensor& x_in,
                                               const at::Tensor& nbr_in, int64_t tpb,
                                               bool with_bias) {
    check_gpu(go_in, "grad_output");
    at::Tensor go = rows_view(go_in);
    at::Tensor x = rows_view(x_in);
    const int64_t c = x.size(-1), n = n_rows(x);
    TORCH_CHECK(go.size(-1) == c && n_rows(go) == n, "grad_output must match x's shape");
    TORCH_CHECK(go.scalar_type() == x.scalar_type(), "grad_output and x dtypes differ");
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    const int dt = dtype_code(x);
    const size_t ws_bytes = svtad_dw_bwd_w_workspace_bytes(n, (int)c, dt);
    TORCH_CHECK(ws_bytes > 0, "dw_bwd_w: ", svtad_last_error());
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    at::Tensor gw = at::empty({9, c}, x.options());
    at::Tensor gb = with_bias ? at::empty({c}, x.options()) : at::empty({0}, x.options());
    const int st = svtad_dw_bwd_w(go.data_ptr(), x.data_ptr(), nbr.data_ptr<int32_t>(), gw.data_ptr(),
                                  with_bias ? gb.data_ptr() : nullptr, ws.data_ptr(), ws_bytes, n,
                                  (int)c, tpb, dt, stream_of(x));
    check_status(st, "dw_bwd_w");
    return {gw, gb};
}

// dw_bwd(grad_output, x, table, weight, tpb, with_bias) -> (grad_in, grad_w, grad_bias):
// dw_bwd_in and dw_bwd_w in one call (one pass over the rows + one reduction)
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_dw_bwd(const at::Tensor& go_in, const at::Tensor& x_in,
                                                         const at::Tensor& nbr_in, const at::Tensor& w_in,
                                                         int64_t tpb, bool with_bias, bool symmetric) {
    check_gpu(go_in, "grad_output");
    at::Tensor go = rows_view(go_in);
    at::Tensor x = rows_view(x_in);
    const int64_t c = x.size(-1), n = n_rows(x);
    TORCH_CHECK(go.size(-1) == c && n_rows(go) == n, "grad_output must match x's shape");
    TORCH_CHECK(go.scalar_type() == x.scalar_type(), "grad_output and x dtypes differ");
    TORCH_CHECK(w_in.dim() == 2 && w_in.size(0) == 9 && w_in.size(1) == c,
                "depthwise weight must be (9, ", c, ")");
    TORCH_CHECK(w_in.scalar_type() == x.scalar_type(), "x and weight dtypes differ");
    at::Tensor w = w_in.contiguous();
    at::Tensor nbr = table_i32(nbr_in, n);
    c10::DeviceGuard g(x.device());
    const int dt = dtype_code(x);
    const size_t ws_bytes = svtad_dw_bwd_workspace_bytes(n, (int)c, dt);
    TORCH_CHECK(ws_bytes > 0, "dw_bwd: ", svtad_last_error());
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
    at::Tensor gi = at::empty({n, c}, x.options());
    at::Tensor gw = at::empty({9, c}, x.options());
    at::Tensor gb = with_bias ? at::empty({c}, x.options()) : at::empty({0}, x.options());
    const int st = svtad_dw_bwd_ex(go.data_ptr(), x.data_ptr(), nbr.data_ptr<int32_t>(), w.data_ptr(),
                                   gi.data_ptr(), gw.data_ptr(), with_bias ? gb.data_ptr() : nullptr, ws.data_ptr(),
                                   ws_bytes, n, (int)c, tpb, dt, table_flags(symmetric), stream_of(x));
    check_status(st, "dw_bwd");
    return {gi, gw, gb};
}

// ---------------------------------------------------------------------------
// neighbor tables
// ---------------------------------------------------------------------------

// build_neighbor_table(mask [..., H, W] bool/uint8) -> int32 [N, 9]
at::Tensor op_build_neighbor_table(const at::Tensor& mask_in) {
    check_gpu(mask_in, "mask");
    TORCH_CHECK(mask_in.dim() >= 2, "mask must be [..., H, W]");
    TORCH_CHECK(mask_in.scalar_type() == at::kBool || mask_in.scalar_type() == at::kByte,
                "mask must be bool or uint8");
    at::Tensor mask = mask_in.contiguous();
    if (mask.scalar_type() == at::kBool) mask = mask.view(at::kByte);
    const int64_t h = mask.size(-2), w = mask.size(-1);
    const int64_t frames = h * w == 0 ? 0 : mask.numel() / (h * w);
    c10::DeviceGuard g(mask.device());
    at::Tensor offs = at::empty({frames + 1}, mask.options().dtype(at::kInt));
    void* s = stream_of(mask);
    check_status(svtad_table_scan(mask.data_ptr<uint8_t>(), frames, (int)h, (int)w,
                                  offs.data_ptr<int32_t>(), s),
                 "build_neighbor_table");
    const int64_t n = offs[frames].item<int32_t>();  // host sync: sizes the output
    at::Tensor table = at::empty({n, 9}, mask.options().dtype(at::kInt));
    if (n == 0) return table;
    check_status(svtad_table_fill(mask.data_ptr<uint8_t>(), offs.data_ptr<int32_t>(), frames, (int)h,
                                  (int)w, table.data_ptr<int32_t>(), s),
                 "build_neighbor_table");
    return table;
}

// build_neighbor_table_n(mask [..., H, W], n_rows, int64_out) -> [n_rows, 9]: no host sync
// (the caller knows the kept count); masks past 4 MiB take scan + fill without a sync
at::Tensor op_build_neighbor_table_n(const at::Tensor& mask_in, int64_t n_rows, bool int64_out) {
    check_gpu(mask_in, "mask");
    TORCH_CHECK(mask_in.dim() >= 2, "mask must be [..., H, W]");
    TORCH_CHECK(mask_in.scalar_type() == at::kBool || mask_in.scalar_type() == at::kByte,
                "mask must be bool or uint8");
    TORCH_CHECK(n_rows >= 0, "n_rows must be >= 0");
    at::Tensor mask = mask_in.contiguous();
    if (mask.scalar_type() == at::kBool) mask = mask.view(at::kByte);
    if (((uintptr_t)mask.data_ptr() & 15) != 0) mask = mask.clone();
    const int64_t h = mask.size(-2), w = mask.size(-1);
    const int64_t frames = h * w == 0 ? 0 : mask.numel() / (h * w);
    c10::DeviceGuard g(mask.device());
    const auto idx_t = int64_out ? at::kLong : at::kInt;
    void* s = stream_of(mask);
    if (frames * h * w <= ((int64_t)4 << 20)) {
        at::Tensor table = at::empty({n_rows, 9}, mask.options().dtype(idx_t));
        check_status(svtad_table_build(mask.data_ptr<uint8_t>(), frames, (int)h, (int)w, n_rows, table.data_ptr(),
                                       int64_out ? 64 : 32, s),
                     "build_neighbor_table");
        return table;
    }
    // large masks: the scan + fill launches, into a buffer with a row for
    // every cell (the fill writes every kept cell, whatever n_rows says),
    // cut to n_rows
    at::Tensor offs = at::empty({frames + 1}, mask.options().dtype(at::kInt));
    check_status(svtad_table_scan(mask.data_ptr<uint8_t>(), frames, (int)h, (int)w, offs.data_ptr<int32_t>(), s),
                 "build_neighbor_table");
    at::Tensor t32 = at::full({std::max(n_rows, frames * h * w), 9}, -1, mask.options().dtype(at::kInt));
    check_status(svtad_table_fill(mask.data_ptr<uint8_t>(), offs.data_ptr<int32_t>(), frames, (int)h, (int)w,
                                  t32.data_ptr<int32_t>(), s),
                 "build_neighbor_table");
    t32 = t32.narrow(0, 0, n_rows).contiguous();
    return int64_out ? t32.to(at::kLong) : t32;
}

// grid_neighbor_table(frames, h, w, int64_out, like) -> [frames * h * w, 9] on like's device
at::Tensor op_grid_neighbor_table(int64_t frames, int64_t h, int64_t w, bool int64_out, const at::Tensor& like) {
    check_gpu(like, "like");
    TORCH_CHECK(frames >= 0 && h > 0 && w > 0, "bad grid");
    c10::DeviceGuard g(like.device());
    at::Tensor table = at::empty({frames * h * w, 9}, like.options().dtype(int64_out ? at::kLong : at::kInt));
    check_status(svtad_table_grid(frames, (int)h, (int)w, table.data_ptr(), int64_out ? 64 : 32, stream_of(like)),
                 "grid_neighbor_table");
    return table;
}

// table_to_global(table [..., 9] int32/int64, tokens_per_batch) -> int32 [rows, 9]: the
// max() < N heuristic on the device (no host sync)
at::Tensor op_table_to_global(const at::Tensor& table_in, int64_t tokens_per_batch) {
    check_gpu(table_in, "neighbor_indices");
    TORCH_CHECK(table_in.scalar_type() == at::kInt || table_in.scalar_type() == at::kLong,
                "neighbor_indices must be int32 or int64");
    TORCH_CHECK(table_in.numel() % 9 == 0, "neighbor_indices must have 9 entries per row");
    TORCH_CHECK(tokens_per_batch >= 0, "tokens_per_batch must be >= 0");
    at::Tensor table = table_in.contiguous();
    const int64_t rows = table.numel() / 9;
    c10::DeviceGuard g(table.device());
    at::Tensor out = at::empty({rows, 9}, table.options().dtype(at::kInt));
    if (rows == 0) return out;
    at::Tensor vmax = table.max();  // device scalar, no sync
    check_status(svtad_table_to_global(table.data_ptr(), table.scalar_type() == at::kLong ? 64 : 32, rows,
                                       tokens_per_batch, vmax.data_ptr(), out.data_ptr<int32_t>(), stream_of(table)),
                 "table_to_global");
    return out;
}

// remap_neighbor_table(table [B, N_prev, 9] int32, keep_idx [B, N_new] int64) -> [B, N_new, 9]
at::Tensor op_remap_neighbor_table(const at::Tensor& table_in, const at::Tensor& keep_in) {
    check_gpu(table_in, "table");
    check_gpu(keep_in, "keep_idx");
    TORCH_CHECK(table_in.dim() == 3 && table_in.size(2) == 9, "table must be [B, N_prev, 9]");
    TORCH_CHECK(table_in.scalar_type() == at::kInt, "table must be int32");
    TORCH_CHECK(keep_in.dim() == 2 && keep_in.size(0) == table_in.size(0), "keep_idx must be [B, N_new]");
    at::Tensor table = table_in.contiguous();
    at::Tensor keep = keep_in.to(at::kLong).contiguous();
    const int64_t B = table.size(0), n_prev = table.size(1), n_new = keep.size(1);
    c10::DeviceGuard g(table.device());
    at::Tensor mapping = at::empty({B * n_prev}, table.options());
    at::Tensor out = at::empty({B, n_new, 9}, table.options());
    check_status(svtad_remap_table(table.data_ptr<int32_t>(), B, n_prev, keep.data_ptr<int64_t>(),
                                   n_new, mapping.data_ptr<int32_t>(), out.data_ptr<int32_t>(),
                                   stream_of(table)),
                 "remap_neighbor_table");
    return out;
}

// prune_tokens(x [B, n_key + N_prev, ...], keep_idx [B, N_new] int64, last_idx [B, N_prev]
// int64 or empty, table [B, N_prev, 9] int32 or empty, n_key)
//   -> (x_out [B, n_key + N_new, ...], idx_out [B, N_new] or empty, table_out [B, N_new, 9] or empty)
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_prune_tokens(const at::Tensor& x_in,
                                                               const at::Tensor& keep_in,
                                                               const at::Tensor& last_in,
                                                               const at::Tensor& table_in,
                                                               int64_t n_key) {
    check_gpu(x_in, "x");
    check_gpu(keep_in, "keep_idx");
    TORCH_CHECK(x_in.dim() >= 2, "x must be [B, n_key + N_prev, ...]");
    TORCH_CHECK(keep_in.dim() == 2 && keep_in.size(0) == x_in.size(0), "keep_idx must be [B, N_new]");
    const int64_t B = x_in.size(0);
    TORCH_CHECK(n_key >= 0 && n_key <= x_in.size(1), "num_key_tokens out of range");
    const int64_t n_prev = x_in.size(1) - n_key, n_new = keep_in.size(1);
    TORCH_CHECK(n_new <= n_prev, "keep_idx keeps more tokens than there are");
    at::Tensor x = x_in.contiguous();
    at::Tensor keep = keep_in.to(at::kLong).contiguous();
    const bool with_idx = last_in.defined() && last_in.numel() > 0;
    const bool with_table = table_in.defined() && table_in.numel() > 0;
    at::Tensor last, table;
    if (with_idx) {
        check_gpu(last_in, "last_idx");
        TORCH_CHECK(last_in.dim() == 2 && last_in.size(0) == B && last_in.size(1) == n_prev,
                    "last_idx must be [B, N_prev]");
        last = last_in.to(at::kLong).contiguous();
    }
    if (with_table) {
        check_gpu(table_in, "neighbor_indices");
        TORCH_CHECK(table_in.dim() == 3 && table_in.size(0) == B && table_in.size(1) == n_prev &&
                        table_in.size(2) == 9,
                    "neighbor_indices must be [B, N_prev, 9]");
        TORCH_CHECK(table_in.scalar_type() == at::kInt, "neighbor_indices must be int32");
        table = table_in.contiguous();
    }
    c10::DeviceGuard g(x.device());
    std::vector<int64_t> shape = x.sizes().vec();
    shape[1] = n_key + n_new;
    at::Tensor x_out = at::empty(shape, x.options());
    const int64_t rows_in = B * x.size(1);
    const int64_t row_bytes = rows_in > 0 ? x.numel() / rows_in * (int64_t)x.element_size() : 0;
    at::Tensor idx_out = with_idx ? at::empty({B, n_new}, last.options()) : at::empty({0}, keep.options());
    at::Tensor table_out = with_table ? at::empty({B, n_new, 9}, table.options())
                                      : at::empty({0}, keep.options().dtype(at::kInt));
    at::Tensor mapping = with_table ? at::empty({B * n_prev}, table.options()) : at::Tensor();
    check_status(svtad_prune_step(x.data_ptr(), B, n_key, n_prev, row_bytes, keep.data_ptr<int64_t>(),
                                  n_new, with_idx ? last.data_ptr<int64_t>() : nullptr,
                                  with_table ? table.data_ptr<int32_t>() : nullptr,
                                  with_table ? mapping.data_ptr<int32_t>() : nullptr, x_out.data_ptr(),
                                  with_idx ? idx_out.data_ptr<int64_t>() : nullptr,
                                  with_table ? table_out.data_ptr<int32_t>() : nullptr, stream_of(x)),
                 "prune_tokens");
    return {x_out, idx_out, table_out};
}

// transpose_neighbor_table(table [N, 9], tokens_per_batch) -> (table_t [N, 9], collisions [1])
std::tuple<at::Tensor, at::Tensor> op_transpose_neighbor_table(const at::Tensor& table_in,
                                                               int64_t tpb) {
    check_gpu(table_in, "table");
    TORCH_CHECK(table_in.scalar_type() == at::kInt, "table must be int32");
    TORCH_CHECK(table_in.numel() % 9 == 0, "table must have 9 entries per row");
    at::Tensor table = table_in.contiguous();
    const int64_t n = table.numel() / 9;
    c10::DeviceGuard g(table.device());
    at::Tensor tt = at::empty({n, 9}, table.options());
    at::Tensor coll = at::zeros({1}, table.options());
    check_status(svtad_transpose_table(table.data_ptr<int32_t>(), n, tpb, tt.data_ptr<int32_t>(),
                                       coll.data_ptr<int32_t>(), stream_of(table)),
                 "transpose_neighbor_table");
    return {tt, coll};
}

// validate_neighbor_table(table, bound) -> int32 [3] = (entries out of range, min, max)
at::Tensor op_validate_neighbor_table(const at::Tensor& table_in, int64_t bound) {
    check_gpu(table_in, "table");
    TORCH_CHECK(table_in.scalar_type() == at::kInt, "table must be int32");
    at::Tensor table = table_in.contiguous();
    c10::DeviceGuard g(table.device());
    at::Tensor stats = at::empty({3}, table.options());
    check_status(svtad_validate_table(table.data_ptr<int32_t>(), table.numel(), bound,
                                      stats.data_ptr<int32_t>(), stream_of(table)),
                 "validate_neighbor_table");
    return stats;
}

// Adapter GEMMs with fused epilogues (f16 / bf16).
void adapter_common(const at::Tensor& t, const at::Tensor& w, const char* name) {
    check_gpu(t, name);
    check_gpu(w, "weight");
    TORCH_CHECK(t.scalar_type() == w.scalar_type(), name, " and weight dtypes differ");
    TORCH_CHECK(t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16,
                "adapter GEMMs take float16 / bfloat16, got ", t.scalar_type());
    TORCH_CHECK(w.dim() == 2, "weight must be (out_features, in_features)");
}

const void* opt_ptr(const c10::optional<at::Tensor>& b, int64_t n, const at::Tensor& like) {
    if (!bias_present(b)) return nullptr;
    TORCH_CHECK(b->numel() == n && b->scalar_type() == like.scalar_type() && b->is_cuda(),
                "bias must have ", n, " elements of the input dtype");
    TORCH_CHECK(b->is_contiguous(), "bias must be contiguous");
    return b->data_ptr();
}

// adapter_down(x [B, N, k], weight [n, k], bias [n] or None, n_special)
//   -> (pre_act [B, N, n], act_special [B, S, n], act_patch [B * (N - S), n])
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_adapter_down(const at::Tensor& x_in, const at::Tensor& w_in,
                                                               const c10::optional<at::Tensor>& bias,
                                                               int64_t n_special) {
    adapter_common(x_in, w_in, "x");
    TORCH_CHECK(x_in.dim() == 3, "x must be [B, N, C]");
    const int64_t B = x_in.size(0), N = x_in.size(1), k = x_in.size(2), n = w_in.size(0);
    TORCH_CHECK(w_in.size(1) == k, "weight must be (n, ", k, ")");
    TORCH_CHECK(n_special >= 0 && n_special <= N, "n_special out of range");
    at::Tensor x = x_in.contiguous(), w = w_in.contiguous();
    c10::DeviceGuard g(x.device());
    at::Tensor pre = at::empty({B, N, n}, x.options());
    at::Tensor sp = at::empty({B, n_special, n}, x.options());
    at::Tensor pa = at::empty({B * (N - n_special), n}, x.options());
    check_status(svtad_adapter_down(x.data_ptr(), w.data_ptr(), opt_ptr(bias, n, x), pre.data_ptr(),
                                    sp.numel() ? sp.data_ptr() : nullptr, pa.numel() ? pa.data_ptr() : nullptr,
                                    B, N, n_special, (int)k, (int)n, dtype_code(x), stream_of(x)),
                 "adapter_down");
    return {pre, sp, pa};
}

// adapter_up(a_special [B, S, k], a_patch [B * (N - S), k], weight [n, k], bias [n] or None,
//            gamma [1], residual [B, N, n], out_float32=False) -> out [B, N, n]
// a_special, a_patch, weight and bias share the compute dtype T (f16 / bf16).
// gamma and the residual are T, or float32 (the reference under autocast,
// where gamma is a float32 parameter): then z * gamma is an fp32 product and
// the add is fp32, and out is float32 with out_float32, else rounded once to
// T. With a T gamma, residual and out are T.
at::Tensor op_adapter_up(const at::Tensor& sp_in, const at::Tensor& pa_in, const at::Tensor& w_in,
                         const c10::optional<at::Tensor>& bias, const at::Tensor& gamma_in,
                         const at::Tensor& res_in, bool out_float32) {
    check_gpu(res_in, "residual");
    adapter_common(pa_in, w_in, "a_patch");
    TORCH_CHECK(res_in.dim() == 3, "residual must be [B, N, C]");
    const int64_t B = res_in.size(0), N = res_in.size(1), n = res_in.size(2), k = w_in.size(1);
    TORCH_CHECK(w_in.size(0) == n, "weight must be (", n, ", k)");
    TORCH_CHECK(sp_in.dim() == 3 && sp_in.size(0) == B && sp_in.size(2) == k, "a_special must be [B, S, k]");
    const int64_t S = sp_in.size(1);
    TORCH_CHECK(S <= N && pa_in.dim() == 2 && pa_in.size(0) == B * (N - S) && pa_in.size(1) == k,
                "a_patch must be [B * (N - S), k]");
    const at::ScalarType t = pa_in.scalar_type();
    TORCH_CHECK(sp_in.scalar_type() == t, "a_special and a_patch must share the dtype");
    auto t_or_f32 = [&](const at::Tensor& v) { return v.scalar_type() == t || v.scalar_type() == at::kFloat; };
    TORCH_CHECK(t_or_f32(gamma_in) && t_or_f32(res_in), "gamma and residual must be of the input dtype or float32");
    const bool g32 = gamma_in.scalar_type() == at::kFloat;
    TORCH_CHECK(g32 || (res_in.scalar_type() == t && !out_float32),
                "a float32 residual or output needs a float32 gamma");
    TORCH_CHECK(gamma_in.numel() == 1 && gamma_in.is_cuda(), "gamma must be one element on the GPU");
    at::Tensor sp = sp_in.contiguous(), pa = pa_in.contiguous(), w = w_in.contiguous(),
               res = res_in.contiguous(), gm = gamma_in.contiguous();
    c10::DeviceGuard g(res.device());
    at::Tensor out = at::empty({B, N, n}, res.options().dtype(out_float32 ? at::kFloat : t));
    const int dt = dtype_code(pa);
    check_status(svtad_adapter_up_mixed(sp.numel() ? sp.data_ptr() : nullptr, pa.numel() ? pa.data_ptr() : nullptr,
                                        w.data_ptr(), opt_ptr(bias, n, pa), gm.data_ptr(), res.data_ptr(),
                                        out.data_ptr(), B, N, S, (int)k, (int)n, dt, dtype_code(gm),
                                        dtype_code(res), dtype_code(out), stream_of(res)),
                 "adapter_up");
    return out;
}

// heatmap_add_(patch [R, C], special [*, C], src_rows int32 [R], gate [1]) -> patch,
// in place: patch[i] += special[src_rows[i]] * gate (rounded as the unfused chain)
at::Tensor op_heatmap_add_(at::Tensor patch, const at::Tensor& special_in, const at::Tensor& src_in,
                           const at::Tensor& gate_in) {
    adapter_common(patch, patch, "patch");
    TORCH_CHECK(patch.dim() == 2 && patch.is_contiguous(), "patch must be a contiguous [rows, cols] tensor");
    check_gpu(special_in, "special");
    check_gpu(src_in, "src_rows");
    check_gpu(gate_in, "gate");
    TORCH_CHECK(special_in.scalar_type() == patch.scalar_type() &&
                    (gate_in.scalar_type() == patch.scalar_type() || gate_in.scalar_type() == at::kFloat),
                "special and patch must share the dtype; gate is of that dtype or float32");
    const int64_t rows = patch.size(0), cols = patch.size(1);
    TORCH_CHECK(special_in.size(-1) == cols, "special must have ", cols, " columns");
    TORCH_CHECK(src_in.scalar_type() == at::kInt && src_in.numel() == rows, "src_rows must be int32 [rows]");
    TORCH_CHECK(gate_in.numel() == 1, "gate must be one element");
    at::Tensor sp = special_in.contiguous(), src = src_in.contiguous(), gate = gate_in.contiguous();
    c10::DeviceGuard g(patch.device());
    check_status(svtad_heatmap_add_mixed(patch.data_ptr(), sp.numel() ? sp.data_ptr() : nullptr,
                                         src.data_ptr<int32_t>(), gate.data_ptr(), rows, n_rows(sp), (int)cols,
                                         dtype_code(patch), dtype_code(gate), stream_of(patch)),
                 "heatmap_add_");
    return patch;
}

// linear_wgrad(g [*, c_g], rows int32 [n] or empty, x [n, c_x], out_float32=False) -> out [c_g, c_x]
// (in x's dtype, or the unrounded fp32 sums with out_float32)
// (out = g[rows]^T x, or g^T x with the first n rows of g when rows is empty)
at::Tensor op_linear_wgrad(const at::Tensor& g_in, const at::Tensor& rows_in, const at::Tensor& x_in,
                           bool out_float32) {
    adapter_common(g_in, g_in, "g");
    check_gpu(x_in, "x");
    TORCH_CHECK(x_in.scalar_type() == g_in.scalar_type(), "g and x dtypes differ");
    TORCH_CHECK(g_in.dim() == 2 && x_in.dim() == 2, "g and x must be 2-D");
    const int64_t n = x_in.size(0), c_g = g_in.size(1), c_x = x_in.size(1);
    const bool with_rows = rows_in.defined() && rows_in.numel() > 0;
    at::Tensor rows;
    if (with_rows) {
        check_gpu(rows_in, "rows");
        TORCH_CHECK(rows_in.scalar_type() == at::kInt && rows_in.numel() == n, "rows must be int32 [n]");
        rows = rows_in.contiguous();
    } else {
        TORCH_CHECK(g_in.size(0) >= n, "g has fewer rows than x");
    }
    at::Tensor g = g_in.contiguous(), x = x_in.contiguous();
    c10::DeviceGuard guard(x.device());
    at::Tensor out = at::empty({c_g, c_x}, x.options().dtype(out_float32 ? at::kFloat : x.scalar_type()));
    const size_t ws = svtad_linear_wgrad_workspace_bytes(n, (int)c_g, (int)c_x, dtype_code(x));
    at::Tensor work = at::empty({(int64_t)std::max<size_t>(ws, 1)}, x.options().dtype(at::kByte));
    check_status(svtad_linear_wgrad_mixed(g.data_ptr(), with_rows ? rows.data_ptr<int32_t>() : nullptr,
                                          x.data_ptr(), out.data_ptr(), work.data_ptr(), ws, n, g.size(0),
                                          (int)c_g, (int)c_x, dtype_code(x), dtype_code(out), stream_of(x)),
                 "linear_wgrad");
    return out;
}

// column_sums(a [rows, cols]) -> [cols]: sum over rows, fp32 accumulation, ordered
at::Tensor op_column_sums(const at::Tensor& a_in) {
    adapter_common(a_in, a_in, "a");
    at::Tensor a = a_in.contiguous();
    const int64_t rows = a.size(0), cols = a.size(1);
    c10::DeviceGuard guard(a.device());
    at::Tensor out = at::empty({cols}, a.options());
    const size_t ws = svtad_column_sums_workspace_bytes(rows, (int)cols, dtype_code(a));
    at::Tensor work = at::empty({(int64_t)std::max<size_t>(ws, 1)}, a.options().dtype(at::kByte));
    check_status(svtad_column_sums(a.data_ptr(), out.data_ptr(), work.data_ptr(), ws, rows, (int)cols,
                                   dtype_code(a), stream_of(a)),
                 "column_sums");
    return out;
}

// gelu_backward_split(grad_special [B, S, n] or None, grad_patch [B * (N - S), n] or None,
//                     pre_act [B, N, n], n_special) -> grad_pre [B, N, n]
at::Tensor op_gelu_backward_split(const c10::optional<at::Tensor>& g_sp, const c10::optional<at::Tensor>& g_pa,
                                  const at::Tensor& pre_in, int64_t n_special) {
    check_gpu(pre_in, "pre_act");
    TORCH_CHECK(pre_in.scalar_type() == at::kHalf || pre_in.scalar_type() == at::kBFloat16,
                "gelu_backward_split takes float16 / bfloat16, got ", pre_in.scalar_type());
    TORCH_CHECK(pre_in.dim() == 3, "pre_act must be [B, N, n]");
    const int64_t B = pre_in.size(0), N = pre_in.size(1), n = pre_in.size(2);
    TORCH_CHECK(n_special >= 0 && n_special <= N, "n_special out of range");
    at::Tensor pre = pre_in.contiguous(), sp, pa;
    if (g_sp.has_value() && g_sp->defined() && g_sp->numel() > 0) {
        check_gpu(*g_sp, "grad_special");
        TORCH_CHECK(g_sp->scalar_type() == pre.scalar_type() && g_sp->numel() == B * n_special * n,
                    "grad_special must be [B, S, n] of the pre_act dtype");
        sp = g_sp->contiguous();
    }
    if (g_pa.has_value() && g_pa->defined() && g_pa->numel() > 0) {
        check_gpu(*g_pa, "grad_patch");
        TORCH_CHECK(g_pa->scalar_type() == pre.scalar_type() && g_pa->numel() == B * (N - n_special) * n,
                    "grad_patch must be [B * (N - S), n] of the pre_act dtype");
        pa = g_pa->contiguous();
    }
    c10::DeviceGuard g(pre.device());
    at::Tensor out = at::empty_like(pre);
    check_status(svtad_gelu_backward_split(sp.defined() ? sp.data_ptr() : nullptr,
                                           pa.defined() ? pa.data_ptr() : nullptr, pre.data_ptr(),
                                           out.data_ptr(), B, N, n_special, (int)n, dtype_code(pre),
                                           stream_of(pre)),
                 "gelu_backward_split");
    return out;
}

// gamma_grad(w, g, b or None, gs or None) -> [1]: sum(w * g) + sum(b * gs), fp32, ordered
at::Tensor op_gamma_grad(const at::Tensor& w_in, const at::Tensor& g_in, const c10::optional<at::Tensor>& b_in,
                         const c10::optional<at::Tensor>& gs_in) {
    check_gpu(w_in, "w");
    check_gpu(g_in, "g");
    TORCH_CHECK(w_in.scalar_type() == g_in.scalar_type(), "w and g dtypes differ");
    TORCH_CHECK(w_in.scalar_type() == at::kHalf || w_in.scalar_type() == at::kBFloat16,
                "gamma_grad takes float16 / bfloat16, got ", w_in.scalar_type());
    TORCH_CHECK(w_in.numel() == g_in.numel(), "w and g must have the same size");
    at::Tensor w = w_in.contiguous(), g = g_in.contiguous(), b, gs;
    if (bias_present(b_in)) {
        TORCH_CHECK(gs_in.has_value() && gs_in->defined() && gs_in->numel() == b_in->numel(),
                    "gs must match b");
        check_gpu(*b_in, "b");
        check_gpu(*gs_in, "gs");
        TORCH_CHECK(b_in->scalar_type() == w.scalar_type() && gs_in->scalar_type() == w.scalar_type(),
                    "b and gs must have the dtype of w");
        b = b_in->contiguous();
        gs = gs_in->contiguous();
    }
    c10::DeviceGuard guard(w.device());
    at::Tensor out = at::empty({1}, w.options());
    const size_t wsb = svtad_gamma_grad_workspace_bytes();
    at::Tensor work = at::empty({(int64_t)wsb}, w.options().dtype(at::kByte));
    check_status(svtad_gamma_grad(w.data_ptr(), g.data_ptr(), w.numel(), b.defined() ? b.data_ptr() : nullptr,
                                  gs.defined() ? gs.data_ptr() : nullptr, b.defined() ? b.numel() : 0,
                                  out.data_ptr(), nullptr, nullptr, nullptr, nullptr, work.data_ptr(), wsb,
                                  dtype_code(w), stream_of(w)),
                 "gamma_grad");
    return out;
}

// up_proj_grads(w, g, b or None, gs or None, gamma [1]) ->
//   (grad_gamma [1], w * gamma, g * gamma, gs * gamma or empty): the gamma
//   gradient and the gamma-scaled tensors of the adapter's up-projection
//   backward in one pass. gamma is of w's dtype or float32 (the reference's
//   autocast training); grad_gamma has gamma's dtype, the scaled tensors w's.
//   g may be float32 (linear_wgrad's unrounded sums): g * gamma is then its
//   only rounding.
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> op_up_proj_grads(
    const at::Tensor& w_in, const at::Tensor& g_in, const c10::optional<at::Tensor>& b_in,
    const c10::optional<at::Tensor>& gs_in, const at::Tensor& gamma_in) {
    check_gpu(w_in, "w");
    check_gpu(g_in, "g");
    check_gpu(gamma_in, "gamma");
    TORCH_CHECK((g_in.scalar_type() == w_in.scalar_type() || g_in.scalar_type() == at::kFloat) &&
                    (gamma_in.scalar_type() == w_in.scalar_type() || gamma_in.scalar_type() == at::kFloat),
                "g and gamma must be of w's dtype or float32");
    TORCH_CHECK(w_in.scalar_type() == at::kHalf || w_in.scalar_type() == at::kBFloat16,
                "up_proj_grads takes float16 / bfloat16, got ", w_in.scalar_type());
    TORCH_CHECK(w_in.numel() == g_in.numel() && gamma_in.numel() == 1, "w and g must match; gamma one element");
    at::Tensor w = w_in.contiguous(), g = g_in.contiguous(), gm = gamma_in.contiguous(), b, gs;
    if (bias_present(b_in)) {
        TORCH_CHECK(gs_in.has_value() && gs_in->defined() && gs_in->numel() == b_in->numel(), "gs must match b");
        check_gpu(*b_in, "b");
        check_gpu(*gs_in, "gs");
        TORCH_CHECK(b_in->scalar_type() == w.scalar_type() && gs_in->scalar_type() == w.scalar_type(),
                    "b and gs must have the dtype of w");
        b = b_in->contiguous();
        gs = gs_in->contiguous();
    }
    c10::DeviceGuard guard(w.device());
    at::Tensor out = at::empty({1}, gm.options());  // the gradient of gamma has gamma's dtype
    at::Tensor w_sc = at::empty_like(w), g_sc = at::empty_like(g, g.options().dtype(w.scalar_type()));
    at::Tensor gs_sc = b.defined() ? at::empty_like(gs) : at::empty({0}, w.options());
    const size_t wsb = svtad_gamma_grad_workspace_bytes();
    at::Tensor work = at::empty({(int64_t)wsb}, w.options().dtype(at::kByte));
    check_status(svtad_gamma_grad_mixed(w.data_ptr(), g.data_ptr(), w.numel(), b.defined() ? b.data_ptr() : nullptr,
                                        gs.defined() ? gs.data_ptr() : nullptr, b.defined() ? b.numel() : 0,
                                        out.data_ptr(), gm.data_ptr(), w_sc.data_ptr(), g_sc.data_ptr(),
                                        b.defined() ? gs_sc.data_ptr() : nullptr, work.data_ptr(), wsb,
                                        dtype_code(w), dtype_code(g), dtype_code(gm), stream_of(w)),
                 "up_proj_grads");
    return {out, w_sc, g_sc, gs_sc};
}

// ---------------------------------------------------------------------------
// The adapter's GEMMs over whole token tiles (svtad_adapter_prep / _rows)
// ---------------------------------------------------------------------------

// whether the adapter of these widths runs on svtad_adapter_rows
bool op_adapter_rows_ok(int64_t embed, int64_t hidden) {
    return svtad_adapter_rows_ok(SVTAD_ROWS_GELU, (int)embed, (int)hidden) &&
           svtad_adapter_rows_ok(SVTAD_ROWS_SPLIT, (int)embed, (int)hidden) &&
           svtad_adapter_rows_ok(SVTAD_ROWS_RES, (int)hidden, (int)embed);
}

// Jobs of one svtad_adapter_prep launch and the tensors they read.
struct PrepList {
    at::TensorOptions opt;  // the compute type
    at::ScalarType t;
    std::vector<svtad_prep_job> jobs;
    std::vector<at::Tensor> keep;

    explicit PrepList(const at::Tensor& like, bool bf16)
        : opt(like.options().dtype(bf16 ? at::kBFloat16 : at::kHalf)), t(bf16 ? at::kBFloat16 : at::kHalf) {}

    at::Tensor param(const at::Tensor& p) {
        TORCH_CHECK(p.is_cuda() && p.device() == opt.device(), "adapter: parameters must share the GPU");
        TORCH_CHECK(p.scalar_type() == t || p.scalar_type() == at::kFloat,
                    "adapter: parameters take the compute type or float32, got ", p.scalar_type());
        return p.contiguous();
    }
    void push(int kind, const at::Tensor& src, const at::Tensor& dst, int off, int64_t n, int64_t k, bool pair,
              const at::Tensor* gamma) {
        jobs.push_back(svtad_prep_job{src.data_ptr(), dst.data_ptr(), gamma ? gamma->data_ptr() : nullptr, kind, off, (int)n,
                                      (int)k, kind != SVTAD_PREP_WIDEN && src.scalar_type() == at::kFloat,
                                      gamma && gamma->scalar_type() == at::kFloat, pair});
        keep.push_back(src);
    }
    at::Tensor add(int kind, const at::Tensor& src, int off, int64_t n, int64_t k, bool pair, const at::Tensor* gamma = nullptr,
                   int64_t extra = 0) {
        at::Tensor dst = at::empty({(int64_t)off * n * k + extra}, opt);
        push(kind, src, dst, off, n, k, pair, gamma);
        return dst;
    }
    at::Tensor cast(const at::Tensor& p_in) {  // in the compute type, 16-byte aligned
        at::Tensor p = param(p_in);
        if (p.scalar_type() == t) return ((uintptr_t)p.data_ptr() & 15) ? p.clone() : p;
        if (p.numel() % 8) return p.to(t);
        return add(SVTAD_PREP_CAST, p, 1, 1, p.numel(), false).view(p.sizes());
    }
    at::Tensor bias(const c10::optional<at::Tensor>& b, int64_t n) {
        if (!bias_present(b)) return at::empty({0}, opt);
        TORCH_CHECK(b->numel() == n, "adapter: a bias must have ", n, " elements");
        return cast(*b);
    }
    // g (the compute type) in the parameter's type: converted by launch() to float32
    at::Tensor grad(const at::Tensor& g, at::ScalarType want) {
        if (!g.defined() || g.numel() == 0 || g.scalar_type() == want) return g;
        if (want != at::kFloat || g.numel() % 8 || ((uintptr_t)g.data_ptr() & 15) || !g.is_contiguous()) return g.to(want);
        at::Tensor dst = at::empty(g.sizes(), opt.dtype(at::kFloat));
        push(SVTAD_PREP_WIDEN, g, dst, 1, 1, g.numel(), false, nullptr);
        return dst;
    }
    // row of the [B * N, .] matrix of each special token, then of each patch token (patch_only: of those)
    at::Tensor token_rows(int64_t B, int64_t N, int64_t S, bool patch_only) {
        const int64_t count = B * (patch_only ? N - S : N);
        at::Tensor rows = at::empty({count}, opt.dtype(at::kInt));
        if (count > 0)
            jobs.push_back(svtad_prep_job{nullptr, rows.data_ptr(), nullptr, SVTAD_PREP_TOKEN_ROWS, (int)B, (int)N, (int)S, 0, 0,
                                          patch_only});
        return rows;
    }
    void launch(void* stream) {
        if (!jobs.empty())
            check_status(svtad_adapter_prep(jobs.data(), (int)jobs.size(), t == at::kHalf ? SVTAD_F16 : SVTAD_BF16, stream),
                         "adapter_prep");
    }
};

// adapter_prep(w_d, b_d, w_c, b_c, w_u, b_u, gamma, bf16, train, pack_conv)
//   -> [wd, b_d, wu, b_u, b_c, w_c, w_u, wdT, wuT, packed_fwd, packed_bwd]
// One launch: the parameters (f32 or the compute type) cast, wd / wu in the
// fragment order of the down / up projection, and with train wdT / wuT in that
// of the input gradient / the up projection's backward (scaled by gamma), w_u
// as is; with pack_conv the SparseConv2D layouts of w_c (packed_bwd with
// train). An item that is not wanted, or a missing bias, is empty.
static std::vector<at::Tensor> adapter_prep_jobs(PrepList& L, const at::Tensor& w_d_in, const c10::optional<at::Tensor>& b_d,
                                                 const at::Tensor& w_c_in, const c10::optional<at::Tensor>& b_c,
                                                 const at::Tensor& w_u_in, const c10::optional<at::Tensor>& b_u,
                                                 const at::Tensor& gamma_in, bool train, bool pack_conv) {
    const int dt = L.t == at::kHalf ? SVTAD_F16 : SVTAD_BF16;
    at::Tensor w_d = L.param(w_d_in), w_c = L.param(w_c_in), w_u = L.param(w_u_in), gm = L.param(gamma_in);
    TORCH_CHECK(w_d.dim() == 2 && w_u.dim() == 2 && w_c.dim() == 3 && w_c.size(0) == 9 && gm.numel() == 1 &&
                    w_u.size(0) == w_d.size(1) && w_u.size(1) == w_d.size(0) && w_c.size(1) == w_d.size(0) &&
                    w_c.size(2) == w_d.size(0),
                "adapter: w_d [h, E], w_c [9, h, h], w_u [E, h] and a gamma of one element");
    const int64_t h = w_d.size(0), E = w_d.size(1);
    std::vector<at::Tensor> out(11, at::empty({0}, L.opt));
    out[0] = L.add(SVTAD_PREP_ROWS, w_d, 1, h, E, true);
    out[1] = L.bias(b_d, h);
    out[2] = L.add(SVTAD_PREP_ROWS, w_u, 1, E, h, false);
    out[3] = L.bias(b_u, E);
    out[4] = L.bias(b_c, h);
    out[5] = L.cast(w_c);
    if (train) {
        out[6] = L.cast(w_u);
        out[7] = L.add(SVTAD_PREP_COLS, w_d, 1, E, h, false);
        L.keep.push_back(gm);
        out[8] = L.add(SVTAD_PREP_COLS, w_u, 1, h, E, true, &gm);
    }
    out[9] = out[10] = at::empty({0}, L.opt.dtype(at::kByte));
    if (pack_conv) {
        const size_t bf = svtad_fwd_workspace_bytes((int)h, (int)h, dt), bb = svtad_bwd_in_workspace_bytes((int)h, (int)h, dt);
        if (bf == (size_t)9 * h * h * 2) out[9] = L.add(SVTAD_PREP_CONV_FWD, w_c, 9, h, h, false).view(at::kByte);
        if (train && bb > bf && bf)
            out[10] = L.add(SVTAD_PREP_CONV_BWD, w_c, 9, h, h, false, nullptr, (int64_t)(bb - bf) / 2).view(at::kByte);
    }
    return out;
}

std::vector<at::Tensor> op_adapter_prep(const at::Tensor& w_d, const c10::optional<at::Tensor>& b_d, const at::Tensor& w_c,
                                        const c10::optional<at::Tensor>& b_c, const at::Tensor& w_u,
                                        const c10::optional<at::Tensor>& b_u, const at::Tensor& gamma, bool bf16, bool train,
                                        bool pack_conv) {
    check_gpu(w_d, "w_d");
    c10::DeviceGuard g(w_d.device());
    PrepList L(w_d, bf16);
    auto out = adapter_prep_jobs(L, w_d, b_d, w_c, b_c, w_u, b_u, gamma, train, pack_conv);
    L.launch(stream_of(w_d));
    return out;
}

// patch_rows(like, B, N, S) -> int32 [B * (N - S)]: the row of like's [B * N, .]
// matrix of each patch token, in the order of the SparseConv2D rows
at::Tensor op_patch_rows(const at::Tensor& like, int64_t B, int64_t N, int64_t S) {
    check_gpu(like, "like");
    TORCH_CHECK(B >= 0 && S >= 0 && S <= N && N < (int64_t)INT32_MAX && B * N < (int64_t)INT32_MAX, "patch_rows: bad sizes");
    c10::DeviceGuard g(like.device());
    PrepList L(like, true);
    at::Tensor rows = L.token_rows(B, N, S, true);
    L.launch(stream_of(like));
    return rows;
}

// x contiguous; a float32 x (whose cast once gave a fresh buffer) on 16 bytes
static at::Tensor rows_input(const at::Tensor& x) {
    at::Tensor c = x.contiguous();
    return c.scalar_type() == at::kFloat && ((uintptr_t)c.data_ptr() & 15) ? c.clone() : c;
}

static svtad_rows_args rows_args(int kind, int64_t B, int64_t N, int64_t S, int64_t k, int64_t n) {
    svtad_rows_args a = {};
    a.kind = kind;
    a.batch = B;
    a.n_tokens = N;
    a.n_special = S;
    a.k = (int)k;
    a.n = (int)n;
    return a;
}

static void rows_check(const at::Tensor& a, const at::Tensor& w, int64_t k, int64_t n, const char* what) {
    check_gpu(a, what);
    check_gpu(w, "w");
    TORCH_CHECK(w.scalar_type() == at::kHalf || w.scalar_type() == at::kBFloat16, "adapter_rows: w must be f16 / bf16");
    TORCH_CHECK(w.numel() == n * k && w.is_contiguous(), "adapter_rows: w does not match ", n, " x ", k);
    TORCH_CHECK(a.scalar_type() == w.scalar_type() || a.scalar_type() == at::kFloat,
                "adapter_rows: ", what, " takes the type of w or float32");
}

// Down projection and GELU of the rows of x [B, N, k] (contiguous): the
// pre-activation, GELU's special rows in sp and patch rows in pa (empty: none),
// and x in the compute type in xc where it is another tensor than x.
static void rows_down(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias, const at::Tensor& pre,
                      const at::Tensor& sp, const at::Tensor& pa, const at::Tensor& xc, int64_t S, const char* what) {
    const int64_t k = x.size(2), n = pre.size(2);
    rows_check(x, w, k, n, "x");
    svtad_rows_args a = rows_args(SVTAD_ROWS_GELU, x.size(0), x.size(1), S, k, n);
    a.a0 = x.data_ptr();
    a.w = w.data_ptr();
    a.bias = opt_ptr(bias, n, w);
    a.a_copy = xc.numel() && !xc.is_same(x) ? xc.data_ptr() : nullptr;
    a.out0 = pre.data_ptr();
    a.out1 = sp.numel() ? sp.data_ptr() : nullptr;
    a.out2 = pa.numel() ? pa.data_ptr() : nullptr;
    a.a_f32 = x.scalar_type() == at::kFloat;
    check_status(svtad_adapter_rows(&a, dtype_code(w), stream_of(x)), what);
}

// adapter_rows_down(x [B, N, k], wd, bias or empty, n, n_special, copy) ->
//   (pre_act [B, N, n], act_special [B, S, n], act_patch [B * (N - S), n], x in the compute type if copy, else empty)
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> op_adapter_rows_down(const at::Tensor& x_in, const at::Tensor& w,
                                                                                const at::Tensor& bias, int64_t n,
                                                                                int64_t S, bool copy) {
    TORCH_CHECK(x_in.dim() == 3, "x must be [B, N, C]");
    const int64_t B = x_in.size(0), N = x_in.size(1), k = x_in.size(2);
    rows_check(x_in, w, k, n, "x");  // before n and S size any buffer
    TORCH_CHECK(S >= 0 && S <= N, "n_special out of range");
    at::Tensor x = rows_input(x_in);
    c10::DeviceGuard g(x.device());
    const auto opt = w.options();
    at::Tensor pre = at::empty({B, N, n}, opt), sp = at::empty({B, S, n}, opt), pa = at::empty({B * (N - S), n}, opt);
    at::Tensor xc = copy && x.scalar_type() == at::kFloat ? at::empty({B, N, k}, opt) : at::empty({0}, opt);
    rows_down(x, w, bias, pre, sp, pa, xc, S, "adapter_rows_down");
    return {pre, sp, pa, xc};
}

// adapter_rows_split(go [B, N, k], wuT, n, n_special, copy) ->
//   (special [B, S, n], patch [B * (N - S), n], go in the compute type if copy, else empty)
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_adapter_rows_split(const at::Tensor& go_in, const at::Tensor& w, int64_t n,
                                                                     int64_t S, bool copy) {
    TORCH_CHECK(go_in.dim() == 3, "go must be [B, N, C]");
    const int64_t B = go_in.size(0), N = go_in.size(1), k = go_in.size(2);
    rows_check(go_in, w, k, n, "go");
    TORCH_CHECK(S >= 0 && S <= N, "n_special out of range");
    at::Tensor go = rows_input(go_in);
    c10::DeviceGuard g(go.device());
    const auto opt = w.options();
    at::Tensor sp = at::empty({B, S, n}, opt), pa = at::empty({B * (N - S), n}, opt);
    const bool f32 = go.scalar_type() == at::kFloat;
    at::Tensor gc = copy && f32 ? at::empty({B, N, k}, opt) : at::empty({0}, opt);
    svtad_rows_args a = rows_args(SVTAD_ROWS_SPLIT, B, N, S, k, n);
    a.a0 = go.data_ptr();
    a.w = w.data_ptr();
    a.a_copy = gc.numel() ? gc.data_ptr() : nullptr;
    a.out1 = sp.numel() ? sp.data_ptr() : nullptr;
    a.out2 = pa.numel() ? pa.data_ptr() : nullptr;
    a.a_f32 = f32;
    check_status(svtad_adapter_rows(&a, dtype_code(w), stream_of(go)), "adapter_rows_split");
    return {sp, pa, gc};
}

// adapter_rows_res(a_special [B, S, k] or None, a, w, bias or empty, gamma or None, residual [B, N, n], out_float32)
//   -> [B, N, n]: adapter_up with a fragment-ordered weight, or without gamma A W^T + residual
// a holds the patch rows [B * (N - S), k] beside a_special, else all rows.
at::Tensor op_adapter_rows_res(const c10::optional<at::Tensor>& sp_in, const at::Tensor& a_in, const at::Tensor& w,
                               const at::Tensor& bias, const c10::optional<at::Tensor>& gamma_in,
                               const at::Tensor& res_in, bool out_float32) {
    TORCH_CHECK(res_in.dim() == 3, "residual must be [B, N, C]");
    const int64_t B = res_in.size(0), N = res_in.size(1), n = res_in.size(2), k = a_in.size(-1);
    rows_check(res_in, w, k, n, "residual");
    check_gpu(a_in, "a");
    TORCH_CHECK(a_in.scalar_type() == w.scalar_type(), "a and w dtypes differ");
    const bool split = sp_in.has_value() && sp_in->defined();
    int64_t S = 0;
    at::Tensor sp;
    if (split) {
        check_gpu(*sp_in, "a_special");
        TORCH_CHECK(sp_in->dim() == 3 && sp_in->size(0) == B && sp_in->size(2) == k && sp_in->scalar_type() == w.scalar_type(),
                    "a_special must be [B, S, k]");
        S = sp_in->size(1);
        sp = sp_in->contiguous();
    }
    TORCH_CHECK(S <= N && a_in.numel() == B * (N - S) * k, "a does not match the residual's rows");
    at::Tensor a = a_in.contiguous(), res = rows_input(res_in), gm;
    c10::DeviceGuard g(res.device());
    at::Tensor out = at::empty({B, N, n}, out_float32 ? res.options().dtype(at::kFloat) : w.options());
    svtad_rows_args r = rows_args(SVTAD_ROWS_RES, B, N, S, k, n);
    if (gamma_in.has_value() && gamma_in->defined()) {
        TORCH_CHECK(gamma_in->is_cuda() && gamma_in->numel() == 1 &&
                        (gamma_in->scalar_type() == w.scalar_type() || gamma_in->scalar_type() == at::kFloat),
                    "gamma must be one element on the GPU, of the type of w or float32");
        gm = gamma_in->contiguous();
        r.gamma = gm.data_ptr();
        r.gamma_f32 = gm.scalar_type() == at::kFloat;
    }
    r.a0 = split ? (sp.numel() ? sp.data_ptr() : nullptr) : a.data_ptr();
    r.a1 = split && a.numel() ? a.data_ptr() : nullptr;
    r.a_patch_split = split;
    r.w = w.data_ptr();
    r.bias = opt_ptr(bias, n, w);
    r.res = res.data_ptr();
    r.out0 = out.data_ptr();
    r.res_f32 = res.scalar_type() == at::kFloat;
    r.out_f32 = out_float32;
    check_status(svtad_adapter_rows(&r, dtype_code(w), stream_of(res)), "adapter_rows_res");
    return out;
}

// ---------------------------------------------------------------------------
// attention to the key tokens
// ---------------------------------------------------------------------------

enum { A_NW, A_NB, A_DW, A_DB, A_QW, A_QB, A_QNW, A_QNB, A_KNW, A_KNB, A_PW, A_PB, A_GAMMA, A_COUNT };

// key_attention_layers_ok(parameters in the order above or None, hidden, heads, n, nk): whether the
// kernels take them: every one there, of the widths that hidden gives (the
// kernels read that many values), norm parameters contiguous and of one type
// per kernel, and svtad_key_attention_ok's sizes
bool op_key_attention_layers_ok(const std::vector<c10::optional<at::Tensor>>& p, int64_t h, int64_t heads, int64_t n, int64_t nk) {
    if (p.size() != A_COUNT || (h != 128 && h != 256) || heads != 4 || nk >= 1024) return false;
    const int64_t a = h / 2, hd = a / 4;
    if (!svtad_key_attention_ok(4, (int)hd, n, (int)nk)) return false;
    for (const auto& t : p)
        if (!t.has_value() || !t->defined()) return false;
    auto rows = [&](int i, int64_t r) { return p[i]->dim() == 1 && p[i]->size(0) == r; };
    auto mat = [&](int i, int64_t r, int64_t c) { return p[i]->dim() == 2 && p[i]->size(0) == r && p[i]->size(1) == c; };
    if (!mat(A_DW, a, h) || !rows(A_DB, a) || !mat(A_QW, 3 * a, a) || !rows(A_QB, 3 * a) || !mat(A_PW, h, a) || !rows(A_PB, h))
        return false;
    for (int i : {A_NW, A_NB, A_QNW, A_QNB, A_KNW, A_KNB}) {
        const int first = i <= A_NB ? A_NW : A_QNW;
        if (!rows(i, i <= A_NB ? h : hd) || !p[i]->is_contiguous() || p[i]->scalar_type() != p[first]->scalar_type()) return false;
    }
    return true;
}

static void attn_params(const at::Tensor& like, std::initializer_list<const at::Tensor*> ps, int64_t n) {
    const at::ScalarType t = (*ps.begin())->scalar_type();
    TORCH_CHECK(t == like.scalar_type() || t == at::kFloat, "norm parameters take the row type or float32");
    for (const at::Tensor* p : ps)
        TORCH_CHECK(p->is_cuda() && p->numel() == n && p->is_contiguous() && p->scalar_type() == t,
                    "norm parameters must be contiguous, of ", n, " elements and one type");
}

// layer_norm_rows(x [..., c], w, b, eps) -> (y, stats [rows, 2] float32)
std::tuple<at::Tensor, at::Tensor> op_layer_norm_rows(const at::Tensor& x_in, const at::Tensor& w, const at::Tensor& b,
                                                      double eps) {
    check_gpu(x_in, "x");
    at::Tensor x = x_in.contiguous();
    const int64_t c = x.size(-1), rows = n_rows(x);
    attn_params(x, {&w, &b}, c);
    c10::DeviceGuard g(x.device());
    at::Tensor y = at::empty_like(x), stats = at::empty({rows, 2}, x.options().dtype(at::kFloat));
    check_status(svtad_layer_norm(nullptr, x.data_ptr(), nullptr, rows, 0, w.data_ptr(), b.data_ptr(), y.data_ptr(), stats.data_ptr<float>(), rows,
                                  (int)c, (float)eps, dtype_code(x), w.scalar_type() == at::kFloat, stream_of(x)),
                 "layer_norm_rows");
    return {y, stats};
}

// layer_norm_rows_bwd(dy, x, stats, w) -> (dx, dwb [2, c] float32)
std::tuple<at::Tensor, at::Tensor> op_layer_norm_rows_bwd(const at::Tensor& dy_in, const at::Tensor& x_in,
                                                          const at::Tensor& stats, const at::Tensor& w) {
    check_gpu(x_in, "x");
    at::Tensor x = x_in.contiguous(), dy = dy_in.contiguous();
    const int64_t c = x.size(-1), rows = n_rows(x);
    TORCH_CHECK(dy.is_cuda() && dy.numel() == x.numel() && dy.scalar_type() == x.scalar_type(), "dy must match x");
    TORCH_CHECK(stats.numel() == 2 * rows && stats.scalar_type() == at::kFloat && stats.is_contiguous(), "bad stats");
    attn_params(x, {&w}, c);
    c10::DeviceGuard g(x.device());
    const auto f = x.options().dtype(at::kFloat);
    at::Tensor dx = at::empty_like(x), dwb = at::empty({2, c}, f);
    const size_t ws = svtad_layer_norm_bwd_workspace_bytes(rows, (int)c);
    at::Tensor work = at::empty({(int64_t)ws}, f.dtype(at::kByte));
    check_status(svtad_layer_norm_bwd(dy.data_ptr(), x.data_ptr(), nullptr, stats.data_ptr<float>(), w.data_ptr(), nullptr,
                                      dx.data_ptr(), rows, 0, dwb.data_ptr<float>(), work.data_ptr(), ws, rows, (int)c, dtype_code(x),
                                      w.scalar_type() == at::kFloat, stream_of(x)),
                 "layer_norm_rows_bwd");
    return {dx, dwb};
}

static void attn_check(const at::Tensor& q, const at::Tensor& kv, const at::Tensor& qw, const at::Tensor& qb,
                       const at::Tensor& kw, const at::Tensor& kb) {
    check_gpu(q, "q");
    check_gpu(kv, "kv");
    TORCH_CHECK(q.dim() == 3 && kv.dim() == 3 && kv.size(0) == q.size(0) && kv.size(2) == 2 * q.size(2) &&
                    kv.scalar_type() == q.scalar_type() && q.is_contiguous() && kv.is_contiguous(),
                "q must be [B, N, a], kv [B, nk, 2 a], contiguous and of one type");
    attn_params(q, {&qw, &qb, &kw, &kb}, q.size(2) / 4);
}

bool op_key_attention_ok(int64_t heads, int64_t head_dim, int64_t n, int64_t nk) {
    return heads < 1024 && head_dim < 1024 && nk < 1024 && svtad_key_attention_ok((int)heads, (int)head_dim, n, (int)nk);
}

// key_attention(q [B, N, a], kv [B, nk, 2a], qn_w, qn_b, kn_w, kn_b, eps) -> [B, N, a]
at::Tensor op_key_attention(const at::Tensor& q, const at::Tensor& kv, const at::Tensor& qw, const at::Tensor& qb,
                            const at::Tensor& kw, const at::Tensor& kb, double eps) {
    attn_check(q, kv, qw, qb, kw, kb);
    c10::DeviceGuard g(q.device());
    at::Tensor out = at::empty_like(q);
    check_status(svtad_key_attention(q.data_ptr(), kv.data_ptr(), qw.data_ptr(), qb.data_ptr(), kw.data_ptr(), kb.data_ptr(),
                                     out.data_ptr(), q.size(0), q.size(1), (int)kv.size(1), (int)q.size(2) / 4, (float)eps,
                                     dtype_code(q), qw.scalar_type() == at::kFloat, stream_of(q)),
                 "key_attention");
    return out;
}

// key_attention_bwd(dout, q, kv, qn_w, qn_b, kn_w, kn_b, eps) -> (dq, dkv, dnorm [4, a / 4] float32)
std::tuple<at::Tensor, at::Tensor, at::Tensor> op_key_attention_bwd(const at::Tensor& dout_in, const at::Tensor& q,
                                                                    const at::Tensor& kv, const at::Tensor& qw,
                                                                    const at::Tensor& qb, const at::Tensor& kw,
                                                                    const at::Tensor& kb, double eps) {
    attn_check(q, kv, qw, qb, kw, kb);
    check_gpu(dout_in, "dout");
    TORCH_CHECK(dout_in.sizes() == q.sizes() && dout_in.scalar_type() == q.scalar_type(), "dout must match q");
    at::Tensor dout = dout_in.contiguous();
    c10::DeviceGuard g(q.device());
    const int64_t B = q.size(0), N = q.size(1), nk = kv.size(1), hd = q.size(2) / 4;
    at::Tensor dq = at::empty_like(q), dkv = at::empty_like(kv), dn = at::empty({4, hd}, q.options().dtype(at::kFloat));
    const size_t ws = svtad_key_attention_bwd_workspace_bytes(B, N, (int)nk, (int)hd);
    at::Tensor work = at::empty({(int64_t)ws}, q.options().dtype(at::kByte));
    check_status(svtad_key_attention_bwd(dout.data_ptr(), q.data_ptr(), kv.data_ptr(), qw.data_ptr(), qb.data_ptr(),
                                         kw.data_ptr(), kb.data_ptr(), dq.data_ptr(), dkv.data_ptr(), dn.data_ptr<float>(),
                                         work.data_ptr(), ws, B, N, (int)nk, (int)hd, (float)eps, dtype_code(q),
                                         qw.scalar_type() == at::kFloat, stream_of(q)),
                 "key_attention_bwd");
    return {dq, dkv, dn};
}

// ---------------------------------------------------------------------------
// the adapter's forward and backward as one call each (widths of adapter_rows_ok)
// ---------------------------------------------------------------------------

enum { S_X, S_PRE, S_CBUF, S_PA, S_WC, S_WU, S_BU, S_WDT, S_WUT, S_PB, S_ROWS, S_COUNT };
enum { S_COMB = S_COUNT, S_STATS, S_XN, S_DW, S_XA, S_QW, S_Q, S_KV, S_ATT, S_PW, S_PBIAS, S_X2, S_DWT, S_QWT, S_PWT, S_ACOUNT };

// x [M, k] W^T + bias, [M, n] in x's type (W in fragment order, pair columns)
static at::Tensor rows_plain(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias, int64_t n) {
    const int64_t M = x.size(0), k = x.size(1);
    at::Tensor out = at::empty({M, n}, x.options());
    at::Tensor b = bias.numel() && ((uintptr_t)bias.data_ptr() & 15) ? bias.clone() : bias;
    svtad_rows_args r = rows_args(SVTAD_ROWS_PLAIN, 1, M, 0, k, n);
    r.a0 = x.data_ptr();
    r.w = w.data_ptr();
    r.bias = b.numel() ? b.data_ptr() : nullptr;
    r.out0 = out.data_ptr();
    check_status(svtad_adapter_rows(&r, dtype_code(x), stream_of(x)), "adapter_rows");
    return out;
}

// adapter_forward(x [B, N, E], w_d, b_d, w_c, b_c, w_u, b_u, gamma, neighbor_indices, n_special, tokens_per_batch, bias_mode,
//                 hm_rows, hm_gate, packed_fwd, packed_bwd, bf16, train, attn, nk, eps_norm, eps_head)
//   -> [out, packed_fwd, packed_bwd, saved tensors of adapter_backward if train]
// packed_fwd None: the SparseConv2D weight is packed here. attn holds the
// parameters of the key-token attention (13 tensors), or nothing.
std::vector<at::Tensor> op_adapter_forward(const at::Tensor& x, const at::Tensor& w_d, const c10::optional<at::Tensor>& b_d,
                                           const at::Tensor& w_c, const c10::optional<at::Tensor>& b_c,
                                           const at::Tensor& w_u, const c10::optional<at::Tensor>& b_u,
                                           const at::Tensor& gamma, const at::Tensor& nbr, int64_t S, int64_t tpb,
                                           int64_t bias_mode, const c10::optional<at::Tensor>& hm_rows,
                                           const c10::optional<at::Tensor>& hm_gate, const c10::optional<at::Tensor>& pf_in,
                                           const c10::optional<at::Tensor>& pb_in, bool bf16, bool train,
                                           const std::vector<at::Tensor>& attn, int64_t nk, double eps_norm, double eps_head) {
    check_gpu(x, "x");
    TORCH_CHECK(x.dim() == 3 && (attn.empty() || attn.size() == A_COUNT), "adapter_forward: x [B, N, E], 0 or 13 attn tensors");
    c10::DeviceGuard g(x.device());
    const int64_t B = x.size(0), N = x.size(1), h = w_d.size(0), M = B * N;
    TORCH_CHECK(S >= 0 && S <= N, "n_special out of range");
    TORCH_CHECK(attn.empty() || op_key_attention_layers_ok({attn.begin(), attn.end()}, h, 4, N, nk),
                "adapter_forward: attention parameters or sizes without a kernel");
    PrepList L(x, bf16);
    const bool pack = !pf_in.has_value();
    auto P = adapter_prep_jobs(L, w_d, b_d, w_c, b_c, w_u, b_u, gamma, train, pack);
    at::Tensor pf = pack ? P[9] : *pf_in, pb = pack ? P[10] : pb_in.has_value() ? *pb_in : P[10];
    at::Tensor dw, db, qw, qb, pw, pwf, pbias, dwf, qwf, dwt, qwt, pwt;
    const int64_t a = attn.empty() ? 0 : attn[A_DW].size(0);
    if (a) {
        dw = L.cast(attn[A_DW]);
        db = L.cast(attn[A_DB]);
        qw = L.cast(attn[A_QW]);
        qb = L.cast(attn[A_QB]);
        pwf = L.add(SVTAD_PREP_ROWS, L.param(attn[A_PW]), 1, h, a, false);
        if (train) pw = L.cast(attn[A_PW]);
        if (svtad_adapter_rows_ok(SVTAD_ROWS_PLAIN, (int)h, (int)a)) {  // and so a -> a, a -> h
            at::Tensor d = L.param(attn[A_DW]), qq = L.param(attn[A_QW]).narrow(0, 0, a);
            dwf = L.add(SVTAD_PREP_ROWS, d, 1, a, h, true);
            qwf = L.add(SVTAD_PREP_ROWS, qq, 1, a, a, true);
            if (train) {
                at::Tensor gm = L.param(attn[A_GAMMA]), pp = L.param(attn[A_PW]);
                L.keep.push_back(gm);
                dwt = L.add(SVTAD_PREP_COLS, d, 1, h, a, true);
                qwt = L.add(SVTAD_PREP_COLS, qq, 1, a, a, true);
                pwt = L.add(SVTAD_PREP_COLS, pp, 1, a, h, true, &gm);
            }
        }
        pbias = L.cast(attn[A_PB]);
    }
    TORCH_CHECK(N < (int64_t)INT32_MAX && M < (int64_t)INT32_MAX, "adapter_forward: 2^31 rows or more");
    // with attention the up projection's operand is in token order
    at::Tensor rows = train && !a ? L.token_rows(B, N, S, false) : at::empty({0}, L.opt.dtype(at::kInt));
    L.launch(stream_of(x));
    // special rows first, then the patch rows' SparseConv2D output: the up
    // projection's operand, and its weight gradient's in one row list
    at::Tensor cbuf = at::empty({M, h}, L.opt);
    at::Tensor sp = cbuf.narrow(0, 0, B * S).view({B, S, h}), conv = cbuf.narrow(0, B * S, M - B * S);
    at::Tensor xin = rows_input(x), pre = at::empty({B, N, h}, L.opt), pa = at::empty({M - B * S, h}, L.opt);
    at::Tensor xc = train && xin.scalar_type() == at::kFloat ? at::empty(x.sizes(), L.opt) : xin;
    void* const st = stream_of(x);
    const int dt = L.t == at::kHalf ? SVTAD_F16 : SVTAD_BF16;
    rows_down(xin, P[0], P[1], pre, sp, pa, xc, S, "adapter_forward");
    if (hm_rows.has_value()) op_heatmap_add_(pa, sp, *hm_rows, *hm_gate);
    at::Tensor tab = table_i32(nbr, pa.size(0));
    int mode = P[4].numel() ? (int)bias_mode : SVTAD_BIAS_NONE;
    if (mode == SVTAD_BIAS_FP32) mode = SVTAD_BIAS_PRE;  // the bias in the compute type, widened exactly
    int packed_st = SVTAD_ERR_UNSUPPORTED;
    if (pf.numel())
        packed_st = svtad_fwd_packed(pa.data_ptr(), tab.data_ptr<int32_t>(), pf.data_ptr(), mode ? P[4].data_ptr() : nullptr,
                                     mode, conv.data_ptr(), pa.size(0), (int)h, (int)h, tpb, dt, st);
    if (packed_st == SVTAD_ERR_UNSUPPORTED)  // no packed layout, or operands of 2^31 bytes: as op_fwd_packed
        conv.copy_(conv_fwd(pa, tab, P[5], P[4], tpb, (int)bias_mode, -1));
    else
        check_status(packed_st, "adapter_forward");
    at::Tensor comb, stats, xn, xa, q, kv, att, x2;
    if (a) {
        attn_params(cbuf, {&attn[A_NW], &attn[A_NB]}, h);
        comb = S ? at::empty({B, N, h}, L.opt) : conv.view({B, N, h});
        xn = at::empty({M, h}, L.opt);
        stats = at::empty({M, 2}, L.opt.dtype(at::kFloat));
        check_status(svtad_layer_norm(S ? sp.data_ptr() : nullptr, conv.data_ptr(), S ? comb.data_ptr() : nullptr, N, S,
                                      attn[A_NW].data_ptr(), attn[A_NB].data_ptr(), xn.data_ptr(), stats.data_ptr<float>(), M,
                                      (int)h, (float)eps_norm, dt, attn[A_NW].scalar_type() == at::kFloat, st),
                     "adapter_forward");
        xa = dwf.defined() ? rows_plain(xn, dwf, db, a) : at::addmm(db, xn, dw.t());
        q = (qwf.defined() ? rows_plain(xa, qwf, qb.narrow(0, 0, a), a) : at::addmm(qb.narrow(0, 0, a), xa, qw.narrow(0, 0, a).t()))
                .view({B, N, a});
        if (B * nk <= 64) {
            kv = at::empty({B, nk, 2 * a}, L.opt);
            check_status(svtad_key_proj(xa.data_ptr(), qw.narrow(0, a, 2 * a).data_ptr(), qb.narrow(0, a, 2 * a).data_ptr(),
                                        kv.data_ptr(), B, N, (int)nk, (int)a, dt, st),
                         "adapter_forward");
        } else {
            at::Tensor xk = xa.view({B, N, a}).narrow(1, 0, nk).reshape({B * nk, a});
            kv = at::addmm(qb.narrow(0, a, 2 * a), xk, qw.narrow(0, a, 2 * a).t()).view({B, nk, 2 * a});
        }
        att = op_key_attention(q, kv, attn[A_QNW], attn[A_QNB], attn[A_KNW], attn[A_KNB], eps_head);
        x2 = op_adapter_rows_res(c10::nullopt, att, pwf, pbias, attn[A_GAMMA], comb, false);
    }
    const bool out32 = gamma.scalar_type() == at::kFloat;
    at::Tensor out = a ? op_adapter_rows_res(c10::nullopt, x2, P[2], P[3], gamma, xin, out32)
                       : op_adapter_rows_res(sp, conv, P[2], P[3], gamma, xin, out32);
    std::vector<at::Tensor> ret{out, pf, pb};
    if (!train) return ret;
    for (const at::Tensor& t : {xc, pre, cbuf, pa, P[5], P[6], P[3], P[7], P[8], pb, rows}) ret.push_back(t);
    if (a)
        for (const at::Tensor& t : {comb, stats, xn, dw, xa, qw, q, kv, att, pw, pbias, x2, dwt, qwt, pwt})
            ret.push_back(t.defined() ? t : at::empty({0}, L.opt));
    return ret;
}

// adapter_backward(go, saved, gamma, neighbor_indices, hm_rows, hm_gate, attn, n_special, tokens_per_batch, nk, eps_head,
//                  symmetric, has_bd, has_bc, need_x, need_wd, param types [w_d, b_d, w_c, b_c, w_u, b_u], x_float32)
//   -> [gx, gw_d, gb_d, gw_c, gb_c, gw_u, gb_u, g_gamma, g_gate, attention parameters]
// Gradients that are not wanted or do not exist are empty.
std::vector<at::Tensor> op_adapter_backward(const at::Tensor& go_in, const std::vector<at::Tensor>& saved,
                                            const at::Tensor& gamma, const at::Tensor& nbr,
                                            const c10::optional<at::Tensor>& hm_rows,
                                            const c10::optional<at::Tensor>& hm_gate,
                                            const std::vector<at::Tensor>& attn, int64_t S, int64_t tpb, int64_t nk,
                                            double eps_head, bool symmetric, bool has_bd, bool has_bc, bool need_x,
                                            bool need_wd, const std::vector<bool>& f32, bool x_f32) {
    const bool with_attn = !attn.empty();
    TORCH_CHECK(saved.size() == (size_t)(with_attn ? S_ACOUNT : S_COUNT) && f32.size() == 6, "adapter_backward: bad saved tensors");
    const at::Tensor &xc = saved[S_X], &pre = saved[S_PRE], &pa = saved[S_PA], &w_u = saved[S_WU], &b_u = saved[S_BU];
    c10::DeviceGuard guard(pre.device());
    const int64_t B = pre.size(0), N = pre.size(1), h = pre.size(2), M = B * N, E = xc.size(2);
    const at::ScalarType t = pre.scalar_type();
    const int dt = dtype_code(pre);
    void* const st = stream_of(pre);
    const auto opt = pre.options();
    const at::Tensor none = at::empty({0}, opt), no_rows = at::empty({0}, opt.dtype(at::kInt));
    PrepList L(pre, t == at::kBFloat16);
    auto want = [&](int i) { return f32[i] ? at::kFloat : t; };
    // gradients of (c W^T + b) gamma from G = go^T c (fp32) and the column sums of go
    auto up_grads = [&](const at::Tensor& w, const at::Tensor& G, const at::Tensor& b, const at::Tensor& gs,
                        const at::Tensor& gm_in, at::Tensor* w_sc, at::Tensor* gw, at::Tensor* gb) {
        at::Tensor gm = gm_in.contiguous(), out = at::empty({1}, gm.options());
        const bool bias = b.numel() > 0;
        if (w_sc) *w_sc = at::empty_like(w);
        *gw = at::empty_like(w);
        *gb = bias ? at::empty_like(gs) : none;
        const size_t wsb = svtad_gamma_grad_workspace_bytes();
        at::Tensor work = at::empty({(int64_t)wsb}, opt.dtype(at::kByte));
        check_status(svtad_gamma_grad_mixed(w.data_ptr(), G.data_ptr(), w.numel(), bias ? b.data_ptr() : nullptr,
                                            bias ? gs.data_ptr() : nullptr, bias ? b.numel() : 0, out.data_ptr(),
                                            gm.data_ptr(), w_sc ? w_sc->data_ptr() : nullptr, gw->data_ptr(),
                                            bias ? gb->data_ptr() : nullptr, work.data_ptr(), wsb, dt, SVTAD_F32,
                                            dtype_code(gm), st),
                     "adapter_backward");
        return out.view(gm_in.sizes());
    };
    at::Tensor go = go_in.contiguous();
    at::Tensor g_sp, g_pa, goc;
    std::tie(g_sp, g_pa, goc) = op_adapter_rows_split(go, saved[S_WUT], h, with_attn ? 0 : S, true);
    if (go.scalar_type() == t) goc = go;
    at::Tensor go2 = goc.view({M, E});
    at::Tensor G = with_attn ? op_linear_wgrad(go2, no_rows, saved[S_X2].view({M, h}), true)
                             : op_linear_wgrad(go2, saved[S_ROWS], saved[S_CBUF], true);
    at::Tensor gsum = b_u.numel() ? op_column_sums(go2) : none, gw_u, gb_u;
    at::Tensor g_gamma = up_grads(w_u, G, b_u, gsum, gamma, nullptr, &gw_u, &gb_u);
    std::vector<at::Tensor> ag;
    if (with_attn) {
        const at::Tensor &xn = saved[S_XN], &dw = saved[S_DW], &xa = saved[S_XA], &qw = saved[S_QW], &q = saved[S_Q],
                         &kv = saved[S_KV], &att = saved[S_ATT], &pw = saved[S_PW], &pbias = saved[S_PBIAS];
        const int64_t a = q.size(2);
        at::Tensor dx2 = g_pa;  // [M, h], token order
        at::Tensor pw_sc, gpw, gpb;
        at::Tensor Gp = op_linear_wgrad(dx2, no_rows, att.view({M, a}), true);
        const bool plain = saved[S_DWT].numel() > 0;
        at::Tensor g_ag = up_grads(pw, Gp, pbias, op_column_sums(dx2), attn[A_GAMMA], plain ? nullptr : &pw_sc, &gpw, &gpb);
        at::Tensor datt = plain ? rows_plain(dx2, saved[S_PWT], none, a) : at::mm(dx2, pw_sc), dq, dkv, dn;
        std::tie(dq, dkv, dn) = op_key_attention_bwd(datt.view({B, N, a}), q, kv, attn[A_QNW], attn[A_QNB], attn[A_KNW],
                                                     attn[A_KNB], eps_head);
        at::Tensor dq2 = dq.view({M, a}), dkv2 = dkv.view({B * nk, 2 * a});
        at::Tensor dxa = plain ? rows_plain(dq2, saved[S_QWT], none, a) : at::mm(dq2, qw.narrow(0, 0, a));
        auto wt = [&](int i) { return attn[i].scalar_type(); };
        at::Tensor gqw, gqb;
        // a key row has no query: its gradient comes from its key and value
        if (B * nk <= 64) {
            gqw = at::empty({3 * a, a}, opt.dtype(wt(A_QW)));
            gqb = at::empty({3 * a}, opt);
            gqw.narrow(0, 0, a).copy_(op_linear_wgrad(dq2, no_rows, xa, wt(A_QW) == at::kFloat));
            gqb.narrow(0, 0, a).copy_(op_column_sums(dq2));
            check_status(svtad_key_proj_bwd(dkv.data_ptr(), xa.data_ptr(), qw.narrow(0, a, 2 * a).data_ptr(), dxa.data_ptr(),
                                            gqw.narrow(0, a, 2 * a).data_ptr(), gqb.narrow(0, a, 2 * a).data_ptr(), B, N,
                                            (int)nk, (int)a, dt, wt(A_QW) == at::kFloat, 0, st),
                         "adapter_backward");
        } else {
            at::Tensor xk = xa.view({B, N, a}).narrow(1, 0, nk).reshape({B * nk, a});
            dxa.view({B, N, a}).narrow(1, 0, nk).copy_(at::mm(dkv2, qw.narrow(0, a, 2 * a)).view({B, nk, a}));
            gqw = at::cat({op_linear_wgrad(dq2, no_rows, xa, false), at::mm(dkv2.t(), xk)});
            gqb = at::cat({op_column_sums(dq2), dkv2.sum(0)});
        }
        at::Tensor gdw = op_linear_wgrad(dxa, no_rows, xn, wt(A_DW) == at::kFloat), gdb = op_column_sums(dxa);
        at::Tensor dxn = plain ? rows_plain(dxa, saved[S_DWT], none, h) : at::mm(dxa, dw), dwb = at::empty({2, h}, opt.dtype(at::kFloat));
        g_sp = at::empty({B, S, h}, opt);
        g_pa = at::empty({M - B * S, h}, opt);
        const size_t ws = svtad_layer_norm_bwd_workspace_bytes(M, (int)h);
        at::Tensor work = at::empty({(int64_t)ws}, opt.dtype(at::kByte));
        check_status(svtad_layer_norm_bwd(dxn.data_ptr(), saved[S_COMB].data_ptr(), dx2.data_ptr(),
                                          saved[S_STATS].data_ptr<float>(), attn[A_NW].data_ptr(),
                                          S ? g_sp.data_ptr() : nullptr, g_pa.data_ptr(), N, S, dwb.data_ptr<float>(),
                                          work.data_ptr(), ws, M, (int)h, dt, attn[A_NW].scalar_type() == at::kFloat, st),
                     "adapter_backward");
        ag.resize(A_COUNT);
        ag[A_NW] = dwb[0].to(wt(A_NW));
        ag[A_NB] = dwb[1].to(wt(A_NB));
        ag[A_DW] = gdw;
        ag[A_DB] = L.grad(gdb, wt(A_DB));
        ag[A_QW] = L.grad(gqw, wt(A_QW));
        ag[A_QB] = L.grad(gqb, wt(A_QB));
        for (int i = 0; i < 4; ++i) ag[A_QNW + i] = dn[i].to(wt(A_QNW + i));
        ag[A_PW] = L.grad(gpw, wt(A_PW));
        ag[A_PB] = L.grad(gpb, wt(A_PB));
        ag[A_GAMMA] = g_ag;
    }
    at::Tensor gi, gw_c, gb_c;
    std::tie(gi, gw_c, gb_c) = op_bwd_packed(g_pa, pa, nbr, saved[S_WC], saved[S_PB], h, tpb, has_bc, symmetric);
    at::Tensor g_gate = none;
    if (hm_rows.has_value()) {
        // backward of patches + special[hm_rows] * gate: the gather's
        // scatter-add into the special-token gradient, summed in float32 and
        // rounded once, and the gate's sum
        at::Tensor sp_rows = saved[S_CBUF].narrow(0, 0, B * S), gf = gi.to(at::kFloat);
        g_gate = (gf * sp_rows.index_select(0, *hm_rows).to(at::kFloat)).sum().view(hm_gate->sizes()).to(hm_gate->scalar_type());
        g_sp = g_sp.reshape({B * S, h}).to(at::kFloat).index_add(0, *hm_rows, gf * hm_gate->to(at::kFloat)).to(t).view({B, S, h});
    }
    at::Tensor du = op_gelu_backward_split(g_sp, gi, pre, S), du2 = du.view({M, h});
    at::Tensor gx = need_x ? op_adapter_rows_res(c10::nullopt, du, saved[S_WDT], none, c10::nullopt, x_f32 ? go : goc, x_f32)
                           : none;
    at::Tensor gw_d = need_wd ? op_linear_wgrad(du2, no_rows, xc.view({M, E}), f32[0]) : none;
    at::Tensor gb_d = has_bd ? L.grad(op_column_sums(du2), want(1)) : none;
    std::vector<at::Tensor> ret{gx, gw_d, gb_d, L.grad(gw_c, want(2)), has_bc ? L.grad(gb_c, want(3)) : none,
                                L.grad(gw_u, want(4)), b_u.numel() ? L.grad(gb_u, want(5)) : none, g_gamma, g_gate};
    L.launch(st);
    ret.insert(ret.end(), ag.begin(), ag.end());
    return ret;
}

PYBIND11_MODULE(opentad_sparse_ops, m) {
    m.def("adapter_forward", &op_adapter_forward, "The sparse-conv adapter's forward over whole token tiles");
    m.def("adapter_backward", &op_adapter_backward, "Its backward");
    m.def("layer_norm_rows", &op_layer_norm_rows, "LayerNorm of rows of 128 or 256 channels (y, stats)", py::arg("x"),
          py::arg("w"), py::arg("b"), py::arg("eps"));
    m.def("layer_norm_rows_bwd", &op_layer_norm_rows_bwd, "LayerNorm backward (dx, [dw, db])", py::arg("dy"), py::arg("x"),
          py::arg("stats"), py::arg("w"));
    m.def("key_attention_ok", &op_key_attention_ok, "Whether key_attention takes these sizes", py::arg("heads"),
          py::arg("head_dim"), py::arg("n"), py::arg("nk"));
    m.def("key_attention_layers_ok", &op_key_attention_layers_ok, "Whether the key-token attention takes these parameters",
          py::arg("parameters"), py::arg("hidden"), py::arg("heads"), py::arg("n"), py::arg("nk"));
    m.def("key_attention", &op_key_attention, "Normalised attention of the visual tokens to the key tokens", py::arg("q"),
          py::arg("kv"), py::arg("qn_w"), py::arg("qn_b"), py::arg("kn_w"), py::arg("kn_b"), py::arg("eps"));
    m.def("key_attention_bwd", &op_key_attention_bwd, "Its gradients (dq, dkv, norm parameters)", py::arg("dout"),
          py::arg("q"), py::arg("kv"), py::arg("qn_w"), py::arg("qn_b"), py::arg("kn_w"), py::arg("kn_b"), py::arg("eps"));
    m.doc() = "MI355X (gfx950) SparseConv2D: drop-in for the reference opentad_sparse_ops";
    m.def("fwd", &op_fwd, "Forward", py::arg("x"), py::arg("neighbor_indices"), py::arg("weight"),
          py::arg("C_out"), py::arg("tokens_per_batch"));
    m.def("bwd_in", &op_bwd_in, "Backward Input", py::arg("grad_output"),
          py::arg("neighbor_indices"), py::arg("weight"), py::arg("n_kept"), py::arg("C_in"),
          py::arg("tokens_per_batch"));
    m.def("bwd_w", &op_bwd_w, "Backward Weight", py::arg("grad_output"), py::arg("x"),
          py::arg("neighbor_indices"), py::arg("C_in"), py::arg("tokens_per_batch"));
    m.def("implicit_gemm_fwd_v2", &op_implicit_gemm_fwd_v2, "Implicit GEMM forward (fused bias)",
          py::arg("x"), py::arg("neighbor_indices"), py::arg("weight"), py::arg("bias"),
          py::arg("tokens_per_batch"));
    m.def("implicit_gemm_fwd_v2_chunked", &op_implicit_gemm_fwd_v2_chunked,
          "Implicit GEMM forward (chunk_size accepted, not needed)", py::arg("x"),
          py::arg("neighbor_indices"), py::arg("weight"), py::arg("bias"),
          py::arg("tokens_per_batch"), py::arg("chunk_size"));
    m.def("fwd_bias", &op_fwd_bias, "Forward with bias_mode 0 none / 1 fp32 / 2 after rounding",
          py::arg("x"), py::arg("neighbor_indices"), py::arg("weight"), py::arg("bias"),
          py::arg("tokens_per_batch"), py::arg("bias_mode"));
    m.def("pack_weight", &op_pack_weight, "Weight in the matrix-core fragment order (fwd, bwd_in)",
          py::arg("weight"), py::arg("fwd") = true, py::arg("bwd") = true);
    m.def("fwd_packed", &op_fwd_packed, "fwd_bias with a packed weight", py::arg("x"),
          py::arg("neighbor_indices"), py::arg("weight"), py::arg("packed_fwd"), py::arg("bias"),
          py::arg("tokens_per_batch"), py::arg("bias_mode"));
    m.def("bwd_in_packed", &op_bwd_in_packed, "bwd_in with a packed weight", py::arg("grad_output"),
          py::arg("neighbor_indices"), py::arg("weight"), py::arg("packed_bwd"), py::arg("n_kept"),
          py::arg("C_in"), py::arg("tokens_per_batch"), py::arg("symmetric") = false);
    m.def("bwd_packed", &op_bwd_packed, "bwd_in_packed + bwd_w_bias in one call",
          py::arg("grad_output"), py::arg("x"), py::arg("neighbor_indices"), py::arg("weight"),
          py::arg("packed_bwd"), py::arg("C_in"), py::arg("tokens_per_batch"), py::arg("with_bias"),
          py::arg("symmetric") = false);
    m.def("bwd_in_gemm", &op_bwd_in_gemm, "Backward-input gathered GEMM only (timing)", py::arg("grad_output"),
          py::arg("neighbor_indices"), py::arg("packed_bwd"), py::arg("C_in"), py::arg("tokens_per_batch"),
          py::arg("symmetric") = false);
    m.def("bwd_w_partials", &op_bwd_w_partials, "Backward-weight partial sums only (timing)",
          py::arg("grad_output"), py::arg("x"), py::arg("neighbor_indices"), py::arg("C_in"),
          py::arg("tokens_per_batch"), py::arg("with_bias"));
    m.def("bwd_w_bias", &op_bwd_w_bias, "Backward weight and bias", py::arg("grad_output"),
          py::arg("x"), py::arg("neighbor_indices"), py::arg("C_in"), py::arg("tokens_per_batch"),
          py::arg("with_bias"));
    m.def("dw_fwd", &op_dw_fwd, "Depthwise forward", py::arg("x"), py::arg("neighbor_indices"),
          py::arg("weight"), py::arg("bias"), py::arg("tokens_per_batch"));
    m.def("dw_bwd_in", &op_dw_bwd_in, "Depthwise backward input", py::arg("grad_output"),
          py::arg("neighbor_indices"), py::arg("weight"), py::arg("tokens_per_batch"),
          py::arg("symmetric") = false);
    m.def("dw_bwd", &op_dw_bwd, "Depthwise backward input, weight and bias in one call",
          py::arg("grad_output"), py::arg("x"), py::arg("neighbor_indices"), py::arg("weight"),
          py::arg("tokens_per_batch"), py::arg("with_bias"), py::arg("symmetric") = false);
    m.def("dw_bwd_w", &op_dw_bwd_w, "Depthwise backward weight and bias", py::arg("grad_output"),
          py::arg("x"), py::arg("neighbor_indices"), py::arg("tokens_per_batch"),
          py::arg("with_bias"));
    m.def("build_neighbor_table", &op_build_neighbor_table, "Neighbor table from a keep mask",
          py::arg("mask"));
    m.def("build_neighbor_table_n", &op_build_neighbor_table_n,
          "Neighbor table from a keep mask with a known row count (one launch, no host sync)",
          py::arg("mask"), py::arg("n_rows"), py::arg("int64_out") = false);
    m.def("grid_neighbor_table", &op_grid_neighbor_table, "Full-grid neighbor table in closed form (one launch)",
          py::arg("frames"), py::arg("h"), py::arg("w"), py::arg("int64_out"), py::arg("like"));
    m.def("table_to_global", &op_table_to_global,
          "int32 global table from a local or global one by the max() < N rule, on the device",
          py::arg("neighbor_indices"), py::arg("tokens_per_batch"));
    m.def("remap_neighbor_table", &op_remap_neighbor_table, "Neighbor table remap after a prune",
          py::arg("table"), py::arg("keep_idx"));
    m.def("prune_tokens", &op_prune_tokens,
          "Fused prune step: kept-token gather, index gather and table remap",
          py::arg("x"), py::arg("keep_idx"), py::arg("last_idx"), py::arg("neighbor_indices"),
          py::arg("num_key_tokens"));
    m.def("transpose_neighbor_table", &op_transpose_neighbor_table, "Transposed neighbor table",
          py::arg("table"), py::arg("tokens_per_batch") = 0);
    m.def("validate_neighbor_table", &op_validate_neighbor_table,
          "(out-of-range count, min, max) of a neighbor table", py::arg("table"), py::arg("bound"));
    m.def("adapter_down", &op_adapter_down, "Adapter down_proj + GELU + special / patch split",
          py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("n_special"));
    m.def("adapter_up", &op_adapter_up, "Adapter up_proj on cat(special, patch) * gamma + residual",
          py::arg("a_special"), py::arg("a_patch"), py::arg("weight"), py::arg("bias"), py::arg("gamma"),
          py::arg("residual"), py::arg("out_float32") = false);
    m.def("adapter_rows_ok", &op_adapter_rows_ok, "Whether the adapter GEMMs over whole token tiles take these widths",
          py::arg("embed"), py::arg("hidden"));
    m.def("adapter_prep", &op_adapter_prep, "Adapter parameters cast and laid out for adapter_rows_*, one launch",
          py::arg("w_d"), py::arg("b_d"), py::arg("w_c"), py::arg("b_c"), py::arg("w_u"), py::arg("b_u"),
          py::arg("gamma"), py::arg("bf16"), py::arg("train"), py::arg("pack_conv"));
    m.def("patch_rows", &op_patch_rows, "Rows of the patch tokens of [B, N, .]", py::arg("like"), py::arg("batch"),
          py::arg("n_tokens"), py::arg("n_special"));
    m.def("adapter_rows_down", &op_adapter_rows_down, "adapter_down over whole token tiles (weight of adapter_prep)",
          py::arg("x"), py::arg("w"), py::arg("bias"), py::arg("n"), py::arg("n_special"), py::arg("copy"));
    m.def("adapter_rows_split", &op_adapter_rows_split, "go W^T split into special and patch rows",
          py::arg("go"), py::arg("w"), py::arg("n"), py::arg("n_special"), py::arg("copy"));
    m.def("adapter_rows_res", &op_adapter_rows_res, "adapter_up over whole token tiles, or A W^T + residual",
          py::arg("a_special"), py::arg("a"), py::arg("w"), py::arg("bias"), py::arg("gamma"), py::arg("residual"),
          py::arg("out_float32") = false);
    m.def("heatmap_add_", &op_heatmap_add_, "In place: patch[i] += special[src_rows[i]] * gate (adapter heatmap injection)",
          py::arg("patch"), py::arg("special"), py::arg("src_rows"), py::arg("gate"));
    m.def("linear_wgrad", &op_linear_wgrad, "Linear-layer weight gradient g[rows]^T x (split rows, ordered sum)",
          py::arg("g"), py::arg("rows"), py::arg("x"), py::arg("out_float32") = false);
    m.def("column_sums", &op_column_sums, "Column sums of a [rows, cols] matrix (ordered, fp32 accumulation)",
          py::arg("a"));
    m.def("gelu_backward_split", &op_gelu_backward_split,
          "GELU backward of the adapter's down projection from split special / patch gradients",
          py::arg("grad_special"), py::arg("grad_patch"), py::arg("pre_act"), py::arg("n_special"));
    m.def("up_proj_grads", &op_up_proj_grads,
          "Adapter up projection: gamma gradient plus w, g, gs scaled by gamma, in one pass",
          py::arg("w"), py::arg("g"), py::arg("b"), py::arg("gs"), py::arg("gamma"));
    m.def("gamma_grad", &op_gamma_grad, "sum(w * g) + sum(b * gs) in fp32 (the adapter's gamma gradient)",
          py::arg("w"), py::arg("g"), py::arg("b"), py::arg("gs"));
    m.def("version", []() { return std::string(svtad_version()); });
}
