// PyTorch module `sc_extension_cuda`: the GPU entry points the reference's Python binds by
// name (utils_functional.py:12, call sites :497-513; C++ side sc_cuda.cpp:21-83), same
// positional signatures, implemented on libgeo_sc.so (gfx950).
#include "sc_torch_common.h"

using namespace geo_sc_torch;

// sc_cuda.cpp:47-63.  dim != 0: y-dimension partial binary accumulation (the default of the
// reference's training script): OR over (c_in, w_k), add over h_k.  dim == 0: z-dimension
// accumulation: OR over the kernel window, add over c_in.
at::Tensor conv2d_add_partial_variable_acc(torch::Tensor input, torch::Tensor weight, int64_t bit_length,
                                           at::IntArrayRef padding, at::IntArrayRef stride, int64_t total_width,
                                           int64_t load_width, int64_t load_wait, bool im2col, int64_t dim)
{
    (void)stride;  // accepted and ignored, as in the reference (stride 1 only)
    (void)im2col;  // selects an equivalent kernel variant in the reference; no effect on results
    // the y/z ops use one load_wait for weights and activations (sc_cuda_kernel.cu:1821-1823, :2119)
    const geo_sc_conv_desc d = make_desc(input, weight, bit_length, padding, total_width, load_width, load_wait,
                                         load_wait, dim == 0 ? GEO_SC_ACC_Z : GEO_SC_ACC_Y);
    return forward_on_device(input, weight, d);
}

// sc_cuda.cpp:34-45: OR over (z_unit consecutive input channels, w_k), add over h_k and over
// the channel groups; separate load_wait for the weight and activation generators.
at::Tensor conv2d_add_yz_variable_acc(torch::Tensor input, torch::Tensor weight, int64_t bit_length,
                                      at::IntArrayRef padding, at::IntArrayRef stride, int64_t total_width,
                                      int64_t load_width, int64_t load_wait_w, int64_t load_wait_a, bool im2col,
                                      int64_t z_unit)
{
    (void)stride;
    (void)im2col;
    const geo_sc_conv_desc d = make_desc(input, weight, bit_length, padding, total_width, load_width, load_wait_w,
                                         load_wait_a, GEO_SC_ACC_YZ, z_unit);
    return forward_on_device(input, weight, d);
}

// sc_cuda.cpp:65-76: y-dimension accumulation with the "accurate random" generator (streams with
// exactly `code` ones).  The reference seeds its generators with constants (37 for the weights, 0
// for the activations, sc_cuda_kernel.cu:1885, :1957), so it returns the same result on every call;
// so does this, with its own counter-based generator: same distribution, other bits.
at::Tensor conv2d_add_partial_acc_acc(torch::Tensor input, torch::Tensor weight, int64_t bit_length,
                                      at::IntArrayRef padding, at::IntArrayRef stride, bool share, int64_t dim)
{
    (void)stride;
    (void)share;  // forced off inside the reference's kernels (sc_cuda_kernel.cu:372, :495)
    (void)dim;    // unused by the reference (sc_cuda.cpp:75)
    const geo_sc_conv_desc d = make_desc(input, weight, bit_length, padding, 7, 8, 1, 1, GEO_SC_ACC_Y, 1,
                                         GEO_SC_GEN_ACC, 37);
    return forward_on_device(input, weight, d);
}

// sc_cuda.cpp:21-32: OR over the whole kernel window and all input channels, Bernoulli random streams.
at::Tensor conv2d_or_acc(torch::Tensor input, torch::Tensor weight, int64_t bit_length, at::IntArrayRef padding,
                         at::IntArrayRef stride, bool im2col)
{
    (void)stride;
    (void)im2col;  // selects where the reference generates its streams; same distribution either way
    const geo_sc_conv_desc d = make_desc(input, weight, bit_length, padding, 7, 8, 1, 1, GEO_SC_ACC_FULL, 1,
                                         GEO_SC_GEN_RAND, 0);
    return forward_on_device(input, weight, d);
}

// The value and the scale of BatchNorm*_fixed on given statistics (utils_class.py:49-64): the weight, its mean as
// PyTorch reduces it (which the chain of operations takes the scale from), the pass over x.  Nothing where the kernel does
// not take the tensors.  In C++ because it is three launches for what was one ctypes call: host time of the 4-layer
// CNN's forward on one image 515 us with ctypes calls, 393 here (423 with the one launch and a mean in double precision).
std::optional<std::tuple<at::Tensor, at::Tensor>> bn_fixed_eval(const at::Tensor& x, const at::Tensor& mean, const at::Tensor& var,
                                                                const std::optional<at::Tensor>& gamma,
                                                                const std::optional<at::Tensor>& beta, double eps)
{
    const auto plain = [&](const at::Tensor& t) {
        return t.is_cuda() && t.device() == x.device() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided &&
               t.is_contiguous() && !t.is_neg();
    };
    if (x.dim() < 2 || !plain(x) || x.numel() < 1 || x.numel() > 0x7fffffff || x.size(1) > 4096) return std::nullopt;
    const int64_t c = x.size(1);
    const auto per_channel = [&](const at::Tensor& t) { return plain(t) && t.dim() == 1 && t.size(0) == c; };
    if (!per_channel(mean) || !per_channel(var) || (gamma && !per_channel(*gamma)) || (beta && !per_channel(*beta)))
        return std::nullopt;
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    geo_sc_stream_t stream = (geo_sc_stream_t)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream();
    const float* gm = gamma ? gamma->const_data_ptr<float>() : nullptr;
    const float* bt = beta ? beta->const_data_ptr<float>() : nullptr;
    const at::Tensor w = at::empty({c}, x.options());
    check_status(geo_sc_bn_eval_weight(var.const_data_ptr<float>(), gm, (int)c, (float)eps, w.data_ptr<float>(), stream),
                 "batch norm weight");
    const at::Tensor w_mean = at::mean(w);
    at::Tensor y = at::empty_like(x), scale = at::empty({}, x.options());
    check_status(geo_sc_bn_fixed_eval_mean(x.const_data_ptr<float>(), (int)x.size(0), (int)c, (int)(x.numel() / (x.size(0) * c)),
                                           mean.const_data_ptr<float>(), var.const_data_ptr<float>(), gm, bt, (float)eps,
                                           w_mean.const_data_ptr<float>(), y.data_ptr<float>(), scale.data_ptr<float>(), stream),
                 "batch norm in eval mode");
    return std::make_tuple(y, scale);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("conv2d_add_partial_variable_acc", &conv2d_add_partial_variable_acc,
          "SC forward conv2d partial (y or z dimension) bin add, variable load, lfsr generator");
    m.def("conv2d_add_yz_variable_acc", &conv2d_add_yz_variable_acc,
          "SC forward conv2d partial (yz dimension) bin add, variable load, lfsr generator");
    m.def("conv2d_add_partial_acc_acc", &conv2d_add_partial_acc_acc,
          "SC forward conv2d partial bin add, accurate random generator");
    m.def("conv2d_or_acc", &conv2d_or_acc, "SC forward conv2d or add, random generator");
    m.def("_bn_fixed_eval", &bn_fixed_eval, "fixed-point batch norm on given statistics: (y, scale), or None");
}
