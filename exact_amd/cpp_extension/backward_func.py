"""Stand-in for the reference's `exact.cpp_extension.backward_func` module
(backward_func.cc:83-107).  The reference only re-exports ATen routines plus
the two-GEMM linear backward, which are reachable from Python as they are;
its one kernel of its own, the ELU derivative, is a kernel of the library."""
import functools

import torch

from .. import _lib
from ..conf import config
from . import _checks


@functools.lru_cache(maxsize=512)
def _scratch_size(entry, *sizes):
    """What a size entry of the library answers: a function of the sizes alone."""
    return int(getattr(_lib.lib(), entry)(*sizes))


def _atomics_allowed():
    """The library's reductions meet in memory through atomics; both the
    framework's deterministic mode and config.deterministic_reductions ask for
    reproducible sums instead."""
    return not (torch.are_deterministic_algorithms_enabled() or config.deterministic_reductions)


def column_sums(matrix):
    """`matrix.sum(0)` of a 2-D tensor.  fp32 device matrices go through the
    library's streaming kernel (the framework's reduction runs far off the
    memory roofline for narrow matrices: 19 ms for [2.4M, 47]); its atomics
    fix no summation order, so deterministic mode
    (config.deterministic_reductions or the framework's own switch) and
    everything else keep the framework's reduction."""
    usable = (matrix.dim() == 2 and matrix.dtype == torch.float32 and _checks.on_device(matrix)
              and matrix.is_contiguous() and 0 < matrix.shape[1] <= 256 and matrix.shape[0] >= 4096
              and _atomics_allowed())
    if not usable:
        return matrix.sum(0)
    out = torch.empty(matrix.shape[1], dtype=torch.float32, device=matrix.device)
    rc = _lib.lib().exact_colsum_f32(_checks.ptr(matrix), matrix.shape[0], matrix.shape[1], _checks.ptr(out),
                                     _checks.stream_ptr(matrix))
    _lib.check(rc, "column_sums")
    return out


def batch_statistics(matrix):
    """(biased variance, mean) of every column of a 2-D tensor by the framework's
    reduction: for the matrices that batch_norm_statistics does not take."""
    return torch.var_mean(matrix, dim=0, unbiased=False)


def _short_weight_gradient(grad_output, input):  # noqa: A002
    """Whether exact_linear_dw_short_f32 takes the product: 4096 to 16383 rows and at
    most 65536 results, on plain tensors that no derivative is recorded for.  Device
    time against the framework's GEMM, from 1 x 1 to 1024 x 64 results: 0.99 to 5.4
    times as fast at 4096 rows, 1.3 to 9.7 at 8192, 2 to 11 at 16383; from 16384 rows on
    the forms of weight_gradient are faster.  More results, 256 x 602: 0.67, 0.80 and
    1.13.  Fewer rows have no one answer, since the framework splits them for some
    shapes and not for others: 256 x 256 takes 16 against 225 us at 1000 rows and 21
    against 17 at 2000, 128 x 512 17 against 11 and 21 against 17, 64 x 64 10 against 20
    and 22; they stay with the framework."""
    return (grad_output.dtype == torch.float32 and input.dtype == torch.float32 and grad_output.dim() == 2 and input.dim() == 2
            and 4096 <= grad_output.shape[0] < 16384 and grad_output.shape[0] == input.shape[0]
            and 0 < grad_output.shape[1] * input.shape[1] <= 65536
            and _checks.on_device(grad_output) and _checks.on_device(input) and grad_output.device == input.device
            and not _checks.recorded(grad_output, input) and _checks.plain_values(grad_output, input)
            and grad_output.stride(1) == 1 and input.stride(1) == 1
            and grad_output.stride(0) >= grad_output.shape[1] and input.stride(0) >= input.shape[1]
            and _atomics_allowed())


def weight_gradient(grad_output, input):  # noqa: A002
    """`grad_output.t().mm(input)` (backward_func.cc:88-89): [N, out]^T . [N, in].
    Tall device operands take the library's matrix-core kernel for this shape: fp32
    ones on the bf16 instruction with operands split in three, or on the fp32
    instruction (config.matrix_cores), whose slabs meet through atomics; fp16 ones on
    the fp16 instruction, whose slabs are added in a fixed order.  Shorter fp32
    operands (_short_weight_gradient) take the fp32 instruction with their slabs in a
    fixed order.  Deterministic mode and everything else keep the framework's GEMM."""
    half = (grad_output.dtype == torch.float16 and input.dtype == torch.float16 and config.matrix_cores == "bf16"
            and not _checks.recorded(grad_output, input))
    usable = (grad_output.dim() == 2 and input.dim() == 2 and (half or (grad_output.dtype == torch.float32
              and input.dtype == torch.float32)) and _checks.on_device(grad_output) and _checks.on_device(input)
              and grad_output.shape[0] == input.shape[0] and grad_output.shape[0] >= 16384
              and 0 < grad_output.shape[1] <= 1024 and 0 < input.shape[1] <= 1024
              and grad_output.stride(1) == 1 and input.stride(1) == 1
              and grad_output.stride(0) >= grad_output.shape[1] and input.stride(0) >= input.shape[1]
              and _atomics_allowed())
    if not usable:
        if _short_weight_gradient(grad_output, input):
            N, K = grad_output.shape
            D = input.shape[1]
            out = torch.empty((K, D), dtype=torch.float32, device=grad_output.device)
            work = torch.empty(_scratch_size("exact_linear_dw_short_work_nbytes", N, K, D), dtype=torch.uint8, device=grad_output.device)
            rc = _lib.lib().exact_linear_dw_short_f32(_checks.ptr(grad_output), grad_output.stride(0), _checks.ptr(input),
                                                      input.stride(0), N, K, D, _checks.ptr(out), _checks.ptr(work),
                                                      _checks.stream_ptr(grad_output))
            _lib.check(rc, "weight_gradient")
            return out
        return grad_output.t().mm(input)
    N, K = grad_output.shape
    D = input.shape[1]
    if half:
        L = _lib.lib()
        out = torch.empty((K, D), dtype=torch.float16, device=grad_output.device)
        work = torch.empty(_scratch_size("exact_linear_dw_f16_work_nbytes", N, K, D), dtype=torch.uint8, device=grad_output.device)
        rc = L.exact_linear_dw_ordered_f16(_checks.ptr(grad_output), grad_output.stride(0), _checks.ptr(input), input.stride(0),
                                           N, K, D, _checks.ptr(out), _checks.ptr(work), _checks.stream_ptr(grad_output))
        _lib.check(rc, "weight_gradient")
        return out
    out = torch.empty((K, D), dtype=torch.float32, device=grad_output.device)
    if config.matrix_cores not in ("bf16", "fp32"):
        raise ValueError("config.matrix_cores must be 'bf16' or 'fp32'")
    kernel = _lib.lib().exact_linear_dw_bf16_f32 if config.matrix_cores == "bf16" else _lib.lib().exact_linear_dw_f32
    rc = kernel(_checks.ptr(grad_output), grad_output.stride(0), _checks.ptr(input), input.stride(0),
                N, K, D, _checks.ptr(out), _checks.stream_ptr(grad_output))
    _lib.check(rc, "weight_gradient")
    return out


# ---- the dense products of a layer on the bf16 matrix cores ---------------------
def _worth_a_tall_product(N, D, K):
    """Whether exact_tall_product_f32 is the faster routine.  Its workgroups take 128
    rows by up to 128 columns and walk the whole depth: where they are too few to
    hide the loads of a step, the framework's GEMM, which can split the depth, wins
    by up to three times.  Measured, kernel / framework: at 128 workgroups (16,384
    rows) 0.87 - 0.97 up to 128 features, 1.0 at 180, 1.2 - 1.4 at 256, 1.4 - 3.1
    from 602 on; at 256 of them the same up to 180, 1.2 - 1.3 beyond; at 313 (40,000
    rows) 0.6 - 0.9 up to 602 and 1.0 - 1.24 beyond, with 32 columns or fewer 0.9 at
    256 and 1.4 from 602 on; from 626 on 0.5 - 0.9 nearly everywhere."""
    groups = -(-N // 128) * -(-K // 128)
    return groups >= 512 or D <= 160 or (groups >= 280 and D <= (800 if K > 32 else 400))


def tall_matmul(x, matrix, transposed=False, bias=None, addend=None, into=None):
    """x[N, D] . M (+ bias[K]) (+ addend[N, K]) -> [N, K], where M = `matrix`
    ([D, K]) or, with transposed=True, the transpose of `matrix` ([K, D]: a weight
    as F.linear holds it).  `into` names the result tensor; it may be `addend`
    itself (accumulate in place).  Tall fp32 device operands (config.tall_gemm_min_rows)
    with an even number of features, where the sizes suit it (_worth_a_tall_product, or
    config.tall_gemm_min_depth and tall_gemm_max_rows_wide), take the library's kernel (six bf16 matrix-core
    products per fp32 product, fp32 accuracy, reproducible, infinities and the ends
    of the range as in fp32; config.matrix_cores == "bf16"); everything else the
    framework's GEMM."""
    M = matrix.t() if transposed else matrix
    usable = (config.matrix_cores == "bf16" and x.dim() == 2 and matrix.dim() == 2 and x.dtype == torch.float32
              and matrix.dtype == torch.float32 and _checks.on_device(x) and _checks.on_device(matrix)
              and x.shape[1] == M.shape[0] and x.shape[0] >= config.tall_gemm_min_rows and x.shape[1] % 2 == 0
              and 0 < x.shape[1] <= 4096 and 0 < M.shape[1] <= 4096
              and (M.shape[1] <= 64 or (x.shape[1] >= config.tall_gemm_min_depth and x.shape[0] <= config.tall_gemm_max_rows_wide))
              and (config.tall_gemm_min_depth != 0 or _worth_a_tall_product(*x.shape, M.shape[1]))
              and x.is_contiguous() and x.data_ptr() % 8 == 0
              and matrix.stride(1) == 1 and matrix.stride(0) >= matrix.shape[1]
              and (bias is None or (bias.dtype == torch.float32 and bias.is_contiguous() and bias.numel() == M.shape[1]
                                    and _checks.on_device(bias)))
              and (addend is None or (addend.dtype == torch.float32 and addend.dim() == 2 and addend.stride(1) == 1
                                      and addend.shape == (x.shape[0], M.shape[1]) and _checks.on_device(addend)))
              and (into is None or (into.dtype == torch.float32 and into.dim() == 2 and into.stride(1) == 1
                                    and into.shape == (x.shape[0], M.shape[1]) and _checks.on_device(into)))
              and not (torch.is_grad_enabled() and (x.requires_grad or matrix.requires_grad
                                                    or (bias is not None and bias.requires_grad)
                                                    or (addend is not None and addend.requires_grad))))
    if not usable:
        if addend is not None:
            out = torch.addmm(addend, x, M) if into is None or into is not addend else addend.addmm_(x, M)
            if bias is not None:
                out += bias
        else:
            out = x.mm(M) if bias is None else torch.addmm(bias, x, M)
        if into is not None and into is not out:
            into.copy_(out)
            out = into
        return out
    N, D = x.shape
    K = M.shape[1]
    out = into if into is not None else torch.empty((N, K), dtype=torch.float32, device=x.device)
    # The weight's fragments are made by every call, on its stream and in scratch of its own (one launch of 5 us), and
    # not remembered: a weight changes through `.data` without raising its version, a captured graph has to read the
    # weight of its replay, and another stream would have to wait for the one that made the copy.
    L = _lib.lib()
    work = torch.empty(_scratch_size("exact_tall_product_work_nbytes", D, K), dtype=torch.uint8, device=x.device)
    rc = L.exact_tall_product_f32(_checks.ptr(x), _checks.ptr(matrix), matrix.stride(0), int(bool(transposed)), N, D, K,
                                  _checks.ptr(bias) if bias is not None else None,
                                  _checks.ptr(addend) if addend is not None else None,
                                  addend.stride(0) if addend is not None else K, _checks.ptr(out), out.stride(0),
                                  _checks.ptr(work), _checks.stream_ptr(x))
    _lib.check(rc, "tall_matmul")
    matrix._exact_gemm_table = (D, K)     # a mark for tests and profiles that the kernel took this operand; nothing reads it here
    return out


def linear_backward(grad_output, input, weight, bias, need_input_grad=True):  # noqa: A002
    """backward_func.cc:83-93.  `need_input_grad=False` leaves out the product
    the caller would discard (the reference forms all three regardless)."""
    grad_input = tall_matmul(grad_output, weight) if need_input_grad else None
    grad_weight = weight_gradient(grad_output, input)
    grad_bias = column_sums(grad_output) if bias is not None else None
    return grad_input, grad_weight, grad_bias


def native_batch_norm(input, weight, bias, running_mean, running_var, training, momentum, eps):  # noqa: A002
    # The check of torch.batch_norm, which the native routine leaves to it: it would read and write past a short vector.
    for name, t in (("running_mean", running_mean), ("running_var", running_var), ("weight", weight), ("bias", bias)):
        if t is not None and input.dim() >= 2 and t.numel() != input.shape[1]:
            raise RuntimeError(f"{name} should contain {input.shape[1]} elements not {t.numel()}")
    return torch.ops.aten.native_batch_norm(input, weight, bias, running_mean, running_var, training, momentum, eps)


def native_batch_norm_backward(grad_out, input, weight, running_mean, running_var, save_mean, save_invstd,  # noqa: A002
                               train, eps, output_mask):
    """at::native_batch_norm_backward as re-exported by backward_func.cc:99-104.
    For a tall fp32 [N, K <= 256] training-mode batch on the device, its two
    column reductions (sum of dy, sum of dy * (x - mean)) run in the library's
    one-pass kernel -- the framework's reduction kernel reads the same two
    matrices at a tenth of the memory bandwidth -- and the element-wise half is
    the framework's batch_norm_backward_elemt, which computes
      dx = (dy - sum_dy / N - (x - mean) * invstd^2 * sum_dy_xmu / N) * invstd * weight
    exactly as the one-call routine does."""
    def stat_ok(t, optional=False):
        if t is None:
            return optional
        return t.dtype == torch.float32 and t.device == grad_out.device and t.numel() == grad_out.shape[1]

    fast = (train and grad_out.dim() == 2 and grad_out.is_cuda and grad_out.dtype == torch.float32
            and input.dtype == torch.float32 and input.device == grad_out.device
            and grad_out.is_contiguous() and input.is_contiguous()
            and 4096 <= grad_out.shape[0] < 2 ** 31 and 0 < grad_out.shape[1] <= 256 and grad_out.shape == input.shape
            and stat_ok(save_mean) and stat_ok(save_invstd) and stat_ok(weight, optional=True)
            and _atomics_allowed())
    if not fast:
        return torch.ops.aten.native_batch_norm_backward(grad_out, input, weight, running_mean, running_var,
                                                         save_mean, save_invstd, train, eps, list(output_mask))
    N, K = grad_out.shape
    mean = save_mean.contiguous()
    sums = torch.empty((2, K), dtype=torch.float32, device=grad_out.device)
    rc = _lib.lib().exact_bn_backward_reduce_f32(_checks.ptr(grad_out), _checks.ptr(input), _checks.ptr(mean), N, K,
                                                 _checks.ptr(sums[0]), _checks.ptr(sums[1]), _checks.stream_ptr(grad_out))
    _lib.check(rc, "native_batch_norm_backward")
    sum_dy, sum_dy_xmu = sums[0], sums[1]
    grad_input = grad_weight = grad_bias = None
    if output_mask[0]:
        count = torch.full((1,), N, dtype=torch.int32, device=grad_out.device)
        grad_input = torch.batch_norm_backward_elemt(grad_out, input, mean, save_invstd, weight, sum_dy, sum_dy_xmu, count)
    if output_mask[1]:
        grad_weight = sum_dy_xmu * save_invstd
    if output_mask[2]:
        grad_bias = sum_dy
    return grad_input, grad_weight, grad_bias


def _column_vector(t, matrix):
    """Whether a kernel may read `t` as one fp32 number per column of `matrix` (None: absent)."""
    return t is None or (t.dtype == torch.float32 and t.device == matrix.device and t.is_contiguous() and t.dim() == 1
                         and t.numel() == matrix.shape[1])


def takes_batch_norm_statistics(matrix, weight, running_mean, running_var, bias=None):
    """Whether batch_norm_statistics takes these operands."""
    return (matrix.dim() == 2 and matrix.dtype == torch.float32 and _checks.on_device(matrix) and matrix.is_contiguous()
            and 0 < matrix.shape[1] <= 8192 and 1024 <= matrix.shape[0] < 2 ** 31
            and all(_column_vector(t, matrix) for t in (weight, bias, running_mean, running_var))
            and (running_mean is None) == (running_var is None) and _atomics_allowed())


def batch_norm_statistics(matrix, weight, running_mean, running_var, momentum, eps, bias=None):
    """The statistics half of native_batch_norm in training mode -> (mean,
    1 / sqrt(var + eps), weight * that), with running_mean / running_var updated
    in place; None where the library's kernels do not apply, `bias` for
    batch_norm_apply among what they need (the caller then takes the framework's
    routines, which refuse what is malformed).  From 1024 rows on: below, the
    framework's reduction is no slower."""
    if momentum is None or not takes_batch_norm_statistics(matrix, weight, running_mean, running_var, bias):
        return None
    N, K = matrix.shape
    L = _lib.lib()
    mean, invstd, mult = torch.empty((3, K), dtype=torch.float32, device=matrix.device)
    work = torch.empty(_scratch_size("exact_bn_work_floats", N, K), dtype=torch.float32, device=matrix.device)
    rc = L.exact_bn_statistics_f32(_checks.ptr(matrix), N, K, float(eps), float(momentum), _checks.ptr(weight),
                                   _checks.ptr(running_mean), _checks.ptr(running_var), _checks.ptr(work),
                                   _checks.ptr(mean), _checks.ptr(invstd), _checks.ptr(mult), _checks.stream_ptr(matrix))
    _lib.check(rc, "batch_norm_statistics")
    if running_mean is not None:
        torch.autograd.graph.increment_version((running_mean, running_var))
    return mean, invstd, mult


def batch_norm_apply(matrix, mean, mult, bias):
    """(matrix - mean) * mult + bias per column, for the statistics above."""
    if not (matrix.dim() == 2 and matrix.dtype == torch.float32 and _checks.on_device(matrix) and matrix.is_contiguous()
            and mean is not None and mult is not None and all(_column_vector(t, matrix) for t in (mean, mult, bias))):
        raise RuntimeError("batch_norm_apply: an fp32 matrix and one fp32 number per column on its device are needed")
    out = torch.empty_like(matrix)
    rc = _lib.lib().exact_bn_apply_f32(_checks.ptr(matrix), _checks.ptr(mean), _checks.ptr(mult), _checks.ptr(bias), *matrix.shape,
                                       _checks.ptr(out), _checks.stream_ptr(matrix))
    _lib.check(rc, "batch_norm_apply")
    return out


def batch_norm_backward_packed(grad_out, mask, p, quantized, weight, mean, invstd, output_mask):
    """native_batch_norm_backward on an input that is still packed, behind a joint
    ReLU / dropout mask where `mask` is given (dropout_bwd): -> (grad_input,
    grad_weight, grad_bias), or None where the kernels do not apply (the caller
    then dequantises and takes the separate routines)."""
    packed, bits, scale, mn = quantized
    vectors = [t for t in (mean, invstd, weight) if t is not None]
    usable = (bits in (1, 2, 4, 8) and grad_out.dim() == 2 and grad_out.dtype == torch.float32 and _checks.on_device(grad_out)
              and grad_out.is_contiguous() and grad_out.data_ptr() % 16 == 0
              and 1024 <= grad_out.shape[0] < 2 ** 31 and 0 < grad_out.shape[1] <= 8192 and grad_out.shape[1] % 4 == 0
              and packed.dtype == torch.int8 and packed.is_contiguous() and packed.data_ptr() % 4 == 0
              and packed.numel() * (8 // bits) >= grad_out.numel()
              and scale.dtype == torch.bfloat16 and mn.dtype == torch.bfloat16
              and scale.numel() == mn.numel() == grad_out.shape[0] and scale.is_contiguous() and mn.is_contiguous()
              and all(t.device == grad_out.device for t in (packed, scale, mn, *vectors))
              and all(_column_vector(t, grad_out) for t in vectors)
              and (mask is None or (mask.dtype == torch.int32 and mask.device == grad_out.device and mask.is_contiguous()
                                    and mask.numel() * 32 >= grad_out.numel()))
              and not _checks.recorded(grad_out, weight)
              and _atomics_allowed())
    if not usable:
        return None
    N, K = grad_out.shape
    L = _lib.lib()
    sums = torch.empty((2, K), dtype=torch.float32, device=grad_out.device)
    work = torch.empty(_scratch_size("exact_bn_work_floats", N, K), dtype=torch.float32, device=grad_out.device)
    grad_input = torch.empty_like(grad_out) if output_mask[0] else None
    grad_weight = torch.empty(K, dtype=torch.float32, device=grad_out.device) if output_mask[1] else None
    rc = L.exact_bn_backward_ordered_f32(_checks.ptr(grad_out), _checks.ptr(mask), float(p), _checks.ptr(packed), bits,
                                         _checks.ptr(scale), _checks.ptr(mn), _checks.ptr(mean), _checks.ptr(invstd),
                                         _checks.ptr(weight), N, K, _checks.ptr(work), _checks.ptr(sums), _checks.ptr(grad_input),
                                         _checks.ptr(grad_weight), _checks.stream_ptr(grad_out))
    _lib.check(rc, "batch_norm_backward_packed")
    return grad_input, grad_weight, sums[0] if output_mask[2] else None


def _elu_backward_cuda(grad_output, data, alpha):
    """backward_func_cuda_kernel.cu:6-36: x >= 0 ? grad : alpha * grad * exp(x)."""
    grad_output, data = grad_output.contiguous(), data.contiguous()
    _checks.check_device_tensor(grad_output, "grad_output", None, _checks.FLOAT_OR_HALF)
    _checks.check_device_tensor(data, "data", None, (grad_output.dtype,))
    if data.numel() != grad_output.numel():
        raise RuntimeError("grad_output and data must have the same number of elements")
    grad_input = torch.empty_like(grad_output)
    fn = getattr(_lib.lib(), "exact_elu_bwd_" + _checks.suffix(grad_output))
    rc = fn(_checks.ptr(grad_output), _checks.ptr(data), float(alpha), grad_output.numel(), _checks.ptr(grad_input),
            _checks.stream_ptr(grad_output))
    _lib.check(rc, "_elu_backward_cuda")
    return grad_input
