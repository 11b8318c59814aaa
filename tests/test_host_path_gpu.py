"""The C++ host path of the per-layer operators (csrc/host.cpp) returns what the operators called one by
one return, bit for bit, at the edges of what it takes: one row, inputs of more than two dimensions, codes
that outgrow the kept scratch, every mode with and without bias; and it leaves to Python what something
watches or what needs a conversion."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from oracle import w8a8_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def loaded(gpu):
    from sglang_amd import _lib

    _lib.load()  # (the host path takes no call before the library's addresses are bound)


def say(*a):
    print(*a, flush=True)


def same(a, b):
    assert a.shape == b.shape and a.dtype == b.dtype
    assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


def block_weight(n, k, gpu, int8=False):
    w = O.gen_weight(n, k, seed=n + k)
    if int8:
        s = torch.rand(((n + 127) // 128, k // 128), generator=torch.Generator().manual_seed(n)) * 1e-3 + 1e-4
        return torch.randint(-127, 128, (n, k), dtype=torch.int8, generator=torch.Generator().manual_seed(k)).to(gpu), s.to(gpu)
    q, s = O.block_quant_weight(w)
    return q.to(gpu), s.to(gpu)


@pytest.mark.parametrize("shape,n,k,dtype", [((1,), 576, 512, torch.bfloat16), ((3, 5), 264, 1152, torch.float16), ((77,), 512, 640, torch.bfloat16),
                                             ((2, 700), 1024, 13056, torch.bfloat16)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_block_linears(gpu, shape, n, k, dtype, with_bias):
    from sglang_amd._lib import native
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8
    from sglang_amd.quantization.fp8_utils import w8a8_block_fp8_linear
    from sglang_amd.quantization.int8_utils import apply_w8a8_block_int8_linear
    from sglang_amd.quantization.int8_kernel import per_token_group_quant_int8, w8a8_block_int8_matmul
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm

    g = torch.Generator().manual_seed(n)
    x = torch.randn((*shape, k), generator=g).to(dtype).to(gpu)
    bias = (torch.randn((n,), generator=g) * 0.1).to(dtype).to(gpu) if with_bias else None
    say("block linears", shape, n, k, dtype, with_bias)
    w, s = block_weight(n, k, gpu)
    assert native.block_linear(x, w, s, bias, 0, 1e-10) is not None
    q, xs = sglang_per_token_group_quant_fp8(x.view(-1, k), 128, column_major_scales=True)
    want = torch.ops.sgl_kernel.fp8_blockwise_scaled_mm(q, w.t(), xs, s.t(), dtype)
    same(fp8_blockwise_scaled_mm(q, w.t(), xs, s.t(), dtype), want)
    if with_bias:
        want = want + bias
    same(w8a8_block_fp8_linear(x, w, [128, 128], s, bias=bias), want.view(*shape, n))
    w, s = block_weight(n, k, gpu, int8=True)
    q, xs = per_token_group_quant_int8(x.view(-1, k), 128)
    want = w8a8_block_int8_matmul(q, w, xs, s, [128, 128], output_dtype=dtype)
    if with_bias:
        want = want + bias
    same(apply_w8a8_block_int8_linear(x, w, [128, 128], s, bias=bias), want.view(*shape, n))


@pytest.mark.parametrize("shape,n,k,dtype", [((1,), 16, 512, torch.bfloat16), ((2, 3), 264, 1136, torch.float16), ((2, 700), 520, 13056, torch.bfloat16)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_token_linears(gpu, shape, n, k, dtype, with_bias):
    from sglang_amd._lib import native
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_quant_fp8
    from sglang_amd.quantization.fp8_utils import apply_fp8_linear
    from sglang_amd.quantization.int8_kernel import per_token_quant_int8
    from sglang_amd.quantization.w8a8_int8 import apply_w8a8_int8_linear

    g = torch.Generator().manual_seed(n)
    x = torch.randn((*shape, k), generator=g).to(dtype).to(gpu)
    bias = (torch.randn((n,), generator=g) * 0.1).to(dtype).to(gpu) if with_bias else None
    s = (torch.rand((n, 1), generator=g) * 1e-2 + 1e-3).to(gpu)
    say("token linears", shape, n, k, dtype, with_bias)
    w = torch.randn((n, k), generator=g).to(torch.float8_e4m3fn).to(gpu).t()
    assert native.token_linear(x, w, s, bias, False) is not None
    q, xs = sglang_per_token_quant_fp8(x.view(-1, k))
    same(apply_fp8_linear(x, w, s, bias=bias), torch.ops.sgl_kernel.fp8_scaled_mm(q, w, xs, s, dtype, bias).view(*shape, n))
    w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).to(gpu).t()
    q, xs = per_token_quant_int8(x)
    assert q.shape == x.shape and xs.shape == (*shape, 1)
    want = torch.ops.sgl_kernel.int8_scaled_mm(q.view(-1, k), w, xs.view(-1, 1), s, dtype, bias)
    same(apply_w8a8_int8_linear(x, w, s, bias), want.view(*shape, n))


def test_scale_layouts(gpu):
    from sglang_amd.quantization.fp8_kernel import create_per_token_group_quant_fp8_output_scale, sglang_per_token_group_quant_fp8

    x = torch.randn((77, 640), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(gpu)
    want_q, want_s = O.per_token_group_quant_fp8(x.cpu(), 128)
    for column, padded in ((False, False), (True, False), (True, True)):
        q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=column, scale_tma_aligned=padded)
        like = create_per_token_group_quant_fp8_output_scale((77, 640), gpu, 128, column, padded, False)
        assert s.stride() == like.stride() and s.shape == like.shape
        same(q.cpu(), want_q)
        assert torch.equal(s.cpu(), want_s)


def test_what_it_leaves_to_python(gpu):
    from sglang_amd._lib import native
    from sglang_amd.quantization.fp8_utils import w8a8_block_fp8_linear

    w, s = block_weight(256, 512, gpu)
    x = torch.randn((4, 512), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(gpu)
    want = w8a8_block_fp8_linear(x, w, [128, 128], s)
    wide = torch.zeros((4, 1024), dtype=torch.bfloat16, device=gpu)[:, :512]
    for args in ((wide, w, s, None), (x.cpu(), w, s, None), (x, w, s[:1], None), (x, w.view(torch.int8), s, None), (x.float(), w, s, None),
                 (x, w, s, torch.zeros(8, dtype=torch.bfloat16, device=gpu)), (x.clone().requires_grad_(), w, s, None)):
        assert native.block_linear(*args, 0, 1e-10) is None

    class Watch(TorchDispatchMode):
        seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    big = x.repeat(3, 1)
    with Watch() as watch:
        got = w8a8_block_fp8_linear(big, w, [128, 128], s)
    assert any("fp8_blockwise_scaled_mm" in name for name in watch.seen)
    same(got[:4], want)
    with pytest.raises(RuntimeError, match="must be CUDA"):
        w8a8_block_fp8_linear(x.cpu(), w.cpu(), [128, 128], s.cpu())
