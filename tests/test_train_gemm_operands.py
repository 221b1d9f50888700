"""Which operands of the training block's projection and weight gradients (the value-embedding gate's too) reach their HIP
kernels, which trust the sizes and addresses they are given: without a GPU, CPU tensors stand for device tensors and a
kernel call is an exception of its own. Operands whose sizes or devices do not agree must meet the library GEMM instead,
which raises."""
import pytest
import torch

from nanochat_amd import attention_op as op
from nanochat_amd import ve_gate


class Reached(BaseException):
    """A kernel entry point would have been called."""


class Library(BaseException):
    """The library GEMM would have been called."""


def library_gemm(*args, **kwargs):
    raise Library


class NoLibrary:
    def __getattr__(self, name):
        raise Reached(name)


@pytest.fixture(autouse=True)
def device_operands(monkeypatch):
    """Every dense aligned tensor counts as a device tensor, and neither kind of product runs."""
    monkeypatch.setattr(op, "_plain", lambda t, dtype, alignment: (t.dtype == dtype and t.is_contiguous()
                                                                   and t.data_ptr() % alignment == 0))
    monkeypatch.setattr(op, "hip_library", NoLibrary)
    monkeypatch.setattr(ve_gate, "hip_library", NoLibrary)
    monkeypatch.setattr(op, "stream", lambda: 0)
    monkeypatch.setattr(torch, "mm", library_gemm)


def bf(*shape, device="cpu"):
    return torch.zeros(*shape, dtype=torch.bfloat16, device=device)


def test_agreeing_operands_reach_the_projection():
    with pytest.raises(Reached):
        op.project(bf(24, 256), bf(128, 256), bf(24, 128))


@pytest.mark.parametrize("x,w,res", [((24, 256), (128, 128), (24, 128)), ((24, 128), (128, 256), (24, 128)),
                                     ((24, 2, 128), (128, 256), (24, 128)), ((24, 256), (128, 256), (23, 128)),
                                     ((24, 256), (128, 256), (24, 256)), ((24, 256), (256,), (24, 128))])
def test_projection_sizes_that_do_not_agree(x, w, res):
    with pytest.raises(Library):
        op.project(bf(*x), bf(*w), bf(*res))


@pytest.mark.parametrize("C,K,met", [(32768, 32640, Reached), (32764, 32768, Reached), (32768, 32768, Library),
                                     (32772, 128, Library)])
def test_projection_weights_at_the_kernels_limit(C, K, met):
    """The kernel's 32-bit offsets end below a 2 GiB weight; that one and wider ones take the library."""
    with pytest.raises(met):
        op.project(bf(1, K), torch.empty(C, K, dtype=torch.bfloat16), bf(1, C))   # never touched


@pytest.mark.parametrize("C,K", [(0, 128), (128, 0)])
def test_empty_projection(C, K):
    """No columns or no inner size: the kernel refuses it, the library gives its empty or zero product."""
    with pytest.raises(Library):
        op.project(bf(3, K), bf(C, K), bf(3, C))


@pytest.mark.parametrize("elsewhere", [0, 1, 2])
def test_projection_operands_on_two_devices(elsewhere):
    args = [bf(*s, device="meta" if i == elsewhere else "cpu") for i, s in enumerate([(24, 256), (128, 256), (24, 128)])]
    with pytest.raises(Library):
        op.project(*args)


def test_agreeing_operands_reach_the_weight_gradient():
    with pytest.raises(Reached):
        op.add_weight_grad(torch.zeros(128, 256), bf(24, 128), bf(24, 256))


@pytest.mark.parametrize("grad,dh,x", [((128, 256), (24, 128), (23, 256)), ((128, 256), (23, 128), (24, 256)),
                                       ((128, 256), (24, 128), (24, 2, 128)), ((128, 256), (24, 128), (24, 128)),
                                       ((256,), (24, 128), (24, 256))])
def test_weight_gradient_sizes_that_do_not_agree(grad, dh, x):
    with pytest.raises(Library):
        op.add_weight_grad(torch.zeros(*grad), bf(*dh), bf(*x))


@pytest.mark.parametrize("elsewhere", [0, 1, 2])
def test_weight_gradient_operands_on_two_devices(elsewhere):
    d = ["meta" if i == elsewhere else "cpu" for i in range(3)]
    with pytest.raises(Library):
        op.add_weight_grad(torch.zeros(128, 256, device=d[0]), bf(24, 128, device=d[1]), bf(24, 256, device=d[2]))


@pytest.mark.parametrize("elsewhere,met", [(None, Reached), (0, Library), (1, Library), (2, Library)])
def test_gate_weight_gradient_operands_on_two_devices(elsewhere, met):
    """n is an operand of this product alone, so its place is checked nowhere before."""
    d = ["meta" if i == elsewhere else "cpu" for i in range(3)]
    with pytest.raises(met):
        ve_gate._weight_grad(bf(24, 2, device=d[0]), bf(24, 256, device=d[1]), torch.zeros(2, 256, device=d[2]))


@pytest.mark.parametrize("tokens,n", [(65536, n) for n in (2304, 2560, 2944, 3072, 3584, 4224, 5120)] + [(9995, 3072)])
def test_wide_weight_gradients_fill_the_chip(lib, tokens, n):
    """Token slices by the workspace they need: of the CUs' turns (256 a round) at least three quarters have work, where one
    slice of 100 to 250 tiles would leave half of them without."""
    slices = max(1, lib.nc_weight_grad_workspace_bytes(tokens, n, n) // (4 * n * n))
    groups = slices * (-(-n // 256)) ** 2
    assert groups / (-(-groups // 256) * 256) >= 0.75, slices


@pytest.mark.parametrize("tokens,n", [(1, 8), (64, 768), (512, 1664), (512, 2560), (2048, 3072)])
def test_few_tokens_take_one_slice(lib, tokens, n):
    """Its tiles are added into the result: no partials, which cost more than the idle CUs."""
    assert 0 < lib.nc_weight_grad_workspace_bytes(tokens, n, n) <= 16
