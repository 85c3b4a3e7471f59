"""Errors found on the host in the middle of a backward pass: they leave the autograd engine as what they are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(pkg, E, dtype, T=64, H=1024, I=256, k=2):
    g = torch.Generator(device="cuda").manual_seed(E)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda") * 0.05
    w = [r(*s).to(dtype).requires_grad_(True) for s in ((E, I, H), (E, I, H), (E, H, I))]
    x = r(T, H).to(torch.bfloat16).requires_grad_(True)
    return x, r(T, E).to(torch.bfloat16), w, r(T, H).to(torch.bfloat16)


# (4 experts: all weight gradients in one launch; 320: the tiled kernel, on more tiles than compute units)
@pytest.mark.parametrize("E", [4, 320])
def test_a_grad_that_is_not_aligned_raises_the_library_s_error(pkg, lib, E):
    print("unaligned .grad", E, flush=True)
    x, logits, w, dy = _step(pkg, E, torch.float32)
    out = pkg.moe_ffn(x, logits, *w, 2, accumulate_into_grad=True)
    w[1].grad = torch.zeros(w[1].numel() + 1, device="cuda")[1:].view_as(w[1])
    with pytest.raises(pkg.lib.MoELibError, match="MOE_ERR_ALIGN"):
        out.backward(dy)
    assert x.grad is None and not w[1].grad.any()


def test_a_weight_type_without_kernels_raises_a_type_error(pkg, lib):
    print("fp16 weights", flush=True)
    x, logits, w, dy = _step(pkg, 4, torch.float16)
    out = pkg.moe_ffn(x, logits, *w, 2)
    with pytest.raises(TypeError, match="bf16 or fp32"):
        out.backward(dy)
    with pytest.raises(pkg.lib.MoELibError, match="MOE_ERR"):  # (and the same type straight from a call)
        pkg.moe_ffn(x, logits, *w, 5)
