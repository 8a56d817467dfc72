"""FlashAttention on three-part bfloat16 products: operands that the parts cannot hold (infinities,
NaN, magnitudes near the ends of FP32's range) and accuracy against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _qkv(B, H, T, D, seed, n=3):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, H, T, D, generator=g) for _ in range(n)]


def _ref(q, k, v, causal, dy=None):
    """Float64 outputs (and gradients), on the CPU."""
    q, k, v = (x.double().requires_grad_(dy is not None) for x in (q, k, v))
    s = (q @ k.mT) * q.shape[-1] ** -0.5
    if causal:
        t = s.shape[-1]
        s = s.masked_fill(torch.ones(t, t, dtype=torch.bool).triu(1), -float("inf"))
    o = torch.softmax(s, -1) @ v
    if dy is None:
        return o
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), dy.double()))


def _rel(x, ref):
    return float((x.double().cpu() - ref).norm() / ref.norm())


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,causal", [(33, True), (160, False), (1100, True)])
def test_forward_outside_the_split_range(cuda, T, causal, D):
    from cuda_transformer.ops import flash_attention_fwd

    q, k, v = _qkv(1, 2, T, D, T + D)
    ref = _ref(q, k, v, causal)
    j = T // 2
    v[0, 0, j, 3] = float("inf")
    q[0, 1, j, 1] = float("nan")
    o, l = (x.cpu() for x in flash_attention_fwd(q.to(cuda), k.to(cuda), v.to(cuda), causal))
    sees = torch.arange(T) >= (j if causal else 0)  # the rows that attend to key j
    assert torch.all(o[0, 0, sees, 3] == float("inf"))
    o[0, 0, :, 3] = ref[0, 0, :, 3].float()  # masked rows of the same tile see 0 x inf
    assert torch.all(torch.isnan(o[0, 1, j]))
    o[0, 1, j] = ref[0, 1, j].float()
    assert torch.isfinite(l[0, 0]).all() and _rel(o, ref) <= 1e-6
    # values of 2^-120: as accurate as ordinary ones
    q, k, v = _qkv(1, 2, T, D, T + D)
    o, _ = flash_attention_fwd(q.to(cuda), k.to(cuda), (v * 2.0 ** -120).to(cuda), causal)
    assert _rel(o.cpu().double() * 2.0 ** 120, ref) <= 1e-6
