"""The GEMM's three-part bfloat16 products: tile and slice edges, operand orders, and the operands
that three bfloat16 parts cannot hold (infinities, NaN, values near the ends of FP32's range)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(x, w):
    """Six accumulator roundings per 16 k (and the bias add), each at most 2^-24 of a partial sum
    and no partial sum above sum |x||w|; the split itself stays below 2^-25 of it."""
    k = x.shape[-1]
    return (6 * ((k + 15) // 16) + 2) * 2.0 ** -24 * (x.abs().double() @ w.abs().double())


def _operands(m, k, n, order, seed):
    """x (1, m, k) and w (k, n) on the GPU, each contiguous, transposed or strided both ways."""
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g)

    def lay(t, how):
        if how == "t":
            return t.t().contiguous().cuda().t()
        if how == "s":  # neither dimension contiguous
            wide = torch.zeros(t.shape[0], t.shape[1], 2)
            wide[..., 0] = t
            return wide.cuda()[..., 0]
        return t.cuda()

    return x, w, lay(x, order[0]).unsqueeze(0), lay(w, order[1])


# Edges of the 64 and 128 tiles, of the 16-deep slices and of the small / narrow / wide / split-K
# choices.
@pytest.mark.parametrize("order", ["nn", "nt", "tn", "tt", "sn", "ns"])
@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (63, 15, 65), (65, 17, 127), (129, 33, 129), (195, 385, 1155), (64, 1030, 64),
    (2049, 35, 769), (4100, 48, 260),
])
def test_gemm_edges(cuda, m, k, n, order):
    from cuda_transformer.ops import cuda_fma

    x, w, xc, wc = _operands(m, k, n, order, m + k + n)
    out = cuda_fma(xc, wc, torch.zeros(n, device=cuda))[0].double().cpu()
    assert torch.all((out - x.double() @ w.double()).abs() <= _bound(x, w))


@pytest.mark.parametrize("m,k,n", [(70, 40, 66), (300, 64, 2000), (130, 2048, 130)])
def test_gemm_outside_the_split_range(cuda, m, k, n):
    """Rows with an infinity, a NaN, FLT_MAX, magnitudes of 2^-120 and zeros: the values FP32
    arithmetic gives, and no effect on the other rows beyond their own rounding."""
    from cuda_transformer.ops import cuda_fma

    x, w, _, _ = _operands(m, k, n, "nn", 5)
    w = w.abs() + 0.5
    x[3, 7] = float("inf")
    x[4, 8] = -float("inf")
    x[5, 9] = float("nan")
    x[6] = 0.0
    x[6, 2] = 3.4028234e38
    w[2, : n // 2] = 0.75
    x[7] *= 2.0 ** -120
    x[8] = 0.0
    out = cuda_fma(x.unsqueeze(0).to(cuda), w.to(cuda), torch.zeros(n, device=cuda))[0].cpu()
    assert torch.all(out[3] == float("inf")) and torch.all(out[4] == -float("inf"))
    assert torch.all(torch.isnan(out[5]))
    ref = x.double() @ w.double()
    assert torch.equal(out[6], (x[6, 2] * w[2]))  # one product: exact in FP32, or infinite
    assert torch.all(out[8] == 0)
    bound = _bound(x, w)
    rows = [i for i in range(m) if i not in (3, 4, 5, 6)]
    assert torch.all((out.double() - ref).abs()[rows] <= bound[rows] + 1e-45)
