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


# Powers of two on the operands: products of ordinary size of one tiny and one large operand, down
# to subnormal x, and up to sums near the top of the range.
SCALES = [(-60, 60), (-100, 20), (-109, 60), (-116, 60), (-120, 40), (-126, 100), (-130, 60),
          (-136, 60), (-136, 20), (-140, 120), (-70, -70), (60, 60), (100, -130), (2, -148)]


@pytest.mark.parametrize("a,b", SCALES)
@pytest.mark.parametrize("m,k,n,order", [(70, 768, 66, "nn"), (300, 40, 2000, "tn"),
                                         (130, 2048, 130, "nt"), (33, 70, 40, "sn")])
def test_gemm_scaled_operands(cuda, m, k, n, order, a, b):
    """Every finite operand takes part with all of its bits, whatever its magnitude and its
    partner's: the bound of ordinary operands, plus FP32's subnormal spacing a step."""
    from cuda_transformer.ops import cuda_fma

    x, w, xc, wc = _operands(m, k, n, order, m + k)
    for t in (x, xc):
        t *= 2.0 ** a
    for t in (w, wc):
        t *= 2.0 ** b
    x, w = xc[0].cpu().contiguous(), wc.cpu().contiguous()  # as rounded to FP32
    out = cuda_fma(xc, wc, torch.zeros(n, device=cuda))[0].double().cpu()
    assert torch.all((out - x.double() @ w.double()).abs() <= _bound(x, w) + k * 2.0 ** -149)


@pytest.mark.parametrize("order", ["nn", "nt", "tn", "tt", "sn", "ns"])
def test_gemm_scales_that_cancel(cuda, order):
    """Column k of x times 2^-e, row k of w times 2^e, e = 124 and -124 in turn: every product is of
    ordinary size, and the result the unscaled operands'."""
    from cuda_transformer.ops import cuda_fma

    m, k, n = 130, 300, 140
    x, w, xc, wc = _operands(m, k, n, order, 17)
    e = torch.tensor([124.0, -124.0]).repeat(k // 2)
    xc *= (2.0 ** -e.double()).float().to(cuda)
    wc *= (2.0 ** e.double()).float().to(cuda)[:, None]
    out = cuda_fma(xc, wc, torch.zeros(n, device=cuda))[0].double().cpu()
    assert torch.all((out - x.double() @ w.double()).abs() <= _bound(x, w))


@pytest.mark.parametrize("order", ["nn", "nt", "tn", "tt", "sn", "ns"])
def test_gemm_second_run_orders(cuda, order):
    """A tile that runs again on FP32 MFMAs (an infinity in one row), in each load order."""
    from cuda_transformer.ops import cuda_fma

    m, k, n = 200, 77, 133
    x, w, xc, wc = _operands(m, k, n, order, 23)
    w, wc = w.abs() + 0.5, wc.abs() + 0.5
    xc[0, 3, 5] = float("inf")
    out = cuda_fma(xc, wc, torch.zeros(n, device=cuda))[0].double().cpu()
    assert torch.all(out[3] == float("inf"))
    rows = [i for i in range(m) if i != 3]
    assert torch.all((out - x.double() @ w.double()).abs()[rows] <= _bound(x, w)[rows])


@pytest.mark.parametrize("rows,k,n", [(300, 70, 65), (3000, 96, 132), (129, 33, 1155)])
def test_weight_bias_grad_second_run(cuda, rows, k, n):
    """dW tiles that run again on FP32 MFMAs beside the column sums that share their LDS, at odd
    and even n, split along the rows and not: dW and db as without the infinity elsewhere."""
    from cuda_transformer_amd.ops import linear_weight_bias_grad

    g = torch.Generator().manual_seed(rows + n)
    x, dy = torch.randn(rows, k, generator=g), torch.randn(rows, n, generator=g)
    x[7, 3] = float("inf")
    dy[7] = dy[7].abs() + 0.5
    dw, db = (t.double().cpu() for t in linear_weight_bias_grad(x.to(cuda), dy.to(cuda)))
    assert torch.all(dw[3] == float("inf"))
    x[:, 3] = 0.0
    dw[3] = 0.0
    assert torch.all((dw - x.double().t() @ dy.double()).abs() <= _bound(x.t(), dy))
    assert torch.all((db - dy.double().sum(0)).abs() <= 1e-6 * dy.double().abs().sum(0))


def test_weight_bias_grad_column_strides(cuda):
    """dy with strided columns: db from the column-sum kernels, not the GEMM's slices."""
    from cuda_transformer_amd.ops import linear_weight_bias_grad

    g = torch.Generator().manual_seed(9)
    x, dy = torch.randn(500, 40, generator=g), torch.randn(500, 50, generator=g)
    wide = torch.zeros(500, 50, 2)
    wide[..., 0] = dy
    dw, db = (t.double().cpu() for t in linear_weight_bias_grad(x.to(cuda), wide.to(cuda)[..., 0]))
    assert torch.all((dw - x.double().t() @ dy.double()).abs() <= _bound(x.t(), dy))
    assert torch.all((db - dy.double().sum(0)).abs() <= 1e-6 * dy.double().abs().sum(0))


# Both sides of the tile choice's lines: 640 | 672 tiles of 64x64, 256 | 288, 320 | 352 tiles of
# 128x128, and the operand orders that never take 64x128.
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,k,n", [(2048, 48, 1280), (2048, 48, 1344), (4096, 48, 1024), (4096, 52, 1152),
                                   (4096, 48, 1280), (4096, 52, 1408), (4096, 35, 1152)])
def test_gemm_tile_lines(cuda, m, k, n, order):
    from cuda_transformer.ops import cuda_fma

    x, w, xc, wc = _operands(m, k, n, order, m + k + n)
    out = cuda_fma(xc, wc, torch.zeros(n, device=cuda))[0].double().cpu()
    assert torch.all((out - x.double() @ w.double()).abs() <= _bound(x, w))
