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


def _grads(cuda, q, k, v, dy, causal):
    from cuda_autograd_fns import CudaFlashAttention

    leaves = [x.to(cuda).requires_grad_() for x in (q, k, v)]
    o, _ = CudaFlashAttention.apply(*leaves, causal)
    return torch.autograd.grad(o, leaves, dy.to(cuda))


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,causal", [(1, True), (33, False), (130, True), (160, False), (1100, True)])
def test_gradients_against_float64(cuda, T, causal, D):
    """FP32 sums of a few thousand terms: a few units of 2^-24 in the 2-norm (T = 1: dQ and dK are
    rounding noise about zero, so only dV is compared)."""
    q, k, v, dy = _qkv(1, 2, T, D, T + D, 4)
    _, *ref = _ref(q, k, v, causal, dy)
    for name, x, r in zip("qkv", _grads(cuda, q, k, v, dy, causal), ref):
        if T > 1 or name == "v":
            assert _rel(x, r) <= 1.5e-6, (name, _rel(x, r))


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,causal", [(33, True), (160, False), (300, True)])
def test_gradients_outside_the_split_range(cuda, T, causal, D):
    q, k, v, dy = _qkv(1, 2, T, D, T + D, 4)
    _, *ref = _ref(q, k, v, causal, dy)
    # gradients of 2^-110: as accurate as ordinary ones
    for x, r in zip(_grads(cuda, q, k, v, dy * 2.0 ** -110, causal), ref):
        assert _rel(x.cpu().double() * 2.0 ** 110, r) <= 1.5e-6
    # an infinite entry of dO: the keys its row sees get an infinite (not NaN) dV there; the
    # other head, and every other column of dV, are untouched
    i, d = T // 2, 3
    dy[0, 0, i, d] = float("inf")
    dq, dk, dv = (x.cpu() for x in _grads(cuda, q, k, v, dy, causal))
    sees = torch.arange(T) <= (i if causal else T)
    assert torch.all(dv[0, 0, sees, d] == float("inf"))
    dv[0, 0, :, d] = ref[2][0, 0, :, d].float()  # a masked key of the same tile: 0 x inf
    assert _rel(dv, ref[2]) <= 1.5e-6
    for x, r in ((dq, ref[0]), (dk, ref[1])):
        assert _rel(x[0, 1], r[0, 1]) <= 1.5e-6
    rows = torch.arange(T) != i
    assert _rel(dq[0, 0, rows], ref[0][0, 0, rows]) <= 1.5e-6


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,causal", [(33, True), (160, False), (1100, True)])
def test_forward_scaled_operands(cuda, T, causal, D):
    """Scores of a tiny and a large operand, and values of any magnitude, a column each: as
    accurate as ordinary ones."""
    from cuda_transformer.ops import flash_attention_fwd

    q, k, v = _qkv(1, 2, T, D, T + D)
    ref = _ref(q, k, v, causal)
    for e in (60, 100, 118, 124):
        for s in (e, -e):
            o, _ = flash_attention_fwd((q * 2.0 ** -s).to(cuda), (k * 2.0 ** s).to(cuda), v.to(cuda),
                                       causal)
            assert _rel(o, ref) <= 1e-6, s
    e = torch.linspace(-124, 100, D).round()
    scale = (2.0 ** e.double()).float()
    o, _ = flash_attention_fwd(q.to(cuda), k.to(cuda), (v * scale).to(cuda), causal)
    assert _rel(o.cpu().double() / scale.double(), ref) <= 1e-6
    # subnormal values: FP32's spacing there, and no zeros in their place
    vs = v.clone()
    vs[..., 1] *= 2.0 ** -137
    o, _ = flash_attention_fwd(q.to(cuda), k.to(cuda), vs.to(cuda), causal)
    assert (o.double().cpu() - _ref(q, k, vs, causal))[..., 1].abs().max() <= 2.0 ** -148


@pytest.mark.parametrize("D", [32, 64, 128])
def test_forward_small_probabilities_of_large_values(cuda, D):
    """A key of probability 2^-124 holds the only nonzero value of its column, 2^100: the output
    of 2^-30 has the accuracy of the exponential, whose argument of 124 sees four roundings of at
    most 2^-24 of it: 4 x 124 x 2^-24 x ln 2 = 2e-5."""
    from cuda_transformer.ops import flash_attention_fwd

    T = 96
    q, k, v = _qkv(1, 1, T, D, D)
    q[..., 0], k[..., 0] = D ** 0.5, 0.0
    q[..., 1:] = 0.0
    k[:, :, 5, 0] = -86.0
    v[..., 2] = 0.0
    v[:, :, 5, 2] = 2.0 ** 100
    ref = _ref(q, k, v, False)
    o, _ = flash_attention_fwd(q.to(cuda), k.to(cuda), v.to(cuda), False)
    assert _rel(o[..., 2], ref[..., 2]) <= 2e-5


def _schedules(cuda, q, k, v, dy, causal):
    """(name, (dq, dk, dv)) through the operator's stored-dS schedule (which splits small grids),
    the schedule without a workspace and the one that forms delta inside dK/dV."""
    from cuda_transformer.ops import flash_attention_bwd, flash_attention_fwd
    from cuda_transformer_amd import capi

    B, H, T, D = q.shape
    q, k, v, dy = (x.to(cuda) for x in (q, k, v, dy))
    O, L = flash_attention_fwd(q, k, v, causal)
    yield "stored", flash_attention_bwd(q, k, v, O, dy, L, causal)
    s4, s3 = capi.strides(q.stride()), capi.strides(L.stride())
    st = torch.cuda.current_stream().cuda_stream
    head = (q.data_ptr(), s4, k.data_ptr(), s4, v.data_ptr(), s4, O.data_ptr(), s4, dy.data_ptr(),
            s4, L.data_ptr(), s3, B, H, T, D, int(causal))
    out = [torch.full_like(q, float("nan")) for _ in range(3)]
    delta = torch.empty(B, H, T, device=cuda)
    capi.call("cta_flash_attention_bwd", *head, *(t.data_ptr() for t in out), delta.data_ptr(),
              None, 0, st)
    yield "recompute", out
    nbytes = capi.call("cta_flash_attention_bwd_workspace", B, H, T, D, int(causal))
    ws = torch.empty(nbytes // 4, device=cuda)
    out = [torch.full_like(q, float("nan")) for _ in range(3)]
    capi.call("cta_flash_attention_bwd_fold_delta", *head, *(t.data_ptr() for t in out),
              ws.data_ptr(), nbytes, st)
    yield "fold_delta", out


# Lengths with and without the small-grid split of dK/dV and dQ (T >= 1024; 2048 at hs 32).
@pytest.mark.parametrize("D,T,causal", [(32, 130, True), (32, 2100, False), (64, 33, False),
                                        (64, 160, True), (64, 1100, True), (128, 96, True),
                                        (128, 1100, False)])
def test_gradients_scaled_operands(cuda, D, T, causal):
    """Operands whose magnitudes differ by up to 2^240 while the gradients stay in range, rows of
    dO at 2^-120 among ordinary ones, and gradients that no part can hold: in every schedule."""
    q, k, v, dy = _qkv(1, 2, T, D, T + D, 4)
    _, *ref = _ref(q, k, v, causal, dy)
    for e in (60, 118, -118):
        for name, (dq, dk, dv) in _schedules(cuda, q * 2.0 ** -e, k * 2.0 ** e, v, dy, causal):
            got = dq.cpu().double() * 2.0 ** -e, dk.cpu().double() * 2.0 ** e, dv
            for x, r in zip(got, ref):
                assert _rel(x, r) <= 1.5e-6, (name, e)
    for e in (60, 110, -110):
        for name, (dq, dk, dv) in _schedules(cuda, q, k, v * 2.0 ** e, dy * 2.0 ** -e, causal):
            for x, r in zip((dq, dk, dv.cpu().double() * 2.0 ** e), ref):
                assert _rel(x, r) <= 1.5e-6, (name, e)
    rows = torch.arange(T) % 3 == 1
    dys = dy.clone()
    dys[:, :, rows] *= 2.0 ** -120
    _, *rref = _ref(q, k, v, causal, dys)
    if causal:
        rows[0] = False  # its dQ is rounding noise about zero
    for name, (dq, dk, dv) in _schedules(cuda, q, k, v, dys, causal):
        for x, r in zip((dq, dk, dv), rref):
            assert _rel(x, r) <= 1.5e-6, name
        x, r = dq.cpu().double() * 2.0 ** 120, rref[0] * 2.0 ** 120
        assert _rel(x[:, :, rows], r[:, :, rows]) <= 3e-6, name
    for name, got in _schedules(cuda, q, k, v, dy * 2.0 ** -110, causal):
        for x, r in zip(got, ref):
            assert _rel(x.cpu().double() * 2.0 ** 110, r) <= 1.5e-6, name


@pytest.mark.parametrize("D,T,causal", [(32, 130, True), (32, 2100, False), (64, 160, True),
                                        (64, 1100, True), (128, 96, True), (128, 1100, False)])
def test_gradients_second_run_schedules(cuda, D, T, causal):
    """An infinite entry of dO sends its passes to FP32 MFMAs in every schedule: split dK/dV and dQ,
    without the dS store, and with delta formed inside."""
    q, k, v, dy = _qkv(1, 2, T, D, T + D, 4)
    _, *ref = _ref(q, k, v, causal, dy)
    i, d = T // 2, 3
    dy[0, 0, i, d] = float("inf")
    sees = torch.arange(T) <= (i if causal else T)
    rows = torch.arange(T) != i
    for name, got in _schedules(cuda, q, k, v, dy, causal):
        dq, dk, dv = (x.cpu() for x in got)
        assert torch.all(dv[0, 0, sees, d] == float("inf")), name
        dv[0, 0, :, d] = ref[2][0, 0, :, d].float()  # a masked key of the same tile: 0 x inf
        assert _rel(dv, ref[2]) <= 1.5e-6, name
        for x, r in ((dq, ref[0]), (dk, ref[1])):
            assert _rel(x[0, 1], r[0, 1]) <= 1.5e-6, name
        assert _rel(dq[0, 0, rows], ref[0][0, 0, rows]) <= 1.5e-6, name


@pytest.mark.parametrize("D,T,H,causal", [(64, 4096, 4, False), (64, 4096, 64, True), (32, 4096, 4, True),
                                          (128, 2048, 4, False)])
def test_gradient_column_sums(cuda, D, T, H, causal):
    """Rounding of dQ and dK has no sign of its own: the sums over the tokens (a bias gradient) are
    off by no more than independent errors of the gradients' own size would leave, three of their
    standard deviations.  A matrix pipe that rounds small addends of a large accumulator downward
    left nine at T = 4096."""
    from cuda_transformer.ops import flash_attention_bwd, flash_attention_fwd

    q, k, v, dy = _qkv(1, H, T, D, T + D, 4)
    dev = [x.to(cuda) for x in (q, k, v, dy)]
    O, L = flash_attention_fwd(*dev[:3], causal)
    got = flash_attention_bwd(*dev[:3], O, dev[3], L, causal)
    _, *ref = _ref(*(x[:, :2] for x in (q, k, v)), causal, dy[:, :2])
    for name, x, r in zip("qk", got, ref):
        e = x[:, :2].double().cpu() - r
        drift = float(e.sum(2).norm() / (r.norm()))  # sqrt(T) sigma, over sqrt(T) rms
        assert drift <= 3 * float(e.norm() / r.norm()), (name, drift)


# Both sides of the lines between two- and four-wave workgroups (hs 64, causal): T = 64 | 65, 128 |
# 129 and 512 | 513, longest-first tiles or pairs, and grids that fill the chip or not.
@pytest.mark.parametrize("heads,T", [(512, 64), (513, 64), (520, 65), (8, 128), (8, 129), (12, 200), (64, 256), (96, 200), (256, 256),
                                     (1024, 256), (64, 512), (128, 512), (256, 512), (16, 513)])
def test_short_causal_heads(cuda, heads, T):
    q, k, v, dy = _qkv(1, heads, T, 64, heads + T, 4)
    from cuda_transformer.ops import flash_attention_bwd, flash_attention_fwd

    dev = [x.to(cuda) for x in (q, k, v, dy)]
    O, L = flash_attention_fwd(*dev[:3], True)
    got = (O, *flash_attention_bwd(*dev[:3], O, dev[3], L, True))
    for h in (0, heads - 1):
        ref = _ref(*(x[:, h : h + 1] for x in (q, k, v)), True, dy[:, h : h + 1])
        for x, r in zip(got, ref):
            assert _rel(x[:, h : h + 1], r) <= 1.5e-6
