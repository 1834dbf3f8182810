"""ltxk_linear (csrc/gemm.hip) against the product in fp64, and the layers that
take it against torch's own linear (GPU)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _case(m, n, k, bias, seed=0):
    g = torch.Generator(device=DEV).manual_seed(m + n + k + seed)
    x = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn(n, device=DEV, generator=g).to(torch.bfloat16) if bias else None
    return x, w, b


def _check(x, w, b, got):
    """The rounding to bf16 moves a result by 2^-8 of it, and each of the k fp32
    additions by 2^-24 of a partial sum.  Partial sums of independent signs stay
    within 4 r, r the root of the summed squared products, and by Hoeffding's
    inequality k independent roundings of at most 2^-24 4 r each add up to more than
    6 sqrt(k) 2^-24 4 r for 3 results in 10^8."""
    k = x.shape[-1]
    for r in range(0, x.shape[0], 512):
        xr = x[r:r + 512].double()
        for c in range(0, w.shape[0], 512):
            wc = w[c:c + 512].double()
            want, square = xr @ wc.T, xr.square() @ wc.square().T
            if b is not None:
                want, square = want + b[c:c + 512].double(), square + b[c:c + 512].double().square()
            err = (got[r:r + 512, c:c + 512].double() - want).abs()
            bound = want.abs() * 2.0**-8 + square.sqrt() * (24 * k**0.5 * 2.0**-24) + 1e-30
            assert bool((err <= bound).all()), f"rows {r}.. columns {c}..: {(err / bound).max().item():.3f}"


@pytest.mark.parametrize("m,n,k,bias", [
    (1, 8, 64, True), (1, 256, 128, False), (255, 264, 192, True), (257, 256, 64 * 9, True), (300, 520, 4096, False),
    (129, 2048, 8192, True), (1000, 1024, 16448, True),
    (4100, 4096, 128, True), (4352, 4096, 1088, False), (4097, 4104, 320, True)])
def test_linear_matches_fp64(m, n, k, bias):
    """One tile and its edges, tiles cut over K, and a full wave of tiles with
    some past it."""
    import ltxk

    x, w, b = _case(m, n, k, bias)
    _check(x, w, b, ltxk.linear(x, w, b))


@pytest.mark.parametrize("m,n,bias", [(300, 6000, False), (130, 40, True)])
def test_feature_projection_matches_fp64(m, n, bias):
    """K 188160: 48 tiles in 5 parts with weight rows past 2^31 bytes, and one tile in
    256 parts."""
    import ltxk

    x, w, b = _case(m, n, 188160, bias)
    _check(x, w, b, ltxk.linear(x, w, b))


@pytest.mark.parametrize("m,k,ns,biased", [
    (1, 128, (8,), (True,)), (126, 2048, (2048, 2048, 2048, 32), (True, True, False, True)),
    (129, 384, (40, 32), (True, True)), (300, 256, (264, 8, 64), (False, True, True)), (128, 896, (72, 96), (True, False)),
    (33, 4096, (128, 128, 128, 32), (True, True, True, True))])
def test_layers_over_few_rows(m, k, ns, biased):
    """One launch for several layers: each equals its product in fp64, over edges
    of the 128-row and 32-column tiles and K of one step to more than its rings."""
    import ltxk

    cases = [_case(m, n, k, b, seed=i) for i, (n, b) in enumerate(zip(ns, biased))]
    x = cases[0][0]
    outs = ltxk.linear_layers(x, [c[1] for c in cases], [c[2] for c in cases])
    for (_, w, b), y in zip(cases, outs):
        _check(x, w, b, y)


@pytest.mark.parametrize("rows,own", [(126, True), (257, False)])
def test_projection_route(rows, own):
    """ltx_nn.project on rows of 2048: one launch up to 2^19 elements of x, the
    layers' own calls above, a missing layer as None."""
    import ltx_nn

    layers = [torch.nn.Linear(2048, n, device=DEV, dtype=torch.bfloat16) for n in (2048, 32)]
    x = torch.randn(1, rows, 2048, device=DEV).to(torch.bfloat16)
    assert (x.numel() <= ltx_nn.FEW_ROWS_MAX) == own
    with torch.no_grad():
        q, none, g = ltx_nn.project(x, layers[0], None, layers[1])
    assert none is None and q.shape == (1, rows, 2048) and g.shape == (1, rows, 32)
    for layer, y in zip(layers, (q, g)):
        _check(x[0], layer.weight.detach(), layer.bias.detach(), y[0])


def test_refusals():
    import ltxk

    lib = ltxk.load()
    x, w, _ = _case(16, 64, 128, False)
    y = torch.empty(16, 64, device=DEV, dtype=torch.bfloat16)

    def call(n=64, k=128, ws=0, shift=0):
        return lib.ltxk_linear(y.data_ptr(), x.data_ptr() + shift, w.data_ptr(), None, 16, n, k, None, ws, None)

    assert call(n=60) == ltxk.E_ARG and call(k=96) == ltxk.E_ARG and call(shift=2) == ltxk.E_ALIGN
    assert lib.ltxk_linear_workspace_bytes(16, 64, 128) > 0 and call() == ltxk.E_ARG  # no workspace
    with pytest.raises(ValueError):
        ltxk.linear(x, w[:, :64].contiguous())
    with pytest.raises(ValueError):
        ltxk.linear_layers(x, [w] * 5, [None] * 5)
    with pytest.raises(RuntimeError):  # n not a multiple of 8
        ltxk.linear_layers(x, [w[:12].contiguous(), w], [None, None])
    with pytest.raises(RuntimeError):  # k not a multiple of 128
        ltxk.linear_layers(x[:, :64].contiguous(), [w[:, :64].contiguous()], [None])


@pytest.mark.parametrize("shape,n,bias,own", [((1, 300), 256, True, True), ((2, 33), 264, False, True),
                                              ((7,), 512, True, True), ((5,), 500, True, False)])
def test_layer_route(shape, n, bias, own):
    """ltx_nn.linear on torch.nn.Linear of K 16384: its route by shape, by hook and
    by recorded gradient, and its values against the layer's own."""
    import ltx_nn

    layer = torch.nn.Linear(16384, n, bias=bias, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(*shape, 16384, device=DEV).to(torch.bfloat16)
    m = x.numel() // 16384
    assert ltx_nn.long_k_tiles(m, n, 16384) == own
    with torch.no_grad():
        got, want = ltx_nn.linear(layer, x), layer(x)
        assert got.shape == want.shape
        _check(x.reshape(m, -1), layer.weight, layer.bias, got.reshape(m, n))
        seen = []
        handle = layer.register_forward_hook(lambda *a: seen.append(1))
        assert torch.equal(ltx_nn.linear(layer, x), want) and seen == [1]
        handle.remove()
    assert ltx_nn.linear(layer, x).requires_grad  # a recorded gradient keeps the layer's own call


@pytest.mark.parametrize("m,n,k,main", [
    (4096, 4096, 4096, 0), (4097, 4096, 4096, 4096), (4864, 4096, 2048, 4096), (4865, 4096, 2048, 0),
    (8200, 4096, 16384, 8192), (5200, 16384, 4096, 5120), (1100, 16384, 4096, 0), (4290, 2048, 4096, 0),
    (4290, 4096, 1024, 0), (4290, 12288, 4096, 0), (4290, 5000, 4096, 0), (4290, 4096, 188160, 0)])
def test_full_wave_rows(m, n, k, main):
    import ltx_nn

    assert ltx_nn.full_wave_rows(m, n, k) == main


@pytest.mark.parametrize("shape,bias", [((1, 4097), True), ((2, 2200), False)])
def test_rows_past_a_full_wave(shape, bias):
    """Both launches' rows against the product in fp64; a hooked layer keeps one call."""
    import ltx_nn

    layer = torch.nn.Linear(2048, 4096, bias=bias, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(*shape, 2048, device=DEV).to(torch.bfloat16)
    m = x.numel() // 2048
    assert ltx_nn.full_wave_rows(m, 4096, 2048) == 4096
    with torch.no_grad():
        got = ltx_nn.linear(layer, x)
        assert got.shape == (*shape, 4096)
        _check(x.view(m, 2048), layer.weight, layer.bias, got.view(m, 4096))
        seen = []
        layer.register_forward_hook(lambda *a: seen.append(1))
        assert torch.equal(ltx_nn.linear(layer, x), layer(x)) and seen == [1, 1]
