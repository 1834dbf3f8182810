"""Which calls ltx_nn hands to the matrix-core entry points and which stay with
torch: the rules that need no GPU."""

import pytest
import torch

BF16 = torch.bfloat16


def _layer(k=128, n=64, bias=True):
    return torch.nn.Linear(k, n, bias=bias, dtype=BF16).requires_grad_(False)


def _param(*shape):
    return torch.nn.Parameter(torch.zeros(*shape, dtype=BF16), requires_grad=False)


def test_layer_of_its_own_shapes_is_plain():
    import ltx_nn

    x = torch.zeros(3, 128, dtype=BF16)
    layer = _layer()
    weight, bias = ltx_nn._plain_layer(layer, x)
    assert weight is layer.weight and bias is layer.bias
    assert ltx_nn._plain_layer(_layer(bias=False), x)[1] is None


@pytest.mark.parametrize("weight,bias", [
    ((64, 128), (1,)), ((64, 128), (32,)), ((64, 128), (128,)), ((64, 128), (64, 1)), ((64, 128), (1, 64)),
    ((40, 128), (64,)), ((60, 128), (60,)), ((128,), (64,)), ((128,), None), ((64, 64), (64,))])
def test_layer_of_other_shapes_keeps_torch(weight, bias):
    """A replaced weight or bias whose shape is not the layer's own (torch broadcasts
    some of them and refuses the others) is not handed to kernels that read
    out_features entries of it."""
    import ltx_nn

    layer = _layer()
    layer.weight = _param(*weight)
    layer.bias = None if bias is None else _param(*bias)
    assert ltx_nn._plain_layer(layer, torch.zeros(3, 128, dtype=BF16)) is None


@pytest.mark.parametrize("name", ["weight", "bias"])
@pytest.mark.parametrize("where", ["attribute", "buffer", "shadow"])
def test_operand_kept_elsewhere_keeps_torch(name, where):
    """A layer whose weight or bias is not (or not only) among its parameters: torch
    reads the attribute, so the parameter dictionary alone does not name the operand."""
    import ltx_nn

    layer = _layer()
    value = torch.ones_like(getattr(layer, name).data)
    if where == "shadow":
        object.__setattr__(layer, name, value)
    else:
        delattr(layer, name)
        layer.register_buffer(name, value) if where == "buffer" else setattr(layer, name, value)
    assert getattr(layer, name) is value
    assert ltx_nn._plain_layer(layer, torch.zeros(3, 128, dtype=BF16)) is None


@pytest.mark.parametrize("m,k,widths,taken", [
    (1, 128, (8, 8), True), (1, 128, (8, 2**24), False), (4, 128, (2**24 + 8, 8), False),
    (126, 2048, (2048, 2048, 2048, 32), True), (256, 2048, (2048, 2048, 2048, 32), True),
    (128, 4096, (4096, 4096, 4096, 32), True), (126, 2048, (2048, 36), False),
    (256, 2048, (2560, 2560), True), (256, 2048, (2568, 2560), False), (4096, 128, (160, 160), True),
    (4096, 128, (1024, 1024, 1024), False), (80, 6144, (2048, 2048), True), (80, 6272, (2048, 2048), False)])
def test_few_rows_widths(m, k, widths, taken):
    """Layers that ltxk_linear_layers refuses, and that it is slower on, keep torch's call."""
    import ltx_nn

    assert ltx_nn.few_rows_widths(m, k, widths) == taken


def test_few_rows_of_a_huge_layer_keep_torch(monkeypatch):
    import ltx_nn
    import ltxk

    monkeypatch.setattr(ltx_nn, "_plain_input", lambda x: True)
    monkeypatch.setattr(ltxk, "_launch_layers", lambda *a: ["launched"] * 2)
    x = torch.zeros(2, 128, dtype=BF16, device="meta")
    for n, taken in ((64, True), (2**24 + 8, False)):
        layers = [torch.nn.Linear(128, n, dtype=BF16, device="meta").requires_grad_(False) for _ in range(2)]
        got = ltx_nn.project(x, *layers)
        assert got == ["launched"] * 2 if taken else [y.shape for y in got] == [(2, n)] * 2


@pytest.mark.parametrize("batch,tokens,heads,fits", [
    (1, 6144, 32, True), (1 << 20, 1, 8, True), ((1 << 20) + 1, 1, 1, False), (1 << 20, 1, 16, False),
    (1 << 19, 128, 16, True), (1 << 19, 129, 16, False), (1, (1 << 28) - (1 << 14), 8, True), (1, 1 << 28, 8, False)])
def test_attention_grid_fits(batch, tokens, heads, fits):
    """Batches and query counts past ltxk_attention's launch keep torch's attention."""
    import ltx_nn

    assert ltx_nn.attention_grid_fits(batch, tokens, heads) == fits


def test_calls_that_torch_watches_are_no_eager_calls():
    """Tracing, function transforms, forward-mode derivatives and dispatch modes see
    only torch's own operations, so calls under them keep those."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    import ltx_nn

    seen = []

    def call(x):
        seen.append(ltx_nn.eager_call())
        return x * 2

    x = torch.ones(2, 3)
    torch.func.vmap(call)(x)
    torch.func.grad(lambda t: call(t).sum())(x)
    torch.func.jvp(call, (x,), (x,))
    torch.jit.trace(call, x, check_trace=False)
    make_fx(call)(x)
    with FlopCounterMode(display=False):
        call(x)
    with forward_ad.dual_level():
        call(forward_ad.make_dual(x, x))
    assert len(seen) >= 7 and not any(seen)
    assert ltx_nn.eager_call()


@pytest.mark.parametrize("batch,tq,tk,heads,dh,torchs", [
    (65, 16, 16, 32, 64, True), (64, 16, 16, 32, 64, False), (65, 17, 16, 32, 64, False), (65, 16, 17, 32, 64, False),
    (65, 32, 1, 32, 128, True), (65, 33, 1, 32, 128, False), (65, 32, 17, 32, 128, False), (4, 16, 16, 32, 64, False)])
def test_many_short_sequences(batch, tq, tk, heads, dh, torchs):
    import ltx_nn

    assert ltx_nn.many_short_sequences(batch, tq, tk, heads, dh) == torchs


@pytest.mark.parametrize("m,n,k,own", [
    (1024, 4096, 188160, True), (1280, 4096, 188160, True), (1281, 4096, 188160, False), (2560, 2048, 188160, True),
    (2561, 2048, 188160, False), (1280, 4096, 65536, True), (1024, 4096, 16384, True), (1025, 4096, 16384, False),
    (23, 2048, 188160, True), (23, 4096, 188160, False), (24, 4096, 188160, True), (64, 5376, 32768, False),
    (65, 5376, 32768, True), (128, 8448, 32768, False), (129, 8448, 32768, True), (64, 4096, 16384, False),
    (65, 4096, 16384, True), (64, 512, 16384, True), (128, 4352, 16384, False), (129, 4352, 16384, True),
    (1280, 4096, 65472, False), (1024, 4096, 16320, False), (64, 4092, 16384, False)])
def test_long_k_tiles(m, n, k, own):
    import ltx_nn

    assert ltx_nn.long_k_tiles(m, n, k) == own


@pytest.mark.parametrize("dtype,shape,dropped", [
    (BF16, (2, 1, 1, 8), True), (BF16, (1, 1, 1, 8), True), (torch.float32, (2, 1, 1, 8), False),
    (torch.bool, (2, 1, 1, 8), False), (BF16, (2, 3, 1, 8), False), (BF16, (2, 1, 8, 8), False),
    (BF16, (2, 1, 5, 8), False), (BF16, (2, 1, 1, 1), False)])
def test_connector_drops_only_masks_that_its_attention_takes(monkeypatch, dtype, shape, dropped):
    """With registers every token is open: the blocks run unmasked, except under a
    mask of a type or shape that the attention is to refuse (or to read another way)."""
    import ltx_te
    import ltxk

    seen = []

    class Block(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.attn1 = torch.nn.Module()
            self.attn1.heads = 2

        def _run(self, x, pending, mask, pe, defer):
            seen.append(mask)
            return x, x

    monkeypatch.setattr(ltxk, "add_norm_modulate", lambda x, f, eps: (x, x))
    connector = ltx_te.Embeddings1DConnector(2, 16, 0, [16], 4, False, True)
    connector.blocks.append(Block())
    connector.learnable_registers.requires_grad_(False).zero_()
    _, mask = connector(torch.zeros(2, 8, 32, dtype=BF16), torch.zeros(shape, dtype=dtype))
    assert mask.shape == shape and mask.dtype == dtype
    assert (seen[0] is None) == dropped
    assert dropped or (seen[0].shape == shape and seen[0].dtype == dtype)
