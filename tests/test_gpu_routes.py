"""Which of ltx_nn's calls reach the matrix-core entry points and which stay with
torch, by counting them (GPU)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
BF16 = torch.bfloat16


@pytest.fixture
def calls(monkeypatch):
    """Counts of the calls that reach each entry point and torch's attention."""
    import ltx_nn
    import ltxk

    counts = {}

    def count(module, name):
        inner = getattr(module, name)

        def counted(*args, **kwargs):
            counts[name] = counts.get(name, 0) + 1
            return inner(*args, **kwargs)

        monkeypatch.setattr(module, name, counted)

    for name in ("attention", "linear", "_launch_layers", "attn_combine"):
        count(ltxk, name)
    for name in ("_two_launches", "sdpa"):
        count(ltx_nn, name)
    return counts


def _attend(heads, dh, tq=70, tk=90, b=2):
    import ltx_nn

    layer = ltx_nn.Attention(256, 256, heads, dh).to(device=DEV, dtype=BF16).requires_grad_(False)
    g = torch.Generator(device=DEV).manual_seed(tq + tk + dh)
    q, k, v = (torch.randn(b, t, heads * dh, device=DEV, generator=g).to(BF16) for t in (tq, tk, tk))
    return layer, q, k, v, torch.randn(b, tq, heads, device=DEV, generator=g).to(BF16)


def _want(layer, q, k, v, gates=None):
    b, tq, d = q.shape
    h = layer.heads
    q, k, v = (t.double().view(b, -1, h, d // h).transpose(1, 2).contiguous() for t in (q, k, v))
    w = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(d // h), -1)
    o = torch.matmul(w, v).transpose(1, 2)
    if gates is not None:
        o = o * 2 * torch.sigmoid(gates.double()).unsqueeze(-1)
    return torch.nn.functional.linear(o.reshape(b, tq, d), layer.to_out.weight.double(), layer.to_out.bias.double())


def _close(got, want):
    # the weights', the output's, the gated output's and the layer's roundings to bf16, 2^-8 of a value each at most
    assert ((got.double() - want).norm() / want.norm()).item() < 4 * 2.0**-8


@pytest.mark.parametrize("heads,dh", [(4, 64), (2, 128)])
def test_attend_on_the_kernel(calls, heads, dh):
    layer, q, k, v, gates = _attend(heads, dh)
    _close(layer.attend(q, k, v, None), _want(layer, q, k, v))
    assert calls == {"attention": 1}
    _close(layer.attend(q, k, v, gates), _want(layer, q, k, v, gates))
    assert calls == {"attention": 2}
    keep = torch.tensor([1.0, 0.0], device=DEV)
    k2, v2 = k[:, :70].contiguous(), v[:, :70].contiguous()
    got = layer.attend(q, k2, v2, gates, perturbation_mask=keep.view(2, 1, 1))
    _close(got[:1], _want(layer, q[:1], k2[:1], v2[:1], gates[:1]))
    assert calls == {"attention": 3}


def _moved(t):
    """The same values, contiguous, two bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:]
    return flat.copy_(t.reshape(-1)).view(t.shape)


def _strided(t):
    """The same values as columns of a wider buffer."""
    wide = torch.zeros(*t.shape[:-1], 2 * t.shape[-1], device=t.device, dtype=t.dtype)
    wide[..., :t.shape[-1]] = t
    return wide[..., :t.shape[-1]]


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("change", ["misaligned", "strided", "gradient"])
def test_attend_of_other_operands_keeps_torch(calls, which, change):
    layer, *qkv, _ = _attend(4, 64)
    want = _want(layer, *qkv)
    how = {"misaligned": _moved, "strided": _strided, "gradient": lambda t: t.requires_grad_()}[change]
    qkv[which] = how(qkv[which])
    _close(layer.attend(*qkv, None).detach(), want)
    assert calls == {"sdpa": 1}


def test_attend_with_a_mask_or_other_heads_keeps_torch(calls):
    layer, q, k, v, gates = _attend(4, 64)
    mask = torch.zeros(1, 1, 70, 90, device=DEV, dtype=BF16)
    _close(layer.attend(q, k, v, gates, mask), _want(layer, q, k, v, gates))
    assert calls == {"sdpa": 1}
    layer, q, k, v, gates = _attend(3, 96)
    _close(layer.attend(q, k, v, gates), _want(layer, q, k, v, gates))
    assert calls == {"sdpa": 2}


def test_attend_cuts_the_keys_of_other_heads_in_torch(calls):
    """Heads that the kernel does not take: few queries over many keys in the
    key-split form, with the gate in its merge."""
    layer, q, k, v, gates = _attend(3, 96, tq=40, tk=2048)
    _close(layer.attend(q, k, v, gates), _want(layer, q, k, v, gates))
    assert calls == {"attn_combine": 1}


def _linear(k, n, rows, bias=True):
    layer = torch.nn.Linear(k, n, bias=bias, device=DEV, dtype=BF16).requires_grad_(False)
    return layer, torch.randn(rows, k, device=DEV).to(BF16)


@pytest.mark.parametrize("k,n,rows,name", [(16384, 256, 70, "linear"), (2048, 4096, 4100, "_two_launches")])
def test_linear_on_its_own_launches(calls, k, n, rows, name):
    """Taken, and not taken with a hook, a patched forward, a gradient to record,
    autocast, or an input that is misaligned or strided."""
    import ltx_nn

    layer, x = _linear(k, n, rows)
    want = layer(x).float()

    def run(x=x):
        got = ltx_nn.linear(layer, x).detach().float()
        assert ((got - want).norm() / want.norm()).item() < 2.0**-7
        return calls.get(name, 0)

    assert run() == 1
    handle = layer.register_forward_pre_hook(lambda *a: None)
    assert run() == 1
    handle.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert run() == 1
    handle.remove()
    own = layer.forward
    layer.forward = lambda x: own(x)
    assert run() == 1
    del layer.forward
    assert run(_moved(x)) == 1 and run(_strided(x)) == 1 and run(x.clone().requires_grad_()) == 1
    layer.requires_grad_(True)
    assert run() == 1
    with torch.no_grad():
        assert run() == 2
    layer.requires_grad_(False)
    with torch.autocast("cuda", dtype=BF16):
        assert run() == 2
    assert run() == 3 and set(calls) == {name}


def test_project_on_one_launch(calls):
    import ltx_nn

    x = torch.randn(2, 50, 512, device=DEV).to(BF16)
    layers = [torch.nn.Linear(512, n, device=DEV, dtype=BF16).requires_grad_(False) for n in (128, 64, 32)]

    def run(x=x, layers=layers):
        for got, layer in zip(ltx_nn.project(x, *layers), layers):
            want = layer(x).float()
            assert ((got.detach().float() - want).norm() / want.norm()).item() < 2.0**-7
        return calls.get("_launch_layers", 0)

    assert run() == 1
    assert run(layers=layers[:1]) == 1                       # a single layer
    assert run(_moved(x)) == 1 and run(_strided(x)) == 1 and run(x.clone().requires_grad_()) == 1
    handle = layers[1].register_forward_hook(lambda *a: None)
    assert run() == 1
    handle.remove()
    with torch.autocast("cuda", dtype=BF16):
        assert run() == 1
    bias = layers[0].bias
    layers[0].bias = torch.nn.Parameter(torch.full((1,), 0.5, device=DEV, dtype=BF16), requires_grad=False)
    assert run() == 1                                        # torch broadcasts it
    layers[0].bias = bias
    assert run() == 2 and set(calls) == {"_launch_layers"}


def test_layers_of_an_attention_and_a_feed_forward(calls):
    """Attention.forward: one launch for the projections of each small input, the
    kernel, the output layer; FeedForward: its long second product."""
    import ltx_nn

    layer = ltx_nn.Attention(256, 256, 8, 64, 1e-6, True).to(device=DEV, dtype=BF16).requires_grad_(False)
    x, context = (torch.randn(1, t, 256, device=DEV).to(BF16) for t in (60, 33))
    layer(x)
    assert calls == {"_launch_layers": 1, "attention": 1}
    layer(x, context=context)
    assert calls == {"_launch_layers": 3, "attention": 2}
    calls.clear()
    ffn = ltx_nn.FeedForward(4096, 256).to(device=DEV, dtype=BF16).requires_grad_(False)
    ffn(torch.randn(1, 40, 4096, device=DEV).to(BF16))
    assert calls == {"linear": 1}


def test_attend_of_many_short_sequences_keeps_torch(calls):
    layer, q, k, v, gates = _attend(32, 64, tq=16, tk=16, b=65)
    _close(layer.attend(q, k, v, gates), _want(layer, q, k, v, gates))
    assert calls == {"sdpa": 1}
    layer.attend(*(t[1:].contiguous() for t in (q, k, v, gates)))
    assert calls == {"sdpa": 1, "attention": 1}


def test_attend_under_autocast(calls):
    """torch's attention casts to autocast's type: to float16 the call stays there
    (and the gate refuses its result), to bfloat16 nothing changes."""
    layer, q, k, v, gates = _attend(4, 64)
    with torch.autocast("cuda", dtype=BF16):
        _close(layer.attend(q, k, v, gates), _want(layer, q, k, v, gates))
    assert calls == {"attention": 1}
    with torch.autocast("cuda", dtype=torch.float16):
        out = layer.attend(q, k, v, None)
        with pytest.raises(RuntimeError):
            layer.attend(q, k, v, gates)
    assert out.dtype == torch.float16 and calls == {"attention": 1, "sdpa": 2}
    _close(out, _want(layer, q, k, v))
