"""ltxk_attention (csrc/flash.hip) against softmax attention in fp64 (GPU), at the
edges of its query and key tiles, where its launches are cut over the keys, and
on inputs whose first key tile weighs nothing."""

import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _check(q, k, v, h, logits, got):
    """Element by element: rounding to bf16 (8 significant bits) moves a value by at
    most 2^-8 of it, so the weights' roundings move the result by at most
    2^-8 sum_j w_j |v_j|, the output's and the gated output's by 2^-8 of their
    value each; the fp32 sums and exponentials are far below that (2 %)."""
    b, tq, d = q.shape
    dh = d // h
    for i in range(b):
        for j in range(h):
            c = slice(j * dh, (j + 1) * dh)
            w = torch.softmax(q[i, :, c].double() @ k[i, :, c].double().T / math.sqrt(dh), -1)
            want, spread = w @ v[i, :, c].double(), w @ v[i, :, c].double().abs()
            bound = spread * 2.0**-8 + want.abs() * 2.0**-8
            if logits is not None:
                gate = 2 * torch.sigmoid(logits[i, :, j].double()).unsqueeze(-1)
                want, bound = want * gate, (bound + want.abs() * 2.0**-8) * gate
            err = (got[i, :, c].double() - want).abs()
            assert bool((err <= bound * 1.02 + 1e-6).all()), f"item {i} head {j}: {(err / (bound + 1e-6)).max().item():.3f}"


@pytest.mark.parametrize("b,tq,tk,h,dh,gated,spread", [
    (1, 1, 1, 2, 64, True, 1.0), (1, 128, 64, 1, 128, False, 1.0), (2, 129, 65, 3, 64, True, 1.0),
    (1, 127, 63, 2, 128, True, 3.0), (3, 257, 191, 3, 128, True, 1.5), (1, 33, 1000, 2, 64, True, 1.5),
    (1, 5, 4099, 9, 128, True, 1.5), (4, 126, 2050, 2, 64, False, 3.0), (1, 8257, 520, 8, 64, True, 1.5),
    (1, 8200, 600, 9, 128, True, 1.5)])
def test_attention_matches_fp64(b, tq, tk, h, dh, gated, spread):
    import ltxk

    g = torch.Generator(device=DEV).manual_seed(tq * 7 + tk)
    q, k, v = ((torch.randn(b, t, h * dh, device=DEV, generator=g) * s).to(torch.bfloat16)
               for t, s in ((tq, spread), (tk, spread), (tk, 1.0)))
    logits = torch.randn(b, tq, h, device=DEV, generator=g).to(torch.bfloat16) if gated else None
    _check(q, k, v, h, logits, ltxk.attention(q, k, v, h, logits))


@pytest.mark.parametrize("tk", [200, 2048])
def test_first_tile_without_weight(tk):
    """Scores of -inf over the whole first key tile (and, with the keys cut, over
    a whole unit) weigh nothing; the other keys' softmax is unaffected."""
    import ltxk

    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.rand(1, 40, 128, device=DEV, generator=g).to(torch.bfloat16) + 0.5
    k, v = (torch.randn(1, tk, 128, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    closed = 64 if tk == 200 else 1024
    k[:, :closed] = -float("inf")
    got = ltxk.attention(q, k, v, 2)
    _check(q, k[:, closed:].contiguous(), v[:, closed:].contiguous(), 2, None, got)


def test_strided_operands_and_refusals():
    """q, k and v as columns of one wider buffer through the C entry equal the
    contiguous call bit for bit; a stride that does not cover the heads, a head
    of 96 and a missing workspace are refused."""
    import ltxk

    lib = ltxk.load()
    b, t, h, dh = 2, 300, 2, 64
    d = h * dh
    qkv = torch.randn(b, t, 3 * d, device=DEV).to(torch.bfloat16)
    q, k, v = (qkv[..., i * d:(i + 1) * d].contiguous() for i in range(3))
    want = ltxk.attention(q, k, v, h)
    out = torch.empty_like(want)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    p, row = qkv.data_ptr(), 3 * d

    def call(tstride=row, head_dim=dh, tk=t, nbytes=0):
        return lib.ltxk_attention(out.data_ptr(), p, t * row, tstride, p + 2 * d, t * row, row, p + 4 * d, t * row, row,
                                  None, b, t, tk, h, head_dim, dh**-0.5, None, nbytes, st)

    assert lib.ltxk_attention_workspace_bytes(b, t, t, h, dh) == 0
    assert call() == 0
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert call(tstride=64) == ltxk.E_ARG and call(tstride=row + 4) == ltxk.E_ALIGN
    assert call(head_dim=96) == ltxk.E_ARG and call(tk=0) == ltxk.E_ARG
    assert lib.ltxk_attention_workspace_bytes(b, t, 4096, h, dh) > 0
    assert call(tk=4096) == ltxk.E_ARG


def test_captured_calls_replay_equal():
    """Attention with cut keys, a linear layer cut over K and layers over few rows in
    one captured graph: every replay, with other inputs and eager work between,
    equals the eager calls bit for bit (their scratch comes from the graph's pool)."""
    import ltxk

    g = torch.Generator(device=DEV).manual_seed(9)

    def fresh(*shape):
        return torch.randn(*shape, device=DEV, generator=g).to(torch.bfloat16)

    q, k, v, logits = fresh(1, 100, 256), fresh(1, 3000, 256), fresh(1, 3000, 256), fresh(1, 100, 4)
    x, w, b = fresh(300, 16384), fresh(256, 16384) * 0.02, fresh(256)
    few, few_w = fresh(70, 512), [fresh(64, 512), fresh(40, 512)]

    def call():
        return [ltxk.attention(q, k, v, 4, logits), ltxk.linear(x, w, b), *ltxk.linear_layers(few, few_w, [None, None])]

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = call()
    for _ in range(4):
        for t in (q, k, v, logits, x, few):
            t.copy_(fresh(*t.shape))
        want = call()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, e in zip(captured, want):
            assert torch.equal(a.view(torch.int16), e.view(torch.int16))


def test_attend_under_a_transform_and_a_mode():
    """Attention.attend without gates, masks and hooks is torch operations under
    vmap and under a dispatch mode that counts them, and gives what eager calls do."""
    from torch.utils.flop_counter import FlopCounterMode

    import ltx_nn

    layer = ltx_nn.Attention(256, 256, 4, 64).to(device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(3, 2, 70, 256, device=DEV, generator=g).to(torch.bfloat16) for _ in range(3))
    want = torch.stack([layer.attend(*t, None) for t in zip(q, k, v)]).float()
    got = torch.func.vmap(lambda *t: layer.attend(*t, None))(q, k, v).float()
    # the attention's bf16 roundings and the output's
    assert ((got - want).norm() / want.norm()).item() < 2.0**-7
    with FlopCounterMode(display=False) as counted:
        layer.attend(q[0], k[0], v[0], None)
    assert counted.get_total_flops() >= 2 * 2 * 70 * 256 * (70 + 70 + 256)


@pytest.mark.parametrize("size", [2.0**10, 2.0**20, 2.0**26, 2.0**34, 2.0**100])
@pytest.mark.parametrize("tk,sign", [(64, 1), (70, -1), (3000, 1)])
def test_large_scores(size, tk, sign):
    """Scores of either sign up to far past 2^31, in which the rounding of a scaled
    score spans whole powers of two, with the largest of a row repeated over the
    units of cut keys: softmax of them as in 64 bits, one-hot or the mean of equals."""
    import ltxk

    q = torch.zeros(1, 40, 128, device=DEV)
    q[..., ::64] = size**0.5 * torch.linspace(1, 1.9, 40, device=DEV).view(1, 40, 1)
    k = torch.zeros(1, tk, 128, device=DEV)
    k[..., ::64] = sign * (torch.arange(tk, device=DEV) % 127 + 129).view(1, tk, 1) * size**0.5 / 256
    v = torch.randn(1, tk, 128, device=DEV, generator=torch.Generator(device=DEV).manual_seed(tk))
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    _check(q, k, v, 2, None, ltxk.attention(q, k, v, 2))
