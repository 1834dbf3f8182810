"""Neural building blocks of the LTX-2.5 DiT with the reference's module API
(standalone/ltx_nn.py), the memory-bound parts running on the ltxk HIP kernels.

Kept as in the reference (names, signatures, shapes): rms_norm, sdpa,
generate_freq_grid_np/_pytorch, precompute_freqs_cis, apply_split_rotary_emb,
TimestepEmbedder, CombinedTimestepEmbeddings, AdaLayerNormSingle, Attention,
FeedForward.  RMSNorm, q/k norm + split RoPE, unmasked attention with the
per-head gate, GELU-tanh, the linear layers of long K that `long_k_tiles` names
and the projections of few rows (`project`) are ltxk kernels, with fp32
arithmetic and one bf16 rounding per output.  The other linear layers, `sdpa` and
masked attention are PyTorch-ROCm's.
"""

import functools
import math

import numpy
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.compiler import is_compiling
from torch.nn.attention import SDPBackend, sdpa_kernel
from torch.nn.modules.module import _has_any_global_hook

import ltxk

SDPA_PRIORITY = [SDPBackend.CUDNN_ATTENTION, SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION,
                 SDPBackend.MATH]


def rms_norm(x: torch.Tensor, eps: float = 1e-6, weight: torch.Tensor | None = None) -> torch.Tensor:
    """RMSNorm over the last dim (reference ltx_nn.py:18-19) on ltxk_rms_norm."""
    return ltxk.rms_norm(x.contiguous(), weight, eps)


def sdpa(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, mask: torch.Tensor | None = None) -> torch.Tensor:
    """q,k,v: (B, H, T, D); PyTorch-ROCm attention with the reference's backend order (ltx_nn.py:22-26).

    Few queries over many keys (126 audio tokens over 6144 video tokens) leave the
    flash kernel a handful of query tiles, so it runs on a few CUs; that shape is
    split over the keys instead (key_split_applies, key_split_partials) and merged
    by ltxk_attn_combine.  Attention comes here with what ltxk_attention does not
    take (fused_attention_applies)."""
    if key_split_applies(q, k, mask):
        b, h, tq, d = q.shape
        merged = ltxk.attn_combine(*key_split_partials(q, k, v, KEY_SPLIT_PARTS), KEY_SPLIT_PARTS)
        return merged.view(b, tq, h, d).transpose(1, 2)
    with sdpa_kernel(SDPA_PRIORITY, set_priority=True):
        return F.scaled_dot_product_attention(q, k, v, attn_mask=mask, dropout_p=0.0, is_causal=False)


KEY_SPLIT_MAX_Q = 256
KEY_SPLIT_MIN_K = 2048
KEY_SPLIT_PARTS = 8


def key_split_applies(q: torch.Tensor, k: torch.Tensor, mask: torch.Tensor | None) -> bool:
    """Whether attention of q over k runs split over the keys: no mask, at most
    KEY_SPLIT_MAX_Q queries over at least KEY_SPLIT_MIN_K keys, in whole chunks."""
    return mask is None and q.is_cuda and q.shape[-2] <= KEY_SPLIT_MAX_Q and k.shape[-2] >= KEY_SPLIT_MIN_K \
        and k.shape[-2] % KEY_SPLIT_PARTS == 0


def key_split_partials(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, parts: int) -> tuple:
    """softmax(q k^T / sqrt(D)) v over `parts` equal chunks of the keys: one
    flash-attention launch with the chunks as extra batch items.  Returns the
    chunk outputs (B*parts, H, Tq, D) bf16 and their log-sum-exps
    (B*parts, H, Tq) fp32, which ltxk.attn_combine merges: out = sum_c
    exp(lse_c - lse) out_c with lse = logsumexp_c lse_c, the same softmax
    evaluated in a different order (each chunk's output is rounded to bf16 by
    the flash kernel before the merge)."""
    b, h, tq, d = q.shape
    tk = k.shape[-2]

    def chunks(x):  # (B, H, T, D) -> (B*parts, H, T/parts, D); a view for token-major storage
        return x.transpose(1, 2).reshape(b * parts, tk // parts, h, d).transpose(1, 2)

    qc = q.unsqueeze(1).expand(b, parts, h, tq, d).reshape(b * parts, h, tq, d)
    out, lse = torch.ops.aten._scaled_dot_product_flash_attention(qc, chunks(k), chunks(v))[:2]
    return out, lse


_dispatch_modes, _transform = torch._C._len_torch_dispatch_stack, torch._C._functorch.peek_interpreter_stack
_tracing = torch._C._is_tracing


def eager_call() -> bool:
    """Whether operations just run as they are called: no compiler, tracer, function
    transform, forward-mode derivative or dispatch mode is to see them.  The ltxk entry
    points bypass torch's dispatcher, so calls that one watches keep torch's operations."""
    return not (is_compiling() or _dispatch_modes() or _tracing() or forward_ad._current_level >= 0
                or _transform() is not None)


def attention_grid_fits(batch: int, tokens: int, heads: int) -> bool:
    """Whether ltxk_attention's launch holds these queries: at most 2^20 batch items,
    and fewer than 2^21 tiles of 128 queries on each of the 8 XCDs (2^32 threads),
    with room for the 64 units that cut keys make there."""
    return batch <= 1 << 20 and -(-batch * heads // 8) * -(-tokens // 128) < (1 << 21) - 64


def many_short_sequences(batch: int, tokens_q: int, tokens_k: int, heads: int, dim_head: int) -> bool:
    """Shapes that torch's attention, in tiles of 16, runs faster than ltxk_attention in
    its tiles of 128 queries and 64 keys.  Measured, torch (with the gate's launch) /
    ltxk_attention, us, for batch * heads of 2048, 4096 and 8192:
      heads of 64, 16 x 16 tokens: 10 / 12, 14 / 22, 21 / 42;  17 x 16: 15 / 12, -, 41 / 43;
        16 x 17: 15 / 12, -, 40 / 43;
      heads of 128, 32 x 16: 19 / 23, 33 / 41, 58 / 77;  40 x 16: 27 / 24, 47 / 44, 88 / 85;
        32 x 17 and more: faster here too (20 x 17: 26 / 22, -, 88 / 74).
    Up to 2048 the second launch costs the host more than is lost here."""
    return tokens_k <= 16 and tokens_q <= dim_head // 4 and batch * heads > 2048


def fused_attention_applies(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, heads: int, dim_head: int) -> bool:
    """Whether unmasked attention of token-major q over k, v runs on
    ltxk_attention: contiguous 16-byte aligned bf16 tensors on one ROCm device,
    heads of 64 or 128, keys of one batch item within the kernel's 32-bit
    offsets, queries within its launch, not many_short_sequences, no gradient to
    record, an eager call and no autocast to another type."""
    if dim_head not in ltxk.ATTENTION_HEAD_DIMS or not q.ndim == k.ndim == 3 or not eager_call():
        return False
    (b, tq, d), (kb, tk, kd) = q.shape, k.shape
    if not (b == kb and d == kd == heads * dim_head and v.shape == k.shape and 0 < tk and (tk + 64) * d < 2**30
            and attention_grid_fits(b, tq, heads)) or many_short_sequences(b, tq, tk, heads, dim_head):
        return False
    if torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != torch.bfloat16:
        return False
    device = q.get_device()
    for t in (q, k, v):
        if not (t.is_cuda and t.get_device() == device and t.dtype == torch.bfloat16 and t.is_contiguous()
                and t.data_ptr() % 16 == 0) or (t.requires_grad and torch.is_grad_enabled()):
            return False
    return True


# ---------------------------------------------------------------------------
# RoPE (LTXRopeType.SPLIT)
# ---------------------------------------------------------------------------


@functools.lru_cache(maxsize=8)
def generate_freq_grid_np(theta: float, n_axes: int, inner_dim: int) -> torch.Tensor:
    """theta ** linspace(0, 1, inner_dim // (2 n_axes)) * pi/2 in fp64, cast to fp32 (ltx_nn.py:34-46)."""
    count = inner_dim // (2 * n_axes)
    exps = numpy.linspace(numpy.log(1.0) / numpy.log(theta), numpy.log(theta) / numpy.log(theta), count,
                          dtype=numpy.float64)
    return torch.as_tensor(numpy.power(theta, exps) * math.pi / 2, dtype=torch.float32)


@functools.lru_cache(maxsize=8)
def generate_freq_grid_pytorch(theta: float, n_axes: int, inner_dim: int) -> torch.Tensor:
    """fp32 variant of the frequency grid (ltx_nn.py:49-60)."""
    count = inner_dim // (2 * n_axes)
    exps = torch.linspace(math.log(1.0, theta), math.log(theta, theta), count, dtype=torch.float32)
    return (theta ** exps).to(torch.float32) * math.pi / 2


def precompute_freqs_cis(
    indices_grid: torch.Tensor,
    dim: int,
    out_dtype: torch.dtype,
    theta: float = 10000.0,
    max_pos: list[int] | None = None,
    use_middle_indices_grid: bool = True,
    num_attention_heads: int = 32,
    double_precision: bool = True,
) -> tuple[torch.Tensor, torch.Tensor]:
    """(cos, sin) tables (B, H, T, D_head/2) for split RoPE (ltx_nn.py:63-96).

    Frequency p = f*n_axes + a (axis fastest) is ind[f] * (2*pos_a/max_pos[a] - 1);
    dim/2 - n_axes*F identity entries are padded in front; the flat table is
    then split per head.  Built once per model call; consumed by
    ltxk_qk_norm_rope.
    """
    if max_pos is None:
        max_pos = [20, 2048, 2048]
    n_axes = indices_grid.shape[1]
    grid_fn = generate_freq_grid_np if double_precision else generate_freq_grid_pytorch
    ind = grid_fn(theta, n_axes, dim).to(indices_grid.device)
    pos = indices_grid
    if pos.ndim == 4:
        pos = (pos[..., 0] + pos[..., 1]) / 2.0 if use_middle_indices_grid else pos[..., 0]
    frac = torch.stack([pos[:, a] / max_pos[a] for a in range(n_axes)], dim=-1)      # (B, T, A)
    ang = (ind * (frac.unsqueeze(-1) * 2 - 1)).transpose(-1, -2).flatten(2)          # (B, T, F*A)
    pad = dim // 2 - ang.shape[-1]
    cos, sin = ang.cos(), ang.sin()
    if pad:
        cos = torch.cat([torch.ones_like(cos[:, :, :pad]), cos], dim=-1)
        sin = torch.cat([torch.zeros_like(sin[:, :, :pad]), sin], dim=-1)
    b, t = cos.shape[0], cos.shape[1]
    cos = cos.reshape(b, t, num_attention_heads, -1).swapaxes(1, 2)
    sin = sin.reshape(b, t, num_attention_heads, -1).swapaxes(1, 2)
    return cos.to(out_dtype).contiguous(), sin.to(out_dtype).contiguous()


def precompute_freqs_cis_compact(
    indices_grid: torch.Tensor,
    dim: int,
    out_dtype: torch.dtype = torch.bfloat16,
    theta: float = 10000.0,
    max_pos: list[int] | None = None,
    use_middle_indices_grid: bool = True,
    num_attention_heads: int = 32,
    double_precision: bool = True,
    merge_slow_axes: bool = True,
) -> ltxk.CompactRope:
    """The tables of precompute_freqs_cis in ltxk's compact form.

    A pair's angle depends on one position axis only, so the table row of a
    token is assembled from one row per axis, keyed by that axis' coordinate:
    for each axis the distinct coordinates (16, 16 and 24 for a 16x16x24 latent
    grid, 16 for the A2V/V2A time axis) get a row holding cos/sin at that
    axis' pairs and 0 elsewhere.  Each distinct angle is computed with the same
    fp32 operations as the full tables, so every combined entry equals the
    full table's bit for bit, while the rows (a few hundred KB) stay in cache.
    With three axes and merge_slow_axes the time and height rows are merged
    into one row per distinct (time, height) pair (256 for the 16x16x24 grid,
    2 MB), so the index has two columns.  One device-to-host read per axis
    (the count of distinct coordinates).
    """
    if max_pos is None:
        max_pos = [20, 2048, 2048]
    b, n_axes, t = indices_grid.shape[0], indices_grid.shape[1], indices_grid.shape[2]
    grid_fn = generate_freq_grid_np if double_precision else generate_freq_grid_pytorch
    ind = grid_fn(theta, n_axes, dim).to(indices_grid.device)
    pos = indices_grid
    if pos.ndim == 4:
        pos = (pos[..., 0] + pos[..., 1]) / 2.0 if use_middle_indices_grid else pos[..., 0]
    nf = ind.numel()
    half = dim // 2
    pad = half - nf * n_axes
    axis_rows = []
    for a in range(n_axes):
        coords, inverse = torch.unique(pos[:, a], return_inverse=True)
        frac = coords / max_pos[a]
        ang = ind * (frac.unsqueeze(-1) * 2 - 1)                        # (U, F)
        cols = pad + torch.arange(nf, device=ang.device) * n_axes + a
        c = torch.zeros(coords.numel(), half, device=ang.device, dtype=torch.float32)
        s = torch.zeros_like(c)
        c[:, cols] = ang.cos()
        s[:, cols] = ang.sin()
        if a == 0 and pad:
            c[:, :pad] = 1.0
        axis_rows.append((c, s, inverse))
    if n_axes == 3 and merge_slow_axes:
        # The two slower axes (time, height) change every w tokens only: one
        # row per distinct (time, height) pair holding both axes' entries
        # (their pairs are disjoint, so the sum is exact) leaves the kernel two
        # table rows per token instead of three.
        (c0, s0, i0), (c1, s1, i1) = axis_rows[0], axis_rows[1]
        pairs, inverse = torch.unique(i0 * c1.shape[0] + i1, return_inverse=True)
        p0, p1 = pairs // c1.shape[0], pairs % c1.shape[0]
        axis_rows = [(c0[p0] + c1[p1], s0[p0] + s1[p1], inverse), axis_rows[2]]
    cos_rows, sin_rows, index = [], [], []
    first = 0
    for c, s, inverse in axis_rows:
        cos_rows.append(c)
        sin_rows.append(s)
        index.append(inverse + first)
        first += c.shape[0]
    cos = torch.cat(cos_rows).to(out_dtype).contiguous()
    sin = torch.cat(sin_rows).to(out_dtype).contiguous()
    idx = torch.stack(index, dim=-1).to(torch.int32).contiguous()  # (B, T, A)
    return ltxk.CompactRope(cos, sin, idx, (b, num_attention_heads, t, half // num_attention_heads), checked=True)


def apply_split_rotary_emb(x: torch.Tensor, freqs_cis) -> torch.Tensor:
    """Split-half rotation per head (ltx_nn.py:99-115) on ltxk_qk_norm_rope.

    x: (B, T, H*D) token-major or (B, H, T, D); freqs: (cos, sin) (B, H, T, D/2)
    or the compact form of precompute_freqs_cis_compact.  Returns a new tensor
    of x's shape.
    """
    if isinstance(freqs_cis, ltxk.CompactRope):
        pe, h = freqs_cis, freqs_cis.shape[1]
    else:
        cos, sin = freqs_cis
        pe, h = (cos.contiguous(), sin.contiguous()), cos.shape[1]
    if x.ndim == 4:
        b, _, t, d = x.shape
        tok = x.transpose(1, 2).reshape(b, t, h * d).contiguous()
        ltxk.qk_norm_rope(tok, None, h, d, q_pe=pe)
        return tok.view(b, t, h, d).transpose(1, 2)
    out = x.contiguous().clone()
    ltxk.qk_norm_rope(out, None, h, x.shape[-1] // h, q_pe=pe)
    return out


# ---------------------------------------------------------------------------
# Timestep embedding (PixArt-alpha style)
# ---------------------------------------------------------------------------


class TimestepEmbedder(torch.nn.Module):
    def __init__(self, in_channels: int, time_embed_dim: int):
        super().__init__()
        self.linear_1 = torch.nn.Linear(in_channels, time_embed_dim)
        self.linear_2 = torch.nn.Linear(time_embed_dim, time_embed_dim)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.linear_2(F.silu(self.linear_1(x)))


class CombinedTimestepEmbeddings(torch.nn.Module):
    """256-wide sinusoidal projection then TimestepEmbedder (ltx_nn.py:133-145)."""

    def __init__(self, embedding_dim: int):
        super().__init__()
        self.timestep_embedder = TimestepEmbedder(256, embedding_dim)

    def forward(self, timestep: torch.Tensor, hidden_dtype: torch.dtype) -> torch.Tensor:
        from common import get_timestep_embedding

        proj = get_timestep_embedding(timestep, 256, max_period=10000)
        return self.timestep_embedder(proj.to(hidden_dtype))


class AdaLayerNormSingle(torch.nn.Module):
    """SiLU -> Linear(embedding_dim -> coefficient*embedding_dim) (ltx_nn.py:148-158)."""

    def __init__(self, embedding_dim: int, embedding_coefficient: int = 6):
        super().__init__()
        self.emb = CombinedTimestepEmbeddings(embedding_dim)
        self.linear = torch.nn.Linear(embedding_dim, embedding_coefficient * embedding_dim, bias=True)

    def forward(self, timestep: torch.Tensor, hidden_dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
        embedded = self.emb(timestep, hidden_dtype=hidden_dtype)
        return self.linear(F.silu(embedded)), embedded


# ---------------------------------------------------------------------------
# Linear layers
# ---------------------------------------------------------------------------


def long_k_tiles(m: int, n: int, k: int) -> bool:
    """Whether a product of (m, k) and (n, k) matrices goes to ltxk_linear: the
    shapes that leave the library's product to few compute units for a long K
    (256 x 256 output tiles, 256 at a time).  Measured, library / ltxk_linear, us:
      K 188160 x N 4096 (2048), M 8: 275 / 337 (358 / 182), 24: 671 / 345, 64: 616 / 352,
        128: 586 / 371 (404 / 192), 512: 1048 / 673 (742 / 363), 1024: 2100 / 1214
        (1087 / 632), 1280: 1807 / 1617, 1536: 1807 / 2112, 2048: 2067 / 2437 (2010 /
        1242), 2560: (1598 / 1593), 4096: 3993 / 4739 (2072 / 2418);
      K 65536 x N 4096, M 8: 116 / 122, 1280: 772 / 572, 2048: 767 / 863;  x N 16384,
        M 24: 382 / 470, 64: 467 / 480, 96: 466 / 490;
      K 32768 x N 3072, M 16: 37 / 46, 24: 73 / 49;  x N 8192, M 32: 100 / 123, 65: 200 / 134;
      K 16384 x N 4096, M 33: 30 / 34, 64: 37 / 36, 65: 40 / 37, 128: 61 / 41, 256: 55 / 52,
        512: 91 / 75, 1024: 130 / 126 (in the text encoder, two blocks: 3864 / 3834 the
        whole call), 1280: 152 / 152, 2048: 207 / 226;  x N 8192, M 65: 57 / 66;
      K 8192 and less: the library's is faster (M 1008, N 2048: 46 / 49)."""
    if n % 8 or k % 64 or k < 16384 or max(m * k, n * k, m * n) >= 2**31:
        return False
    if m < 24:
        most = 8 if k >= 32768 else 2
    elif m <= 64:
        most = 20 if k >= 32768 else 2
    elif m <= 128:
        most = 32 if k >= 32768 else 16
    else:
        most = 80 if k >= 65536 else 64
    return -(-m // 256) * -(-n // 256) <= most


def full_wave_rows(m: int, n: int, k: int) -> int:
    """The rows of a large (m, k) x (n, k) product that fill whole waves of 256 tiles
    of 256 x 256, where few rows are left past them: those then go in a launch of
    their own, because the library gives them a whole further wave, or other tiles
    to all of it.  0: one launch.  Measured, one launch / two, us, N x K:
      4096 x 4096, M 4160: 131 / 104, 4290: 131 / 110, 4800: 141 / 122, 8580: 221 / 205,
        12500: 388 / 289, 24676: 657 / 548;  4096 x 2048, M 4290: 78 / 60, 12500: 223 / 156;
      4096 x 8192, M 4290: 240 / 204;  4096 x 16384, M 4290: 844 / 401, 8448: 1198 / 760,
        24776: 2386 / 2196;  4096 x 32768, M 4290: 1579 / 857;
      8192 x 2048, M 4352: 145 / 117, 8900: 222 / 219;  8192 x 4096, M 4100: 305 / 192,
        4600: 229 / 218, 8892: 412 / 403, 17084: 883 / 761;  8192 x 16384, M 4200: 1207 / 772;
      16384 x 2048, M 4290: 253 / 215;  16384 x 4096, M 4290: 427 / 391, 4800: 572 / 438,
        8892: 928 / 791, 17084: 1609 / 1504, 24776: 2207 / 2176.
    Above 768 rows the two are less often apart, and three times the other way (4096 x
    16384, 1769 rows past 4096: 584 / 746; 16384 x 4096, 808 past 8192: 790 / 812, 776
    past 16384: 1517 / 1524)."""
    across = -(-n // 256)
    if n < 4096 or not 2048 <= k < 65536 or across > 64 or 256 % across:
        return 0
    wave = 256 // across * 256
    main = m // wave * wave
    return main if main >= 4096 and 0 < m - main <= 768 else 0


def _plain_input(x: torch.Tensor) -> bool:
    """Whether the ltxk products can read x: contiguous aligned bf16 on a ROCm
    device, no autocast, no gradient to record, an eager call without module hooks."""
    return x.is_cuda and x.dtype == torch.bfloat16 and eager_call() and x.is_contiguous() and x.data_ptr() % 16 == 0 \
        and x.numel() > 0 and not (x.requires_grad and torch.is_grad_enabled()) \
        and not torch.is_autocast_enabled("cuda") and not _has_any_global_hook()


_PLAIN = (torch.nn.Parameter, torch.Tensor)


def _plain_layer(layer: torch.nn.Linear, x: torch.Tensor) -> tuple | None:
    """(weight, bias) of a bare torch.nn.Linear (no hooks, its own forward, plain
    tensors) whose operands fit x like _plain_input, else None.  They must have the
    layer's own shapes: torch broadcasts a bias of one entry, the kernels read
    out_features of them.  Reads the module's dictionaries: its attribute lookup
    costs more than the rest (`project` over four layers takes the host 30 us with
    it, 16 without)."""
    own = layer.__dict__
    if type(layer) is not torch.nn.Linear or own["_forward_hooks"] or own["_forward_pre_hooks"] \
            or "forward" in own or "weight" in own or "bias" in own:  # attributes come before class and parameters
        return None
    params = own["_parameters"]
    w, b, n = params.get("weight"), params.get("bias", False), own["out_features"]
    if w is None or b is False:  # kept elsewhere
        return None
    if w.shape != (n, x.shape[-1]) or (b is not None and b.shape != (n,)):
        return None
    device, bf16 = x.get_device(), torch.bfloat16
    for t in (w,) if b is None else (w, b):
        if not (type(t) in _PLAIN and t.get_device() == device and t.dtype == bf16 and t.is_contiguous()
                and t.data_ptr() % 16 == 0) or (t.requires_grad and torch.is_grad_enabled()):
            return None
    return w, b


def linear(layer: torch.nn.Linear, x: torch.Tensor) -> torch.Tensor:
    """layer(x): on ltxk_linear where long_k_tiles says so, in two launches where
    full_wave_rows does."""
    if type(layer) is not torch.nn.Linear:
        return layer(x)
    k, n = x.shape[-1], layer.out_features
    m = x.numel() // max(k, 1)
    own = k >= 16384 and long_k_tiles(m, n, k)
    main = 0 if own or m <= 4096 else full_wave_rows(m, n, k)
    if (own or main) and _plain_input(x):
        plain = _plain_layer(layer, x)
        if plain is not None:
            return ltxk.linear(x, *plain) if own else _two_launches(x, *plain, main)
    return layer(x)


def _two_launches(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, main: int) -> torch.Tensor:
    """x weight^T + bias, the first `main` rows and the others apart."""
    k, n = x.shape[-1], weight.shape[0]
    out = x.new_empty((*x.shape[:-1], n))
    rows, to, wt = x.view(-1, k), out.view(-1, n), weight.t()
    for part in (slice(0, main), slice(main, None)):
        if bias is None:
            torch.mm(rows[part], wt, out=to[part])
        else:
            torch.addmm(bias, rows[part], wt, out=to[part])
    return out


# ltxk_linear_layers takes the projections of an input of at most this many
# elements: a launch and about 20 us of the host for all of them instead of for
# each.  Measured, layer by layer / ltxk_linear_layers, device us (eager calls):
#   x [126, 2048], N 3 x 2048 + 32: 45 / 16 (77 / 16); [252, 2048]: 47 / 27;
#   [504, 2048]: 49 / 50; x [126, 4096], N 3 x 4096 + 32: 62 / 50; [256, 4096]: 79 / 87;
#   one layer alone, x [126, 2048], N 2048: 9 / 13, so single layers stay as they are.
FEW_ROWS_MAX = 1 << 19


def few_rows_widths(m: int, k: int, widths) -> bool:
    """Whether layers of these widths over m rows of k go to ltxk_linear_layers: each a
    multiple of 8, weights and outputs of fewer than 2^31 elements, K up to 6144, and
    up to 160 of its tiles of 128 x 32 a layer (a launch takes 256 at a time, and what
    it saves is a launch a layer).  Measured, layer by layer / ltxk_linear_layers,
    device us:
      x [256, 2048], N 2 x 2048 (128 tiles a layer): 19 / 13, 2 x 3072 (192): 21 / 25,
        3 x 2560 (160): 31 / 25;  [126, 2048], 4 x 4096 (128): 38 / 27;
      x [1024, 512], 3 x 576 (144): 18 / 12, 2 x 2048 (512): 14 / 23;  [4096, 128],
        3 x 1024 (1024): 19 / 45;
      x [80, 6144], 3 x 2048: 39 / 29, 3 x 4096: 54 / 55;  [64, 8192], 3 x 2048: 52 / 38,
        2 x 2048: 35 / 36, 3 x 4096: 56 / 74, 8192 + 32: 39 / 72;  [32, 16384],
        2 x 4096: 59 / 69."""
    if k > 6144:
        return False
    tiles = 0
    for n in widths:
        if n % 8 or max(m, k) * n >= 2**31:
            return False
        tiles += (n + 31) // 32
    return -(-m // 128) * tiles <= 160 * len(widths)


def project(x: torch.Tensor, *layers: torch.nn.Linear | None) -> list:
    """[layer(x) for each layer], None for None, in one launch where x is small."""
    real = [layer for layer in layers if layer is not None]
    size, k = x.numel(), x.shape[-1]
    if 2 <= len(real) <= ltxk.MAX_LINEAR_LAYERS and 0 < size <= FEW_ROWS_MAX and k % 128 == 0 \
            and few_rows_widths(size // k, k, [i.out_features if type(i) is torch.nn.Linear else 1 for i in real]) \
            and _plain_input(x):
        plain = [_plain_layer(layer, x) for layer in real]
        if None not in plain:
            weights, biases = zip(*plain)
            done = iter(ltxk._launch_layers(x, weights, biases))
            return [None if layer is None else next(done) for layer in layers]
    return [None if layer is None else linear(layer, x) for layer in layers]


# ---------------------------------------------------------------------------
# Attention + FFN
# ---------------------------------------------------------------------------


class Attention(torch.nn.Module):
    """Multi-head attention with RMS q/k-norm, split RoPE and per-head gating (ltx_nn.py:166-236).

    q/k/v/gate projections are PyTorch-ROCm, or one ltxk_linear_layers launch
    over few rows (`project`).  q_norm/k_norm + RoPE run as one in-place
    ltxk_qk_norm_rope launch on the fresh projections; attention, the head merge
    and the per-head 2*sigmoid gate are one ltxk_attention call (`attend`).
    """

    def __init__(self, query_dim: int, context_dim: int | None = None, heads: int = 8, dim_head: int = 64,
                 norm_eps: float = 1e-6, apply_gated_attention: bool = False):
        super().__init__()
        self.heads = heads
        self.dim_head = dim_head
        inner_dim = heads * dim_head
        context_dim = query_dim if context_dim is None else context_dim
        self.q_norm = torch.nn.RMSNorm(inner_dim, eps=norm_eps)
        self.k_norm = torch.nn.RMSNorm(inner_dim, eps=norm_eps)
        self.to_q = torch.nn.Linear(query_dim, inner_dim, bias=True)
        self.to_k = torch.nn.Linear(context_dim, inner_dim, bias=True)
        self.to_v = torch.nn.Linear(context_dim, inner_dim, bias=True)
        self.to_gate_logits = torch.nn.Linear(query_dim, heads, bias=True) if apply_gated_attention else None
        self.to_out = torch.nn.Linear(inner_dim, query_dim, bias=True)

    def forward(self, x: torch.Tensor, context: torch.Tensor | None = None, mask: torch.Tensor | None = None,
                pe: tuple[torch.Tensor, torch.Tensor] | None = None,
                k_pe: tuple[torch.Tensor, torch.Tensor] | None = None,
                perturbation_mask: torch.Tensor | None = None, all_perturbed: bool = False) -> torch.Tensor:
        context = x if context is None else context
        h, dh = self.heads, self.dim_head
        if all_perturbed:
            v = self.to_v(context)
            gates = self.to_gate_logits(x).contiguous() if self.to_gate_logits is not None else None
            out = v if gates is None else ltxk.head_gate(v, gates)
            return linear(self.to_out, out)
        if context is x:
            q, k, v, gates = project(x, self.to_q, self.to_k, self.to_v, self.to_gate_logits)
        else:
            q, gates = project(x, self.to_q, self.to_gate_logits)
            k, v = project(context, self.to_k, self.to_v)
        gates = gates.contiguous() if gates is not None else None
        ltxk.qk_norm_rope(q, k, h, dh, q_weight=self.q_norm.weight, k_weight=self.k_norm.weight,
                          q_pe=pe, k_pe=pe if k_pe is None else k_pe, eps=self.eps)
        return self.attend(q, k, v, gates, mask, perturbation_mask)

    @property
    def eps(self) -> float:
        return self.q_norm.eps if self.q_norm.eps is not None else 1e-6

    def attend(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, gates: torch.Tensor | None,
               mask: torch.Tensor | None = None, perturbation_mask: torch.Tensor | None = None) -> torch.Tensor:
        """The part of forward after q/k norm + RoPE (ltx_nn.py:219-236): attention
        on token-major q, k, v (B, T, H*Dh), the head merge [+ perturbation blend]
        [+ per-head gate], then to_out.  Without a mask and for heads of 64 or 128
        that is ltxk_attention with the gate inside it (the blend as an
        ltxk_head_gate pass after it); otherwise torch's SDPA, then ltxk_head_gate.
        Lets a caller prepare the q/k of two attentions in one launch (Block's
        A2V/V2A)."""
        b = q.shape[0]
        h, dh = self.heads, self.dim_head
        pm = None
        if perturbation_mask is not None:
            pm = perturbation_mask.reshape(-1).to(torch.bfloat16).contiguous()
        if mask is None and fused_attention_applies(q, k, v, h, dh):
            if pm is None:
                return linear(self.to_out, ltxk.attention(q, k, v, h, gates))
            return linear(self.to_out, ltxk.head_gate(ltxk.attention(q, k, v, h), gates, v=v, mask=pm, heads=h))
        q4 = q.view(b, -1, h, dh).transpose(1, 2)
        k4 = k.view(b, -1, h, dh).transpose(1, 2)
        v4 = v.view(b, -1, h, dh).transpose(1, 2)
        if mask is not None:
            if mask.ndim == 2:
                mask = mask.unsqueeze(0)
            if mask.ndim == 3:
                mask = mask.unsqueeze(1)
        if perturbation_mask is None and key_split_applies(q4, k4, mask):
            # key-split attention (of heads that ltxk_attention does not take): its merge, the
            # head merge and the gate in one pass
            part, lse = key_split_partials(q4, k4, v4, KEY_SPLIT_PARTS)
            return self.to_out(ltxk.attn_combine(part, lse, KEY_SPLIT_PARTS, gates))
        attn = sdpa(q4, k4, v4, mask)  # (B, H, T, D) view
        if perturbation_mask is None and gates is None:
            out = attn.transpose(1, 2).reshape(b, -1, h * dh)
        else:
            # head merge [+ perturbation blend] [+ per-head gate] in one pass
            out = ltxk.head_gate(attn, gates, v=v.contiguous() if pm is not None else None, mask=pm)
        return self.to_out(out)


class FeedForward(torch.nn.Module):
    """proj_in -> GELU-tanh (ltxk, in place) -> proj_out (ltx_nn.py:239-248)."""

    def __init__(self, dim: int, dim_out: int | None = None, mult: int = 4, bias: bool = True):
        super().__init__()
        dim_out = dim if dim_out is None else dim_out
        inner = int(dim * mult)
        self.proj_in = torch.nn.Linear(dim, inner, bias=bias)
        self.proj_out = torch.nn.Linear(inner, dim_out, bias=bias)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        hdn = linear(self.proj_in, x)
        ltxk.gelu_tanh(hdn, out=hdn)
        return linear(self.proj_out, hdn)
