"""GPT-2 decoder whose four Linear slots take :class:`QuantLinear` modules.

This is the inference model of the quantized path: pre-LN GPT-2 blocks with
learned positions, the tanh GELU and a tied head. The reference's ablation
switches (post-LN, sinusoidal positions, other activations, grouped-query
heads, attention / neuron masks, activation taps) are not part of that path
and are refused at construction.

Three things are interface and therefore fixed:

* the module names (``wte``, ``wpe``, ``h.<i>.ln_1``, ``h.<i>.attn.c_attn``,
  ``h.<i>.attn.c_proj``, ``h.<i>.ln_2``, ``h.<i>.mlp.c_fc``,
  ``h.<i>.mlp.c_proj``, ``ln_f``, ``lm_head``): ``quantize_model`` finds its
  targets by these suffixes and checkpoints are keyed by them;
* the order of the random draws at construction and initialisation, which
  fixes the seed-0 weights every benchmark is quoted on
  (``src/transformer_internals/model.py:457-518``; see :meth:`GPT._seeded_init`);
* ``forward(idx, targets=None, cache=None)`` returning ``{"logits", "loss"}``
  and the ``KVCache`` calls made by the greedy loop
  (``sampling.py:100-181``, ``model.py:106-172``).

The arithmetic is GPT-2's (``model.py:57-75,227-320,351-355,528-599``); on the
GPU the quantized projections are the library's HIP kernels and the prefill's
GELU is one HIP pass.
"""

from __future__ import annotations

import math
from typing import Any

import torch
import torch.nn as nn
import torch.nn.functional as F

from .config import GPTConfig
from .qlinear import QuantLinear

__all__ = ["GPT", "MLP", "Block", "CausalSelfAttention", "KVCache", "gelu_tanh"]

_SQRT_2_OVER_PI = math.sqrt(2.0 / math.pi)


def gelu_tanh(x: torch.Tensor) -> torch.Tensor:
    """GELU in GPT-2's tanh form, ``0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))``.

    An fp32 GPU tensor that needs no gradient goes through one HIP pass
    (``tiq_gelu_tanh``: one read and one write instead of the eight passes
    of the op chain). Anything else -- CPU tensors, other dtypes, or a tensor
    autograd must differentiate -- is computed with torch ops, which carry the
    gradient.
    """
    if x.is_cuda and x.dtype == torch.float32 and not (torch.is_grad_enabled() and x.requires_grad):
        from . import _lib

        src = x.contiguous()
        if src.data_ptr() % 16:
            src = src.clone()  # fresh allocations are 16-byte aligned
        out = torch.empty_like(src)
        _lib.check(_lib.lib().tiq_gelu_tanh(src.data_ptr(), out.data_ptr(), src.numel(), _lib.stream_of(src)),
                   "gelu_tanh")
        return out
    inner = _SQRT_2_OVER_PI * (x + 0.044715 * x.pow(3))
    return 0.5 * x * (1.0 + torch.tanh(inner))


class KVCache:
    """Per-layer key / value history for cached decoding.

    Each layer owns a buffer ``(B, heads, capacity, head_dim)`` that grows by
    doubling, so appending a step writes only the new rows (the reference's
    ``torch.cat`` copies the whole history every step, ``model.py:153-172``).
    ``length(layer)`` is that layer's own fill level -- inside one forward
    pass the earlier layers already hold the current step, so the causal
    offset of a layer must come from it, not from :attr:`seq_len`
    (``model.py:139-151``).
    """

    def __init__(self, keys: int | list[torch.Tensor | None], values: list[torch.Tensor | None] | None = None) -> None:
        """``KVCache(n_layer)``: an empty cache. ``KVCache(keys=[...],
        values=[...])`` (the reference's dataclass fields, ``model.py:106-126``):
        per layer a filled ``(B, heads, T, head_dim)`` history or ``None``;
        those tensors become the layers' buffers (full: the next append grows
        them by a copy)."""
        if isinstance(keys, int):
            if values is not None:
                raise ValueError("KVCache(n_layer) takes no values")
            self._k: list[torch.Tensor | None] = [None] * keys
            self._v: list[torch.Tensor | None] = [None] * keys
            self._len = [0] * keys
            return
        if values is None or len(keys) != len(values):
            raise ValueError("KVCache needs keys and values lists of the same length")
        for k, v in zip(keys, values):
            if (k is None) != (v is None) or (k is not None and k.shape != v.shape):
                raise ValueError("each layer's keys and values must both be None or tensors of one shape")
        self._k, self._v = list(keys), list(values)
        self._len = [0 if k is None else int(k.shape[-2]) for k in keys]

    @classmethod
    def empty(cls, n_layer: int) -> KVCache:
        return cls(n_layer)

    @classmethod
    def over(cls, keys: list[torch.Tensor], values: list[torch.Tensor]) -> KVCache:
        """An empty cache whose layer buffers are the given ``(B, heads,
        capacity, head_dim)`` tensors (a decoder's preallocated cache): a
        prefill appends into them in place (past ``capacity`` they grow by a
        copy, as an empty cache's do)."""
        cache = cls(len(keys))
        cache._k, cache._v = list(keys), list(values)  # buffers, 0 positions filled
        return cache

    @property
    def seq_len(self) -> int:
        """Positions already processed (layer 0's fill level): the absolute
        position of the tokens a forward pass is about to add."""
        return self._len[0]

    def length(self, layer: int) -> int:
        return self._len[layer]

    @property
    def keys(self) -> list[torch.Tensor | None]:
        """Each layer's filled history (views; append with :meth:`update`)."""
        return [None if b is None else b[:, :, :n] for b, n in zip(self._k, self._len)]

    @property
    def values(self) -> list[torch.Tensor | None]:
        return [None if b is None else b[:, :, :n] for b, n in zip(self._v, self._len)]

    def _room(self, layer: int, t: int, dims: tuple[int, ...], like_k: torch.Tensor,
              like_v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """The layer's buffers, grown (a copy) if ``t`` more positions do not
        fit; a first buffer is ``(*dims[:-1], capacity, dims[-1])``."""
        n = self._len[layer]
        buf_k, buf_v = self._k[layer], self._v[layer]
        if buf_k is None or n + t > buf_k.shape[-2]:
            cap = max(16, 2 * (n + t))
            grown_k = like_k.new_empty(*dims[:-1], cap, dims[-1])
            grown_v = like_v.new_empty(*dims[:-1], cap, dims[-1])
            if buf_k is not None:
                grown_k[:, :, :n] = buf_k[:, :, :n]
                grown_v[:, :, :n] = buf_v[:, :, :n]
            self._k[layer], self._v[layer] = buf_k, buf_v = grown_k, grown_v
        return buf_k, buf_v

    def _append_slots(self, layer: int, batch: int, heads: int, t: int,
                      like: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor] | None:
        """The ``(batch, heads, t, 64)`` slots the next ``t`` positions of an fp32
        GPU cache take, for a kernel that writes them (then :meth:`_advance`);
        None where :meth:`update` has to copy: another type, device, shape or
        layout, a tensor that autograd follows."""
        buf = self._k[layer]
        if buf is not None and (buf.dim() != 4 or buf.shape[:2] != (batch, heads) or buf.shape[3] != 64):
            return None
        bk, bv = self._room(layer, t, (batch, heads, 64), like, like)
        n, s = self._len[layer], bk.stride()
        if (bk.dtype != torch.float32 or bv.dtype != torch.float32 or bk.get_device() != like.get_device()
                or bv.get_device() != like.get_device() or bk.requires_grad or bv.requires_grad
                or bv.shape != bk.shape or bv.stride() != s or s[3] != 1 or min(s[:3]) < 64):
            return None
        return bk[:, :, n : n + t], bv[:, :, n : n + t]

    def _advance(self, layer: int, t: int) -> tuple[torch.Tensor, torch.Tensor]:
        n = self._len[layer] = self._len[layer] + t
        return self._k[layer][:, :, :n], self._v[layer][:, :, :n]

    def update(self, layer: int, k: torch.Tensor, v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """Append ``k, v`` ``(B, heads, T_new, head_dim)`` to ``layer``; return
        views of the whole history ``(B, heads, length, head_dim)``."""
        n, t = self._len[layer], k.shape[-2]
        buf_k, buf_v = self._room(layer, t, (*k.shape[:-2], k.shape[-1]), k, v)
        buf_k[:, :, n : n + t] = k
        buf_v[:, :, n : n + t] = v
        self._len[layer] = n + t
        return buf_k[:, :, : n + t], buf_v[:, :, : n + t]


def _causal_softmax_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int,
                              p_drop: float) -> torch.Tensor:
    """``softmax(q k^T / sqrt(hd) + mask) v`` for queries at absolute positions
    ``first .. first + T - 1`` over keys ``0 .. S - 1`` (``model.py:284-309``).

    Key ``j`` is visible to query ``i`` iff ``j <= first + i``; hidden scores
    are ``-inf``, so they get probability exactly 0. A query block that sees
    every key (one new token over the cache) needs no mask at all.
    """
    T, S = q.shape[-2], k.shape[-2]
    scores = torch.matmul(q, k.transpose(-2, -1)) / math.sqrt(q.shape[-1])
    if not (T == 1 and first + 1 == S):
        qpos = torch.arange(first, first + T, device=q.device).unsqueeze(1)
        kpos = torch.arange(S, device=q.device).unsqueeze(0)
        scores = scores.masked_fill(kpos > qpos, float("-inf"))
    probs = torch.softmax(scores, dim=-1)
    if p_drop:
        probs = F.dropout(probs, p_drop, training=True)
    return torch.matmul(probs, v)


def _fused_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int,
                     p_drop: float) -> torch.Tensor | None:
    """``_causal_softmax_attention`` as one HIP kernel (``tiq_prefill_attention``),
    its output as ``(B, T, heads * head_dim)`` rows, for fp32 GPU tensors with
    64-dim heads that need no gradient and no dropout; ``None`` otherwise. q, k
    and v are read in place through their strides (the projection's rows, a
    cache's buffers): no copies."""
    B, H, T, hd = q.shape
    ok = (q.is_cuda and hd == 64 and p_drop == 0.0 and k.shape[-2] == first + T
          and all(t.dtype == torch.float32 and t.stride(-1) == 1 for t in (q, k, v))
          and not (torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad)))
    if not ok:
        return None
    from . import _lib

    y = torch.empty(B, T, H * hd, device=q.device, dtype=torch.float32)
    rc = _lib.lib().tiq_prefill_attention(
        q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(), *v.stride()[:3], B, H, T, first, hd,
        y.data_ptr(), T * H * hd, hd, H * hd, _lib.stream_of(q))
    if rc in (_lib.EALIGN, _lib.EUNSUPPORTED):
        return None  # strides or sizes the kernel does not take: the torch ops below
    _lib.check(rc, "prefill attention")
    return y


def _as_is(module: nn.Module, cls: type) -> bool:
    """A plain ``cls`` without hooks, whose call may be replaced by a kernel that
    does the same."""
    return (type(module) is cls and "forward" not in module.__dict__ and not module._forward_hooks
            and not module._forward_pre_hooks and not module._backward_hooks and not module._backward_pre_hooks)


def _prefill_rows(x: torch.Tensor) -> bool:
    """Contiguous fp32 GPU rows that no gradient, tangent or global hook follows,
    as :meth:`QuantLinear.forward_prefill` takes them."""
    return (x.is_cuda and x.dtype is torch.float32 and x.dim() == 3 and x.numel() > 4 * x.shape[2]
            and x.is_contiguous() and not (torch.is_grad_enabled() and x.requires_grad)
            and torch.autograd.forward_ad._current_level < 0 and not nn.modules.module._has_any_global_hook())


def _plain_ln(ln: nn.Module, x: torch.Tensor) -> bool:
    """An nn.LayerNorm over the rows of ``x`` with fp32 parameters that no
    gradient follows."""
    if not _as_is(ln, nn.LayerNorm) or ln.normalized_shape != x.shape[2:]:
        return False
    w, b = ln.weight, ln.bias
    return (w is not None and b is not None and w.dtype is torch.float32 and b.dtype is torch.float32
            and w.get_device() == x.get_device() and b.get_device() == x.get_device() and w.is_contiguous()
            and b.is_contiguous() and not (torch.is_grad_enabled() and (w.requires_grad or b.requires_grad)))


def _head_logits(head: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``head(x)``; a plain bias-free fp32 ``nn.Linear`` over more than 64 rows that no
    gradient follows goes through ``tiq_linear_f32_ws``."""
    if _prefill_rows(x) and _as_is(head, nn.Linear) and head.bias is None:
        w = head.weight
        B, T, C = x.shape
        if (type(w) is nn.Parameter and w.dtype is torch.float32 and w.get_device() == x.get_device()
                and w.is_contiguous() and w.shape[1] == C and not (torch.is_grad_enabled() and w.requires_grad)
                and not torch.is_autocast_enabled("cuda")):
            from . import _lib

            L, M, N = _lib.lib(), B * T, w.shape[0]
            ws_bytes = L.tiq_linear_f32_workspace(M, C, N)
            if ws_bytes and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0:
                y = x.new_empty((B, T, N))
                ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
                _lib.check(L.tiq_linear_f32_ws(x.data_ptr(), M, C, C, w.data_ptr(), C, N, y.data_ptr(), N,
                                               ws.data_ptr(), ws_bytes, _lib.stream_of(x)), "lm_head over a batch")
                return y
    return head(x)


class CausalSelfAttention(nn.Module):
    """Fused ``c_attn`` (q, k, v side by side), heads of 64 columns, causal
    attention over the cache, ``c_proj``."""

    def __init__(self, config: GPTConfig, layer_idx: int = 0) -> None:
        super().__init__()
        self.config = config
        self.layer_idx = layer_idx
        self.n_head, self.head_dim, self.n_embd = config.n_head, config.head_dim, config.n_embd
        self.c_attn = nn.Linear(config.n_embd, 3 * config.n_embd, bias=config.attn_bias)
        self.c_proj = nn.Linear(config.n_embd, config.n_embd, bias=config.attn_bias)

    def forward(self, x: torch.Tensor, cache: KVCache | None = None) -> torch.Tensor:
        return self.c_proj(self._heads(x, cache))

    def _heads(self, x: torch.Tensor, cache: KVCache | None, ln: nn.LayerNorm | None = None) -> torch.Tensor | None:
        """The attention of (the LayerNorm of) ``x`` before ``c_proj``, ``(B, T, C)``
        rows. A quantized ``c_attn`` over a prompt applies ``ln`` itself and puts
        keys and values straight into the cache, which saves their copies (two
        of 10 us beside a 96 us product at 4096 rows of width 1600). With ``ln``:
        None, nothing done, where the product does not apply it."""
        B, T, C = x.shape
        first = 0 if cache is None else cache.length(self.layer_idx)
        qkv = None
        if (ln is not None or (cache is not None and _prefill_rows(x))) and _as_is(self.c_attn, QuantLinear):
            x2 = x.view(B * T, C)
            # (a cache of another class, or whose update a caller replaced, is filled through it)
            plain = type(cache) is KVCache and "update" not in cache.__dict__
            # (asked for few rows only: from 256 on no GPT-2 width's product is split, and a
            # refusal costs no more than the attempt)
            if (plain and self.head_dim == 64 and self.c_attn.out_features == 3 * 64 * self.n_head
                    and (B * T >= 256 or self.c_attn.writes_kv(B * T))):
                slots = cache._append_slots(self.layer_idx, B, self.n_head, T, x)
                q = None if slots is None else self.c_attn.forward_prefill(x2, ln=ln, kv=(*slots, T))
                if q is not None:
                    k, v = cache._advance(self.layer_idx, T)
                    return self._attend(q.view(B, T, self.n_head, 64).transpose(1, 2), k, v, first)
            if ln is not None:
                qkv = self.c_attn.forward_prefill(x2, ln=ln)
        if qkv is None:
            if ln is not None:
                return None
            qkv = self.c_attn(x)
        # (B, T, 3C) -> (3, B, heads, T, hd): q, k, v heads in one permute
        q, k, v = qkv.view(B, T, 3, self.n_head, self.head_dim).permute(2, 0, 3, 1, 4).unbind(0)
        if cache is not None:
            k, v = cache.update(self.layer_idx, k, v)
        return self._attend(q, k, v, first)

    def _attend(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
        p = self.config.dropout if self.training else 0.0
        y = _fused_attention(q, k, v, first, p)
        if y is None:
            y = _causal_softmax_attention(q, k, v, first, p).transpose(1, 2).flatten(2)
        return y


class MLP(nn.Module):
    """``c_proj(gelu_tanh(c_fc(x)))``, 4x expansion."""

    def __init__(self, config: GPTConfig) -> None:
        super().__init__()
        self.c_fc = nn.Linear(config.n_embd, 4 * config.n_embd, bias=config.mlp_bias)
        self.c_proj = nn.Linear(4 * config.n_embd, config.n_embd, bias=config.mlp_bias)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self._project(self.c_fc(x))

    def _project(self, h: torch.Tensor, residual: torch.Tensor | None = None) -> torch.Tensor:
        """``c_proj(gelu_tanh(h))``, plus ``residual``."""
        if _prefill_rows(h) and _as_is(self.c_proj, QuantLinear):
            y = self.c_proj.forward_prefill(h.view(-1, h.shape[2]), gelu=True, residual=residual)
            if y is not None:
                return y.view(*h.shape[:2], -1)
        fused = getattr(self.c_proj, "forward_gelu_in", None)  # a quantized c_proj over a prefill's rows
        y = fused(h) if fused is not None else None
        if y is None:
            y = self.c_proj(gelu_tanh(h))
        return y if residual is None else residual + y


class Block(nn.Module):
    """Pre-LN block: ``x + attn(ln_1(x))``, then ``x + mlp(ln_2(x))``."""

    def __init__(self, config: GPTConfig, layer_idx: int = 0) -> None:
        super().__init__()
        self.p_drop = config.dropout
        # construction order = registration order = the order of the RNG draws
        self.ln_1 = nn.LayerNorm(config.n_embd, eps=config.layer_norm_epsilon)
        self.attn = CausalSelfAttention(config, layer_idx=layer_idx)
        self.ln_2 = nn.LayerNorm(config.n_embd, eps=config.layer_norm_epsilon)
        self.mlp = MLP(config)

    def _drop(self, t: torch.Tensor) -> torch.Tensor:
        return F.dropout(t, self.p_drop, training=True) if self.training and self.p_drop else t

    def forward(self, x: torch.Tensor, cache: KVCache | None = None) -> torch.Tensor:
        y = self._prefill(x, cache)
        if y is not None:
            return y
        x = x + self._drop(self.attn(self.ln_1(x), cache))
        return x + self._drop(self.mlp(self.ln_2(x)))

    def _prefill(self, x: torch.Tensor, cache: KVCache | None) -> torch.Tensor | None:
        """The block over a prompt's rows with quantized Linears: both
        LayerNorms inside the Linear that follows, both residual adds at the end
        of the Linear before (four passes over x fewer; each step that a Linear
        does not take runs as its own op). None, nothing done, where the block
        has to run module by module: hooks, replaced modules, a gradient,
        dropout, rows that ``c_attn`` does not take as digit planes."""
        attn, mlp = self.attn, self.mlp
        if not (_prefill_rows(x) and _as_is(attn.c_attn, QuantLinear) and _as_is(attn.c_proj, QuantLinear)
                and _as_is(mlp.c_fc, QuantLinear) and _as_is(mlp.c_proj, QuantLinear)
                and _as_is(attn, CausalSelfAttention) and _as_is(mlp, MLP)
                and _plain_ln(self.ln_1, x) and _plain_ln(self.ln_2, x)
                and not (self.training and (self.p_drop or attn.config.dropout))):
            return None
        B, T, C = x.shape
        heads = attn._heads(x, cache, self.ln_1)
        if heads is None:
            return None
        y = attn.c_proj.forward_prefill(heads.view(B * T, -1), residual=x)
        x = x + attn.c_proj(heads) if y is None else y.view(B, T, C)
        h = mlp.c_fc.forward_prefill(x.view(B * T, C), ln=self.ln_2)
        h = mlp.c_fc(self.ln_2(x)) if h is None else h.view(B, T, -1)
        return mlp._project(h, x)


def _refuse_unsupported(config: GPTConfig) -> None:
    """The layouts of the quantized path only: GPT-2 as released."""
    unsupported = {
        "norm_position": (config.norm_position, "pre"),
        "pos_embedding": (config.pos_embedding, "learned"),
        "activation": (config.activation, "gelu_tanh"),
        "n_kv_head": (config.kv_heads, config.n_head),
        "use_sdpa": (config.use_sdpa, False),
    }
    for field, (got, want) in unsupported.items():
        if got != want:
            raise NotImplementedError(
                f"{field}={got!r}: this model implements GPT-2's inference layout only ({field}={want!r})")


class GPT(nn.Module):
    """GPT-2 with a tied head (``lm_head.weight is wte.weight``)."""

    def __init__(self, config: GPTConfig) -> None:
        super().__init__()
        _refuse_unsupported(config)
        if not config.tie_weights:
            raise NotImplementedError("tie_weights=False: GPT-2's head is the embedding matrix")
        self.config = config
        self.wte = nn.Embedding(config.vocab_size, config.n_embd)
        self.wpe = nn.Embedding(config.n_positions, config.n_embd)
        self.h = nn.ModuleList(Block(config, layer_idx=i) for i in range(config.n_layer))
        self.ln_f = nn.LayerNorm(config.n_embd, eps=config.layer_norm_epsilon)
        self.lm_head = nn.Linear(config.n_embd, config.vocab_size, bias=False)
        self.lm_head.weight = self.wte.weight
        self._seeded_init()

    @torch.no_grad()
    def _seeded_init(self) -> None:
        """GPT-2's initialisation, drawn in the reference's order.

        Every Linear and Embedding weight ~ N(0, 0.02), biases 0, LayerNorm
        scale 1 and shift 0, visiting the leaf modules in registration order
        (so the tied ``lm_head``, last, redraws the embedding); then the two
        residual-writing projections of each block are redrawn with
        ``std = 0.02 / sqrt(2 * n_layer)``, attention's before the MLP's. With
        the construction draws of the ``nn`` modules before it, this sequence
        reproduces the reference's seed-0 weights bit for bit
        (``model.py:457-518``).
        """
        for mod in self.modules():
            if isinstance(mod, (nn.Linear, nn.Embedding)):
                mod.weight.normal_(0.0, 0.02)
                if getattr(mod, "bias", None) is not None:
                    mod.bias.zero_()
            elif isinstance(mod, nn.LayerNorm):
                mod.weight.fill_(1.0)
                mod.bias.zero_()
        if self.config.residual_scaled_init:
            std = 0.02 / math.sqrt(2 * self.config.n_layer)
            for block in self.h:
                block.attn.c_proj.weight.normal_(0.0, std)
                block.mlp.c_proj.weight.normal_(0.0, std)

    def position_embeddings(self, pos: torch.Tensor) -> torch.Tensor:
        return self.wpe(pos)

    def forward(
        self,
        idx: torch.Tensor,
        targets: torch.Tensor | None = None,
        cache: KVCache | None = None,
        last_only: bool = False,
    ) -> dict[str, Any]:
        """Logits ``(B, T, vocab)`` of ``idx`` ``(B, T)`` (``model.py:528-599``).

        With a ``cache``, ``idx`` holds only the new tokens, placed after the
        cached ones. ``targets`` adds the mean cross entropy (``-100``
        ignored) as ``loss``. ``last_only`` returns the last position's logits
        ``(B, 1, vocab)`` only -- all a prefill needs, and the head is the
        largest product of a long prompt.
        """
        T = idx.shape[1]
        first = 0 if cache is None else cache.seq_len
        if first + T > self.config.n_positions:
            raise ValueError(
                f"sequence of length {first + T} exceeds n_positions={self.config.n_positions}; "
                f"learned position embeddings cannot extrapolate"
            )
        if last_only and targets is not None:
            raise ValueError("last_only computes no loss: the loss needs every position's logits")
        pos = torch.arange(first, first + T, device=idx.device)
        x = self.wte(idx) + self.wpe(pos)
        if self.training and self.config.dropout:
            x = F.dropout(x, self.config.dropout, training=True)
        for block in self.h:
            x = block(x, cache)
        if last_only:
            x = x[:, -1:]
        logits = _head_logits(self.lm_head, self.ln_f(x))
        out: dict[str, Any] = {"logits": logits}
        if targets is not None:
            out["loss"] = F.cross_entropy(logits.flatten(0, 1), targets.reshape(-1), ignore_index=-100)
        return out
