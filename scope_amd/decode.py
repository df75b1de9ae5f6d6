"""Token-loop decoding of the 16-layer SCOPE decoder on one MI355X.

The model mirrors ``GPT`` of scoped_medium.py:266-639 — token and value
embeddings (the 012 ... 012 pattern, :592), per block ``lambdas`` mixing with
x0, QK-norm, half-truncated rotary, value-embedding mix, ReLU² MLP, the
U-net skip connections with ``skip_weights``, no attention in block 7
(:499), and the soft-capped logits ``30·σ(logits/7.5)`` (:618) over the
vocabulary padded to a multiple of 128 (:529).  Every attention layer is a
SCOPE layer with the block-scoring pointer mask (window W, budget B, G
document-start globals) and no spectral bias.  Weights are random (the
reference zero-initialises its output projections and lm_head, which would
make greedy decoding trivial).

* ``prefill(tokens)``: one forward over the prompt (T a multiple of the
  block size) with the block-sparse attention kernel; fills every layer's KV
  cache and key-block means.
* ``step(token)``: one new position t.  When t opens a q-block, every layer
  reselects that block's list over its cache (the query block mean is the
  new token's query, the only one known), and keeps it for the block's other
  positions; the attention of the token runs ``scope_decode_attn`` over the
  list.  When t closes a block, its key mean joins the candidates.
* At the default width a step that opens no block runs every layer in one
  launch (``ops.decoder_step``); other configurations take a chain of fused
  kernels per layer.
* The steps inside a block (neither opening nor closing it) run as one
  captured HIP graph (``torch.cuda.CUDAGraph``), replayed per token: the
  position lives on the device (``_t_dev``; cache and document writes index
  with it, ``scope_decode_attn_at`` reads it), the lists sit in fixed
  per-layer buffers that a reselection refills, so every replay sees the
  current state.  The eager steps run the same operations, so both paths
  give the same logits.

The reference has no decode path; this is the row of the scope table that
puts the hot-path kernels under a token loop.
"""
from __future__ import annotations

import math
import operator
import threading
from dataclasses import dataclass

import torch
import torch.nn.functional as F
from torch import nn

from . import ops

EOT = 50256

# Held while a step's launches are enqueued (a graph's as well as single ones):
# the launch that takes the step lock and the step behind it come in a row also
# where the streams of two threads share a hardware queue.  A lock waited for in
# front of its holder's step would be waited for until its limit.
_ENQUEUE = threading.Lock()


@dataclass
class DecoderConfig:
    vocab_size: int = 50257
    num_layers: int = 16
    num_heads: int = 8
    model_dim: int = 1024
    head_dim: int = 128
    block_size: int = 128
    window: int = 4
    budget: int = 4
    n_global: int = 1
    attn_scale: float = 0.12
    no_attn_layer: int = 7

    @property
    def vocab_padded(self) -> int:
        return ((self.vocab_size + 127) // 128) * 128


def _norm(x: torch.Tensor) -> torch.Tensor:
    return F.rms_norm(x, (x.size(-1),))


def _mix(a: float, b: float, x: torch.Tensor, x0: torch.Tensor) -> torch.Tensor:
    """a·x + b·x0 (scoped_medium.py:505); a = 1, b = 0 is x itself, exactly."""
    return x if (a == 1.0 and b == 0.0) else a * x + b * x0


def _skip(x: torch.Tensor, w: float, s: torch.Tensor) -> torch.Tensor:
    """x + w·s (scoped_medium.py:607); w = 1 is a plain sum, exactly."""
    return x + s if w == 1.0 else x + w * s


_CFG_NUMBERS = operator.attrgetter("attn_scale", "block_size", "num_layers", "num_heads", "head_dim", "model_dim",
                                   "vocab_size", "window", "budget", "n_global")


class _StepInputs:
    """What a step inside a block reaches by address or bakes in, at one moment:
    its tensors (kept alive here) and its numbers.  ``same`` compares with the
    decoder's state now: a replaced tensor, one with other memory, and
    (``layout``) one with other strides."""

    def __init__(self, dec: "ScopeDecoder"):
        self.tensors, self.numbers = self._of(dec)
        self.addresses = list(map(torch.Tensor.data_ptr, self.tensors))
        self.strides = list(map(torch.Tensor.stride, self.tensors))

    @staticmethod
    def _of(dec):
        ts = [t for lay in dec.layers for n in ("qkv", "proj", "mlp_fc", "mlp_proj") if (t := lay.get(n)) is not None]
        for per_layer in (dec.k_cache, dec.v_cache, dec.list_num, dec.list_idx):
            ts += [t for t in per_layer if t is not None]
        ts += dec.value_embeds
        ts += [dec.embed, dec.lm_head, dec.rotary.cos, dec.rotary.sin, dec.docs, dec.tokens, dec._t_dev, dec._ws]
        return ts, (_CFG_NUMBERS(dec.cfg), tuple(dec.skip_weights),
                    [(tuple(lay["lambdas"]), tuple(lay.get("vlam", ())), "qkv" in lay) for lay in dec.layers])

    def same(self, dec, layout: bool = True) -> bool:
        ts, numbers = self._of(dec)
        return (numbers == self.numbers and len(ts) == len(self.tensors)
                and all(map(operator.is_, ts, self.tensors))
                and list(map(torch.Tensor.data_ptr, ts)) == self.addresses
                and (not layout or list(map(torch.Tensor.stride, ts)) == self.strides))


class _Rotary:
    """Half-truncated RoPE tables (scoped_medium.py:282-299)."""

    def __init__(self, dim: int, max_len: int, device):
        freq = (1 / 1024) ** torch.linspace(0, 1, steps=dim // 4, dtype=torch.float32)
        freq = torch.cat([freq, freq.new_zeros(dim // 4)])
        theta = torch.arange(max_len, dtype=torch.float32)[:, None] * freq[None]
        self.cos, self.sin = theta.cos().to(device), theta.sin().to(device)

    def __call__(self, x: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
        """x [T, H, D] at positions pos [T]."""
        cos, sin = self.cos[pos][:, None, :], self.sin[pos][:, None, :]
        x1, x2 = x.float().chunk(2, dim=-1)
        return torch.cat((x1 * cos + x2 * sin, x1 * (-sin) + x2 * cos), -1).type_as(x)


class ScopeDecoder(nn.Module):
    def __init__(self, cfg: DecoderConfig, *, max_len: int, device="cuda", seed: int = 0, use_graph: bool = True):
        super().__init__()
        self.cfg = cfg
        g = torch.Generator(device="cpu").manual_seed(seed)
        d, H, D, L = cfg.model_dim, cfg.num_heads, cfg.head_dim, cfg.num_layers
        hd = H * D

        def uni(*shape, fan_in):
            b = math.sqrt(3.0) * 0.5 * fan_in ** -0.5  # CastedLinear / qkv init bound (:270-274, :305-306)
            return ((torch.rand(shape, generator=g) * 2 - 1) * b).to(torch.bfloat16).to(device)

        self.embed = (torch.randn((cfg.vocab_size, d), generator=g)).to(torch.bfloat16).to(device)
        self.value_embeds = [torch.randn((cfg.vocab_size, d), generator=g).to(torch.bfloat16).to(device)
                             for _ in range(3)]
        self.layers = []
        for i in range(L):
            lay = dict(lambdas=(1.0, 0.0), mlp_fc=uni(4 * d, d, fan_in=d), mlp_proj=uni(d, 4 * d, fan_in=4 * d))
            if i != cfg.no_attn_layer:
                lay.update(qkv=uni(3 * hd, d, fan_in=d), proj=uni(d, hd, fan_in=hd), vlam=(0.5, 0.5))
            self.layers.append(lay)
        self.skip_weights = [1.0] * (L // 2)
        self.lm_head = uni(cfg.vocab_padded, d, fan_in=d)
        self.rotary = _Rotary(D, max_len, device)
        self.device = torch.device(device)
        self.max_len = max_len
        # caches
        nbc = max_len // cfg.block_size
        z = dict(dtype=torch.bfloat16, device=device)
        self.k_cache = [torch.zeros((H, max_len, D), **z) if "qkv" in lay else None for lay in self.layers]
        self.v_cache = [torch.zeros((H, max_len, D), **z) if "qkv" in lay else None for lay in self.layers]
        self.kbar = [torch.zeros((H, nbc, D), dtype=torch.float32, device=device) if "qkv" in lay else None
                     for lay in self.layers]
        # current q-block's list per layer, in fixed buffers of the full width
        # (window + budget + globals) that each reselection refills
        width = cfg.window + cfg.budget + cfg.n_global
        self.list_num = [torch.zeros(H, dtype=torch.int32, device=device) if "qkv" in lay else None
                         for lay in self.layers]
        self.list_idx = [torch.zeros((H, width), dtype=torch.int32, device=device) if "qkv" in lay else None
                         for lay in self.layers]
        self.have_lists = False
        # a dict here makes every reselection record, per attention layer, the
        # query row it chose from, its logits and its lists (eager steps only)
        self.record: dict | None = None
        self.docs = torch.zeros(max_len, dtype=torch.int32, device=device)
        self.tokens = torch.zeros(max_len, dtype=torch.int64, device=device)
        self.t = 0
        self._t_dev = torch.zeros(1, dtype=torch.int64, device=device)  # = t, on the device
        self._ws = torch.empty(H * width * (D + 2) * 4, dtype=torch.uint8, device=device)
        self.use_graph = bool(use_graph) and self.device.type == "cuda"
        self._graph = None
        self._g_inputs: _StepInputs | None = None  # what it was captured with
        self._g_tok = None
        self._g_out = None
        self._g_warm = 0
        # the one-launch step (``_fused``): the table of the layers' tensors, what
        # it was made from, and the status its waits set (pinned)
        self._step_inputs: _StepInputs | None = None
        self._step_table = None
        self._step_status = None

    # ---- pieces shared by prefill and step -------------------------------------
    def _ve(self, tok: torch.Tensor):
        ve = [F.embedding(tok, w) for w in self.value_embeds]
        L = self.cfg.num_layers
        return [ve[0], ve[1], ve[2]] + [None] * (L - 6) + [ve[0], ve[1], ve[2]]

    def _qkv(self, lay, x: torch.Tensor, ve, pos: torch.Tensor, i: int | None = None):
        """x [T, d] (normed) -> q [T, H, D] (normed and rotated) and k, v: with
        a layer index i, k and v go to rows pos of that layer's caches (which
        are returned); otherwise they are new [T, H, D] tensors.  The glue runs
        as one kernel (``ops.decoder_qkv_glue``)."""
        cfg = self.cfg
        qkv = F.linear(x, lay["qkv"])
        a, b = lay["vlam"]
        kc = self.k_cache[i] if i is not None else None
        vc = self.v_cache[i] if i is not None else None
        return ops.decoder_qkv_glue(qkv, ve, pos, self.rotary.cos, self.rotary.sin, heads=cfg.num_heads, va=a,
                                    vb=b if ve is not None else 0.0, k_out=kc, v_out=vc)

    def _logits(self, x: torch.Tensor) -> torch.Tensor:
        return 30 * torch.sigmoid(F.linear(_norm(x), self.lm_head).float() / 7.5)

    def _select(self, qbar: torch.Tensor, kbar: torch.Tensor, nb: int, return_logits: bool = False, ds=None):
        """Block-scoring lists of blocks 0..nb-1 from q̄, k̄ [H, nb, D]; ``ds``:
        their document starts, when the caller has them."""
        cfg = self.cfg
        T = nb * cfg.block_size
        ds_ptr, ds_local, _ = ds or ops.doc_starts(self.docs[:T], cfg.block_size)
        return ops.pointer_select(ds_ptr, ds_local, bs=cfg.block_size, NB=nb, H=cfg.num_heads, window=cfg.window,
                                  n_global=cfg.n_global, budget=cfg.budget, qbar=qbar, kbar=kbar, temp=1.0,
                                  logit_scale=cfg.block_size / math.sqrt(cfg.head_dim), noise="none",
                                  return_logits=return_logits)

    # ---- prefill ---------------------------------------------------------------
    @torch.no_grad()
    def prefill(self, tokens: torch.Tensor, *, all_logits: bool = False) -> torch.Tensor:
        """Forward over the prompt; returns the logits of the last position
        (or of every position with ``all_logits``)."""
        cfg = self.cfg
        T = tokens.numel()
        bs = cfg.block_size
        if T % bs or T > self.max_len:
            raise ValueError(f"prefill: T={T} must be a multiple of {bs} and at most {self.max_len}")
        if self._step_status is not None and int(self._step_status[0]):
            # a wait of an earlier one-launch step expired: its workspace and the
            # graph that uses it are left behind, once nothing runs on them
            torch.cuda.synchronize(self.device)
            self._graph = self._g_table = self._step_inputs = self._step_table = self._step_status = None
        tok = tokens.to(self.device).long()
        self.tokens[:T] = tok
        self.docs[:T] = (tok == EOT).cumsum(0).to(torch.int32)
        docs = self.docs[:T]
        ds = ops.doc_starts(docs, bs)
        pos = torch.arange(T, device=self.device)
        ve = self._ve(tok)
        x = x0 = _norm(F.embedding(tok, self.embed))
        skips: list = []
        n, L = len(self.skip_weights), len(self.layers)
        # with the model's initial mixing weights the residual adds, the U-net
        # skips and the norms between the products run as one pass each
        plain = all(w == 1.0 for w in self.skip_weights) and L == 2 * n and cfg.model_dim % 8 == 0 \
            and cfg.model_dim <= 4096 and all(lay["lambdas"] == (1.0, 0.0) for lay in self.layers)
        xn = _norm(x)
        for i, lay in enumerate(self.layers):
            if not plain:
                if i >= n:
                    x = _skip(x, self.skip_weights[i - n], skips.pop())
                a, b = lay["lambdas"]
                x = _mix(a, b, x, x0)
                xn = _norm(x)
            if "qkv" in lay:
                q, kc, vc = self._qkv(lay, xn, ve[i], pos, i)  # k, v into cache rows 0 .. T-1
                qh, kh, vh = q.transpose(0, 1), kc[:, :T], vc[:, :T]  # [H, T, D] views
                qbar, kbar = ops.block_means(qh, kh, bs)
                self.kbar[i][:, :T // bs] = kbar
                kv_num, kv_idx, _ = self._select(qbar, kbar, T // bs, ds=ds)
                y, _ = ops.attn_fwd(qh[None], kh[None], vh[None], kv_num, kv_idx, docs, ds[2], bs=bs,
                                    scale=cfg.attn_scale, check=False)
                y = F.linear(y[0].transpose(0, 1).reshape(T, -1), lay["proj"])
                if plain:
                    x, xn = ops.decoder_add_norm(x, y)
                else:
                    x = x + y
                    xn = _norm(x)
            y = F.linear(ops.decoder_relu2(F.linear(xn, lay["mlp_fc"])), lay["mlp_proj"])
            if not plain:
                x = x + y
                if i < n:
                    skips.append(x)
            elif i == L - 1:
                x = x + y
            elif i == n - 1:  # layer n takes this layer's own output as its skip
                x, xn = ops.decoder_add_norm(x, y, skip_self=True)
            else:
                x, xn = ops.decoder_add_norm(x, y, skip=skips.pop() if i >= n else None)
                if i < n:
                    skips.append(x)
        self.t = T
        self._t_dev.fill_(T)
        self.have_lists = False
        return self._logits(x) if all_logits else self._logits(x[-1:])[0]

    # ---- one decode step ---------------------------------------------------------
    def _fused(self):
        """The arguments of ``ops.decoder_step`` (table of the layers' current
        tensors, workspace), or None when a step has to run layer by layer:
        other sizes than the library serves, mixing weights other than the
        model's initial ones, or a device too small for it."""
        cfg, n = self.cfg, len(self.skip_weights)
        if self.device.type != "cuda" or any(w != 1.0 for w in self.skip_weights) \
                or any(lay["lambdas"] != (1.0, 0.0) for lay in self.layers) or len(self.layers) != 2 * n:
            return None
        if self._step_inputs is None or not self._step_inputs.same(self):
            if self._step_table is not None:  # left behind once no step runs on it, on whatever stream
                torch.cuda.synchronize(self.device)
            ve = [0, 1, 2] + [-1] * (cfg.num_layers - 6) + [0, 1, 2]
            layers = []
            for i, lay in enumerate(self.layers):
                va, vb = lay.get("vlam", (0.0, 0.0))
                layers.append(dict(qkv=lay.get("qkv"), proj=lay.get("proj"), mlp_fc=lay["mlp_fc"],
                                   mlp_proj=lay["mlp_proj"], k_cache=self.k_cache[i], v_cache=self.v_cache[i],
                                   kv_num=self.list_num[i], kv_idx=self.list_idx[i], ve=ve[i], va=va, vb=vb))
            cache, vcache = (next((c for c in cs if c is not None), None) for cs in (self.k_cache, self.v_cache))
            self._step_table = None
            if cache is not None and vcache is not None and cfg.num_layers >= 6:
                self._step_table = ops.decoder_step_table(layers, dict(
                    layers=cfg.num_layers, H=cfg.num_heads, D=cfg.head_dim, dm=cfg.model_dim, mlp=4 * cfg.model_dim,
                    bs=cfg.block_size, maxkv=cfg.window + cfg.budget + cfg.n_global, scale=cfg.attn_scale,
                    eps=torch.finfo(torch.float32).eps, T_cap=self.max_len, vocab=cfg.vocab_size, eot=EOT,
                    rot_rows=self.rotary.cos.shape[0], rot_st=self.rotary.cos.stride(0), k_sh=cache.stride(0),
                    k_st=cache.stride(1), v_sh=vcache.stride(0), v_st=vcache.stride(1),
                    spin_ticks=20 * 100_000_000, gang_ticks=50_000), cache.device)  # 20 s; 0.5 ms, about a step
            if self._step_status is None:
                self._step_status = torch.zeros(1, dtype=torch.int32, pin_memory=True)
            self._step_inputs = _StepInputs(self)
        return self._step_table

    def _body(self, tok: torch.Tensor, t: int, opens: bool, closes: bool) -> torch.Tensor:
        """The step at the position held in ``_t_dev`` (= t), then _t_dev += 1.
        ``opens`` / ``closes`` (eager steps only) add the block's reselection /
        its key-mean update; with both false the body is graph-capturable."""
        cfg = self.cfg
        bs = cfg.block_size
        td = self._t_dev
        fused = None if opens else self._fused()
        if fused is not None:
            with _ENQUEUE:
                x = ops.decoder_step(*fused, tok, td, self.tokens, self.docs, self.embed, self.value_embeds,
                                     self.rotary.cos, self.rotary.sin, self._step_status)
            if closes:  # the block is complete: its key means join the candidates
                for kbar, kc in zip(self.kbar, self.k_cache):
                    if kbar is not None:
                        kbar[:, t // bs] = kc[:, t // bs * bs:t + 1].float().mean(dim=1)
            return ops.decoder_gemv(x, self.lm_head, norm=True, epi="logit")
        # token and document bookkeeping, the embedding, its norm and the
        # value embeddings in one kernel
        x0, ve3 = ops.decoder_step_prologue(tok, td, self.tokens, self.docs, self.embed, self.value_embeds, eot=EOT)
        qb = t // bs
        if opens:  # positions of the new block not yet written carry the current document
            self.docs[t + 1:(qb + 1) * bs] = self.docs[t]
        v0, v1, v2 = ve3[0:1], ve3[1:2], ve3[2:3]
        ve = [v0, v1, v2] + [None] * (cfg.num_layers - 6) + [v0, v1, v2]
        x = x0
        skips = []
        n = len(self.skip_weights)
        H, D = cfg.num_heads, cfg.head_dim
        gemv = ops.decoder_gemv
        for i, lay in enumerate(self.layers):
            # the row-vector products run fused with their norms, activations
            # and residual adds (ops.decoder_gemv); the U-net skip (weight 1)
            # joins the next normed product
            skip = None
            a, b = lay["lambdas"]
            if i >= n:
                if self.skip_weights[i - n] == 1.0 and "qkv" in lay and (a, b) == (1.0, 0.0):
                    skip = skips.pop()
                else:
                    x = _skip(x, self.skip_weights[i - n], skips.pop())
            x = _mix(a, b, x, x0)
            if "qkv" in lay:
                if skip is not None:
                    qkv, x = gemv(x, lay["qkv"], norm=True, addx=skip)
                else:
                    qkv = gemv(x, lay["qkv"], norm=True)
                va, vb = lay["vlam"]
                vb = vb if ve[i] is not None else 0.0
                if opens:
                    # the block's lists are chosen from this token's q: the glue
                    # (k, v into cache row t), the reselection, then the attention
                    q, _, _ = ops.decoder_qkv_glue(qkv[None], ve[i], td, self.rotary.cos, self.rotary.sin, heads=H,
                                                   va=va, vb=vb, k_out=self.k_cache[i], v_out=self.v_cache[i])
                    nb = qb + 1
                    qbar = torch.zeros((H, nb, D), dtype=torch.float32, device=self.device)
                    qbar[:, qb] = q[0].float()
                    if self.record is None:
                        kv_num, kv_idx, _ = self._select(qbar, self.kbar[i][:, :nb].contiguous(), nb)
                    else:
                        kv_num, kv_idx, _, lg = self._select(qbar, self.kbar[i][:, :nb].contiguous(), nb,
                                                             return_logits=True)
                        self.record[i] = dict(q=qbar[:, qb].clone(), logits=lg.clone(), kv_num=kv_num.clone(),
                                              kv_idx=kv_idx.clone())
                    self.list_num[i].copy_(kv_num[:, qb])
                    self.list_idx[i].zero_()
                    self.list_idx[i][:, :kv_idx.shape[-1]].copy_(kv_idx[:, qb])
                    y, _ = ops.decode_attn(q[0], self.k_cache[i], self.v_cache[i], self.list_num[i], self.list_idx[i],
                                           self.docs, td, bs=bs, scale=cfg.attn_scale, workspace=self._ws, check=False)
                else:
                    # lists fixed within the block: the glue runs inside the attention
                    # (k, v into cache row t there)
                    y, _, _ = ops.decode_attn_glue(qkv, ve[i], td, self.rotary.cos, self.rotary.sin, self.k_cache[i],
                                                   self.v_cache[i], self.list_num[i], self.list_idx[i], self.docs,
                                                   heads=H, va=va, vb=vb, bs=bs, scale=cfg.attn_scale,
                                                   workspace=self._ws, check=False)
                x = gemv(y.reshape(H * D), lay["proj"], epi="resid", res=x)
                if closes:  # the block is complete: its key mean joins the candidates
                    self.kbar[i][:, qb] = self.k_cache[i][:, qb * bs:(qb + 1) * bs].float().mean(dim=1)
            h2 = gemv(x, lay["mlp_fc"], norm=True, epi="relu2")
            x = gemv(h2, lay["mlp_proj"], epi="resid", res=x)
            if i < n:
                skips.append(x)
        logits = gemv(x, self.lm_head, norm=True, epi="logit")
        td.add_(1)
        return logits

    def _check_waits(self, who: str) -> None:
        """Raises if a wait inside a one-launch step that has run expired."""
        if self._step_status is not None and int(self._step_status[0]):
            raise RuntimeError(f"{who}: an earlier step's workgroups waited too long for each other; its logits are NaN")

    @torch.no_grad()
    def step(self, token: int | torch.Tensor) -> torch.Tensor:
        """Append one token at position t; returns its logits [vocab_padded]
        (all NaN where a wait inside the one-launch step expired; the next call
        raises then).  It does not wait for the GPU."""
        bs = self.cfg.block_size
        t = self.t
        if t >= self.max_len:
            raise ValueError("step: the cache is full")
        self._check_waits("step")
        if not isinstance(token, torch.Tensor) or not token.is_cuda:  # a host token is checked here
            if not 0 <= int(token) < self.cfg.vocab_size:
                raise ValueError(f"step: token {int(token)} outside the vocabulary [0, {self.cfg.vocab_size})")
        tok = torch.as_tensor(token, device=self.device).reshape(1).long()
        opens = t % bs == 0 or not self.have_lists
        closes = t % bs == bs - 1
        if self.use_graph and not opens and not closes:
            out = self._graph_step(tok, t)
        else:
            out = self._body(tok, t, opens, closes)
            self.have_lists = True
        self.t = t + 1
        return out

    def _graph_step(self, tok: torch.Tensor, t: int) -> torch.Tensor:
        """A step inside a block: one eager run of the body first (library
        warm-up), then a capture; every later such step replays the graph, which
        is captured anew when what it reaches has been replaced."""
        if self._graph is not None and not self._g_inputs.same(self, layout=False):
            torch.cuda.synchronize(self.device)  # no replay of the old graph is running
            self._graph = None
        if self._graph is None and self._g_warm == 0:
            self._g_warm = 1
            self._fused()  # its table and workspace belong to the caller's stream, not to the side stream
            side = torch.cuda.Stream(self.device)
            side.wait_stream(torch.cuda.current_stream(self.device))
            with torch.cuda.stream(side):
                out = self._body(tok, t, False, False)
            torch.cuda.current_stream(self.device).wait_stream(side)
            return out
        if self._graph is None:
            self._g_tok = tok.clone()
            self._g_table = self._fused()  # made outside the capture, alive as long as the graph
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                self._g_out = self._body(self._g_tok, -1, False, False)
            self._graph = g  # the capture ran nothing: replay for this token below
            self._g_inputs = _StepInputs(self)
        else:
            self._g_tok.copy_(tok)
        with _ENQUEUE:
            self._graph.replay()
        return self._g_out.clone()

    @torch.no_grad()
    def generate(self, n_steps: int, first: int | torch.Tensor) -> torch.Tensor:
        """Greedy decoding: feeds ``first``, then each argmax, for n_steps.
        With the one-launch step it returns when the tokens are there: a step
        whose waits expired has no other step after it to say so."""
        out = torch.empty(n_steps, dtype=torch.int64, device=self.device)
        tok = torch.as_tensor(first, device=self.device)
        for s in range(n_steps):
            logits = self.step(tok)
            tok = ops.argmax(logits[:self.cfg.vocab_size], out=out[s:s + 1])  # written in place
        if self._step_status is not None:
            torch.cuda.current_stream(self.device).synchronize()
            self._check_waits("generate")
        return out
