"""LAPrune decode attention inside a transformers Llama model.

Mirrors the reference's model plumbing for the decode path:
  * ``Decoder`` (laprune/llm/modifiers/aq_evaluation.py:496-540) patches
    every attention layer; layers in ``apply_layers`` are LAPrune layers, the
    rest stay dense;
  * ``self_attn_forward`` (:279-322): q/k/v projections, RoPE, append to the
    layer's K/V cache, encode new keys (prefill: all of them; decode: in
    64-token groups), causal SDPA at prefill, sparse retrieval at decode;
  * ``AQGeneration.generate`` (aq_generation.py:114-151): prefill all prompt
    tokens but the last, then greedy decode one token at a time.

Each layer owns a :class:`~laprune_amd.cache.DecodeKVCache`; LAPrune layers
decode through :class:`~laprune_amd.retrieval.SparseDecoder` (LUT -> fused
score -> top-k -> sparse attention, all HIP), dense layers through
:class:`~laprune_amd.retrieval.DenseDecoder`.  Sequences of one batch may have
different lengths (ragged): prefill them one row at a time with
:meth:`LAPruneLlama.prefill_row`, then decode the batch together.

The model is a plain ``transformers`` ``LlamaForCausalLM``; nothing here
downloads anything (build it from a local ``LlamaConfig``).
"""
from __future__ import annotations

import functools
import math
from dataclasses import dataclass, field
from types import MethodType

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.nn.attention import SDPBackend, sdpa_kernel

from ._ops import ops
from .cache import DecodeKVCache
from .retrieval import DenseDecoder, RetrievalConfig, SparseDecoder, check_step_health


# looked up once: every wrapped call of an eager step asks them
_compiling, _grad_on = torch.compiler.is_compiling, torch.is_grad_enabled
_transforms, _modes = torch._C._functorch.peek_interpreter_stack, torch._C._len_torch_dispatch_stack
_trace = torch._C._get_tracing_state


def _unwatched() -> bool:
    """Whether the calling ops only have to compute: no compiler, gradient, function
    transform (vmap, jvp), forward-mode level, dispatch mode (fake tensors, op
    counters) or trace looks at them, all of which a kernel call would pass by."""
    return not (_compiling() or _grad_on() or forward_ad._current_level >= 0 or
                _transforms() is not None or _modes() or _trace() is not None)


def _plain_tensor(x: torch.Tensor) -> bool:
    """A tensor of no other class, contiguous and aligned to 16 bytes."""
    return (type(x) in (torch.Tensor, torch.nn.Parameter) and x.is_contiguous() and
            x.data_ptr() % 16 == 0)


def _one_token(x: torch.Tensor) -> bool:
    """Whether x [B, 1, n] is a decode step's activation that the fused
    element-wise kernels serve; anything else keeps the model's own code."""
    return (_unwatched() and x.dim() == 3 and x.shape[1] == 1 and x.numel() > 0 and x.is_cuda and
            x.dtype in (torch.bfloat16, torch.float16) and _plain_tensor(x))


def _weight_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the projection kernel serves weight w with the tokens of x, and faster
    than the library: many short rows are the library's (us in a captured loop,
    library / kernel, bf16: 14336 x 64 4.4 / 4.6, 32000 x 256 8.2 / 8.7, 151936 x 384
    34.3 / 35.4; 8192 x 64 4.2 / 3.2, and from 512 columns on the kernel at every
    height)."""
    return (w.dim() == 2 and w.dtype == x.dtype and w.device == x.device and
            x.shape[-1] == w.shape[1] and w.shape[1] % 8 == 0 and w.numel() > 0 and
            _plain_tensor(w) and (w.shape[1] >= 512 or w.shape[0] <= 8192) and
            not torch.is_autocast_enabled(x.device.type))


def _one_vector(x: torch.Tensor, w: torch.Tensor, b=None) -> bool:
    """Whether x is one token for the projection kernel with weight w."""
    return b is None and _one_token(x) and x.numel() == x.shape[-1] and _weight_fits(x, w)


def _linear(x: torch.Tensor, w: torch.Tensor, b=None) -> torch.Tensor:
    """F.linear; one token of one sequence goes to the projection kernel."""
    if _one_vector(x, w, b):
        out = x.new_empty((1, 1, w.shape[0]))
        ops().gemv(x, w, out)
        return out
    return F.linear(x, w, b)


def _own_forward(mod) -> bool:
    """Whether mod runs its class's forward (unpickled modules hold it bound) or the
    one bound to it here, and not a replacement (one that wraps either included)."""
    f = mod.__dict__.get("forward")
    return f is None or (isinstance(f, MethodType) and f.__self__ is mod and
                         (f.__func__ in _DECODE_FORWARDS or f.__func__ is type(mod).forward))


def _unhooked(mod) -> bool:
    """Whether a call of mod is its class's forward and no more: the fused MLP
    leaves such a call out."""
    g = torch.nn.modules.module
    return (_own_forward(mod) and
            not (mod._forward_hooks or mod._forward_pre_hooks or mod._backward_hooks or
                 mod._backward_pre_hooks or g._global_forward_hooks or
                 g._global_forward_pre_hooks or g._global_backward_hooks or
                 g._global_backward_pre_hooks))


def _plain(mod) -> bool:
    """A bias-free nn.Linear whose call is its weight's product and no more."""
    return type(mod) is torch.nn.Linear and mod.bias is None and _unhooked(mod)


# Single-token forwards, bound to the modules as methods: a deep copy of a module
# runs on its own weights, and a pickled one finds its class's forward (hence the
# name).  Other inputs run the class's forward.

def _norm_forward(self, hidden_states):
    x, w = hidden_states, self.weight
    if (_one_token(x) and x.shape[-1] % 8 == 0 and w.dtype == x.dtype and
            w.device == x.device and _plain_tensor(w)):
        out = torch.empty_like(x)
        ops().rms_norm(x, w, self.variance_epsilon, out)
        return out
    return type(self).forward(self, x)


def _mlp_forward(self, x):
    if not (_one_token(x) and type(self.act_fn) in _silu_types() and _unhooked(self.act_fn)):
        return type(self).forward(self, x)
    gp, up = self.gate_proj, self.up_proj
    if (x.numel() == x.shape[-1] and _plain(gp) and _plain(up) and
            gp.weight.shape == up.weight.shape and _weight_fits(x, gp.weight) and
            _weight_fits(x, up.weight)):
        out = x.new_empty((1, 1, gp.weight.shape[0]))
        ops().gemv_glu(x, gp.weight, up.weight, out)
        return self.down_proj(out)
    g, u = gp(x), up(x)
    if (_one_token(g) and _one_token(u) and g.dtype == u.dtype and g.shape == u.shape and
            g.numel() % 2 == 0):
        out = torch.empty_like(g)
        ops().silu_mul(g, u, out)
    else:
        out = self.act_fn(g) * u
    return self.down_proj(out)


def _linear_forward(self, input):
    return _linear(input, self.weight, self.bias)


def _rotary_forward(self, x, position_ids):
    f, p = self.inv_freq, position_ids
    if (_one_token(x) and p.dtype == torch.long and p.dim() == 2 and p.shape[1] == 1 and
            p.device == x.device and f.device == x.device and p.is_contiguous() and
            f.is_contiguous() and type(p) is torch.Tensor and type(f) is torch.Tensor and
            0 < f.numel() <= 128 and
            f.dtype in (torch.float32, torch.bfloat16, torch.float16) and
            "dynamic" not in self.rope_type and self.rope_type != "longrope"):
        cos = x.new_empty((p.shape[0], 1, 2 * f.numel()))
        sin = torch.empty_like(cos)
        ops().rope_tables(p, f, self.attention_scaling, cos, sin)
        return cos, sin
    return type(self).forward(self, x, p)


_DECODE_FORWARDS = (_norm_forward, _mlp_forward, _linear_forward, _rotary_forward)
for _f in _DECODE_FORWARDS:
    _f.__name__ = "forward"
del _f


@functools.lru_cache(None)
def _silu_types() -> tuple:
    from transformers.activations import ACT2FN
    return torch.nn.SiLU, type(ACT2FN["silu"])


def _fuse_decode_ops(model) -> None:
    """Single-token forwards of the model's RMSNorms, MLPs, rotary tables and
    projections as one kernel each where the module is the stock class and
    nobody replaced its forward; other inputs run the class's forward."""
    from transformers.models.llama import modeling_llama as hf

    def wrap(mod, cls, forward):
        if type(mod) is cls and _own_forward(mod):
            mod.forward = MethodType(forward, mod)

    def part(mod, name):  # None: a model without it (another MLP, no rotary module)
        return getattr(mod, name, None)

    m = model.model
    wrap(part(m, "norm"), hf.LlamaRMSNorm, _norm_forward)
    wrap(part(m, "rotary_emb"), hf.LlamaRotaryEmbedding, _rotary_forward)
    for layer in m.layers:
        wrap(part(layer, "input_layernorm"), hf.LlamaRMSNorm, _norm_forward)
        wrap(part(layer, "post_attention_layernorm"), hf.LlamaRMSNorm, _norm_forward)
        mlp = part(layer, "mlp")
        wrap(mlp, hf.LlamaMLP, _mlp_forward)
        for mod in (part(layer.self_attn, "o_proj"), part(mlp, "gate_proj"),
                    part(mlp, "up_proj"), part(mlp, "down_proj")):
            wrap(mod, torch.nn.Linear, _linear_forward)
    wrap(part(model, "lm_head"), torch.nn.Linear, _linear_forward)


def _step_mask(model, batch: int, device):
    """Attention mask of a single-token forward.  Every layer's attention ignores
    it; a 4-D one, which LlamaModel hands through as it is, spares the step the
    launches that build one.  Another model class gets none, as for a prompt."""
    from transformers.models.llama import modeling_llama as hf
    if type(model.model) is not hf.LlamaModel:
        return None
    return torch.ones((batch, 1, 1, 1), dtype=torch.bool, device=device)


@dataclass
class LAPruneSettings:
    """Decode settings (the reference's ``draft_kwargs`` keys on this path)."""

    apply_layers: list[int] = field(default_factory=list)  # LAPrune layers
    retrieval: RetrievalConfig = field(default_factory=RetrievalConfig)
    group_size: int = 64                                   # decode encode buffer

    def __post_init__(self):
        if self.retrieval.local_window < self.group_size - 1:
            raise ValueError("local_window must cover the encode buffer "
                             "(local_window >= group_size - 1)")


class _LayerState:
    def __init__(self, cache: DecodeKVCache, sparse: SparseDecoder | None, dense: DenseDecoder):
        self.cache = cache
        self.sparse = sparse
        self.dense = dense


class LAPruneLlama:
    """A Llama model whose attention layers run the LAPrune decode path.

    Args:
      model: ``transformers`` ``LlamaForCausalLM`` on the GPU (bf16 or fp16).
      codebooks: {layer index: [M=32, K=256, head_dim] fp32 codebooks} for the
        layers in ``settings.apply_layers``.
      settings: which layers are LAPrune layers and the selection settings.
      batch: sequences decoded together.
      capacity: token capacity of every layer's cache (prompt + new tokens).
      health_every: decode steps between reads of the one-launch steps'
        health counters (one synchronisation each; 0 reads only at the end
        of ``generate``).  A non-zero counter raises
        :class:`~laprune_amd.retrieval.StepHealthError`.
    """

    def __init__(self, model, codebooks: dict[int, torch.Tensor], settings: LAPruneSettings,
                 batch: int, capacity: int, health_every: int = 64):
        from transformers.models.llama.modeling_llama import apply_rotary_pos_emb
        self._rope = apply_rotary_pos_emb
        self.model = model
        self.settings = settings
        cfg = model.config
        self.B = batch
        self.Hq = cfg.num_attention_heads
        self.Hkv = cfg.num_key_value_heads
        self.D = getattr(cfg, "head_dim", None) or cfg.hidden_size // self.Hq
        self.capacity = capacity
        p = next(model.parameters())
        self.dev, self.dtype = p.device, p.dtype
        missing = [i for i in settings.apply_layers if i not in codebooks]
        if missing:
            raise RuntimeError(f"no codebooks for LAPrune layers {missing}")
        self.layers = model.model.layers
        self.states: list[_LayerState] = []
        for i, layer in enumerate(self.layers):
            cb = codebooks[i].to(self.dev, torch.float32) if i in settings.apply_layers else None
            cache = DecodeKVCache(cb, batch, self.Hkv, self.D, capacity, dtype=self.dtype,
                                  group_size=settings.group_size, device=self.dev)
            sparse = None
            if cb is not None:
                sparse = SparseDecoder(cb, batch, self.Hq, self.Hkv, self.D, capacity,
                                       settings.retrieval, dtype=self.dtype)
            dense = DenseDecoder(batch, self.Hq, self.Hkv, self.D, capacity, self.dev, self.dtype)
            self.states.append(_LayerState(cache, sparse, dense))
            attn = layer.self_attn
            self._fuse_qkv(attn)
            attn.forward = self._make_forward(i, attn)
        _fuse_decode_ops(model)
        self._mask = _step_mask(model, batch, self.dev)
        self._row = None  # sequence being prefilled alone (ragged prefill)
        self.health_every = health_every
        self._since_check = 0
        self._dev_mode = False
        self._graph = None
        self._g = None

    # ------------------------------------------------------------ attention
    @staticmethod
    @torch.no_grad()
    def _fuse_qkv(attn) -> None:
        """One [q; k; v] weight per layer, so that a step projects with one
        GEMV instead of three; the modules' own weights become views of it
        (no second copy).  Layers whose biases are mixed keep three GEMVs."""
        mods = (attn.q_proj, attn.k_proj, attn.v_proj)
        has_b = [m.bias is not None for m in mods]
        if any(has_b) and not all(has_b):
            attn._lap_qkv = None
            return
        w = torch.cat([m.weight for m in mods], 0)
        b = torch.cat([m.bias for m in mods], 0) if all(has_b) else None
        sizes = [m.weight.shape[0] for m in mods]
        o = 0
        for m, n in zip(mods, sizes):
            m.weight = torch.nn.Parameter(w[o:o + n], requires_grad=False)
            if b is not None:
                m.bias = torch.nn.Parameter(b[o:o + n], requires_grad=False)
            o += n
        attn._lap_qkv = (w, b, sizes)

    @staticmethod
    def _fused_current(attn) -> bool:
        """Whether the modules' weights (and biases) are still the views of
        the fused tensors.  ``model.to(...)`` or ``load_state_dict(assign=True)``
        replace the parameters; the fused copy is then stale."""
        w, b, sizes = attn._lap_qkv
        mods = (attn.q_proj, attn.k_proj, attn.v_proj)
        off = 0
        for m, n in zip(mods, sizes):
            mw = m.weight
            if (mw.dtype != w.dtype or mw.device != w.device or
                    mw.data_ptr() != w.data_ptr() + off * w.stride(0) * w.element_size()):
                return False
            if b is not None and (m.bias is None or m.bias.dtype != b.dtype or
                                  m.bias.data_ptr() != b.data_ptr() + off * b.element_size()):
                return False
            off += n
        return True

    @classmethod
    def _project(cls, attn, h):
        """q, k, v projections of h [B, T, hidden] as [B, T, n] (views of one
        fused GEMV output when the layer's weights are fused).  A layer whose
        parameters were replaced after wrapping is fused again first."""
        f = getattr(attn, "_lap_qkv", None)
        if f is not None and not cls._fused_current(attn):
            cls._fuse_qkv(attn)
            f = attn._lap_qkv
        if f is None:
            return attn.q_proj(h), attn.k_proj(h), attn.v_proj(h)
        w, b, sizes = f
        return _linear(h, w, b).split(sizes, dim=-1)

    def _make_forward(self, idx: int, attn):
        def forward(hidden_states, position_embeddings=None, attention_mask=None,
                    past_key_values=None, **kwargs):
            return self._attention(idx, attn, hidden_states, position_embeddings)
        return forward

    def _attention(self, idx, attn, h, position_embeddings):
        B, T, _ = h.shape
        Hq, Hkv, D = self.Hq, self.Hkv, self.D
        cos, sin = position_embeddings
        st = self.states[idx]
        if T == 1 and self._dev_mode:
            # fixed launches, every per-step value in device memory; RoPE and
            # the cache write are one kernel
            qp, kp, vp = self._project(attn, h)
            q = st.cache.rope_append(qp, kp, vp, cos, sin, self._g_pos, self._q_rope)
            if st.sparse is not None:
                if self._g_flush:
                    st.cache.encode_ranges(self._g_ranges)
                o = st.sparse.step_dev(q, st.cache.codes, st.cache.k, st.cache.v,
                                       self._g_plan_sparse)
            else:
                o = st.dense.step_dev(q, st.cache.k, st.cache.v, self._g_plan_dense)
            o = o.transpose(1, 2).reshape(B, T, Hq * D)
            return attn.o_proj(o), None
        qp, kp, vp = self._project(attn, h)
        q = qp.reshape(B, T, Hq, D).transpose(1, 2)
        k = kp.reshape(B, T, Hkv, D).transpose(1, 2)
        v = vp.reshape(B, T, Hkv, D).transpose(1, 2)
        q, k = self._rope(q, k, cos, sin)
        if T > 1:  # prefill: causal attention over the prompt, encode all its keys
            if self._row is None:
                if any(n != 0 for n in st.cache.lengths):
                    raise RuntimeError("batched prefill needs empty caches (use reset())")
                st.cache.append(k, v, prefill=True)
            else:
                st.cache.append_row(self._row, k, v, prefill=True)
            G = Hq // Hkv
            kk = k.repeat_interleave(G, dim=1)
            vv = v.repeat_interleave(G, dim=1)
            # fused kernels only: the math fallback would materialise T x T scores
            with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
                o = F.scaled_dot_product_attention(q, kk, vv, is_causal=True,
                                                   scale=1.0 / math.sqrt(D))
        else:
            if self._row is not None:
                raise RuntimeError("single-token steps decode the whole batch")
            st.cache.append(k, v)  # encodes each sequence's 64-token groups
            if st.sparse is not None:
                o = st.sparse.step_cached(q, st.cache)
            else:
                o = st.dense.step(q, st.cache.k, st.cache.v, lengths=st.cache.lengths)
        o = o.transpose(1, 2).reshape(B, T, Hq * D)
        return attn.o_proj(o), None

    # ------------------------------------------------------------ model calls
    def reset(self) -> None:
        """Forget every sequence (the reference's Decoder.reset)."""
        for st in self.states:
            st.cache.lengths = [0] * self.B
            st.cache.encoded_lens = [0] * self.B

    @property
    def lengths(self) -> list[int]:
        return list(self.states[0].cache.lengths)

    def _check_room(self, new: int, rows=None) -> None:
        """Raise before any layer runs when ``new`` more tokens for the given
        sequences (all by default) would exceed ``capacity``, which sized
        every layer's decoder and workspaces; nothing is appended then, so
        the layers' caches stay consistent."""
        lens = self.lengths
        rows = range(self.B) if rows is None else rows
        need = max(lens[b] for b in rows) + new
        if need > self.capacity:
            raise RuntimeError(f"{need} tokens exceed the capacity of {self.capacity} the "
                               "model was wrapped with (wrap it with a larger capacity)")

    def _forward(self, ids: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
        mask = self._mask if ids.shape[1] == 1 else None
        out = self.model(input_ids=ids, attention_mask=mask, position_ids=pos, use_cache=False,
                         logits_to_keep=1)
        return out.logits[:, -1]

    @torch.no_grad()
    def prefill(self, input_ids: torch.Tensor) -> torch.Tensor:
        """Prefill [B, T] prompts of one length; returns last-position logits [B, V]."""
        if input_ids.shape[0] != self.B:
            raise RuntimeError(f"expected {self.B} sequences, got {input_ids.shape[0]}")
        T = input_ids.shape[1]
        if any(n != 0 for n in self.lengths):
            raise RuntimeError("batched prefill needs empty caches (use reset())")
        self._check_room(T)
        pos = torch.arange(T, device=self.dev)[None].expand(self.B, T)
        return self._forward(input_ids.to(self.dev), pos)

    @torch.no_grad()
    def prefill_row(self, b: int, input_ids: torch.Tensor) -> torch.Tensor:
        """Prefill sequence b alone ([1, T_b] prompt); returns its logits [1, V]."""
        T = input_ids.shape[-1]
        if not 0 <= b < self.B:
            raise RuntimeError(f"sequence {b} out of range for batch {self.B}")
        self._check_room(T, rows=[b])
        self._row = b
        try:
            pos = torch.arange(T, device=self.dev)[None]
            return self._forward(input_ids.reshape(1, T).to(self.dev), pos)
        finally:
            self._row = None

    @torch.no_grad()
    def decode(self, tokens: torch.Tensor) -> torch.Tensor:
        """One decode step for all sequences: tokens [B, 1]; returns logits [B, V]."""
        self._check_room(1)
        pos = torch.tensor(self.lengths, device=self.dev)[:, None]
        logits = self._forward(tokens.reshape(self.B, 1).to(self.dev), pos)
        self._count_step()
        return logits

    # ------------------------------------------------------------ health
    def check_health(self) -> None:
        """Read every LAPrune layer's health counters (one gather, one
        synchronising copy) and raise StepHealthError naming the layers
        whose one-launch steps split a row over XCDs or timed out a barrier."""
        self._since_check = 0
        decs = [(i, st.sparse) for i, st in enumerate(self.states) if st.sparse is not None]
        if not decs:
            return
        words = torch.stack([d.status_words() for _, d in decs]).cpu()
        bad = [(i, int(w[0]), int(w[1])) for (i, _), w in zip(decs, words.tolist())
               if w[0] or w[1]]
        if bad:
            check_step_health(sum(b[1] for b in bad), sum(b[2] for b in bad),
                              who=f"LAPruneLlama (layers {[b[0] for b in bad]})")

    def reset_health(self) -> None:
        """Zero every LAPrune layer's step workspace after an unhealthy step."""
        for st in self.states:
            if st.sparse is not None:
                st.sparse.reset_health()

    def _count_step(self) -> None:
        self._since_check += 1
        if self.health_every and self._since_check >= self.health_every:
            self.check_health()

    # ------------------------------------------------------------ captured decode
    # One decode step of the whole model as one HIP graph.  Per-step values
    # (positions, the sequences' plans, encode-flush ranges) live in one
    # device int32 buffer that the host rewrites before each replay; every
    # kernel of the step reads them there, so the captured launches stay
    # valid.  The host keeps the lengths and flush bookkeeping.

    def _graph_buffers(self):
        B, dev = self.B, self.dev
        flat = torch.zeros(20 * B, dtype=torch.int32, device=dev)
        self._g_flat = flat
        self._g_plan_sparse = flat[:8 * B].view(B, 8)
        self._g_plan_dense = flat[8 * B:16 * B].view(B, 8)
        self._g_ranges = flat[16 * B:18 * B].view(B, 2)
        self._g_pos = flat[18 * B:].view(torch.long).view(B, 1)
        self._q_rope = torch.empty((B, self.Hq, self.D), dtype=self.dtype, device=dev)
        self._g_flush = False
        self._g_tok = torch.zeros((B, 1), dtype=torch.long, device=dev)
        self._g_next = torch.zeros((B, 1), dtype=torch.long, device=dev)
        self._g_logits = None
        self._g_host = [torch.zeros(20 * B, dtype=torch.int32).pin_memory() for _ in range(4)]
        self._g_done = [None] * 4
        self._g_slot = 0
        self._g = True

    def _graph_body(self):
        self._dev_mode = True
        try:
            logits = self._forward(self._g_tok, self._g_pos)
        finally:
            self._dev_mode = False
        if self._g_logits is None:
            self._g_logits = torch.empty_like(logits, memory_format=torch.contiguous_format)
        if logits.dtype in (torch.bfloat16, torch.float16) and logits.stride(-1) == 1:
            ops().argmax_rows(logits, self._g_next, self._g_logits)
        else:
            self._g_logits.copy_(logits)
            self._g_next.copy_(logits.argmax(dim=-1, keepdim=True))

    def _upload_step(self) -> None:
        """Advance every layer's bookkeeping by one token and upload the
        step's positions, plans and flush ranges."""
        B = self.B
        pos = self.lengths
        ranges = None
        for st in self.states:
            r = st.cache.advance_decode()
            if st.sparse is not None:
                ranges = r
        # steps on which no sequence fills its encode buffer replay the graph
        # without the encode launches
        self._g_flush = ranges is not None and any(hi > lo for lo, hi in ranges)
        c0 = next((st for st in self.states if st.sparse is not None), self.states[0])
        t_total = c0.cache.lengths
        rows = [0] * (20 * B)  # the last 2 B words are B int64 positions
        if c0.sparse is not None:
            from .retrieval import PLAN_FIELDS
            for b, p in enumerate(c0.sparse.row_plans(c0.cache.encoded_lens, t_total)):
                rows[8 * b:8 * b + 8] = [p[f] for f in PLAN_FIELDS]
        for b in range(B):
            t = t_total[b]
            rows[8 * B + 8 * b:8 * B + 8 * b + 8] = [t, t, 0, 0, 0, 0, 0, t]
            if ranges is not None:
                rows[16 * B + 2 * b:16 * B + 2 * b + 2] = list(ranges[b])
            rows[18 * B + 2 * b] = pos[b]
        i = self._g_slot
        self._g_slot = (i + 1) % len(self._g_host)
        if self._g_done[i] is not None:
            self._g_done[i].synchronize()
        h = self._g_host[i]
        h.copy_(torch.tensor(rows, dtype=torch.int32))
        self._g_flat.copy_(h, non_blocking=True)
        ev = torch.cuda.Event()
        ev.record(torch.cuda.current_stream(self.dev))
        self._g_done[i] = ev

    @torch.no_grad()
    def decode_graph(self, tokens: torch.Tensor | None = None) -> torch.Tensor:
        """One decode step for all sequences as one graph replay.  tokens
        [B, 1] (device or host); None feeds the previous step's greedy
        tokens.  Returns the logits [B, V] (a buffer the next step reuses)."""
        self._check_room(1)
        if self._g is None:
            self._graph_buffers()
        if tokens is not None:
            self._g_tok.copy_(tokens.reshape(self.B, 1), non_blocking=True)
        else:
            self._g_tok.copy_(self._g_next)
        self._upload_step()
        sig = tuple((st.cache.k.data_ptr(), st.cache.v.data_ptr(), st.cache.codes.data_ptr())
                    for st in self.states)
        if self._graph is not None and sig != self._graph_sig:
            self._graph = None  # a cache was reallocated (grown): capture again
        if self._graph is None:
            self._graph = {}
            self._graph_sig = sig
        g = self._graph.get(self._g_flush)
        if g is None:
            # the first step of each variant (with or without encode flushes)
            # runs eagerly (it also warms up every kernel), then the same body
            # is captured for the following steps
            side = torch.cuda.Stream(self.dev)
            side.wait_stream(torch.cuda.current_stream(self.dev))
            with torch.cuda.stream(side):
                self._graph_body()
            torch.cuda.current_stream(self.dev).wait_stream(side)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                self._graph_body()
            self._graph[self._g_flush] = g
        else:
            g.replay()
        self._count_step()
        return self._g_logits

    def next_tokens(self) -> torch.Tensor:
        """Greedy tokens [B, 1] of the last captured step (device)."""
        return self._g_next

    @torch.no_grad()
    def generate(self, input_ids: torch.Tensor, max_new_tokens: int,
                 eos_token_id: int | None = None, graph: bool = False) -> torch.Tensor:
        """Greedy generation as AQGeneration.generate: prefill all prompt
        tokens but the last, then decode from it.  Returns [B, T + n] ids.
        graph=True decodes with captured steps (the cache capacity must hold
        the whole generation)."""
        self.reset()
        ids = input_ids.to(self.dev)
        if ids.shape[1] > 1:
            self.prefill(ids[:, :-1])
        tok = ids[:, -1:]
        new = []
        for i in range(max_new_tokens):
            if graph:
                self.decode_graph(tok if i == 0 else None)
                tok = self._g_next.clone()
            else:
                tok = self.decode(tok).argmax(dim=-1, keepdim=True)
            new.append(tok)
            if eos_token_id is not None and bool((tok == eos_token_id).all()):
                break
        self.check_health()
        return torch.cat([ids] + new, dim=1)


def llama31_8b_config(num_layers: int = 32, max_position_embeddings: int = 131072):
    """A local LlamaConfig with Llama-3.1-8B's public geometry (no download)."""
    from transformers import LlamaConfig
    return LlamaConfig(
        vocab_size=128256, hidden_size=4096, intermediate_size=14336,
        num_hidden_layers=num_layers, num_attention_heads=32, num_key_value_heads=8,
        head_dim=128, max_position_embeddings=max_position_embeddings, rms_norm_eps=1e-5,
        rope_theta=500000.0, tie_word_embeddings=False,
        rope_scaling={"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0,
                      "high_freq_factor": 4.0, "original_max_position_embeddings": 8192},
        attn_implementation="sdpa")


def random_model(config, device, dtype=torch.bfloat16, seed: int = 0, std: float = 0.02):
    """Random-init LlamaForCausalLM: every weight N(0, std), norms at 1."""
    from transformers import LlamaForCausalLM
    torch.manual_seed(seed)
    with torch.device(device):
        model = LlamaForCausalLM(config).to(dtype)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.dim() >= 2:
                p.normal_(0.0, std)
            else:
                p.fill_(1.0)
    return model.eval()
