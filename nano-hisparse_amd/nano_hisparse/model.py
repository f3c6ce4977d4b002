"""A small Qwen2-shaped decoder that drives the sparse decode path.

Reference: nano_hisparse/model.py:19-221. Projections and SwiGLU are torch
operations; in the prompt pass of a bf16/fp16 GPU model RMSNorm (with the
residual add), RoPE and the causal attention are kernels
(nhs_add_rmsnorm, nhs_rope, nhs_prefill_attention), elsewhere torch too. Each
decode step appends K/V through the cache, selects pages with Quest on the
GPU and attends over the selected rows with the HIP kernels; the batched one
runs its dense layers on kernels as well. The module tree
(names and construction order) is the reference's, which is HF Qwen2's, so
state dicts load either way and a seeded random init draws the same weights.
"""

from __future__ import annotations

import sys
from dataclasses import dataclass
from typing import NamedTuple

import torch
from torch import nn
from torch.nn import functional as F

from .selection import Selection, quest_selection, select_pages
from .storage import upload


ROPE_TABLE_ROWS = 1 << 17  # longest cos/sin tables a model keeps (32 MB at head_dim 128 in 16 bits)


@dataclass
class ModelConfig:
    vocab_size: int = 256
    hidden_size: int = 128
    intermediate_size: int = 256
    num_hidden_layers: int = 2
    num_attention_heads: int = 4
    num_key_value_heads: int = 2
    rms_norm_eps: float = 1e-6
    rope_theta: float = 10000.0

    @property
    def head_dim(self):
        return self.hidden_size // self.num_attention_heads

    def __post_init__(self):
        if (
            self.hidden_size % self.num_attention_heads
            or self.num_attention_heads % self.num_key_value_heads
            or self.head_dim % 2
        ):
            raise ValueError("model dimensions must support grouped-query attention and RoPE")


class RMSNorm(nn.Module):
    def __init__(self, width, eps):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(width))
        self.eps = eps

    def forward(self, x):
        xf = x.float()
        return (xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + self.eps)).to(x.dtype) * self.weight


class Projections(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        kv_width = cfg.num_key_value_heads * cfg.head_dim
        self.q_proj = nn.Linear(cfg.hidden_size, cfg.hidden_size, bias=True)
        self.k_proj = nn.Linear(cfg.hidden_size, kv_width, bias=True)
        self.v_proj = nn.Linear(cfg.hidden_size, kv_width, bias=True)
        self.o_proj = nn.Linear(cfg.hidden_size, cfg.hidden_size, bias=False)


class MLP(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.gate_proj = nn.Linear(cfg.hidden_size, cfg.intermediate_size, bias=False)
        self.up_proj = nn.Linear(cfg.hidden_size, cfg.intermediate_size, bias=False)
        self.down_proj = nn.Linear(cfg.intermediate_size, cfg.hidden_size, bias=False)

    def forward(self, x):
        return self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


class Block(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.self_attn = Projections(cfg)
        self.mlp = MLP(cfg)


class Decoder(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(Block(cfg) for _ in range(cfg.num_hidden_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)


class Model(nn.Module):
    def __init__(self, config: ModelConfig | None = None):
        super().__init__()
        self.config = config or ModelConfig()
        self.model = Decoder(self.config)
        self.lm_head = nn.Linear(self.config.hidden_size, self.config.vocab_size, bias=False)

    @classmethod
    def from_pretrained(cls, name: str, device="cuda", dtype=torch.bfloat16):
        """Qwen2/Qwen2.5 weights with standard RoPE from a local directory or
        an already-cached hub name (no network is assumed)."""
        from transformers import AutoConfig, AutoModelForCausalLM

        hf_cfg = AutoConfig.from_pretrained(name)
        rope = getattr(hf_cfg, "rope_parameters", None) or getattr(hf_cfg, "rope_scaling", None) or {}
        if hf_cfg.model_type != "qwen2" or rope.get("rope_type", rope.get("type", "default")) != "default":
            raise ValueError("only Qwen2/Qwen2.5 with standard RoPE are supported")
        if getattr(hf_cfg, "use_sliding_window", False) or hf_cfg.hidden_act != "silu":
            raise ValueError("sliding window / non-SiLU models are unsupported")
        hf = AutoModelForCausalLM.from_pretrained(name, torch_dtype=dtype).eval().to(device)
        model = cls.__new__(cls)
        nn.Module.__init__(model)
        fields = {f: getattr(hf_cfg, f) for f in ModelConfig.__dataclass_fields__ if f != "rope_theta"}
        fields["rope_theta"] = rope.get("rope_theta", getattr(hf_cfg, "rope_theta", 10000.0))
        model.config = ModelConfig(**fields)
        model.model, model.lm_head = hf.model, hf.lm_head
        return model.eval()

    @property
    def device(self):
        return self.model.embed_tokens.weight.device

    @property
    def dtype(self):
        return self.model.embed_tokens.weight.dtype

    def _project(self, layer, x, start):
        """RMSNorm, q/k/v projections and rotary embedding for tokens at
        positions start .. start + len(x) - 1."""
        return self._project_at(layer, x, torch.arange(start, start + len(x), device=x.device))

    def _project_at(self, layer, x, positions):
        """_project for rows at arbitrary positions (an int tensor [len(x)])."""
        cfg, n = self.config, len(x)
        h = layer.input_layernorm(x)
        attn = layer.self_attn
        q = attn.q_proj(h).view(n, cfg.num_attention_heads, cfg.head_dim)
        k = attn.k_proj(h).view(n, cfg.num_key_value_heads, cfg.head_dim)
        v = attn.v_proj(h).view(n, cfg.num_key_value_heads, cfg.head_dim)
        inv_freq = cfg.rope_theta ** (-torch.arange(0, cfg.head_dim, 2, device=x.device).float() / cfg.head_dim)
        angle = positions.float()[:, None] * inv_freq[None, :]
        angle = torch.cat((angle, angle), -1)[:, None, :]
        cos, sin = angle.cos().to(x.dtype), angle.sin().to(x.dtype)

        def rope(t):
            lo, hi = t.chunk(2, -1)
            return t * cos + torch.cat((-hi, lo), -1) * sin

        return rope(q), rope(k), v

    @staticmethod
    def _finish(layer, residual, attention):
        x = residual + layer.self_attn.o_proj(attention.reshape(len(residual), -1))
        return x + layer.mlp(layer.post_attention_layernorm(x))

    @torch.inference_mode()
    def prefill(self, tokens: list[int], cache=None, request_id=None):
        """Dense causal forward over the prompt, writing K/V to the cache;
        returns the last position's logits (fp32)."""
        if not tokens:
            raise ValueError("prompt cannot be empty")
        if cache is not None and any(cache.storage.requests[request_id].lengths):
            raise ValueError("prefill is allowed exactly once per request")
        cfg = self.config
        groups = cfg.num_attention_heads // cfg.num_key_value_heads
        # bf16/fp16 models on a GPU run the causal attention as the MFMA
        # flash kernel (nhs_prefill_attention): O(S) memory where the dense
        # path materialises S x S scores per head; fp32 and CPU models keep
        # the dense causal attention.
        flash = (self.device.type == "cuda" and self.dtype in (torch.bfloat16, torch.float16)
                 and cfg.head_dim in (64, 128))
        if flash:
            from . import row_kernels as rk
        x = self.model.embed_tokens(upload(tokens, torch.int64, self.device))
        layers = self.model.layers
        if flash and len(layers) and all(_plain_layer(layer, x.dtype) for layer in layers):
            if not _plain(self.model.embed_tokens, nn.Embedding):
                x = x.clone()  # a hook may hold the rows, which are updated in place
            return self._prefill_layers(x, cache, request_id)
        for index, layer in enumerate(self.model.layers):
            q, k, v = self._project(layer, x, 0)
            if cache is not None:
                cache.write(request_id, index, k, v)
            if flash:
                attention = rk.prefill_attention(q, k, v)
            else:
                attention = F.scaled_dot_product_attention(
                    q.transpose(0, 1),
                    k.repeat_interleave(groups, 1).transpose(0, 1),
                    v.repeat_interleave(groups, 1).transpose(0, 1),
                    is_causal=True,
                ).transpose(0, 1)
            x = self._finish(layer, x, attention)
        return self.lm_head(self.model.norm(x[-1])).float()

    def _prefill_layers(self, x, cache, request_id):
        """The prompt pass of a bf16/fp16 GPU model from its embedded tokens
        x (updated in place): the residual add and RMSNorm are one kernel and
        q and k rotate in place by cos/sin computed once per prompt, where
        the torch expressions take some thirty passes over [tokens, hidden]
        per layer (4000 tokens x 4096, two layers: 5.6 -> 5.1 ms)."""
        from . import row_kernels as rk

        cfg, n = self.config, len(x)
        D, Hq, Hkv = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
        cos, sin = _rope_rows(cfg, torch.arange(n, device=x.device), x.dtype)
        x, delta = x.contiguous(), None
        for index, layer in enumerate(self.model.layers):
            attn, norm1, norm2 = layer.self_attn, layer.input_layernorm, layer.post_attention_layernorm
            h = rk.add_rmsnorm(x, delta, norm1.weight, _eps(norm1, cfg))
            q, k, v = attn.q_proj(h), attn.k_proj(h), attn.v_proj(h)
            rk.rope_(q, Hq, D, cos, sin)
            rk.rope_(k, Hkv, D, cos, sin)
            q, k, v = q.view(n, Hq, D), k.view(n, Hkv, D), v.view(n, Hkv, D)
            if cache is not None:
                cache.write(request_id, index, k, v)
            o = attn.o_proj(rk.prefill_attention(q, k, v).reshape(n, -1)).contiguous()
            delta = layer.mlp(rk.add_rmsnorm(x, o, norm2.weight, _eps(norm2, cfg))).contiguous()
        if _plain_norm(self.model.norm, x.dtype) and _plain(self.lm_head, nn.Linear):
            return self._head([_Last(x[-1:], delta[-1:])])[0]
        return self.lm_head(self.model.norm(x[-1] + delta[-1])).float()

    @torch.inference_mode()
    def decode(self, token: int, request_id, cache, top_k=None, backend="auto", selector="quest"):
        """One decode step: per layer append K/V, select (Quest top_k pages,
        or the page-mean selector, or everything for top_k=None) and attend
        over the selected rows. Returns fp32 logits."""
        lengths = cache.storage.requests[request_id].lengths
        if len(set(lengths)) != 1 or lengths[0] == 0:
            raise ValueError("all layers must have the same nonempty history")
        position = lengths[0]
        P = cache.config.page_size
        x = self.model.embed_tokens(upload([token], torch.int64, self.device))
        for index, layer in enumerate(self.model.layers):
            q, k, v = self._project(layer, x, position)
            cache.write(request_id, index, k, v)
            request = cache.storage.requests[request_id]
            if selector == "quest" and top_k is not None:
                selection = quest_selection(
                    q[0], request.minimum[index], request.maximum[index], request.lengths[index], P, top_k
                )
            elif selector in ("quest", "mean"):
                pages = select_pages(cache, request_id, index, q[0], top_k)
                selection = Selection.from_pages(pages, request.lengths[index], P, q.shape[1])
            else:
                raise ValueError("selector must be quest or mean")
            attention = cache.attention(q[0], request_id, index, selection, backend)
            x = self._finish(layer, x, attention.unsqueeze(0))
        return self.lm_head(self.model.norm(x[0])).float()

    def _fused_projections(self):
        """Per layer: the q/k/v weights and biases and the gate/up weights as
        one tensor each, for one GEMM apiece in the batched decode. The
        module parameters become views of the fused tensors (names, state
        dicts and the per-request path are unchanged); fusing again happens
        only if a parameter was replaced since (e.g. by .to())."""
        fused = getattr(self, "_fused", None)
        if fused is not None and fused[0].unchanged():
            return fused[1]
        layers, modules = [], [self.model.layers]
        for layer in self.model.layers:
            attn, mlp = layer.self_attn, layer.mlp
            qkv, gate_up = (attn.q_proj, attn.k_proj, attn.v_proj), (mlp.gate_proj, mlp.up_proj)
            layers.append((_fuse(qkv, "weight"), _fuse(qkv, "bias"), _fuse(gate_up, "weight")))
            modules += (layer, attn, mlp, *qkv, *gate_up)
        self._fused = (_Held(modules), layers)
        return layers

    @torch.inference_mode()
    def decode_batch(self, tokens: list[int], request_ids: list, cache, top_k: int, micro_batches: int = 1,
                     graph: bool = False):
        """One decode step for several requests at once (Quest top_k pages).

        Dense layers run on the batch with fused projections (one q/k/v
        GEMM, one gate/up GEMM) and libnhs_hip.so's fused residual-add +
        RMSNorm, RoPE (cos/sin computed once per step) and SiLU * up
        kernels; the sparse stages run once per layer for all requests
        (cache.decode_batch). With micro_batches=2 the requests form two
        groups that run half a layer apart, so each group's host-row gather
        (transfer stream) runs beside the other group's layer compute; the
        gather's grid is capped meanwhile to leave compute units to that
        work. Returns fp32 logits [B, vocab]; row b equals decode(tokens[b],
        request_ids[b]) up to the order of the dense layers' reductions.

        graph=True replays the step's launches from a HIP graph
        captured at the first step of this batch composition (see
        _decode_batch_graph): the same kernels on the same buffers, with no
        per-launch host work."""
        from . import row_kernels as rk

        if len(tokens) != len(request_ids):
            raise ValueError("one token per request")
        if top_k is None or top_k < 1:
            raise ValueError("batched decode needs a positive Quest top_k")
        if micro_batches not in (1, 2):
            raise ValueError("micro_batches must be 1 or 2")
        n = len(tokens)
        embed = self.model.embed_tokens
        if n and _plain(embed, nn.Embedding) and not 0 <= min(tokens) <= max(tokens) < len(embed.weight):
            raise IndexError("token id outside the vocabulary")
        if n < 2:
            micro_batches = 1
        cuts = [0, n] if micro_batches == 1 else [0, (n + 1) // 2, n]
        if graph:
            return self._decode_batch_graph(tokens, request_ids, cache, top_k, cuts)
        overlap = len(cuts) > 2
        groups = [_Group(self, tokens[a:b], request_ids[a:b], cache, overlap) for a, b in zip(cuts, cuts[1:])]
        logits = self._run_groups(groups, top_k)
        for g in groups:
            g.step.end()
        return logits

    def _run_groups(self, groups, top_k):
        """Every layer of one group, or of two groups half a layer apart (each
        group's gather on the transfer stream beside the other's compute,
        with the gather's grid capped meanwhile), then the final norm and the
        lm_head; returns the logits."""
        from . import row_kernels as rk

        fused = self._fused_projections()
        layers = self.model.layers
        if len(groups) == 1:
            g = groups[0]
            for index, layer in enumerate(layers):
                g.pre(index, layer, fused[index], top_k)
                g.post(layer)
        else:
            a, b = groups
            rk.set_gather_workgroups(32)
            try:
                a.pre(0, layers[0], fused[0], top_k)
                b.pre(0, layers[0], fused[0], top_k)
                for index, layer in enumerate(layers):
                    following = index + 1 < len(layers)
                    a.post(layer)
                    if following:
                        a.pre(index + 1, layers[index + 1], fused[index + 1], top_k)
                    b.post(layer)
                    if following:
                        b.pre(index + 1, layers[index + 1], fused[index + 1], top_k)
            finally:
                rk.set_gather_workgroups(0)
        return self._head(groups)

    def _head(self, groups):
        """The last residual add, the final norm and the lm_head of every
        group's rows: fused kernels in place of a plain norm and head, else
        the modules themselves."""
        from . import row_kernels as rk

        norm, head = self.model.norm, self.lm_head
        plain = _plain_norm(norm, self.dtype)
        rows = [rk.add_rmsnorm(g.x, g.delta, norm.weight, _eps(norm, self.config), write_back=False) if plain
                else g.x + g.delta for g in groups]
        x = rows[0] if len(rows) == 1 else torch.cat(rows)
        if not plain:
            x = norm(x)
        return (_linear(x, head.weight, head.bias) if _plain(head, nn.Linear) else head(x)).float()

    def _rope_tables(self, limit):
        """cos and sin [rows, head_dim / 2] in the model dtype of every
        position below `limit` (None beyond ROPE_TABLE_ROWS positions): kept
        with the model while its device, dtype and RoPE stay, longer ones
        (twice as long each) made on demand. A decode step then reads its
        rows instead of computing them in eleven launches. Inside a graph
        capture, which cannot wait for a table, none is made (None where no
        kept one is long enough)."""
        if limit > ROPE_TABLE_ROWS:
            return None
        cfg = self.config
        key = (self.device, self.dtype, cfg.rope_theta, cfg.head_dim)
        stream = torch.cuda.current_stream(self.device) if self.device.type == "cuda" else None
        made = [entry for entry in self.__dict__.get("_rope", ()) if entry[0] == key]
        for _, tables, home in reversed(made):
            if len(tables[0]) >= limit:
                if stream != home:
                    for t in tables:
                        t.record_stream(stream)
                return tables
        if stream is not None and torch.cuda.is_current_stream_capturing():
            return None
        rows = min(ROPE_TABLE_ROWS, max(4096, 1 << (limit - 1).bit_length()))
        tables = _rope_rows(cfg, torch.arange(rows, device=self.device), self.dtype)
        if stream is not None:
            stream.synchronize()  # complete for every stream from here on
        self.__dict__["_rope"] = [*made, (key, tables, stream)]
        return tables

    def _span_tables(self, store, request_ids, spans):
        """The cos/sin tables of each group's own positions (each by its
        longest reservation: a group beyond ROPE_TABLE_ROWS has none, beside
        another that does), for a capture that must make none."""
        return [self._rope_tables(max(store.requests[r].max_tokens for r in request_ids[a:b])) for a, b in spans]

    def clear_decode_graphs(self):
        """Drops every captured decode-step graph, with the cache, buffers and
        graph memory each one holds, and the kept cos/sin tables."""
        self.__dict__.pop("_decode_graphs", None)
        self.__dict__.pop("_rope", None)

    def __getstate__(self):
        # graphs, tables and fused projections stay with this object: a copy makes its own
        return {k: v for k, v in self.__dict__.items() if k not in ("_decode_graphs", "_rope", "_fused")}

    def _decode_batch_graph(self, tokens, request_ids, cache, top_k, cuts):
        """decode_batch with the step's launches (every layer of every group,
        the final norm and the lm_head) captured once per batch composition
        into a HIP graph and replayed from then on. With two groups (cuts
        [0, m, n]) the capture holds both groups' schedule: each gather is a
        branch forked from the capture stream by an event and joined back by
        the attention that waits for it, so the replay runs it beside the
        other group's compute as the eager steps do.

        Per step, outside the graph: the page placement and residency policy
        (BatchDecode's constructor; its table writes precede the replay on
        the compute stream), the upload of the lengths and token ids into the
        buffers the graph reads, the waits for the tables' pending events,
        and after the replay the pages' host state and the policy tick
        (end()). Every launch's shape depends only on the batch, the budget
        and the requests' reserved pages, so the replayed step is the eager
        one. A graph is reused only while the cache's device item tables of
        the groups are the same objects (they hold the pointers the graph
        read) and the model's modules and parameters are those it read
        (model.to() replaces them and frees the old ones); otherwise it is
        captured again."""
        store = cache.storage
        store.check_stream()
        graphs = self.__dict__.setdefault("_decode_graphs", {})
        # graphs captured against another cache hold that cache (its pool),
        # their buffers and their private memory: drop them
        for stale in [k for k, e in graphs.items() if e["cache"] is not cache]:
            del graphs[stale]
        spans = list(zip(cuts, cuts[1:]))
        overlap = len(spans) > 1
        key = (tuple(request_ids), top_k, len(spans))
        items = [cache._layer_items(request_ids[a:b]) for a, b in spans]
        entry = graphs.get(key)
        if entry is not None and (entry["cache"] is not cache or not entry["read"].unchanged()
                                  or any(x is not y for x, y in zip(entry["items"], items))):
            del graphs[key]
            entry = None
        token_ids = [torch.tensor(tokens[a:b], dtype=torch.int64).pin_memory() for a, b in spans]

        def open_steps(buffers):
            steps = []
            for (a, b), (lengths, _) in zip(spans, buffers):
                step = cache.decode_batch(request_ids[a:b], overlap, lengths_buffer=lengths)
                step.sync_tables()
                step.clear_reads()
                steps.append(step)
            for (_, ids), t in zip(buffers, token_ids):
                ids.copy_(t, non_blocking=True)
            return steps

        if entry is None:
            # Fuse before the capture: a fusion inside it would be recorded and not run, and every replay would
            # read the separate weights, which fusing frees.
            self._fused_projections()
            # The same holds for each group's cos/sin tables, and a workspace made inside it would be cleared by every
            # replay.
            tables = self._span_tables(store, request_ids, spans)
            buffers = [(torch.empty(2, b - a, dtype=torch.int64, device=cache.device),
                        torch.empty(b - a, dtype=torch.int64, device=cache.device)) for a, b in spans]
            steps = open_steps(buffers)
            for step in steps:
                step.make_workspace(self.config.num_attention_heads, top_k)
            graph = torch.cuda.CUDAGraph()
            side = torch.cuda.Stream(device=cache.device)
            side.wait_stream(store.compute)
            if overlap:
                side.wait_stream(store.transfer)
            with store.capturing(side), torch.cuda.graph(graph, stream=side):
                groups = [_Group(self, None, request_ids[a:b], cache, overlap, step=step, ids=ids, tables=made)
                          for (a, b), step, (_, ids), made in zip(spans, steps, buffers, tables)]
                logits = self._run_groups(groups, top_k)
            for step in steps:
                step.forget_capture_events()
            # what the graph reads outside its own memory lives as long as it does
            entry = {"cache": cache, "read": _Held(_tree(self)), "items": items, "buffers": buffers, "graph": graph,
                     "logits": logits, "stream": side, "tables": tables,
                     "workspaces": [step.workspace for step in steps]}
            graphs[key] = entry
            while len(graphs) > 8:  # the most recent compositions keep their graphs
                del graphs[next(iter(graphs))]
        else:
            steps = open_steps(entry["buffers"])
            for step in steps:
                step.account_replayed()
        entry["graph"].replay()
        for step in steps:
            step.end()
        return entry["logits"].clone()


def _tree(module):
    """A module and every module below it."""
    modules = [module]
    for m in modules:
        modules.extend(c for c in m._modules.values() if c is not None)
    return modules


class _Held:
    """The parameters and child modules that some modules hold at one time,
    to tell later whether they hold the same ones at the same addresses."""

    def __init__(self, modules):
        self.dicts = [d for m in modules for d in (m._parameters, m._buffers, m._modules) if d]
        self.children = [c for m in modules for c in m._modules.values()]  # held: their identities stay their own
        self.state = self._now()

    def _now(self):
        from . import row_kernels as rk

        return (rk._launch or rk._load_launch()).held_state(self.dicts)

    def unchanged(self):
        return self._now() == self.state


class _Last(NamedTuple):
    """A prompt's last row, as _head takes a group."""

    x: torch.Tensor
    delta: torch.Tensor


class _Group:
    """One batch group of decode_batch: its residual stream, RoPE tables,
    cache step and the gather handle in flight. Within a capture the step,
    its token ids and its tables (or None) are made before and handed in."""

    def __init__(self, model, tokens, request_ids, cache, overlap, step=None, ids=None, tables=None):
        cfg = model.config
        self.model, self.cfg = model, cfg
        self.step = cache.decode_batch(request_ids, overlap) if step is None else step
        positions = self.step.dev_lengths[0]  # already on the device
        if step is None:
            tables = model._rope_tables(self.step.max_tokens)
        if ids is None:
            ids = torch.tensor(tokens, dtype=torch.int64).pin_memory().to(model.device, non_blocking=True)
        embed = model.model.embed_tokens
        read = _decode_rows(embed, ids, positions, tables)
        if read is not None:
            self.x, self.cos, self.sin = read
        else:
            if tables is None:
                self.cos, self.sin = _rope_rows(cfg, positions, model.dtype)
            else:
                self.cos, self.sin = (F.embedding(positions, t) for t in tables)
            self.x = embed(ids).contiguous()
        self.delta = None
        self.handle = None

    def pre(self, index, layer, fused, top_k):
        """Norm, projections, RoPE, append, selection; the gather is left in flight."""
        from . import row_kernels as rk

        cfg, B = self.cfg, len(self.x)
        D, Hq, Hkv = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
        qkv_w, qkv_b, _ = fused
        self.gu_w = fused[2]
        h = rk.add_rmsnorm(self.x, self.delta, layer.input_layernorm.weight, _eps(layer.input_layernorm, cfg))
        if _small_m(h, qkv_w, qkv_b) and D % 16 == 0:  # projection and RoPE in one launch
            qkv = rk.linear_rope(h, qkv_w, qkv_b, Hq + Hkv, D, self.cos, self.sin)
        else:
            qkv = _linear(h, qkv_w, qkv_b)
            rk.rope_(qkv, Hq + Hkv, D, self.cos, self.sin)
        q = qkv[:, : Hq * D].view(B, Hq, D)
        k = qkv[:, Hq * D: (Hq + Hkv) * D].view(B, Hkv, D)
        v = qkv[:, (Hq + Hkv) * D:].view(B, Hkv, D)
        self.step.append(index, k, v)
        self.handle = self.step.select(index, q, top_k)

    def post(self, layer):
        """Attention once the gather is in, output projection, MLP."""
        from . import row_kernels as rk

        cfg, B = self.cfg, len(self.x)
        attention = self.step.finish(self.handle)
        o_proj = layer.self_attn.o_proj
        o = _linear(attention.reshape(B, -1), o_proj.weight, o_proj.bias)
        norm2 = layer.post_attention_layernorm
        h = rk.add_rmsnorm(self.x, o, norm2.weight, _eps(norm2, cfg))
        down = layer.mlp.down_proj
        if _small_m(h, self.gu_w, None) and self.gu_w.shape[0] % 16 == 0:  # gate/up and SiLU in one launch
            act = rk.linear_silu_mul(h, self.gu_w)
        else:
            act = rk.silu_mul(_linear(h, self.gu_w, None))
        self.delta = _linear(act, down.weight, down.bias)


def _decode_rows(embed, ids, positions, tables):
    """The step's embedded tokens and cos/sin rows in one launch, of a plain
    embedding and kept tables; else None (a step of 8 requests and two layers:
    472 us against 492 with three torch lookups)."""
    from . import row_kernels as rk

    if tables is None or not _plain(embed, nn.Embedding) or embed.max_norm is not None:
        return None
    return rk.decode_rows(ids, positions, embed.weight, *tables)


def _linear(x, weight, bias):
    """x @ weight.T + bias for a decode batch: the MFMA weight-stream kernel
    (nhs_linear_small_m) for bf16/fp16 batches of up to 16 rows whose shapes
    it takes, else torch."""
    from . import row_kernels as rk

    if _small_m(x, weight, bias):
        return rk.linear_small_m(x, weight, bias)
    return F.linear(x, weight, bias)


def _small_m(x, weight, bias):
    """Whether the decode projection x @ weight.T (+ bias) fits the
    weight-stream kernels (nhs_linear_small_m and its fused forms)."""
    m, k = x.shape
    n = weight.shape[0]
    return (x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and weight.dtype == x.dtype and m <= 16
            and n % 16 == 0 and k % 2048 == 0 and x.stride(1) == 1 and weight.is_contiguous()
            and (bias is None or bias.is_contiguous()))


def _rope_rows(cfg, positions, dtype):
    """cos and sin [len(positions), head_dim / 2] in `dtype`."""
    D = cfg.head_dim
    inv_freq = cfg.rope_theta ** (-torch.arange(0, D, 2, device=positions.device).float() / D)
    angle = positions.float()[:, None] * inv_freq[None, :]
    return angle.cos().to(dtype).contiguous(), angle.sin().to(dtype).contiguous()


def _plain(module, *kinds):
    """Whether a call of `module` is the forward of one of the `kinds` and
    nothing more, so that a kernel may compute it from the weights: no
    subclass, no forward of the instance's own, no hook."""
    hooks = torch.nn.modules.module
    return (type(module) in kinds and "forward" not in vars(module)
            and not (module._forward_hooks or module._forward_pre_hooks or hooks._global_forward_hooks
                     or hooks._global_forward_pre_hooks))


def _plain_norm(norm, dtype):
    """Whether `norm` is an RMSNorm that nhs_add_rmsnorm computes: this
    module's or Qwen2's (from_pretrained), its weight in the activations'
    dtype."""
    qwen2 = sys.modules.get("transformers.models.qwen2.modeling_qwen2")
    kinds = (RMSNorm,) if qwen2 is None else (RMSNorm, qwen2.Qwen2RMSNorm)
    return _plain(norm, *kinds) and norm.weight.dtype == dtype and norm.weight.is_contiguous()


def _plain_layer(layer, dtype):
    """Whether _prefill_layers computes a layer's prompt pass: plain norms,
    and plain q and k projections, whose outputs it rotates in place."""
    attn = layer.self_attn
    return (_plain_norm(layer.input_layernorm, dtype) and _plain_norm(layer.post_attention_layernorm, dtype)
            and _plain(attn.q_proj, nn.Linear) and _plain(attn.k_proj, nn.Linear))


def _eps(norm, cfg):
    return getattr(norm, "eps", getattr(norm, "variance_epsilon", cfg.rms_norm_eps))


def _fuse(modules, name):
    """Concatenate the modules' `name` parameters along dim 0 and make each
    module's parameter a view of the result (None if any is missing)."""
    params = [getattr(m, name) for m in modules]
    if any(p is None for p in params):
        return None
    whole = torch.cat([p.detach() for p in params], 0)
    row = 0
    for m, p in zip(modules, params):
        n = p.shape[0]
        setattr(m, name, nn.Parameter(whole[row: row + n], requires_grad=p.requires_grad))
        row += n
    return whole
