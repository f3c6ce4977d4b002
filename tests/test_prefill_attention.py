"""Causal GQA prefill attention (nhs_prefill_attention) against an fp32
reference of the dense causal softmax attention that Model.prefill computes
(reference model.py:170-180): bf16 within 2e-2 and fp16 within 1e-2 max-abs,
over ragged lengths (not multiples of the 64-row tiles), GQA groups of 1, 4
and 7, head_dim 64 and 128, and strided q/k/v views of one fused projection."""

import pytest
import torch

from nano_hisparse import row_kernels as rk


def reference(q, k, v):
    S, Hq, D = q.shape
    g = Hq // k.shape[1]
    qf = q.float().transpose(0, 1)  # [Hq, S, D]
    kf = k.float().repeat_interleave(g, 1).transpose(0, 1).contiguous()
    vf = v.float().repeat_interleave(g, 1).transpose(0, 1).contiguous()
    scores = torch.matmul(qf, kf.transpose(1, 2).contiguous()) / D**0.5
    mask = torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1)
    scores.masked_fill_(mask, float("-inf"))
    return torch.matmul(scores.softmax(-1), vf).transpose(0, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2e-2), (torch.float16, 1e-2)])
@pytest.mark.parametrize("S,Hq,Hkv,D", [(1, 8, 8, 128), (7, 4, 1, 64), (64, 8, 2, 128), (65, 28, 4, 128),
                                          (200, 32, 8, 128), (1000, 8, 2, 64), (513, 4, 4, 128)])
def test_prefill_attention_matches_fp32_reference(gpu, dtype, tol, S, Hq, Hkv, D):
    print("case:", dict(S=S, Hq=Hq, Hkv=Hkv, D=D, dtype=str(dtype)), flush=True)
    g = torch.Generator(device=gpu).manual_seed(S * 31 + Hq)
    fused = torch.randn(S, (Hq + 2 * Hkv) * D, generator=g, device=gpu).to(dtype)
    q = fused[:, : Hq * D].view(S, Hq, D)
    k = fused[:, Hq * D: (Hq + Hkv) * D].view(S, Hkv, D)
    v = fused[:, (Hq + Hkv) * D:].view(S, Hkv, D)
    out = rk.prefill_attention(q, k, v)
    want = reference(q, k, v)
    err = (out.float() - want).abs().max().item()
    assert err <= tol, err


@pytest.mark.gpu
def test_prefill_attention_rejects_unsupported_inputs(gpu):
    q = torch.randn(8, 4, 96, device=gpu, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="head_dim"):
        rk.prefill_attention(q, q[:, :2], q[:, :2])
    with pytest.raises(ValueError, match="bf16 or fp16"):
        x = torch.randn(8, 4, 64, device=gpu)
        rk.prefill_attention(x, x, x)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_model_prefill_runs_the_flash_kernel(gpu, dtype, monkeypatch):
    """A bf16/fp16 GPU model's prefill calls nhs_prefill_attention; its
    logits match the same model with the attention swapped for the fp32
    reference (rounded to the model dtype)."""
    from nano_hisparse.model import Model, ModelConfig

    print("case:", dict(test="model-prefill", dtype=str(dtype)), flush=True)
    torch.manual_seed(3)
    cfg = ModelConfig(hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=4,
                      num_key_value_heads=2, vocab_size=128)
    model = Model(cfg).to(gpu, dtype).eval()
    tokens = list(torch.randint(0, 128, (150,)).tolist())
    calls = []
    kernel = rk.prefill_attention

    def counted(q, k, v):
        calls.append(q.shape)
        return kernel(q, k, v)

    monkeypatch.setattr(rk, "prefill_attention", counted)
    got = model.prefill(tokens)
    assert len(calls) == cfg.num_hidden_layers
    monkeypatch.setattr(rk, "prefill_attention", lambda q, k, v: reference(q, k, v).to(q.dtype))
    want = model.prefill(tokens)
    err = (got - want).abs().max().item()
    assert err <= 5e-2 * max(1.0, want.abs().max().item()), err


@pytest.mark.gpu
@pytest.mark.parametrize("S,Hq,Hkv,D", [
    # rounds of two 64-key tiles, workgroups of 128 queries: one tile short of, at and past their edges
    (63, 8, 2, 128), (127, 3, 1, 64), (128, 3, 1, 128), (129, 8, 2, 64), (191, 5, 5, 128), (193, 2, 2, 64),
    (255, 1, 1, 128), (257, 28, 4, 128), (384, 14, 2, 64), (641, 4, 2, 64),
    # enough workgroups of 256 queries that each takes every tile
    (769, 128, 4, 128), (1025, 96, 8, 64), (3073, 32, 8, 128),
])
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2e-2), (torch.float16, 1e-2)])
def test_prefill_attention_at_the_edges_of_tiles_and_rounds(gpu, dtype, tol, S, Hq, Hkv, D):
    test_prefill_attention_matches_fp32_reference(gpu, dtype, tol, S, Hq, Hkv, D)


@pytest.mark.gpu
def test_prefill_attention_of_infinite_and_nan_scores(gpu):
    """A query that is NaN or meets an infinite score is NaN as in the dense
    softmax, and the queries before the key that is infinite are untouched;
    keys whose scores are -inf carry no weight."""
    g = torch.Generator(device=gpu).manual_seed(9)
    S, Hq, Hkv, D = 300, 2, 1, 64
    q, k, v = (torch.randn(S, h, D, generator=g, device=gpu).half() for h in (Hq, Hkv, Hkv))
    q[10, 0, 0] = float("nan")
    q[:, 1, 3] = q[:, 1, 3].abs() + 0.5
    k[200, 0] = 0
    k[200, 0, 3] = float("-inf")  # -inf for head 1's queries (0 * inf is not met: the rest of the key is finite)
    q[:, 0, 3] = -q[:, 0, 3].abs() - 0.5  # +inf for head 0's
    out = rk.prefill_attention(q, k, v)
    want = reference(q, k, v)
    for h in (0, 1):
        a, b = out[:, h].float(), want[:, h]
        assert torch.equal(a.isnan(), b.isnan())
        assert (a - b)[~b.isnan()].abs().max().item() <= 1e-2
    assert out[10, 0].isnan().all() and out[200:, 0].isnan().all() and not out[:, 1].isnan().any()


@pytest.mark.gpu
@pytest.mark.parametrize("S,Hq,Hkv,D", [(500, 2, 1, 64), (4001, 2, 1, 128), (3100, 32, 8, 128)])
@pytest.mark.parametrize("dtype,subnormal", [(torch.float16, 16), (torch.float16, 22), (torch.bfloat16, 16)])
def test_prefill_attention_of_one_dominating_key_and_many_small_ones(gpu, dtype, subnormal, S, Hq, Hkv, D):
    """Weights of 2^-subnormal beside one of 1 (fp16: subnormal numbers) count
    alike in the numerator (MFMA) and the denominator (packed dot products):
    the values are 0 for the dominating key and 1 for the others, so an
    output is S / (1 + S) with S the small weights' sum, and flushing them in
    either sum alone would show as S or as S^2.

    A weight is rounded to the dtype: by half a unit in the last place, 2^-25
    at most for an fp16 weight below 2^-13 and 2^-8 of itself in bf16 (eight
    significant bits). So S is off by at most n * 2^-25 or 2^-8 * S, and the
    output by that and its own rounding, 2^-11 or 2^-8 of itself (plus one
    subnormal unit, 2^-24)."""
    print("case:", dict(S=S, Hq=Hq, Hkv=Hkv, D=D, dtype=str(dtype), subnormal=subnormal), flush=True)
    q, k, v = (torch.zeros(S, h, D, device=gpu, dtype=dtype) for h in (Hq, Hkv, Hkv))
    q[..., 0] = 8
    k[0, :, 0] = subnormal * 0.6931471805599453 * D**0.5 / 8
    v[1:] = 1
    out = rk.prefill_attention(q, k, v).double()
    small = torch.exp(-8 * k[0, 0, 0].double() * D**-0.5)  # a small key's weight, the dominating one's being 1
    n = torch.arange(S, device=gpu, dtype=torch.float64)  # small keys that a query sees
    total = n * small
    want = (total / (1 + total))[:, None, None].expand_as(out)
    half_unit, rounding = (2.0**-25 * n, 2.0**-11) if dtype == torch.float16 else (2.0**-8 * total, 2.0**-8)
    bound = half_unit[:, None, None] + rounding * want + 2.0**-24
    assert ((out - want).abs() <= bound).all(), ((out - want).abs() / bound).max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2e-2), (torch.float16, 1e-2)])
@pytest.mark.parametrize("S,Hq,Hkv,D", [(12345, 4, 2, 128), (24000, 2, 1, 64)])
def test_prefill_attention_of_long_prompts(gpu, dtype, tol, S, Hq, Hkv, D):
    """The last 300 queries, which see every tile of a long prompt."""
    print("case:", dict(S=S, Hq=Hq, Hkv=Hkv, D=D, dtype=str(dtype)), flush=True)
    g = torch.Generator(device=gpu).manual_seed(S)
    q, k, v = (torch.randn(S, h, D, generator=g, device=gpu).to(dtype) for h in (Hq, Hkv, Hkv))
    out = rk.prefill_attention(q, k, v)[-300:].float()
    mask = torch.arange(S, device=gpu) > torch.arange(S - 300, S, device=gpu)[:, None]
    for h in range(Hq):
        scores = q[-300:, h].float() @ k[:, h * Hkv // Hq].float().t().contiguous() * D**-0.5
        want = scores.masked_fill_(mask, float("-inf")).softmax(-1) @ v[:, h * Hkv // Hq].float()
        # outputs are sums of thousands of values of 1 / thousands each: hundredths, not ones
        assert (out[:, h] - want).abs().max().item() <= tol * 0.1, h


# ---- the prompt pass ------------------------------------------------------------------------


def rms_norm(x, weight, eps):
    xf = x.float()
    return (xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + eps)).to(x.dtype) * weight


@pytest.fixture(params=["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)])
def prompt_device(request, monkeypatch):
    """The device of a model whose prompt pass is the one of a GPU model: on
    the CPU its kernels are their torch expressions."""
    from nano_hisparse import model as model_module

    if request.param != "cpu":
        return request.getfixturevalue("gpu")

    def add_rmsnorm(x, delta, weight, eps, write_back=True):
        h = x if delta is None else x.add_(delta) if write_back else x + delta
        return rms_norm(h, weight, eps)

    def rope_(t, heads, head_dim, cos, sin):
        view = t.view(len(t), heads, head_dim)
        lo, hi = view.chunk(2, -1)
        c, s = torch.cat((cos, cos), -1)[:, None], torch.cat((sin, sin), -1)[:, None]
        view.copy_(view * c + torch.cat((-hi, lo), -1) * s)

    monkeypatch.setattr(model_module.Model, "device", property(lambda self: torch.device("cuda:0")))
    monkeypatch.setattr(model_module, "upload", lambda values, dtype, device: torch.tensor(values, dtype=dtype))
    monkeypatch.setattr(rk, "add_rmsnorm", add_rmsnorm)
    monkeypatch.setattr(rk, "rope_", rope_)
    monkeypatch.setattr(rk, "prefill_attention", lambda q, k, v: reference(q, k, v).to(q.dtype))
    return "cpu"


def prompt_model(device, dtype, head_dim=64, layers=2, seed=3):
    from nano_hisparse.model import Model, ModelConfig

    torch.manual_seed(seed)
    cfg = ModelConfig(hidden_size=4 * head_dim, intermediate_size=512, num_hidden_layers=layers,
                      num_attention_heads=4, num_key_value_heads=2, vocab_size=128)
    model = Model(cfg).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name:
                p.copy_(1 + 0.2 * torch.randn_like(p))
    return model.to(device, dtype)


TOKENS = [(7 * i * i + 3 * i) % 128 for i in range(70)]


@pytest.mark.parametrize("where", ["norm1", "norm2", "norm", "lm_head"])
def test_prompt_pass_calls_the_modules_that_are_not_plain(prompt_device, where):
    """Forward hooks on the norms and the head run, and a norm or head of
    another kind computes what it defines."""
    print("case:", dict(test="prompt-modules", device=str(prompt_device), where=where), flush=True)
    dtype = torch.bfloat16
    plain = prompt_model(prompt_device, dtype)
    want = plain.prefill(TOKENS)

    def replace(model, make):
        layer = model.model.layers[1]
        owner, name = {"norm1": (layer, "input_layernorm"), "norm2": (layer, "post_attention_layernorm"),
                       "norm": (model.model, "norm"), "lm_head": (model, "lm_head")}[where]
        setattr(owner, name, make(getattr(owner, name)))

    class Scaled(torch.nn.Module):  # the module with another parametrisation of its weight, exact: 4 * (w / 4)
        def __init__(self, inner):
            super().__init__()
            self.inner = inner
            with torch.no_grad():
                inner.weight.div_(4)
            self.eps, self.bias = getattr(inner, "eps", None), None

        @property
        def weight(self):
            return self.inner.weight

        def forward(self, x):
            w = self.inner.weight * 4
            return torch.nn.functional.linear(x, w) if self.eps is None else rms_norm(x, w, self.eps)

    calls = []

    def hooked(module):
        module.register_forward_hook(lambda m, args, out: calls.append(out.shape))
        return module

    def hooked_first(module):
        module.register_forward_pre_hook(lambda m, args: calls.append(args[0].shape))
        return module

    def own_forward(module):
        forward = module.forward
        module.forward = lambda x: calls.append(x.shape) or forward(x)
        return module

    for make in (hooked, hooked_first, own_forward):
        calls.clear()
        model = prompt_model(prompt_device, dtype)
        replace(model, make)
        got = model.prefill(TOKENS)
        assert len(calls) == 1, make.__name__
        assert (got - want).norm() <= 2e-2 * want.norm(), make.__name__
    model = prompt_model(prompt_device, dtype)
    replace(model, Scaled)
    got = model.prefill(TOKENS)
    assert (got - want).norm() <= 2e-2 * want.norm()


def test_prompt_pass_leaves_what_hooks_hold(prompt_device):
    """q, k and the embedded rows that a hook keeps are the modules' outputs,
    not the rotated and accumulated rows."""
    print("case:", dict(test="prompt-hooks", device=str(prompt_device)), flush=True)
    model = prompt_model(prompt_device, torch.bfloat16)
    want = model.prefill(TOKENS)
    attn = model.model.layers[0].self_attn
    for module in (model.model.embed_tokens, attn.q_proj, attn.k_proj):
        held = []
        hook = module.register_forward_hook(lambda m, args, out: held.append((args[0], out, out.clone())))
        got = model.prefill(TOKENS)
        hook.remove()
        (_, out, copy), = held
        assert torch.equal(out, copy)
        assert (got - want).norm() <= 2e-2 * want.norm()


def test_the_norms_of_both_model_sources_are_plain():
    """Qwen2's own norm and layer (from_pretrained) take the fused prompt pass
    as this package's do; a subclass does not."""
    from nano_hisparse.model import RMSNorm, _plain, _plain_layer, _plain_norm

    modeling = pytest.importorskip("transformers.models.qwen2.modeling_qwen2")
    transformers = pytest.importorskip("transformers")
    cfg = transformers.Qwen2Config(vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1,
                                   num_attention_heads=4, num_key_value_heads=2)
    hf = transformers.Qwen2ForCausalLM(cfg).eval()
    model = prompt_model("cpu", torch.float32, layers=1)
    for m in (hf, model):
        assert _plain_layer(m.model.layers[0], torch.float32) and _plain_norm(m.model.norm, torch.float32)
        assert not _plain_norm(m.model.norm, torch.bfloat16)
        assert _plain(m.lm_head, torch.nn.Linear) and _plain(m.model.embed_tokens, torch.nn.Embedding)

    class Other(RMSNorm):
        pass

    assert not _plain_norm(Other(8, 1e-6), torch.float32) and _plain_norm(RMSNorm(8, 1e-6), torch.float32)
    assert isinstance(hf.model.norm, modeling.Qwen2RMSNorm)
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not _plain_norm(model.model.norm, torch.float32)
    handle.remove()


def test_the_batched_steps_head_calls_modules_that_are_not_plain():
    """The decode step's last norm and lm_head (of one group and of two): a
    hooked norm sees every row once, a hooked head too."""
    from nano_hisparse.model import _Last

    model = prompt_model("cpu", torch.float32, layers=1)
    x, delta = torch.randn(5, 256), torch.randn(5, 256)
    want = torch.nn.functional.linear(rms_norm(x + delta, model.model.norm.weight, 1e-6), model.lm_head.weight)
    seen = []
    model.model.norm.register_forward_hook(lambda m, args, out: seen.append(("norm", out.shape)))
    model.lm_head.register_forward_hook(lambda m, args, out: seen.append(("lm_head", out.shape)))
    for cuts in ([0, 5], [0, 3, 5]):
        seen.clear()
        with torch.inference_mode():
            got = model._head([_Last(x[a:b], delta[a:b]) for a, b in zip(cuts, cuts[1:])])
        assert seen == [("norm", (5, 256)), ("lm_head", (5, 128))]
        torch.testing.assert_close(got, want)


def test_prompt_pass_of_no_layers(prompt_device):
    print("case:", dict(test="prompt-no-layers", device=str(prompt_device)), flush=True)
    model = prompt_model(prompt_device, torch.bfloat16, layers=0)
    with torch.inference_mode():
        row = model.model.embed_tokens.weight[TOKENS[-1]]
        want = torch.nn.functional.linear(rms_norm(row, model.model.norm.weight, 1e-6), model.lm_head.weight)
    assert torch.equal(model.prefill(TOKENS), want.float())


def exact_prompt(model, tokens):
    """Logits of the last token and each layer's keys and values, in float64
    from the model's weights."""
    cfg, n = model.config, len(tokens)
    D, groups = cfg.head_dim, cfg.num_attention_heads // cfg.num_key_value_heads

    def norm(x, m):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + m.eps) * m.weight.double()

    def linear(x, m):
        y = x @ m.weight.double().t().contiguous()
        return y if m.bias is None else y + m.bias.double()

    x = model.model.embed_tokens.weight[tokens].double()
    angle = torch.arange(n, device=x.device).double()[:, None] * cfg.rope_theta ** (
        -torch.arange(0, D, 2, device=x.device).double() / D)
    cos, sin = (torch.cat((f, f), -1)[:, None] for f in (angle.cos(), angle.sin()))
    mask = torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1)
    kv = []
    for layer in model.model.layers:
        h, a = norm(x, layer.input_layernorm), layer.self_attn
        q, k, v = (linear(h, p).view(n, -1, D) for p in (a.q_proj, a.k_proj, a.v_proj))
        q, k = (t * cos + torch.cat((-t[..., D // 2:], t[..., : D // 2]), -1) * sin for t in (q, k))
        kv += [k, v]
        heads = []
        for i in range(cfg.num_attention_heads):
            scores = (q[:, i] @ k[:, i // groups].t().contiguous() * D**-0.5).masked_fill(mask, float("-inf"))
            heads.append(scores.softmax(-1) @ v[:, i // groups])
        x = x + linear(torch.cat(heads, -1), a.o_proj)
        h = norm(x, layer.post_attention_layernorm)
        x = x + linear(torch.nn.functional.silu(linear(h, layer.mlp.gate_proj)) * linear(h, layer.mlp.up_proj),
                       layer.mlp.down_proj)
    return [linear(norm(x[-1], model.model.norm), model.lm_head), *kv]


class Written:
    """A cache that keeps what is written to it."""

    def __init__(self):
        from types import SimpleNamespace

        self.rows = []
        self.storage = SimpleNamespace(requests={"r": SimpleNamespace(lengths=[0])})

    def write(self, request_id, layer, k, v):
        assert request_id == "r" and layer == len(self.rows) // 2
        self.rows += [k.clone(), v.clone()]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n", [1, 70, 333])
def test_prompt_pass_is_as_exact_as_the_general_one(prompt_device, monkeypatch, dtype, head_dim, n):
    """Logits and the keys and values of every layer, of the fused prompt pass
    and of the general expressions, against float64. Both round at the same
    places of each layer, so their errors are the same but for single
    roundings that fall the other way: a quarter more is allowed, where a
    residual, a norm, a position or a row that is not the right one would
    show as an error of the size of the result."""
    from nano_hisparse import model as model_module

    print("case:", dict(test="prompt-exact", device=str(prompt_device), dtype=str(dtype), D=head_dim, n=n), flush=True)
    model = prompt_model(prompt_device, dtype, head_dim, layers=3)
    tokens = [(7 * i * i + 3 * i) % 128 for i in range(n)]
    with torch.inference_mode():
        want = exact_prompt(model, tokens)
    passes = []
    fused_pass = model_module.Model._prefill_layers

    def counted(self, *a):
        passes.append(1)
        return fused_pass(self, *a)

    monkeypatch.setattr(model_module.Model, "_prefill_layers", counted)
    results = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(model_module, "_plain_layer", lambda layer, dtype: False)
        cache = Written()
        logits = model.prefill(tokens, cache, "r")
        assert torch.equal(logits, model.prefill(tokens))  # without a cache
        results.append([logits, *cache.rows])
    assert len(passes) == 2  # the fused pass ran, with and without the cache, and only in the first round
    for name, exact, fused, general in zip(["logits", *"kvkvkv"], want, *results):
        size = exact.norm()
        a, b = ((r.double() - exact).norm() / size for r in (fused, general))
        assert a <= 1.25 * b and b <= 3e-2, (name, a.item(), b.item())
