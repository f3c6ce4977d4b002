"""The batched decode layer's fused elementwise kernels against the torch
expressions they replace (reference model.py:43-71, 140-158), and the fused
batched model step against per-request decoding.

RoPE and the residual adds reproduce torch's roundings exactly (bit-exact);
RMSNorm's mean and SiLU's exp may differ from torch's by their last fp32
bits. For SiLU that shows as at most one unit in the last place after
rounding to bf16/fp16; RMSNorm rounds twice after the mean
(round(round(h * r) * weight)), so a flip of the inner rounding by one unit
can become two units of the output (seen at fp16, 4 x 8192: 0.46 * r rounds
one unit apart, times a weight of 1.06 two units apart). fp32: a relative
1e-6.
"""

import pytest
import torch
from torch.nn import functional as F

from nano_hisparse import row_kernels as rk
from nano_hisparse.config import CacheConfig
from nano_hisparse.hybrid import HotConfig, HybridKVCache
from nano_hisparse.model import Model, ModelConfig, RMSNorm

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def ulp_close(a, b, units=1):
    """|a - b| within `units` units in the last place of b's dtype (fp32: a
    relative 1e-6 per unit, the spread of the mean's reduction order over
    rows of thousands)."""
    a, b = a.float(), b.float()
    eps = units * {torch.float32: 1e-6, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}[ULP_DTYPE[0]]
    tiny = {torch.float32: 1e-30, torch.float16: 6e-8, torch.bfloat16: 1e-30}[ULP_DTYPE[0]]
    return bool(((a - b).abs() <= eps * b.abs() + tiny).all())


ULP_DTYPE = [torch.float32]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
def test_add_rmsnorm_matches_torch(gpu, dtype):
    ULP_DTYPE[0] = dtype
    g = torch.Generator(device=gpu).manual_seed(1)
    for rows, width in ((8, 4096), (16, 3584), (2, 512), (4, 8192), (3, 96), (1, 1000), (2, 8704), (3, 1004)):
        x = torch.randn(rows, width, generator=g, device=gpu).to(dtype)
        delta = torch.randn(rows, width, generator=g, device=gpu).to(dtype)
        norm = RMSNorm(width, 1e-6).to(gpu)
        norm.weight.data = (1 + 0.1 * torch.randn(width, generator=g, device=gpu)).to(dtype)
        want_h = x + delta
        want = norm(want_h)
        got_x = x.clone()
        got = rk.add_rmsnorm(got_x, delta, norm.weight, 1e-6)
        assert torch.equal(got_x, want_h)  # the residual add is exact
        assert ulp_close(got, want, units=2), (rows, width)
        plain = rk.add_rmsnorm(x.clone(), None, norm.weight, 1e-6)
        assert ulp_close(plain, norm(x), units=2), (rows, width)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
def test_rope_matches_the_torch_rotation_bit_exactly(gpu, dtype):
    g = torch.Generator(device=gpu).manual_seed(2)
    rows, heads, D, extra = 5, 12, 64, 3 * 64
    t = torch.randn(rows, heads * D + extra, generator=g, device=gpu).to(dtype)
    angle = torch.rand(rows, D // 2, generator=g, device=gpu) * 1000
    cos, sin = angle.cos().to(dtype), angle.sin().to(dtype)
    # the model's expression: t * cos + cat(-hi, lo) * sin with cos/sin repeated
    view = t[:, : heads * D].view(rows, heads, D)
    c2, s2 = torch.cat((cos, cos), -1)[:, None, :], torch.cat((sin, sin), -1)[:, None, :]
    lo, hi = view.chunk(2, -1)
    want = view * c2 + torch.cat((-hi, lo), -1) * s2
    tail = t[:, heads * D:].clone()
    rk.rope_(t, heads, D, cos.contiguous(), sin.contiguous())
    assert torch.equal(t[:, : heads * D].view(rows, heads, D), want)
    assert torch.equal(t[:, heads * D:], tail)  # v columns untouched


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul_matches_torch(gpu, dtype):
    ULP_DTYPE[0] = dtype
    g = torch.Generator(device=gpu).manual_seed(3)
    gu = (3 * torch.randn(8, 2 * 1000, generator=g, device=gpu)).to(dtype)
    want = F.silu(gu[:, :1000]) * gu[:, 1000:]
    assert ulp_close(rk.silu_mul(gu), want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
# the smallest rows, the edge of a workgroup (256 chunks of 16 bytes) and past it
@pytest.mark.parametrize("B,hidden,half", [(1, 8, 8), (16, 2048, 64), (3, 1936, 64), (7, 4096, 64), (2, 4104, 8)])
def test_decode_rows_reads_the_tables_bit_for_bit(gpu, dtype, B, hidden, half):
    g = torch.Generator(device=gpu).manual_seed(B)
    embed = torch.randn(50, hidden, generator=g, device=gpu).to(dtype)
    cos, sin = (torch.randn(90, half, generator=g, device=gpu).to(dtype) for _ in range(2))
    ids = torch.randint(0, 50, (B,), generator=g, device=gpu)
    positions = torch.randint(0, 90, (B,), generator=g, device=gpu)
    ids[-1], positions[-1] = 49, 89
    x, c, s = rk.decode_rows(ids, positions, embed, cos, sin)
    assert torch.equal(x, embed[ids]) and torch.equal(c, cos[positions]) and torch.equal(s, sin[positions])
    assert rk.decode_rows(ids, positions, embed[:, :-1].contiguous(), cos, sin) is None  # no whole chunks
    assert rk.decode_rows(ids, positions, embed, cos[:, :-1].contiguous(), sin[:, :-1].contiguous()) is None


@pytest.mark.gpu
# (2048, 16, 4): q/k/v and o take nhs_linear_small_m in bf16
@pytest.mark.parametrize("hidden,heads,kv_heads", [(128, 8, 2), (2048, 16, 4)])
@pytest.mark.parametrize("micro_batches", [1, 2])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 0.15)])
def test_fused_batched_step_matches_per_request_decode(gpu, dtype, tol, micro_batches, hidden, heads, kv_heads):
    print("case:", dict(dtype=str(dtype), micro_batches=micro_batches, hidden=hidden), flush=True)
    torch.manual_seed(7)
    cfg = ModelConfig(hidden_size=hidden, intermediate_size=2 * hidden, num_hidden_layers=2,
                      num_attention_heads=heads, num_key_value_heads=kv_heads, vocab_size=100)
    model = Model(cfg).eval().to(gpu).to(dtype)
    caches = [
        HybridKVCache(CacheConfig(gpu_pages=64, host_pages=256, page_size=4, kv_heads=kv_heads,
                                  head_dim=hidden // heads, dtype=dtype, device=gpu),
                      HotConfig(16, 32, resident_window_pages=4))
        for _ in range(2)
    ]
    prompts = {"a": list(range(3, 40)), "b": list(range(1, 23)), "c": list(range(9, 60))}
    tokens = {}
    for c in caches:
        for name, prompt in prompts.items():
            c.reserve(name, len(prompt) + 16, cfg.num_hidden_layers)
            tokens[name] = int(model.prefill(prompt, c, name).argmax())
    for _ in range(6):
        batch = model.decode_batch([tokens[n] for n in prompts], list(prompts), caches[1], 4, micro_batches)
        for i, name in enumerate(prompts):
            single = model.decode(tokens[name], name, caches[0], top_k=4)
            scale = single.abs().max().item()
            assert (batch[i] - single).abs().max().item() <= tol * max(scale, 1.0), name
        tokens = {n: int(batch[i].argmax()) for i, n in enumerate(prompts)}
    for c in caches:
        c.assert_invariants()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,heads,D,extra,offset", [
    (3, 1, 16, 0, 0), (300, 32, 128, 0, 0), (2, 33, 128, 8, 0),  # one chunk; two and three workgroups per row
    (3, 5, 24, 0, 0), (4, 3, 64, 4, 0), (4, 3, 64, 8, 2),  # halves, row strides and addresses off the 16-byte chunks
])
def test_rope_at_the_edges_of_its_chunks(gpu, dtype, rows, heads, D, extra, offset):
    g = torch.Generator(device=gpu).manual_seed(rows)
    width = heads * D + extra
    t = torch.randn(rows * width + offset, generator=g, device=gpu).to(dtype)[offset:].view(rows, width)
    angle = torch.rand(rows, D // 2, generator=g, device=gpu) * 1000
    cos, sin = angle.cos().to(dtype), angle.sin().to(dtype)
    view = t[:, : heads * D].reshape(rows, heads, D)
    c2, s2 = torch.cat((cos, cos), -1)[:, None, :], torch.cat((sin, sin), -1)[:, None, :]
    lo, hi = view.chunk(2, -1)
    want = view * c2 + torch.cat((-hi, lo), -1) * s2
    tail = t[:, heads * D:].clone()
    rk.rope_(t, heads, D, cos, sin)
    assert torch.equal(t[:, : heads * D].reshape(rows, heads, D), want)
    assert torch.equal(t[:, heads * D:], tail)


@pytest.mark.parametrize("dtype", DTYPES)
def test_rope_tables_hold_the_rows_that_a_step_would_compute(monkeypatch, dtype):
    from nano_hisparse import model as model_module

    monkeypatch.setattr(model_module, "ROPE_TABLE_ROWS", 9000)
    model = Model(ModelConfig(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, num_hidden_layers=1)).to(dtype)
    short = model._rope_tables(100)
    assert len(short[0]) == 4096 and model._rope_tables(4096)[0] is short[0]
    long = model._rope_tables(4097)
    assert len(long[0]) == 8192 and model._rope_tables(5)[0] is long[0]
    assert len(model._rope_tables(8500)[0]) == 9000 and model._rope_tables(9001) is None
    positions = torch.tensor([0, 1, 4095, 4096, 8191])
    for table, rows in zip(long, model_module._rope_rows(model.config, positions, dtype)):
        assert torch.equal(F.embedding(positions, table), rows)
    other = {torch.float32: torch.bfloat16}.get(dtype, torch.float32)
    assert model.to(other)._rope_tables(10)[0].dtype == other  # tables of another dtype are made anew


def test_a_captured_groups_tables_are_made_before_it(monkeypatch):
    """Each group of a graph step has tables by its own longest reservation
    (none beyond ROPE_TABLE_ROWS, beside a group that has some), made before
    the capture: a group that is handed its step asks for none."""
    from types import SimpleNamespace

    from nano_hisparse import model as model_module

    monkeypatch.setattr(model_module, "ROPE_TABLE_ROWS", 64)
    model = Model(ModelConfig(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, num_hidden_layers=1))
    lengths = {"long": 65, "short": 50, "shorter": 20}
    store = SimpleNamespace(requests={r: SimpleNamespace(max_tokens=n) for r, n in lengths.items()})
    long, short = model._span_tables(store, list(lengths), [(0, 1), (1, 3)])
    assert long is None and len(short[0]) == 64

    def refused(limit):
        raise AssertionError("a table was asked for within the capture")

    monkeypatch.setattr(model, "_rope_tables", refused)
    monkeypatch.setattr(model_module, "_decode_rows", lambda *a: None)  # a GPU kernel
    positions = torch.tensor([7, 41])
    step = SimpleNamespace(dev_lengths=torch.stack((positions, positions + 1)), max_tokens=50)
    groups = [model_module._Group(model, None, None, None, False, step=step, ids=torch.tensor([1, 2]), tables=t)
              for t in (long, short)]
    assert torch.equal(groups[0].cos, groups[1].cos) and torch.equal(groups[0].sin, groups[1].sin)


def test_no_table_is_made_while_a_stream_is_captured(monkeypatch):
    monkeypatch.setattr(Model, "device", property(lambda self: torch.device("cuda:0")))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: "stream")
    model = Model(ModelConfig(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, num_hidden_layers=1))
    assert model._rope_tables(10) is None and "_rope" not in model.__dict__
    kept = (torch.empty(20, 8), torch.empty(20, 8))
    model._rope = [((model.device, model.dtype, model.config.rope_theta, 16), kept, "stream")]
    assert model._rope_tables(20) is kept and model._rope_tables(21) is None


def test_rope_tables_go_with_what_they_were_made_for(native_launchers):
    """Tables of an earlier dtype are dropped when new ones are made,
    clear_decode_graphs() drops all of them, and a copy of the model carries
    none along."""
    import copy
    import io
    import weakref

    model = Model(ModelConfig(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, num_hidden_layers=1))
    old = [weakref.ref(model._rope_tables(n)[0]) for n in (10, 5000)]
    assert len(model._rope) == 2
    new = model.to(torch.bfloat16)._rope_tables(10)
    assert len(model._rope) == 1 and model._rope_tables(10) is new and all(r() is None for r in old)
    model._fused_projections()
    buffer = io.BytesIO()
    torch.save(model, buffer)
    buffer.seek(0)
    for other in (copy.deepcopy(model), torch.load(buffer, weights_only=False)):
        assert not {"_rope", "_fused", "_decode_graphs"} & set(other.__dict__)
        assert all(torch.equal(a, b) for a, b in zip(other.parameters(), model.parameters()))
        qkv = other._fused_projections()[0][0]
        assert torch.equal(qkv, model._fused_projections()[0][0]) and qkv is not model._fused_projections()[0][0]
    gone = weakref.ref(new[0])
    model.clear_decode_graphs()
    del new
    assert gone() is None
