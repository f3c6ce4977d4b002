"""The native launchers (csrc/launch.cpp) against the Python ones: the same
bits for every form of a call that they take, and every call that they leave
to the Python launchers (wrong shapes, dtypes, devices, or values) raises
what it raised there."""

import pytest
import torch

from nano_hisparse import row_kernels as rk

pytestmark = pytest.mark.gpu

bf16, f16, f32 = torch.bfloat16, torch.float16, torch.float32


class PythonOnly:
    """Stands in for the module: declines every call."""

    def __getattr__(self, name):
        return lambda *a: None


class Counting:
    """The module, counting the calls that it takes."""

    def __init__(self, module):
        self.module, self.taken = module, 0

    def __getattr__(self, name):
        def call(*a):
            done = getattr(self.module, name)(*a)
            self.taken += done is not None
            return done

        return call


def both(monkeypatch, call):
    """call() through the native launchers and through the Python ones; returns whether the native one took it."""
    counting = Counting(rk._load_launch())
    results = []
    for module in (counting, PythonOnly()):
        monkeypatch.setattr(rk, "_launch", module)
        results.append(call())
    for a, b in zip(*[r if isinstance(r, tuple) else (r,) for r in results]):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and a.device == b.device
            assert torch.equal(a, b)
    return counting.taken == 1


@pytest.mark.parametrize("dtype", [bf16, f16])
@pytest.mark.parametrize("m", [1, 16])
def test_linear_launchers(gpu, monkeypatch, dtype, m):
    print("case:", dict(dtype=dtype, m=m), flush=True)
    g = torch.Generator(device=gpu).manual_seed(m)
    k, n = 2048, 96

    def t(*shape):
        return torch.randn(*shape, generator=g, device=gpu).to(dtype)

    x, w, bias, wide = t(m, k), t(n, k), t(n), t(m, 2 * k)
    cos, sin, norm, delta = t(m, 16), t(m, 16), t(k), t(m, k)
    out = torch.empty(m, 2 * n, device=gpu, dtype=dtype)
    assert both(monkeypatch, lambda: rk.linear_small_m(x, w))
    assert both(monkeypatch, lambda: rk.linear_small_m(wide[:, k:], w, bias))
    assert both(monkeypatch, lambda: rk.linear_small_m(x, w, bias, out=out[:, :n]).clone())
    assert both(monkeypatch, lambda: rk.linear_small_m(x, torch.nn.Parameter(w)).detach())
    assert both(monkeypatch, lambda: rk.linear_silu_mul(wide[:, :k], w))
    assert both(monkeypatch, lambda: rk.linear_rope(x, w, bias, 2, 32, cos, sin))
    assert both(monkeypatch, lambda: rk.linear_rope(x, w, None, 0, 32, cos, sin))

    def norm_of(write_back):
        h = x.clone()
        return rk.add_rmsnorm(h, delta, norm, 1e-6, write_back), h

    assert both(monkeypatch, lambda: norm_of(True)) and both(monkeypatch, lambda: norm_of(False))
    assert both(monkeypatch, lambda: rk.add_rmsnorm(x, None, norm, 1e-6))
    assert both(monkeypatch, lambda: rk.add_rmsnorm(x, None, norm, 1))


@pytest.mark.parametrize("dtype,q_dtype", [(bf16, bf16), (f16, f16), (f32, f32), (bf16, f32)])
def test_attention_launchers(gpu, monkeypatch, dtype, q_dtype):
    print("case:", dict(dtype=dtype, q_dtype=q_dtype), flush=True)
    g = torch.Generator(device=gpu).manual_seed(3)
    B, Hq, Hkv, D, P = 3, 4, 2, 64, 8
    pool = rk.padded_pool(40, P, Hkv, D, dtype, gpu)
    pool.copy_(torch.randn(pool.shape, generator=g, device=gpu))
    q = torch.randn(B, Hq + 2, D, generator=g, device=gpu).to(q_dtype)[:, :Hq]  # a batch stride of its own
    rows = torch.randint(-1, 40 * P, (B, Hq, 50), generator=g, device=gpu)
    shared, expanded = rows[:, 0], rows[:, :1].expand(B, Hq, 50)
    rk.attend_batched(q, pool, rows, P)  # the stream's workspace is there from here on
    out = torch.empty(B, 2 * Hq, D, dtype=q_dtype, device=gpu)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu)
    assert both(monkeypatch, lambda: rk.attend_batched(q, pool, shared, P))
    assert both(monkeypatch, lambda: rk.attend_batched(q, pool, rows, P))
    assert both(monkeypatch, lambda: rk.attend_batched(q, pool, expanded, P))
    assert both(monkeypatch, lambda: rk.attend_batched(q, pool, rows[:, 0, ::2], P))
    assert both(monkeypatch, lambda: rk.attend_batched(q, pool, shared, P, out=out[:, ::2], workspace=ws).clone())
    assert not both(monkeypatch, lambda: rk.attend_batched(q, pool, shared[:, :0], P))  # no rows: zeros, no launch
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # a stream without a workspace: the Python launcher makes it
        first = rk.attend_batched(q, pool, shared, P)
    torch.cuda.current_stream().wait_stream(side)
    first.record_stream(torch.cuda.current_stream())
    assert torch.equal(first, rk.attend_batched(q, pool, shared, P))
    if dtype == q_dtype and dtype != f32:
        fused = torch.randn(70, (Hq + 2 * Hkv) * D, generator=g, device=gpu).to(dtype)
        pq, pk, pv = (a.view(70, -1, D) for a in fused.split([Hq * D, Hkv * D, Hkv * D], 1))
        assert both(monkeypatch, lambda: rk.prefill_attention(pq, pk, pv))


@pytest.mark.parametrize("dtype", [bf16, f32])
@pytest.mark.parametrize("as_int", [False, True])
def test_selection_launchers(gpu, monkeypatch, dtype, as_int):
    print("case:", dict(dtype=dtype, as_int=as_int), flush=True)
    g = torch.Generator(device=gpu).manual_seed(4)
    B, Hq, Hkv, D, P, n, top, H = 3, 4, 2, 64, 8, 20, 4, 64
    q = torch.randn(B, Hq, D, generator=g, device=gpu).to(dtype)
    both_bounds = torch.randn(2, B, n + 1, Hkv, D, generator=g, device=gpu).to(dtype)[:, :, :n]
    lo, hi = both_bounds.amin(0).contiguous(), both_bounds.amax(0).contiguous()
    lengths = 150 if as_int else torch.tensor([150, 160, 7], device=gpu)
    for select in (True, False):
        # unselected scores past a request's last page are not written: compare what is
        assert both(monkeypatch, lambda: rk.quest_batched(q, lo, hi, lengths, P, top, select=select)[:2])
    source = torch.arange(B * n, dtype=torch.int32, device=gpu).view(B, n)
    resident = torch.where(source % 3 == 0, source, -1).int()
    hot = torch.arange(B * n, B * n + B * (H // P), dtype=torch.int32, device=gpu).view(B, -1)
    scores = torch.randn(B, n, generator=g, device=gpu)

    def resolve(mode="quest", total=None):
        tags = torch.full((B, H), -1, dtype=torch.int32, device=gpu)
        lru = torch.arange(H, device=gpu).repeat(B, 1)
        return rk.select_resolve_batched(scores, source, resident, hot, tags, lru, lengths, P, top, mode=mode,
                                         counts_total=total) + (tags, lru)

    total = torch.zeros(3, dtype=torch.int64, device=gpu)
    assert both(monkeypatch, resolve)
    assert both(monkeypatch, lambda: resolve("mean", total))
    if not as_int:  # lengths of another type are converted by the Python launcher
        lengths = lengths.int()
        assert not both(monkeypatch, resolve)


def test_calls_the_native_launchers_decline_are_refused_as_before(gpu):
    x, w = torch.randn(1, 2048, device=gpu, dtype=bf16), torch.randn(32, 2048, device=gpu, dtype=bf16)
    with pytest.raises(ValueError, match="x .m, k., weight"):
        rk.linear_small_m(x, w[:, :1024])
    with pytest.raises(ValueError, match="of one dtype"):
        rk.linear_small_m(x, w.half())
    with pytest.raises(ValueError, match="all tensors must be on"):
        rk.linear_silu_mul(x, w.cpu())
    with pytest.raises(ValueError, match="tensors must be on a GPU"):
        rk.linear_silu_mul(x.cpu(), w.cpu())
    with pytest.raises(RuntimeError, match="nhs_linear_small_m failed with status .*m <= 16"):
        rk.linear_small_m(x.expand(17, -1).contiguous(), w)
    pool = rk.padded_pool(4, 8, 2, 64, f32, gpu)
    q, rows = torch.randn(1, 4, 64, device=gpu), torch.zeros(1, 8, dtype=torch.int64, device=gpu)
    with pytest.raises(ValueError, match="int64 rows"):
        rk.attend_batched(q, pool, rows.int(), 8)
    with pytest.raises(ValueError, match="head shape mismatch"):
        rk.attend_batched(q, pool, rows, 16)
    with pytest.raises(ValueError, match="workspace holds"):
        rk.attend_batched(q, pool, rows, 8, workspace=torch.zeros(8, device=gpu))
    with pytest.raises(ValueError, match="share dtype and layout"):
        rk.quest_batched(q, pool[:1, 0].float(), pool[:1, 0].half(), 8, 8, 2)
