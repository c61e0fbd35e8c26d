"""The native host path (csrc/host_ext.cpp) against the Python code that takes every form of a call: the same bits, or the same
exception with the same words, for each form -- with the native functions answering None the general path runs alone."""
import threading

import pytest
import torch

import sparse_transformers_amd as st
from sparse_transformers_amd import _lib

DEV = "cuda:0"


class _Nothing:
    def __getattr__(self, name):
        return lambda *a: None


def test_native_functions_leave_everything_else_to_python():
    """On the CPU: other devices, subclasses, transforms' wrappers, wrong counts and types of arguments."""
    nat = _lib.native()
    x, A, Bm = torch.zeros(1, 16), torch.zeros(8, 16), torch.zeros(32, 8)
    assert nat.predictor_mask(x, A, Bm, 0.0, True, None, None, None, 0, 0) is None
    assert nat.predictor_mask(x, A) is None and nat.update_forward() is None and nat.mlp_forward(1, 2, 3) is None
    assert nat.predictor_mask(None, "a", 3, [], {}, 1.5, x, x, x, x) is None
    assert nat.update_forward(*[x] * 10) is None and nat.mlp_forward(*[None] * 13) is None

    class Sub(torch.Tensor):
        pass
    assert nat.predictor_mask(x.as_subclass(Sub), A, Bm, 0.0, True, None, None, None, 0, 0) is None
    seen = []
    torch.func.vmap(lambda v: (seen.append(nat.mlp_forward(v, None, v, v, 1, None, None, None, 0, v, 0, 0, False)), v)[1])(torch.zeros(2, 3, 4))
    torch.func.grad(lambda v: (seen.append(nat.mlp_forward(v, None, v, v, 1, None, None, None, 0, v, 0, 0, False)), v.sum())[1])(torch.zeros(3, 4))
    assert seen == [None, None]
    with pytest.raises(TypeError):
        nat.bind(1)


def _both(monkeypatch, f):
    """f() with and without the native path: (kind, payload) of each."""
    got = []
    for native in (None, _Nothing()):
        with monkeypatch.context() as m:
            if native is not None:
                m.setattr(_lib, "native", lambda: native)
            try:
                r = f()
                r = r if isinstance(r, (tuple, list)) else (r,)
                torch.cuda.synchronize()
                got.append(("value", [(t.clone(), tuple(t.shape), t.stride(), t.dtype) for t in r]))
            except Exception as e:
                got.append((type(e).__name__, str(e)))
    return got


def _same(a, b):
    if a[0] != "value" or b[0] != "value":
        assert a == b
        return
    for x, y in zip(a[1], b[1]):
        assert x[1:] == y[1:] and torch.equal(x[0], y[0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64, torch.int32])
def test_predictor_mask_forms(monkeypatch, dtype):
    H, r, I, B = 64, 16, 200, 3
    g = torch.Generator().manual_seed(1)
    x, A, Bm = ((torch.randn(s, generator=g) * 2).to(dtype).to(DEV) for s in ((B, H), (r, H), (I, r)))
    f32 = dict(dtype=torch.float32, device=DEV)
    forms = [
        lambda: st.predictor_mask(x, A, Bm, 0.5), lambda: st.predictor_mask(x, A, Bm, 0.5, False, True),
        lambda: st.predictor_mask(x[:1], A, Bm, 0.5, round_to_storage=True), lambda: st.predictor_mask(x[0], A, Bm),
        lambda: st.predictor_mask(x.view(1, B, H), A, Bm), lambda: st.predictor_mask(x.t().contiguous().t(), A, Bm),
        lambda: st.predictor_mask(x, A.t().contiguous().t(), Bm), lambda: st.predictor_mask(x, A, Bm[::2]),
        lambda: st.predictor_mask(x, torch.nn.Parameter(A) if dtype.is_floating_point else A, Bm),
        lambda: st.predictor_mask(x, A[:, :32], Bm), lambda: st.predictor_mask(x, A, Bm[:, :8]), lambda: st.predictor_mask(x, A[0], Bm),
        lambda: st.predictor_mask(x, A.to(torch.float16), Bm), lambda: st.predictor_mask(x, A.cpu(), Bm), lambda: st.predictor_mask(x.cpu(), A, Bm),
        lambda: st.predictor_mask(x, A, Bm, out=torch.zeros(I, dtype=torch.bool, device=DEV)),
        lambda: st.predictor_mask(x, A, Bm, out=torch.zeros(I - 1, dtype=torch.bool, device=DEV)),
        lambda: st.predictor_mask(x, A, Bm, out=torch.zeros(I, dtype=torch.uint8, device=DEV)),
        lambda: st.predictor_mask(x, A, Bm, out=torch.zeros(2 * I, dtype=torch.bool, device=DEV)[::2]),
        lambda: st.predictor_mask(x, A, Bm, t_ws=torch.zeros(B * r, **f32)), lambda: st.predictor_mask(x, A, Bm, t_ws=torch.zeros(3, **f32)),
        lambda: st.predictor_mask(x, A, Bm, t_ws=torch.zeros(B * r)),
        lambda: st.predictor_mask(x, A, Bm, scores_out=torch.zeros(2 * B * I, **f32)),
        lambda: st.predictor_mask(x, A, Bm, scores_out=torch.zeros(3, **f32)), lambda: st.predictor_mask(x, A, Bm, "a"),
        lambda: st.predictor_scores(x[:0], A, Bm), lambda: st.predictor_scores(x, A, Bm),
    ]
    for f in forms:
        _same(*_both(monkeypatch, f))


def _cache(dtype=torch.float16, H=256, I=512, gated=True, seed=2):
    g = torch.Generator().manual_seed(seed)
    gate, up, down = ((torch.randn(s, generator=g) * 0.1).to(dtype).to(DEV) for s in ((I, H), (I, H), (H, I)))
    ones = torch.ones(I, dtype=torch.bool, device=DEV)
    return st.WeightCache(ones, H, gate if gated else None, up, down, gated), g


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [True, False])
def test_cache_call_forms(monkeypatch, gated):
    H, I, B = 256, 512, 4
    x = torch.randn(B, H, generator=torch.Generator().manual_seed(5)).half().to(DEV)
    mask = (torch.rand(I, generator=torch.Generator().manual_seed(6)) < 0.4).to(DEV)

    def fresh(f):
        def run():
            c, _ = _cache(gated=gated)
            r = f(c)
            return (r, c.get_active_indices()) if isinstance(r, torch.Tensor) else (*r, c.get_active_indices())
        return run

    def lazy(c):
        c.lazy_updates = True
        c.update_active_weights(mask)
        return c.update_and_forward(~mask, x)

    def held(c):
        w = c.get_concat_weight()           # alive across the update: filled first
        return c.update_and_forward(mask, x), w + 0
    half = lambda *s: torch.zeros(*s, dtype=torch.float16, device=DEV)
    forms = [
        lambda c: c.update_and_forward(mask, x), lambda c: c.update_and_forward(mask, x[:1], "relu"), lambda c: c.update_and_forward(mask, x[0]),
        lambda c: c.update_and_forward(mask, x.view(2, 2, H)), lambda c: c.update_and_forward(mask.to(torch.uint8) * 3, x),
        lambda c: c.update_and_forward(mask.int(), x), lambda c: c.update_and_forward(mask.cpu(), x), lambda c: c.update_and_forward(mask[:-1], x),
        lambda c: c.update_and_forward(torch.stack([mask, mask], 1)[:, 0], x), lambda c: c.update_and_forward(mask, x.float()),
        lambda c: c.update_and_forward(mask, x[:, :-8]), lambda c: c.update_and_forward(mask, x.t().contiguous().t()),
        lambda c: c.update_and_forward(mask, x, "tanh"), lambda c: c.update_and_forward(mask, x.cpu()), lambda c: c.update_and_forward(mask, x[:0]),
        lambda c: c.update_and_forward(mask, x, out=half(B, H)), lambda c: c.update_and_forward(mask, x, out=half(B, H + 1)),
        lambda c: c.update_and_forward(mask, x, out=half(B, H).float()), lambda c: c.update_and_forward(mask, x, out=half(H, B).t()),
        lambda c: c.update_and_forward(mask, x, workspace=torch.zeros(1 << 24, dtype=torch.uint8, device=DEV)),
        lambda c: c.update_and_forward(mask, x, workspace=torch.zeros(64, dtype=torch.uint8, device=DEV)),
        lambda c: c.update_and_forward(mask, x, workspace=torch.zeros(1 << 24, dtype=torch.int8, device=DEV)),
        lambda c: c.update_and_forward(mask, x, combined=half(B, 2 * I)), lambda c: c.update_and_forward(mask, x, n_hint=7),
        lazy, held,
        lambda c: c.forward(x), lambda c: c.forward(x.view(1, B, H), "relu"), lambda c: c.forward(x[:1], out=half(1, H)),
        lambda c: c.forward(x, out=half(B + 1, H)), lambda c: c.forward(x.float()), lambda c: c.forward(x, "swish"),
        lambda c: c.forward(x, workspace=torch.zeros(8, dtype=torch.uint8, device=DEV)), lambda c: c.forward(x[:, ::1], "gelu_pytorch_tanh"),
    ]
    for f in forms:
        _same(*_both(monkeypatch, fresh(f)))


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [True, False])
def test_operator_forms(monkeypatch, gated):
    monkeypatch.setattr(st.ops, "_warned_layout", True)    # (warns once per process; restored for the test of that)
    H, I, B = 256, 512, 2
    x = torch.randn(B, H, generator=torch.Generator().manual_seed(7)).half().to(DEV)
    mask = (torch.rand(I, generator=torch.Generator().manual_seed(8)) < 0.3).to(DEV)
    half = lambda *s: torch.zeros(*s, dtype=torch.float16, device=DEV)

    def call(f):
        def run():
            c, _ = _cache(gated=gated)
            c.update_active_weights(mask)
            n = c.get_num_active()
            bufs = [half(B, H), half(B, (2 if gated else 1) * n)]
            return (f(c, bufs, n), *bufs)
        return run
    F = st.sparse_mlp_forward
    forms = [
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), *b, "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight() + 0, c.get_active_down_weight(), *b, "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight().contiguous(), *b, "relu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight()[:, :-1], *b, "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight().t(), *b, "silu", gated),        # packed rows are not the
        lambda c, b, n: F(x, c.get_concat_weight(), c.down_active, *b, "silu", gated),                         # operator's [H, n]
        lambda c, b, n: F(x, c.get_concat_weight(), c.down_active[:n], *b, "silu", gated),
        lambda c, b, n: F(x[:1], c.get_concat_weight(), c.get_active_down_weight(), *b, "silu", gated),        # resized
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), b[0].resize_(1, 8), b[1].resize_(3), "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), half(H, B).t(), b[1], "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), b[0], b[1].float(), "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), b[0].cpu(), b[1], "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), b[0], b[0], "silu", gated),   # one buffer for both
        lambda c, b, n: F(x.view(B, 1, H), c.get_concat_weight(), c.get_active_down_weight(), *b, "silu", gated),
        lambda c, b, n: F(x.float(), c.get_concat_weight(), c.get_active_down_weight(), *b, "silu", gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), *b, "silu", not gated),
        lambda c, b, n: F(x, c.get_concat_weight(), c.get_active_down_weight(), *b, "cube", gated),
        lambda c, b, n: (lambda w, d: (c.update_active_weights(~mask), F(x, w, d, *b, "silu", gated))[1])(c.get_concat_weight(), c.get_active_down_weight()),
    ]
    for f in forms:
        _same(*_both(monkeypatch, call(f)))


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [True, False])
def test_operator_with_as_many_active_rows_as_columns(monkeypatch, gated):
    """n = H: the shape does not tell [H, n] from packed [n, H] rows.  A row-major down weight is the matrix it says it is."""
    monkeypatch.setattr(st.ops, "_warned_layout", True)
    H, I, B = 256, 1024, 3
    c, g = _cache(H=H, I=I, gated=gated)
    c.update_active_weights((torch.randperm(I, generator=g) < H).to(DEV))
    x = torch.randn(B, H, generator=g).half().to(DEV)
    view = c.get_active_down_weight()
    assert tuple(view.shape) == (H, H)
    h = torch.nn.functional.silu(x.float() @ (c.gate_active if gated else c.up_active)[:H].float().t())
    if gated:
        h = h * (x.float() @ c.up_active[:H].float().t())
    for down in (view, view.contiguous(), view.t(), c.down_active[:H]):
        def call():
            bufs = [torch.zeros(B, k, dtype=torch.float16, device=DEV) for k in (H, (2 if gated else 1) * H)]
            return (st.sparse_mlp_forward(x, c.get_concat_weight(), down, *bufs, "silu", gated), *bufs)
        a, b = _both(monkeypatch, call)
        _same(a, b)
        # (fp32 sums of fp16 operands, the intermediate in fp32 or rounded once, one rounding of the output: 2^-11 each)
        want = h @ down.float().t()
        assert (a[1][0][0].float() - want).abs().max() <= 2 * 2.0 ** -11 * (h.abs() @ down.float().abs().t()).max()


@pytest.mark.gpu
def test_refused_calls_leave_the_workspace_alone(monkeypatch):
    """Calls whose x the general path refuses must not have grown the scratch that is kept for the process."""
    c, _ = _cache()
    mask = torch.ones(512, dtype=torch.bool, device=DEV)
    w, d = c.get_concat_weight(), c.get_active_down_weight()
    asked = []
    kept = st.ops._kept_workspace
    for module in (st.ops, st.weight_cache):
        monkeypatch.setattr(module, "_kept_workspace", lambda dev, need: (asked.append(need), kept(dev, need))[1])
    half = lambda *s: torch.zeros(*s, dtype=torch.float16, device=DEV)
    for x in (half(4000, 248), torch.zeros(4000, 256, device=DEV), half(30, 100, 248), torch.zeros(30, 100, 256, dtype=torch.bfloat16, device=DEV)):
        for call in (lambda: c.forward(x), lambda: c.update_and_forward(mask, x), lambda: st.sparse_mlp_forward(x, w, d, half(1, 256), half(1, 8))):
            with pytest.raises((ValueError, TypeError)):
                call()
    assert asked == []
    for rows in (0, 5000):
        with pytest.raises(ValueError):
            c.forward(half(rows, 256))
    assert not {0, 5000} & set(c._ws_need)


@pytest.mark.gpu
def test_threads_and_streams():
    """Several threads, each with a cache and a stream of its own, through the native path: the results of one thread alone."""
    c0, _ = _cache()
    x = torch.randn(1, 256, generator=torch.Generator().manual_seed(9)).half().to(DEV)
    masks = [(torch.rand(512, generator=torch.Generator().manual_seed(i)) < 0.3).to(DEV) for i in range(6)]
    sequence = lambda c: [c.update_and_forward(m, x).clone() for _ in range(20) for m in masks]   # (the list's order has a history)
    want = sequence(c0)
    caches = [_cache()[0] for _ in range(4)]
    torch.cuda.synchronize()
    got = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = sequence(caches[i])
            torch.cuda.current_stream().synchronize()
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert all(torch.equal(a, b) for g in got for a, b in zip(g, want))


@pytest.mark.gpu
@pytest.mark.parametrize("I,H,gated,dtype", [(1, 64, True, torch.float32), (203, 72, False, torch.float16), (2048, 256, True, torch.bfloat16)])
def test_cache_construction_forms(I, H, gated, dtype, monkeypatch):
    """A cache built by the native path and by the general one, which takes every other form of the arguments (strided weights, a
    mask of numbers or on the host), hold the same; sizes and types that do not fit are refused by either."""
    g = torch.Generator(device=DEV).manual_seed(I)
    gate, up, down = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((I, H), (I, H), (H, I)))
    mask = torch.rand(I, generator=g, device=DEV) < 0.7
    mask[0] = True
    native = st._lib.native()
    with monkeypatch.context() as m:
        m.setattr(st.WeightCache, "_build", None)          # only the native path can make it
        fast = st.WeightCache(mask, H, gate if gated else None, up, down, gated)
    strided = down.t().contiguous().t()
    for args in ((mask.float(), H, gate, up, down), (mask.cpu(), H, gate, up, down), (mask, H, gate, up, strided)):
        if args[4] is strided and I == 1:
            continue                                       # (one column: contiguous either way)
        assert native.cache_build(args[2] if gated else None, args[3], args[4], args[0], H, st._lib.STATE_WORDS,
                                  torch.cuda.current_stream().cuda_stream) is None
        slow = st.WeightCache(args[0], args[1], args[2] if gated else None, *args[3:], gated)
        assert fast.sync_state() == slow.sync_state() and (fast.intermediate_size, fast.hidden_size) == (I, H)
        n = fast.get_num_active()
        for name in ("gate_pool", "up_pool", "downT_pool", "gate_active", "up_active", "down_active", "indices", "cur_mask", "state"):
            a, b = getattr(fast, name), getattr(slow, name)
            assert (a is None) == (b is None) == (name.startswith("gate") and not gated)
            if a is not None:
                assert a.shape == b.shape and a.dtype == b.dtype
                e = int(fast.sync_state()["epoch"])
                rows = slice(0, n) if name.endswith("active") else e if name == "cur_mask" else slice(None)
                assert torch.equal(a[e, :n], b[e, :n]) if name == "indices" else torch.equal(a[rows], b[rows]), name
    for bad in ((mask, H + 8, gate, up, down), (mask, H, gate, up, down[:, :-1] if I > 1 else down[:-1]), (mask[:-1], H, gate, up, down),
                (mask, H, gate.double(), up.double(), down.double())):
        with pytest.raises((ValueError, TypeError)):
            st.WeightCache(bad[0], bad[1], bad[2] if gated else None, *bad[3:], gated)
    # (weight_cache.h:223-226,237-240: a first mask that is all False is the mask the cache begins with, and no error)
    assert st.WeightCache(torch.zeros_like(mask), H, gate if gated else None, up, down, gated).get_num_active() == 0
