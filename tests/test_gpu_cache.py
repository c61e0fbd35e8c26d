"""Differential weight cache on the GPU vs the oracle / golden traces: ordered index list and cache
layout must be bit-exact (integer and byte work)."""
import numpy as np
import pytest
import torch

import oracle
import sparse_transformers_amd as st
from sparse_transformers_amd import synthetic as syn
from conftest import bits_to_mask, golden_weights

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _t(a, dtype=torch.float32):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(DEV, dtype)


def _check_layout(wc, oc_order, gate, up, down, has_gate):
    n = len(oc_order)
    assert wc.get_num_active() == n
    assert wc.get_active_indices().cpu().tolist() == list(oc_order)
    cw = wc.get_concat_weight()
    assert cw.is_contiguous() and cw.shape == ((2 if has_gate else 1) * n, up.shape[1])
    cw = cw.float().cpu().numpy()
    if has_gate:
        assert np.array_equal(cw[:n], gate[oc_order])
    assert np.array_equal(cw[-n:] if n else cw, up[oc_order])
    dw = wc.get_active_down_weight()
    assert dw.shape == (up.shape[1], n) and (n == 0 or dw.stride() == (1, up.shape[1]))
    assert np.array_equal(dw.float().cpu().numpy(), down[:, oc_order])


def test_golden_traces_from_reference(golden_traces):
    for trace in golden_traces:
        I, H, hg = trace["I"], trace["H"], trace["has_gate"]
        gate, up, down = golden_weights(I, H)
        wc = st.WeightCache(_t(bits_to_mask(trace["init_mask"]), torch.bool), H, _t(gate) if hg else None, _t(up),
                            _t(down), hg)
        _check_layout(wc, trace["init_order"], gate, up, down, hg)
        for step in trace["steps"]:
            m = _t(bits_to_mask(step["mask"]), torch.bool)
            if step["error"]:
                with pytest.raises(RuntimeError, match="No active weights"):
                    wc.update_active_weights(m)
                continue
            wc.update_active_weights(m)
            assert wc.get_active_indices().cpu().tolist() == step["order"], trace["seed"]
        _check_layout(wc, trace["steps"][-1]["order"], gate, up, down, hg)


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("has_gate", [True, False])
def test_ragged_traces_vs_oracle(dtype, has_gate):
    tdt = getattr(torch, dtype)
    rng = np.random.default_rng(7)
    for I, H in [(5, 8), (64, 8), (1000, 24), (2051, 16)]:
        g = torch.randn(I, H).to(tdt)
        u = torch.randn(I, H).to(tdt)
        d = torch.randn(H, I).to(tdt)
        gf, uf, df = g.float().numpy(), u.float().numpy(), d.float().numpy()
        trace = syn.ragged_mask_trace(int(rng.integers(1 << 30)), I, 80)
        oc = oracle.OracleWeightCache(trace[0], H, gf if has_gate else None, uf, df, has_gate)
        wc = st.WeightCache(_t(trace[0], torch.bool), H, g.to(DEV) if has_gate else None, u.to(DEV), d.to(DEV), has_gate)
        for t in range(1, len(trace)):
            oc.update_active_weights(trace[t])
            wc.update_active_weights(_t(trace[t], torch.bool))
            assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist(), (I, t)
            if t % 16 == 0:
                _check_layout(wc, oc.get_active_indices().tolist(), gf, uf, df, has_gate)
        _check_layout(wc, oc.get_active_indices().tolist(), gf, uf, df, has_gate)


@pytest.mark.parametrize("I,n,lo,hi", [(8192, 2867, 0.05, 0.15), (14336, 3584, 0.10, 0.10), (11008, 1100, 0.2, 0.2)])
def test_full_size_index_order(I, n, lo, hi):
    """Index order at the real intermediate sizes (the order does not depend on H, so H is kept small)."""
    H = 8
    rng = np.random.default_rng(1)
    g = rng.standard_normal((I, H)).astype(np.float32)
    u = rng.standard_normal((I, H)).astype(np.float32)
    d = rng.standard_normal((H, I)).astype(np.float32)
    trace = syn.mask_trace(5, 1, I, n, 128, lo, hi)[:, 0]
    oc = oracle.OracleWeightCache(np.ones(I, bool), H, g, u, d, True)
    wc = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, _t(g), _t(u), _t(d), True)
    for t in range(len(trace)):
        oc.update_active_weights(trace[t])
        wc.update_active_weights_async(_t(trace[t], torch.bool))   # no read-back between updates
        if t % 32 == 0 or t == len(trace) - 1:
            assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist(), t
    _check_layout(wc, oc.get_active_indices().tolist(), g, u, d, True)
    st_ = wc.sync_state()
    assert st_["n_active"] == n and st_["n_added"] == st_["n_removed"] > 0


@pytest.mark.parametrize("I", [7, 1025, 8192, 14336, 16001, 22000])
def test_surplus_removals(I):
    """Updates that remove more than they add, in the stand-alone update kernel: everything but one index at once, a few
    and a few thousand, removals that sit at the end of the list (each step's moved entry is itself removed later) or
    spread over it, with additions beside them."""
    H = 8
    rng = np.random.default_rng(I)
    g, u, d = (rng.standard_normal(s).astype(np.float32) for s in ((I, H), (I, H), (H, I)))
    oc = oracle.OracleWeightCache(np.ones(I, bool), H, g, u, d, True)
    wc = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, _t(g), _t(u), _t(d), True)
    cur = np.ones(I, bool)

    def step(m):
        nonlocal cur
        cur = m
        oc.update_active_weights(m)
        wc.update_active_weights_async(_t(m, torch.bool))
        assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist()

    for frac in (0.35, 0.9, 0.2, 0.95, 0.6):
        for _ in range(3):
            step(rng.random(I) < frac)
        for removed in (1, 3, 65, 1100, I // 3):      # from the end of the list, a few additions beside them
            order = oc.get_active_indices()
            m = cur.copy()
            m[order[-removed:]] = False
            off = np.flatnonzero(~cur)
            m[off[: min(len(off), removed // 4)]] = True
            if not m.any():
                m[I // 2] = True
            step(m)
            m = cur | (rng.random(I) < 0.3)           # and room for the next one
            step(m)
    one = np.zeros(I, bool)
    one[I // 2] = True
    step(one)
    step(np.ones(I, bool))
    _check_layout(wc, oc.get_active_indices().tolist(), g, u, d, True)


@pytest.mark.parametrize("I,unaligned", [(64, 0), (8192, 0), (8192, 1), (16001, 0), (22000, 0), (28672, 0)])
def test_surplus_removals_in_one_chain(I, unaligned):
    """A block of removals leaves the end of the list in descending order; removing index 0 and that end then moves every
    step's entry to where the next step takes it from again.  With a few additions beside them, and once more behind."""
    H, k = 8, max(8, I // 4)
    rng = np.random.default_rng(I)
    g, u, d = (rng.standard_normal(s).astype(np.float32) for s in ((I, H), (I, H), (H, I)))
    oc = oracle.OracleWeightCache(np.ones(I, bool), H, g, u, d, True)
    wc, fused = (st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, _t(g), _t(u), _t(d), True) for _ in range(2))
    x = torch.ones(1, H, device=DEV)

    def step(m):
        oc.update_active_weights(m)
        buf = torch.zeros(I + unaligned, dtype=torch.bool, device=DEV)[unaligned:]
        buf.copy_(_t(m, torch.bool))
        wc.update_active_weights_async(buf)
        fused.update_and_forward(buf, x)
        want = oc.get_active_indices().tolist()
        assert wc.get_active_indices().cpu().tolist() == want and fused.get_active_indices().cpu().tolist() == want

    for added in (0, 3):
        m = np.ones(I, bool)
        step(m)
        m[I // 2:I // 2 + k] = False
        step(m)
        m = m.copy()
        m[0] = False
        m[oc.get_active_indices()[-k:]] = False
        m[I // 2:I // 2 + added] = True
        step(m)
    _check_layout(wc, oc.get_active_indices().tolist(), g, u, d, True)


@pytest.mark.parametrize("I,has_gate", [(28672, True), (32768, False), (22016, True)])
def test_large_intermediate_sizes(I, has_gate):
    """Intermediate sizes of the 70B-class models (28672), above what the index lists of the smaller kernels allow:
    index order and layout against the oracle over a trace that starts with every row active, shrinks to a quarter
    (thousands of sequential removals), then churns with the active count drifting both ways, with a no-op update,
    the error of an emptying mask and the state after it."""
    H = 16
    rng = np.random.default_rng(I)
    g = rng.standard_normal((I, H)).astype(np.float32)
    u = rng.standard_normal((I, H)).astype(np.float32)
    d = rng.standard_normal((H, I)).astype(np.float32)
    oc = oracle.OracleWeightCache(np.ones(I, bool), H, g if has_gate else None, u, d, has_gate)
    wc = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, _t(g) if has_gate else None, _t(u), _t(d), has_gate)
    assert wc.get_active_indices().cpu().tolist() == list(range(I))
    m = rng.random(I) < 0.25
    masks = [m.copy()]
    for t in range(24):
        m = m ^ (rng.random(I) < rng.choice([0.003, 0.02, 0.1]))
        masks.append(m.copy())
        if t == 9:
            masks.append(m.copy())           # unchanged mask
    for t, mk in enumerate(masks):
        oc.update_active_weights(mk)
        wc.update_active_weights(_t(mk, torch.bool))
        assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist(), (I, t)
        if t in (0, 5, len(masks) - 1):
            _check_layout(wc, oc.get_active_indices().tolist(), g, u, d, has_gate)
    with pytest.raises(RuntimeError, match="No active weights"):
        wc.update_active_weights(torch.zeros(I, dtype=torch.bool, device=DEV))
    with pytest.raises(RuntimeError):
        oc.update_active_weights(np.zeros(I, bool))
    # (the remembered mask is still the last good one: only indices outside it are added now)
    oc.update_active_weights(np.ones(I, bool))
    wc.update_active_weights(torch.ones(I, dtype=torch.bool, device=DEV))
    assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist()
    assert 0 < wc.get_num_active() < I
    # update + MLP in one call at this size (two launches underneath) against the oracle
    x = rng.standard_normal((1, H)).astype(np.float32)
    oc.update_active_weights(masks[7])
    y = wc.update_and_forward(_t(masks[7], torch.bool), _t(x), "silu" if has_gate else "relu")
    want, _ = oracle.mlp_forward(x, oc.get_concat_weight(), oc.get_active_down_weight(), "silu" if has_gate else "relu",
                                 has_gate)
    assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist()
    scale = np.abs(want).max()
    assert np.abs(y.cpu().numpy() - want).max() <= 1e-5 * scale + 1e-6


def test_full_size_layout_invariants_fp16():
    """cfg-2 shapes: every active row is a bit-copy of its pool row; set(indices) == nonzero(mask)."""
    I, H, n = 8192, 3072, 2867
    gen = torch.Generator(device=DEV).manual_seed(3)
    g = (torch.randn(I, H, device=DEV, generator=gen) * 0.02).half()
    u = (torch.randn(I, H, device=DEV, generator=gen) * 0.02).half()
    d = (torch.randn(H, I, device=DEV, generator=gen) * 0.02).half()
    wc = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, g, u, d, True)
    assert torch.equal(wc.get_concat_weight(), torch.cat([g, u]))          # init: all rows, ascending
    assert torch.equal(wc.get_active_down_weight(), d)
    trace = syn.mask_trace(9, 1, I, n, 12, 0.05, 0.15)[:, 0]
    for t in range(len(trace)):
        m = _t(trace[t], torch.bool)
        wc.update_active_weights(m)
        idx = wc.get_active_indices()
        assert idx.numel() == n and torch.equal(torch.sort(idx)[0], torch.nonzero(m).flatten())
        cw = wc.get_concat_weight()
        assert torch.equal(cw[:n], g[idx]) and torch.equal(cw[n:], u[idx])
        assert torch.equal(wc.get_active_down_weight(), d[:, idx])


def test_noop_and_error_semantics():
    I, H = 32, 8
    gate, up, down = golden_weights(I, H)
    m0 = np.zeros(I, bool)
    m0[[3, 5, 9]] = True
    wc = st.WeightCache(_t(m0, torch.bool), H, _t(gate), _t(up), _t(down), True)
    s0 = wc.sync_state()
    wc.update_active_weights(_t(m0, torch.bool))           # unchanged mask: nothing happens
    s1 = wc.sync_state()
    assert s1["serial"] == s0["serial"] and s1["n_changed"] == 0 and s1["n_active"] == 3
    with pytest.raises(RuntimeError, match="No active weights"):
        wc.update_active_weights(torch.zeros(I, dtype=torch.bool, device=DEV))
    # the remembered mask is still m0 (the reference stores the new mask only after a successful rebuild), so m0 is
    # an unchanged mask now: the reference returns before touching anything, and so does this -- no second error
    wc.update_active_weights(_t(m0, torch.bool))
    assert wc.get_num_active() == 0
    with pytest.raises(RuntimeError, match="No active weights"):      # all-false again differs from m0: it raises again
        wc.update_active_weights(torch.zeros(I, dtype=torch.bool, device=DEV))
    # an all-false init mask is an unchanged mask for the constructor's update (weight_cache.h:223-226,237-240):
    # nothing is built, and the getters then refuse like the reference's TORCH_CHECK(cache_valid)
    empty = st.WeightCache(torch.zeros(I, dtype=torch.bool, device=DEV), H, _t(gate), _t(up), _t(down), True)
    with pytest.raises(RuntimeError, match="Cache is not valid"):
        empty.get_concat_weight()
    with pytest.raises(RuntimeError, match="Cache is not valid"):
        empty.get_active_down_weight()
    empty.update_active_weights(_t(m0, torch.bool))
    assert empty.get_active_indices().cpu().tolist() == [3, 5, 9]
    with pytest.raises(ValueError):
        wc.update_active_weights(torch.ones(I + 1, dtype=torch.bool, device=DEV))
    # masks of other integer types and on the host are accepted like a bool tensor
    m1 = m0.copy()
    m1[[1, 2]] = True
    oc = oracle.OracleWeightCache(m0, H, gate, up, down, True)
    with pytest.raises(RuntimeError):
        oc.update_active_weights(np.zeros(I, bool))
    oc.update_active_weights(m1)
    wc.update_active_weights(torch.from_numpy(m1.astype(np.int64)))
    assert wc.get_active_indices().cpu().tolist() == oc.get_active_indices().tolist()


def test_constructor_validation():
    I, H = 16, 8
    gate, up, down = golden_weights(I, H)
    ones = torch.ones(I, dtype=torch.bool, device=DEV)
    with pytest.raises(ValueError):
        st.WeightCache(ones, H, _t(gate), _t(up), _t(down.T.copy()), True)          # down must be [H, I]
    with pytest.raises(TypeError):
        st.WeightCache(ones, H, _t(gate), _t(up), _t(down).double(), True)
    with pytest.raises(ValueError):
        st.WeightCache(ones, H, None, _t(up), _t(down), True)
    wc = st.WeightCache(ones, H, None, _t(up), _t(down), False)                       # ungated: gate may be None
    assert wc.get_concat_weight().shape == (I, H)
    with pytest.raises(ValueError):                                                   # rows must be 16-byte multiples
        st.WeightCache(ones, 6, _t(gate[:, :6]), _t(up[:, :6]), _t(down[:6]), True)


def test_fast_path_argument_errors():
    """forward / update_and_forward check x, out and combined against the cache on the host: a wrong dtype, a
    short output or a combined buffer that cannot hold every possible count raises instead of reaching a kernel."""
    I, H = 256, 128
    g = torch.Generator().manual_seed(3)
    mk = lambda *s: (torch.randn(*s, generator=g) * 0.05).half().to(DEV)
    cache = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, mk(I, H), mk(I, H), mk(H, I), True)
    mask = (torch.rand(I, generator=g) < 0.5).to(DEV)
    x = mk(1, H)
    for call in (lambda **kw: cache.forward(kw.pop("x", x), "silu", **kw),
                 lambda **kw: cache.update_and_forward(mask, kw.pop("x", x), "silu", **kw)):
        with pytest.raises(TypeError):
            call(x=x.float())                                   # fp32 x on an fp16 cache
        with pytest.raises(ValueError):
            call(x=mk(1, H // 2))                               # wrong hidden size
        with pytest.raises(TypeError):
            call(out=torch.empty(1, H, dtype=torch.float32, device=DEV))
        with pytest.raises(ValueError):
            call(out=torch.empty(1, H // 2, dtype=torch.float16, device=DEV))
        with pytest.raises(ValueError):
            call(combined=torch.empty(1, I, dtype=torch.float16, device=DEV))   # gated: needs 2*I columns
        with pytest.raises(ValueError):
            call(workspace=torch.empty(16, dtype=torch.uint8, device=DEV))
        with pytest.raises((TypeError, RuntimeError)):
            call(x=x.cpu())
    # and the C entry point itself refuses a short row pitch for `combined`
    from sparse_transformers_amd import _lib
    comb = torch.empty(1, I, dtype=torch.float16, device=DEV)
    out = torch.empty(1, H, dtype=torch.float16, device=DEV)
    ws = torch.empty(int(_lib.lib().st_mlp_workspace_bytes(1, H, I)), dtype=torch.uint8, device=DEV)
    rc = _lib.lib().st_cache_update_forward(cache._h, mask.data_ptr(), x.data_ptr(), 1, 0, out.data_ptr(), comb.data_ptr(),
                                            I, ws.data_ptr(), ws.numel(), 1, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.ST_ERR_ARG and "ldc" in _lib.last_error()
    # nothing above changed the cache
    assert cache.get_num_active() == I


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("I,H", [(5, 8), (127, 136), (128, 64), (1000, 264), (2051, 48), (4104, 4160), (32768, 8)])
def test_construction_equals_load_then_update(dtype, I, H):
    """One pass over the weights gives what loading them and a first update give: pools, packed rows, lists, masks, state.
    (tile edges both ways, sizes that cannot be read in vectors, rows of more than one pass, sources off their alignment)"""
    import ctypes as C

    from sparse_transformers_amd import _lib
    tdt, L = getattr(torch, dtype), _lib.lib()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(I + H)
    for has_gate, fill, off in [(True, "some", 0), (False, "all", 0), (True, "none", 0), (True, "last", 1), (False, "some", 1)]:
        def src(a, b):
            return torch.randn(a * b + off, generator=gen, device=DEV).to(tdt)[off:].view(a, b)
        gate, up, down = src(I, H) if has_gate else None, src(I, H), src(H, I)
        mask = torch.zeros(I + off, dtype=torch.uint8, device=DEV)[off:]
        if fill == "some":
            mask.copy_(torch.randint(0, 3, (I,), generator=gen, device=DEV) * 64)   # any nonzero byte counts
        elif fill != "none":
            mask[0 if fill == "all" else I - 1:] = 1
        one = st.WeightCache(mask, H, gate, up, down, has_gate)
        two = st.WeightCache(torch.ones(I, dtype=torch.bool, device=DEV), H, gate, up, down, has_gate)
        _lib.check(L.st_cache_load_weights(two._h, gate.data_ptr() if has_gate else None, up.data_ptr(), down.data_ptr(),
                                           torch.cuda.current_stream().cuda_stream), "st_cache_load_weights")
        two._dirty = True
        assert two.get_num_active() == 0
        m2 = mask.clone()
        rc = L.st_cache_update_sync(two._h, m2.data_ptr(), two._host_state, torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.ST_OK, (fill, rc)
        n = two.get_num_active()
        assert n == int((mask != 0).sum())
        for c in (one, two):   # the words a wait leaves on the host are the device's, all of them
            assert list(c._host_state) == c.state.tolist()
        for name in ("gate_pool", "up_pool", "downT_pool", "gate_active", "up_active", "down_active", "indices", "cur_mask", "state"):
            a, b = getattr(one, name), getattr(two, name)
            if a is not None:
                assert torch.equal(a[:n], b[:n]) if name.endswith("active") else torch.equal(a, b), (name, has_gate, fill)


@pytest.mark.parametrize("I,H,dtype", [(8192, 3072, "float16"), (2051, 1024, "float32"), (28672, 512, "bfloat16")])
def test_waiting_calls_are_done_when_they_return(I, H, dtype):
    """The constructor and update_active_weights wait: what they read (the mask, the module's weights) may be rewritten and
    what they wrote (pools, packed rows) may be read on another stream right after they return, without an event."""
    tdt = getattr(torch, dtype)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(I)
    side = torch.cuda.Stream(device=DEV)
    want = [torch.randn(*s, generator=gen, device=DEV).to(tdt) for s in ((I, H), (I, H), (H, I))]
    weights = [w.clone() for w in want]
    rows = [torch.empty(I, H, dtype=tdt, device=DEV) for _ in range(3)]
    want_rows = [want[0], want[1], want[2].t().contiguous()]

    def take(wc):   # on the other stream: the packed rows as they are now, then the inputs are gone
        with torch.cuda.stream(side):
            for r, a in zip(rows, (wc.gate_active, wc.up_active, wc.down_active)):
                r.copy_(a)

    for _ in range(3):
        mask = torch.rand(I, generator=gen, device=DEV) < 0.6
        first = mask.clone()
        for w, v in zip(weights, want):
            w.copy_(v)
        torch.cuda.synchronize()
        wc = st.WeightCache(mask, H, *weights, True)
        take(wc)
        with torch.cuda.stream(side):
            for t in (mask, *weights):
                t.zero_()
        torch.cuda.synchronize()
        idx = torch.nonzero(first).flatten()
        for r, w in zip(rows, want_rows):
            assert torch.equal(r[: len(idx)], w[idx])
        for pool, w in zip((wc.gate_pool, wc.up_pool, wc.downT_pool), want_rows):
            assert torch.equal(pool, w)
        for density in (0.55, 0.2, 0.9):
            mask.copy_(torch.rand(I, generator=gen, device=DEV) < density)
            second = mask.clone()
            torch.cuda.synchronize()
            wc.update_active_weights(mask)
            take(wc)
            with torch.cuda.stream(side):
                mask.zero_()
            torch.cuda.synchronize()
            idx = wc.get_active_indices()
            assert torch.equal(torch.sort(idx)[0], torch.nonzero(second).flatten())
            for r, w in zip(rows, want_rows):
                assert torch.equal(r[: len(idx)], w[idx])
            assert list(wc._host_state) == wc.state.tolist()


def test_host_words_are_shared_and_reused():
    """More caches than one slab of pinned words holds, in any order of construction and destruction."""
    w = torch.randn(64, 8, device=DEV)
    down = torch.randn(8, 64, device=DEV)
    for order in (1, -1):
        caches = []
        for k in range(150):
            mask = torch.zeros(64, dtype=torch.bool, device=DEV)
            mask[:1 + k % 64] = True
            caches.append(st.WeightCache(mask, 8, w, w, down))
            assert caches[-1].get_num_active() == 1 + k % 64
        for k, c in enumerate(caches):
            assert c._seen.value == 1 + k % 64
            c.update_active_weights(torch.ones(64, dtype=torch.bool, device=DEV))
            assert c.get_num_active() == 64
        while caches:
            caches.pop(0 if order == 1 else -1)


@pytest.mark.parametrize("I,unaligned", [(64, 0), (8192, 1), (2051, 0), (28672, 0), (32768, 0)])
def test_every_update_tells_its_count(I, unaligned):
    """The count that launches take as their guess is the last update's in every form of the update, and after construction."""
    H = 8
    g, u, d = (torch.randn(*s, device=DEV) for s in ((I, H), (I, H), (H, I)))
    masks = [torch.rand(I, device=DEV) < f for f in (0.5, 0.3, 0.3, 0.8)]
    masks.append(masks[-1].clone())   # an unchanged mask
    wc = st.WeightCache(masks[0], H, g, u, d, True)
    assert wc._seen.value == int(masks[0].sum())
    for m in masks[1:]:
        buf = torch.zeros(I + unaligned, dtype=torch.bool, device=DEV)[unaligned:]
        wc._seen.value = -1
        wc.update_active_weights(buf.copy_(m))
        assert wc._seen.value == int(m.sum())
