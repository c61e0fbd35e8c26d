"""Fused sparse MLP on the GPU vs the oracle (float64-accumulating CPU restatement), through the C ABI.

Tolerances: fp32 1e-5 relative; fp16 / bf16 2e-2 absolute, 1e-2 relative, against an fp32
evaluation of the dtype-rounded weights and inputs."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import oracle
import sparse_transformers_amd as st
from sparse_transformers_amd.ops import mlp_forward_rows
from conftest import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _case(seed, B, H, n, dtype, has_gate, std=0.02, lead_shape=None):
    g = torch.Generator().manual_seed(seed)
    tdt = getattr(torch, dtype)
    cw = (torch.randn((2 if has_gate else 1) * n, H, generator=g) * std).to(tdt)
    dn = (torch.randn(n, H, generator=g) * std).to(tdt)
    x = torch.randn(*(lead_shape or (B,)), H, generator=g).to(tdt)
    return x, cw, dn


def _run(x, cw, dn, act, has_gate):
    H = x.shape[-1]
    db = torch.zeros(1, H, dtype=x.dtype, device=DEV)
    cb = torch.zeros(1, 2, dtype=x.dtype, device=DEV)
    out = st.sparse_mlp_forward(x.to(DEV), cw.to(DEV), dn.to(DEV).t(), db, cb, act, has_gate)
    torch.cuda.synchronize()
    return out, db, cb


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("act", ["silu", "relu", "gelu_pytorch_tanh", "sigmoid"])
@pytest.mark.parametrize("has_gate", [True, False])
def test_forward_vs_oracle_small(dtype, act, has_gate):
    for seed, (B, H, n) in enumerate([(1, 64, 5), (1, 256, 300), (2, 128, 77), (3, 1024, 129), (5, 512, 1000)]):
        x, cw, dn = _case(seed, B, H, n, dtype, has_gate, std=0.05)
        out, db, cb = _run(x, cw, dn, act, has_gate)
        want, wantc = oracle.mlp_forward(x.float().numpy(), cw.float().numpy(), dn.float().numpy().T, act, has_gate)
        assert out.shape == x.shape and out.data_ptr() == db.data_ptr()        # aliases down_proj_buffer
        assert tuple(db.shape) == (B, H) and tuple(cb.shape) == (B, cw.shape[0])  # buffers resized in place
        assert_close(out.float().cpu().numpy(), want, dtype, f"out B={B} H={H} n={n}")
        assert_close(cb.float().cpu().numpy(), wantc, dtype, "combined_proj_buffer")


@pytest.mark.parametrize("name,B,H,n,dtype,act,has_gate", [
    ("llama-1b layer fp32", 1, 2048, 2457, "float32", "silu", True),
    ("llama-3b layer fp16", 1, 3072, 2867, "float16", "silu", True),
    ("llama-3b bf16, 4 rows, union of masks", 4, 3072, 4620, "bfloat16", "silu", True),
    ("llama-3b bf16, 8 rows, union of masks", 8, 3072, 6300, "bfloat16", "silu", True),
    ("mistral-7b layer", 1, 4096, 3584, "bfloat16", "silu", True),
    ("mistral-7b layer, 2 rows", 2, 4096, 3584, "bfloat16", "silu", True),
    ("relu-llama-7b gated", 1, 4096, 1100, "float16", "relu", True),
    ("relu-llama-7b ungated", 1, 4096, 1100, "float16", "relu", False),
    ("fp32 wide rows (two chunks per thread)", 1, 4096, 700, "float32", "silu", True),
    ("fp32 8192 hidden", 1, 8192, 300, "float32", "relu", True),
    ("fp16 8192 hidden", 3, 8192, 900, "float16", "silu", True),
])
def test_forward_vs_oracle_config_shapes(name, B, H, n, dtype, act, has_gate):
    x, cw, dn = _case(11, B, H, n, dtype, has_gate, lead_shape=(B, 1))
    out, _, cb = _run(x, cw, dn, act, has_gate)
    want, wantc = oracle.mlp_forward(x.float().numpy(), cw.float().numpy(), dn.float().numpy().T, act, has_gate)
    assert out.shape == (B, 1, H)
    assert_close(out.float().cpu().numpy(), want, dtype, name)
    assert_close(cb.float().cpu().numpy(), wantc, dtype, name + " combined")


@pytest.mark.parametrize("act", ["silu", "relu", "gelu_pytorch_tanh", "sigmoid"])
@pytest.mark.parametrize("has_gate", [True, False])
def test_forward_float64(act, has_gate):
    """Double precision (the reference's operator is dtype-generic, sparse_mlp_op.cpp:151-161): against numpy's
    float64 matrix products (1e-12 of the output's scale: only the order of the sums differs) and, on inputs that
    float32 holds exactly, against the oracle (whose sums are in double and whose outputs are rounded to float32)."""
    acts = {"silu": lambda v: v / (1 + np.exp(-v)), "relu": lambda v: np.maximum(v, 0), "sigmoid": lambda v: 1 / (1 + np.exp(-v)),
            "gelu_pytorch_tanh": lambda v: 0.5 * v * (1 + np.tanh(np.sqrt(2 / np.pi) * (v + 0.044715 * v ** 3)))}
    for seed, (B, H, n) in enumerate([(1, 64, 5), (1, 3072, 700), (3, 256, 300), (8, 130, 77), (9, 1024, 129), (19, 512, 1000)]):
        x, cw, dn = _case(seed, B, H, n, "float32", has_gate, std=0.05)      # float32 values, held in double
        out, db, cb = _run(x.double(), cw.double(), dn.double(), act, has_gate)
        assert out.dtype == torch.float64 and tuple(cb.shape) == (B, cw.shape[0])
        xd, cwd, dnd = x.double().numpy(), cw.double().numpy(), dn.double().numpy()
        up = xd @ cwd[n:].T if has_gate else xd @ cwd.T
        h = acts[act](xd @ cwd[:n].T) * up if has_gate else acts[act](up)
        assert_close(out.cpu().numpy(), h @ dnd, "float64", f"float64 out B={B} H={H} n={n}")
        assert_close(cb.cpu().numpy()[:, :n], h, "float64", "float64 combined")
        if has_gate:
            assert_close(cb.cpu().numpy()[:, n:], up, "float64", "float64 combined, up half")
        want, wantc = oracle.mlp_forward(x.numpy(), cw.numpy(), dn.numpy().T, act, has_gate)
        assert_close(out.cpu().numpy(), want, "float32", "float64 against the oracle")
        assert_close(cb.cpu().numpy(), wantc, "float32", "float64 combined against the oracle")
    # an odd hidden size has rows that are not 16-byte multiples
    x, cw, dn = _case(3, 1, 33, 8, "float32", True)
    with pytest.raises(ValueError, match="16-byte"):
        _run(x.double(), cw.double(), dn.double(), "silu", True)
    # caches and the predictor do not take double
    with pytest.raises(TypeError, match="float64"):
        st.WeightCache(torch.ones(8, dtype=torch.bool, device=DEV), 16, torch.zeros(8, 16, dtype=torch.float64, device=DEV),
                       torch.zeros(8, 16, dtype=torch.float64, device=DEV), torch.zeros(16, 8, dtype=torch.float64, device=DEV))


def test_matches_reference_operator_vectors(golden_mlp):
    """Outputs of the reference's compiled ReLU operator (tests/golden/mlp_forward.json)."""
    for case in golden_mlp:
        H, n, hg = case["H"], case["n"], case["has_gate"]
        x = torch.tensor(case["x"]).reshape(case["x_shape"])
        cw = torch.tensor(case["concat"]).reshape(-1, H)
        dn = torch.tensor(case["down_rows"]).reshape(n, H)
        out, _, cb = _run(x, cw, dn, "relu", hg)
        np.testing.assert_allclose(out.cpu().numpy().ravel(), np.array(case["out"], np.float32), rtol=2e-5, atol=2e-5)
        np.testing.assert_allclose(cb.cpu().numpy().ravel(), np.array(case["combined"], np.float32), rtol=2e-5,
                                   atol=2e-5)


def test_device_count_and_hint_paths():
    """With a device-side count the result must not depend on the host's hint (too low, exact, too
    high, absent) nor on rows beyond the count."""
    I, H, n = 4096, 3072, 1500
    g = torch.Generator().manual_seed(2)
    gate = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    up = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    dn = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    x = torch.randn(1, H, generator=g).half().to(DEV)
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    ref = torch.empty(1, H, dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate, up, dn, n, None, ref, None, "silu", True)
    want, _ = oracle.mlp_forward(x.float().cpu().numpy(), torch.cat([gate[:n], up[:n]]).float().cpu().numpy(),
                                 dn[:n].float().cpu().numpy().T, "silu", True)
    assert_close(ref.float().cpu().numpy(), want, "float16", "host count")
    for hint in (0, 1, 700, n, n + 500, I):
        out = torch.full((1, H), float("nan"), dtype=torch.float16, device=DEV)
        mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True, n_hint=hint)
        assert torch.equal(out, ref), f"hint {hint}"
    n_dev.fill_(0)
    out = torch.full((1, H), 1.0, dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True, n_hint=n)
    assert not out.any()                                       # empty active set -> zeros


@pytest.mark.parametrize("B,H,dt", [(4, 3072, "float16"), (20, 2048, "bfloat16"), (6, 1536, "bfloat16")])
def test_batch_device_count_and_hint_paths(B, H, dt):
    """The batch kernels deal rows to blocks for the count the host expects before the device's count has arrived:
    whatever that guess (absent, too low, exact, too high), the result carries the bits of a call with the exact host
    count, and an empty set gives zeros."""
    I, n = 4096, 1777
    dtype = getattr(torch, dt)
    g = torch.Generator().manual_seed(5)
    gate = (torch.randn(I, H, generator=g) * 0.02).to(dtype).to(DEV)
    up = (torch.randn(I, H, generator=g) * 0.02).to(dtype).to(DEV)
    dn = (torch.randn(I, H, generator=g) * 0.02).to(dtype).to(DEV)
    x = torch.randn(B, H, generator=g).to(dtype).to(DEV)
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    ref = torch.empty(B, H, dtype=dtype, device=DEV)
    mlp_forward_rows(x, gate, up, dn, n, None, ref, None, "silu", True)
    want, _ = oracle.mlp_forward(x.float().cpu().numpy(), torch.cat([gate[:n], up[:n]]).float().cpu().numpy(),
                                 dn[:n].float().cpu().numpy().T, "silu", True)
    assert_close(ref.float().cpu().numpy(), want, dt, "host count")
    for hint in (0, 1, 900, n - 1, n, n + 1, n + 700, I):
        out = torch.full((B, H), float("nan"), dtype=dtype, device=DEV)
        mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True, n_hint=hint)
        assert torch.equal(out, ref), f"hint {hint}"
    n_dev.fill_(0)
    out = torch.full((B, H), 1.0, dtype=dtype, device=DEV)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True, n_hint=n)
    assert not out.any()                                       # empty active set -> zeros


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("n", [1, 2049, 6144, 6145, 8192, 12288, 12289, 14337])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_streaming_kernel_slots(B, n, dtype):
    """The forms of the streaming kernel by rows per thread group (three, six, seven, double-buffered twos: the guess of the
    count chooses) sum the same rows in the same order: the same bits for every guess, rows past the count NaN."""
    H, I = 1024, 16000                    # eight thread groups per block: n / 2048 rows per group
    g = torch.Generator().manual_seed(n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.03).to(getattr(torch, dtype)).to(DEV) for _ in range(3))
    x = torch.randn(B, H, generator=g).to(gate.dtype).to(DEV)
    h = torch.nn.functional.silu(x.float() @ gate[:n].float().t()) * (x.float() @ up[:n].float().t())
    want = (h @ dn[:n].float()).cpu().numpy()
    for t in (gate, up, dn):
        t[n:] = float("nan")
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    first = None
    for hint in (0, 1, n - 1, n, 6144, 8192, 12288, I):
        out = torch.full((B, H), float("nan"), dtype=gate.dtype, device=DEV)
        mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True, n_hint=hint)
        torch.cuda.synchronize()
        assert_close(out.float().cpu().numpy(), want, dtype, f"{n} active, guess {hint}")
        first = out if first is None else first
        assert torch.equal(first, out), hint


def test_float64_device_count_and_empty_set():
    """Double precision with the count on the device: rows beyond it are ignored, the result carries the same bits
    as with the host's count (fixed summation order), and an empty set gives zeros."""
    I, H, n = 700, 256, 333
    g = torch.Generator().manual_seed(4)
    gate = torch.randn(I, H, generator=g, dtype=torch.float64).to(DEV)
    up = torch.randn(I, H, generator=g, dtype=torch.float64).to(DEV)
    dn = torch.randn(I, H, generator=g, dtype=torch.float64).to(DEV)
    x = torch.randn(3, H, generator=g, dtype=torch.float64).to(DEV)
    ref = torch.empty(3, H, dtype=torch.float64, device=DEV)
    mlp_forward_rows(x, gate, up, dn, n, None, ref, None, "silu", True)
    gu = x @ gate[:n].T
    want = ((gu / (1 + torch.exp(-gu))) * (x @ up[:n].T)) @ dn[:n]
    assert_close(ref.cpu().numpy(), want.cpu().numpy(), "float64", "float64, host count")
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    out = torch.full((3, H), float("nan"), dtype=torch.float64, device=DEV)
    comb = torch.zeros(3, 2 * I, dtype=torch.float64, device=DEV)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, comb, "silu", True)
    assert_close(out.cpu().numpy(), want.cpu().numpy(), "float64", "float64, device count")
    n_dev.fill_(0)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True)
    assert not out.any()
    out.fill_(1.0)
    mlp_forward_rows(x, gate, up, dn, 0, None, out, None, "silu", True)
    assert not out.any()


def test_run_to_run_determinism_and_linearity_full_size():
    x, cw, dn = _case(5, 1, 3072, 2867, "float16", True)
    a, _, _ = _run(x, cw, dn, "silu", True)
    b, _, _ = _run(x, cw, dn, "silu", True)
    assert torch.equal(a, b)                                   # fixed summation order
    # identity activation, ungated: the op is linear in x
    xs = torch.randn(2, 3072, generator=torch.Generator().manual_seed(1)).float()
    cwu, dnf = cw[2867:].float(), dn.float()
    y0, _, _ = _run(xs[:1], cwu, dnf, "identity", False)
    y0 = y0.clone()
    y1, _, _ = _run(xs[1:], cwu, dnf, "identity", False)
    y1 = y1.clone()
    ys, _, _ = _run(xs[:1] + xs[1:], cwu, dnf, "identity", False)
    assert_close((y0 + y1).cpu().numpy(), ys.cpu().numpy(), "float32", "linearity")


def test_argument_errors():
    x, cw, dn = _case(0, 1, 64, 8, "float32", True)
    db = torch.zeros(1, 64, device=DEV)
    cb = torch.zeros(1, 2, device=DEV)
    with pytest.raises(ValueError):
        st.sparse_mlp_forward(x.to(DEV), cw.to(DEV)[:-1], dn.to(DEV).t(), db, cb, "silu")      # odd row count
    with pytest.raises(ValueError):
        st.sparse_mlp_forward(x.to(DEV), cw.to(DEV), dn.to(DEV)[:-1].t(), db, cb, "silu")      # n mismatch
    with pytest.raises(ValueError):
        st.sparse_mlp_forward(x.to(DEV), cw.to(DEV), dn.to(DEV).t(), db, cb, "tanh")           # unknown act
    with pytest.raises(TypeError):
        st.sparse_mlp_forward(x.to(DEV), cw.to(DEV).half(), dn.to(DEV).t(), db, cb, "silu")    # dtype mismatch
    # a contiguous [H, n] down matrix (not the cache's view) still gives the right answer
    dwc = dn.to(DEV).t().contiguous()
    with pytest.warns(UserWarning):
        out = st.sparse_mlp_forward(x.to(DEV), cw.to(DEV), dwc, db, cb, "silu")
    want, _ = oracle.mlp_forward(x.numpy(), cw.numpy(), dn.numpy().T, "silu", True)
    assert_close(out.cpu().numpy(), want, "float32", "repacked down")


@pytest.mark.parametrize("name,M,H,n,dtype,act,has_gate", [
    ("small ragged", 130, 256, 200, "float16", "silu", True),
    ("one row tile, n below a K step", 32, 128, 20, "bfloat16", "relu", True),
    ("ungated", 77, 512, 333, "float16", "relu", False),
    ("llama-3b prefill shape, part of the active set", 512, 3072, 1000, "bfloat16", "silu", True),
    ("wide hidden", 96, 4096, 600, "float16", "gelu_pytorch_tanh", True),
    ("narrow tiles, two K groups, many tiles", 100, 512, 7000, "bfloat16", "silu", True),
    ("64-row weight tiles, two K groups", 512, 256, 2457, "float16", "silu", True),
    ("narrow tiles, one K group (more tiles than CUs, one row tile)", 64, 256, 17000, "float16", "silu", True),
    ("the same, ungated", 500, 384, 2300, "bfloat16", "relu", False),
    ("up to 64 rows of x: four K groups", 50, 768, 900, "bfloat16", "silu", True),
    ("four K groups, ungated", 64, 512, 333, "float16", "sigmoid", False),
    ("one active row", 40, 256, 1, "float16", "silu", True),
    ("three active rows, several row tiles", 300, 256, 3, "bfloat16", "silu", True),
])
def test_prefill_mfma_vs_oracle(name, M, H, n, dtype, act, has_gate):
    """More than 32 rows (32 where the batch kernels do not apply) in fp16 / bf16 run on the MFMA GEMM kernels; same
    tolerance as decode."""
    x, cw, dn = _case(21, M, H, n, dtype, has_gate)
    out, _, cb = _run(x, cw, dn, act, has_gate)
    want, wantc = oracle.mlp_forward(x.float().numpy(), cw.float().numpy(), dn.float().numpy().T, act, has_gate)
    assert_close(out.float().cpu().numpy(), want, dtype, name)
    assert_close(cb.float().cpu().numpy()[:, :n], wantc[:, :n], dtype, name + " combined[:, :n]")


@pytest.mark.parametrize("M", [40, 200, 512])
def test_prefill_device_count(M):
    """The GEMM kernels with the active count read on the device: the tile geometry is laid out for the host's
    upper bound, rows beyond the device count may hold anything (here NaN), and the result is the one for the
    exact count."""
    I, H, n = 6144, 1024, 1500
    g = torch.Generator().manual_seed(31)
    gate = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    up = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    dn = (torch.randn(I, H, generator=g) * 0.02).half().to(DEV)
    x = torch.randn(M, H, generator=g).half().to(DEV)
    ref = torch.empty(M, H, dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate, up, dn, n, None, ref, None, "silu", True)
    for t in (gate, up, dn):
        t[n:] = float("nan")
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), ref.float().cpu().numpy(), "float16", f"device count, {M} rows")
    want, _ = oracle.mlp_forward(x[:4].float().cpu().numpy(), torch.cat([gate[:n], up[:n]]).float().cpu().numpy(),
                                 dn[:n].float().cpu().numpy().T, "silu", True)
    assert_close(out[:4].float().cpu().numpy(), want, "float16", "device count vs oracle")
    n_dev.fill_(0)
    out.fill_(1.0)
    mlp_forward_rows(x, gate, up, dn, I, n_dev, out, None, "silu", True)
    assert not out.any()                                       # empty active set -> zeros


@pytest.mark.parametrize("M", [40, 130, 300])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 1025, 3000, 6143, 6144])
def test_prefill_tiles_follow_the_device_count(M, n):
    """The tiles of weight rows are dealt out over the count the device holds: counts around the tile edges, from one row to
    the capacity, in every form of the gate / up kernel; every column of the intermediate has to be written by some tile."""
    I, H = 6144, 512
    g = torch.Generator().manual_seed(n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.05).half().to(DEV) for _ in range(3))
    x = torch.randn(M, H, generator=g).half().to(DEV)
    h = torch.nn.functional.silu(x.float() @ gate[:n].float().t()) * (x.float() @ up[:n].float().t())
    want = h @ dn[:n].float()
    for t in (gate, up, dn):
        t[n:] = float("nan")
    out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
    comb = torch.full((M, 2 * I), float("nan"), dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate, up, dn, I, torch.tensor([n], dtype=torch.int32, device=DEV), out, comb, "silu", True)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), want.cpu().numpy(), "float16", f"{M} rows, {n} active")
    assert_close(comb[:, :n].float().cpu().numpy(), h.cpu().numpy(), "float16", f"intermediate, {M} rows, {n} active")


@pytest.mark.parametrize("M,H,I,n,gated", [
    # 256-row tiles of x by 128 (gated) or 256 active rows: t of them; rest = t modulo the CUs (256)
    (1030, 384, 8192, 3000, True),     # t = 120: all halved
    (1030, 384, 8192, 3201, True),     # t = 130: all big, the last row tile of x nearly empty
    (1030, 128, 8192, 6527, True),     # t = 255; two K stages
    (1030, 256, 8192, 6529, True),     # t = 260: 256 big, 4 quartered
    (1030, 256, 8192, 8192, True),     # t = 320: 256 big, 64 quartered
    (2030, 256, 8448, 8200, False),    # t = 264: 256 big, 8 quartered, of which the last two quarters are past the padded count
    (2030, 384, 8448, 8447, False),    # the same with all quarters
    (150, 256, 8448, 8447, False),     # t = 33: all quartered, one row tile
    (1030, 384, 8448, 3001, False),    # t = 60: all quartered
    (2030, 128, 8448, 2048, False),    # t = 64: the last that is quartered
    (1030, 640, 8448, 3210, False),    # t = 65: all halved
    (2030, 128, 8448, 4000, False),    # t = 128: all halved
    (2030, 640, 8448, 4200, False),    # t = 136: all big
])
def test_prefill_big_tiles(M, H, I, n, gated):
    """The 256 x 256 tiles of the gate / up kernel and the halves of those that do not fill a round of CUs: every element of
    the output and of the intermediate, rows past the device's count NaN.  Bounds as in the tests above (fp32 sums of the
    same fp16 operands, a rounding of the intermediate and of the output)."""
    g = torch.Generator().manual_seed(n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.05).half().to(DEV) for _ in range(3))
    x = torch.randn(M, H, generator=g).half().to(DEV)
    h = torch.nn.functional.silu((x.float() @ (gate if gated else up)[:n].float().t()))
    if gated:
        h = h * (x.float() @ up[:n].float().t())
    want = h @ dn[:n].float()
    for t in (gate, up, dn):
        t[n:] = float("nan")
    out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
    comb = torch.full((M, (2 if gated else 1) * I), float("nan"), dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate if gated else None, up, dn, I, torch.tensor([n], dtype=torch.int32, device=DEV), out, comb, "silu",
                     gated)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), want.cpu().numpy(), "float16", f"{M} rows, {n} active")
    assert_close(comb[:, :n].float().cpu().numpy(), h.cpu().numpy(), "float16", f"intermediate, {M} rows, {n} active")


@pytest.mark.parametrize("M,H,I,n", [
    (129, 64, 9000, 1), (129, 64, 9000, 8192), (256, 192, 9000, 8129), (257, 128, 9000, 4095), (384, 256, 9000, 4033),
    (385, 320, 9000, 4096), (1100, 128, 9000, 6700),
])
def test_prefill_quarters_of_gated_tiles(M, H, I, n):
    """Rests of up to a quarter of the CUs, which go out as 128 rows of x by 64 active ones: one tile of them, the most, K loops
    of one stage to five, rows of x that leave a tile's lower half out or with one row, counts that leave an active half out.
    Checked as the tiles above are."""
    test_prefill_big_tiles(M, H, I, n, True)


@pytest.mark.parametrize("M,n", [(300, 3000), (300, 4096), (300, 4097), (512, 6500), (1030, 6529)])
def test_prefill_guess_of_the_count_picks_the_kernel_only(M, n, H=256, I=9000):
    """Counts whose rest of gated tiles goes out in quarters, in halves or whole, under guesses that pick either kernel: the same bits."""
    g = torch.Generator().manual_seed(M + n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.05).half().to(DEV) for _ in range(3))
    x = torch.randn(M, H, generator=g).half().to(DEV)
    outs = []
    for hint in (0, n, 3000, 6500, I):
        out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
        comb = torch.full((M, 2 * I), float("nan"), dtype=torch.float16, device=DEV)
        mlp_forward_rows(x, gate, up, dn, I, torch.tensor([n], dtype=torch.int32, device=DEV), out, comb, "silu", True, n_hint=hint)
        torch.cuda.synchronize()
        outs.append((out, comb[:, :n]))
    h = torch.nn.functional.silu(x.float() @ gate[:n].float().t()) * (x.float() @ up[:n].float().t())
    assert_close(outs[0][1].float().cpu().numpy(), h.cpu().numpy(), "float16", "intermediate")
    for o, c in outs[1:]:
        assert torch.equal(o, outs[0][0]) and torch.equal(c, outs[0][1])


@pytest.mark.parametrize("M,H,I,n,gated", [
    (33, 128, 1000, 1, True), (64, 384, 9000, 8192, True), (65, 1152, 9000, 8193, True), (96, 640, 8448, 8447, True),
    (97, 128, 4096, 4033, True), (128, 1024, 8200, 8200, True),
    (48, 256, 9000, 8192, False), (64, 1152, 520, 33, False), (77, 2560, 9000, 6144, False), (97, 384, 8300, 8300, False),
    (128, 128, 8320, 8257, False), (96, 768, 300, 300, False),
])
def test_prefill_few_rows(M, H, I, n, gated):
    """Up to 128 rows of x: every form of the two kernels (64, 96, 128 rows; the fewer or the more active rows per block, which
    the guess of the count chooses and which must not show in a bit), K loops shorter and longer than the ring, splits of the
    down projection without stages, rows past the device's count NaN.  Bounds as in the tests above."""
    g = torch.Generator().manual_seed(M + n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.05).half().to(DEV) for _ in range(3))
    x = torch.randn(M, H, generator=g).half().to(DEV)
    h = torch.nn.functional.silu((x.float() @ (gate if gated else up)[:n].float().t()))
    if gated:
        h = h * (x.float() @ up[:n].float().t())
    want = h @ dn[:n].float()
    for t in (gate, up, dn):
        t[n:] = float("nan")
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    first = None
    for hint in (0, 1, n, I):
        out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
        comb = torch.full((M, (2 if gated else 1) * I), float("nan"), dtype=torch.float16, device=DEV)
        mlp_forward_rows(x, gate if gated else None, up, dn, I, n_dev, out, comb, "silu", gated, n_hint=hint)
        torch.cuda.synchronize()
        assert_close(out.float().cpu().numpy(), want.cpu().numpy(), "float16", f"{M} rows, {n} active, guess {hint}")
        assert_close(comb[:, :n].float().cpu().numpy(), h.cpu().numpy(), "float16", f"intermediate, {M} rows, {n} active")
        first = out if first is None else first
        assert torch.equal(first, out)


@pytest.mark.parametrize("M,H,I,n,gated", [
    (33, 128, 1000, 1, True), (48, 256, 9000, 8191, False), (64, 1152, 520, 63, False), (65, 1152, 9000, 8129, True),
    (77, 2560, 9000, 6081, False), (96, 640, 8448, 8384, True), (128, 512, 4096, 2500, True), (128, 1024, 8200, 8199, True),
])
def test_prefill_few_rows_infinite_last_row(M, H, I, n, gated):
    """An infinity and a NaN in the last active row of the down weights, 33 to 128 rows of x and a count that is not a multiple
    of the padding: the padding's zeros must not meet them, so that an infinite element is infinite with the intermediate's
    sign and the other columns are finite.  Bounds as in the tests above."""
    g = torch.Generator().manual_seed(M * n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * 0.05).half().to(DEV) for _ in range(3))
    x = torch.randn(M, H, generator=g).half().to(DEV)
    x[:, 0], x[:, 1] = 8.0, torch.where(torch.arange(M, device=DEV) % 3 > 0, 1.0, -1.0).half()
    gate[n - 1], up[n - 1] = 0.0, 0.0
    (gate if gated else up)[n - 1, 0] = 1.0                  # the last intermediate: silu(8), times 1 or -1 with a gate
    if gated:
        up[n - 1, 1] = 1.0
    h = torch.nn.functional.silu(x.float() @ (gate if gated else up)[:n].float().t())
    if gated:
        h = h * (x.float() @ up[:n].float().t())
    dn[n - 1, 1], dn[n - 1, H // 2], dn[n - 1, H - 1] = float("inf"), float("-inf"), float("nan")
    finite = torch.ones(H, dtype=torch.bool, device=DEV)
    finite[[1, H // 2, H - 1]] = False
    want = h @ torch.where(torch.isfinite(dn[:n]), dn[:n], 0).float()
    for t in (gate, up, dn):
        t[n:] = float("nan")
    out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
    mlp_forward_rows(x, gate if gated else None, up, dn, I, torch.tensor([n], dtype=torch.int32, device=DEV), out, None, "silu",
                     gated)
    torch.cuda.synchronize()
    sign = x[:, 1].float() if gated else torch.ones(M, device=DEV)
    assert torch.equal(out[:, 1].float(), sign * float("inf")) and torch.equal(out[:, H // 2].float(), -sign * float("inf"))
    assert bool(torch.isnan(out[:, H - 1]).all())
    assert_close(out[:, finite].float().cpu().numpy(), want[:, finite].cpu().numpy(), "float16", f"{M} rows, {n} active")


@pytest.mark.parametrize("M,H,I,n,gated", [
    (17, 1024, 33000, 8129, True), (31, 2048, 16500, 63, False), (32, 640, 9000, 8191, True), (32, 128, 40, 1, True),
    (24, 768, 44000, 6143, False),
])
def test_prefill_of_17_to_32_rows(M, H, I, n, gated):
    """17 to 32 rows at both sides of the line between the batch kernels and the few-row form: the checks of the two tests above.
    (At most 2048 wide: rounding the intermediate to fp16 puts sqrt(n) * 0.05 * rms(h) * 1e-4 on a result, 0.0016 at rms(h) = 3.6 and
    8129 rows, against a bound of 0.02; at 4096, rms(h) near 10, two of 69632 results pass it.)"""
    test_prefill_few_rows(M, H, I, n, gated)
    test_prefill_few_rows_infinite_last_row(M, H, I, n, gated)


@pytest.mark.parametrize("M,H,n,gated,stride", [
    (200, 65536, 33000, False, 0),                # weights of 4.3 GB
    (4096, 128, 524416, False, 0),                # an intermediate of 4.3 GB
    (128, 128, 520, True, (1 << 24) + 8),         # rows of the combined buffer 2^24 + 8 elements apart, 4.3 GB
    (300, 128, 520, True, (1 << 24) + 8),
    (128, (1 << 24) + 128, 3, False, 0),          # 128 rows of x of 33.6 MB
])
def test_prefill_beyond_4_gib(M, H, n, gated, stride):
    """Operands whose offsets from their own start do not fit 32 bits.  Bounds as in the tests above (the down weights are
    scaled so that the roundings of the intermediate, at random, add up to about 1e-3 of an output of about 2)."""
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, H, generator=g, device=DEV).half()
    gate, up, dn = (torch.empty(n if i or gated else 1, H, dtype=torch.float16, device=DEV).normal_(0, s, generator=g)
                    for i, s in enumerate((H ** -0.5, H ** -0.5, 4 * n ** -0.5)))
    comb = torch.empty(M, stride, dtype=torch.float16, device=DEV)[:, :2 * n] if stride else None
    out = torch.full((M, H), float("nan"), dtype=torch.float16, device=DEV)
    need = st.ops.mlp_workspace_bytes(M, H, n)               # (140 GB for the widest x; kept by the test, not by the process)
    if torch.cuda.mem_get_info()[0] < need + (40 << 30):
        pytest.skip(f"needs {need >> 30} GB of scratch")
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    mlp_forward_rows(x, gate if gated else None, up, dn, n, None, out, comb, "silu", gated, workspace=ws)
    for rows in torch.arange(M, device=DEV).split(512):
        h = torch.nn.functional.silu(x[rows].float() @ (gate if gated else up).float().t())
        if gated:
            h = h * (x[rows].float() @ up.float().t())
        # (with few active rows and many columns some sums cancel: the intermediate is off by its rounding, at most 2^-11 of it,
        # and by its fp32 sum, 2^-12 for 2^24 products in 2^18 steps of a wave; three such errors add up to less than 1.8 times
        # their root of squares, many at random to less.  Reference products of no more than 2^31 elements.)
        for cols in range(0, H, 1 << 20):
            d = dn[:, cols:cols + (1 << 20)].float()
            want, got = h @ d, out[rows, cols:cols + (1 << 20)].float()
            bound = 2e-2 + 1e-2 * want.abs() + 2.0 ** -9 * ((h * h) @ (d * d)).sqrt()
            assert bool(((got - want).abs() <= bound).all()) and float(want.abs().max()) > 0.5
        if comb is not None:
            assert_close(comb[rows, :n].float().cpu().numpy(), h.cpu().numpy(), "float16", f"intermediate, {M} rows")
    del x, gate, up, dn, comb, out, ws, h, d, want, got, bound
    torch.cuda.empty_cache()


def test_prefill_agrees_with_decode_kernel():
    """The MFMA path (B = 40) and the streaming path (the same rows, 4 at a time) agree to rounding."""
    x, cw, dn = _case(22, 40, 1024, 700, "float16", True)
    big, _, _ = _run(x, cw, dn, "silu", True)
    big = big.clone()
    for b0 in range(0, 40, 8):
        small, _, _ = _run(x[b0:b0 + 8], cw, dn, "silu", True)
        assert_close(small.float().cpu().numpy(), big[b0:b0 + 8].float().cpu().numpy(), "float16", f"rows {b0}")


@pytest.mark.parametrize("name,M,H,n,dtype,act,has_gate", [
    ("ragged rows and columns, K loop with whole groups and a tail", 300, 1152, 6000, "bfloat16", "silu", True),
    ("ungated, K loop shorter than one group", 260, 256, 8500, "float16", "relu", False),
    ("llama-3b prefill, every row active", 512, 3072, 8192, "bfloat16", "silu", True),
    ("ragged 256-row tile through both wide kernels, intermediate kept in the combined buffer", 448, 1024, 4096, "float16", "silu", True),
    ("the same with an odd count: combined rows not 16-byte aligned, intermediate in the workspace", 448, 1024, 3001, "bfloat16", "silu", True),
    ("ungated, combined buffer exactly as wide as the padded intermediate", 512, 512, 5120, "float16", "relu", False),
    ("more 256-row tiles than CUs: down projection without a K split", 2800, 3072, 640, "bfloat16", "silu", True),
    ("two K stages in gate/up; down projection with splits that have nothing to do", 512, 128, 8200, "float16", "silu", True),
])
def test_prefill_wide_blocks(name, M, H, n, dtype, act, has_gate):
    """With more 128-row tiles than CUs the gate/up kernel switches to 256-row blocks, and from 256 rows on the down
    projection to 256-row tiles with the K range split over the CUs.  Every row of the output and of the
    intermediate is held against the oracle; a sample of row groups is also compared with the streaming decode
    kernel."""
    x, cw, dn = _case(23, M, H, n, dtype, has_gate)
    out, _, cb = _run(x, cw, dn, act, has_gate)
    out, cb = out.float().cpu().numpy().copy(), cb.float().cpu().numpy().copy()
    xf, cwf, dnf = x.float().numpy(), cw.float().numpy(), np.ascontiguousarray(dn.float().numpy().T)
    for r0 in range(0, M, 128):
        rows = slice(r0, min(M, r0 + 128))
        want, wantc = oracle.mlp_forward(xf[rows], cwf, dnf, act, has_gate)
        assert_close(out[rows], want, dtype, f"{name} rows {rows}")
        assert_close(cb[rows, :n], wantc[:, :n], dtype, f"{name} combined rows {rows}")
    step = 8
    for b0 in range(0, M, 64):   # a sample of row groups through the streaming kernel
        small, _, cs = _run(x[b0:b0 + step], cw, dn, act, has_gate)
        assert_close(out[b0:b0 + step], small.float().cpu().numpy(), dtype, f"{name} rows {b0}.. vs decode kernel")
        assert_close(cb[b0:b0 + step, :n], cs.float().cpu().numpy()[:, :n], dtype, f"{name} combined rows {b0}..")


def test_prefill_leaves_the_parent_of_a_column_slice_alone():
    """`combined` given as a column slice of a wider tensor (ungated, 64 rows of x, n not a multiple of 128): the
    GEMM kernels keep their intermediate in a buffer whose row stride has room for n rounded up to 128 and zero the
    padding, which must not happen to the parent's columns."""
    B, H, n = 64, 512, 700
    x, cw, dn = _case(29, B, H, n, "float16", False)
    parent = torch.full((B, 1024), 7.0, dtype=torch.float16, device=DEV)
    out = torch.empty(B, H, dtype=torch.float16, device=DEV)
    mlp_forward_rows(x.to(DEV), None, cw.to(DEV), dn.to(DEV), n, None, out, parent[:, :n], "relu", False)
    torch.cuda.synchronize()
    assert bool((parent[:, n:] == 7.0).all()), "columns outside the view were written"
    want, wantc = oracle.mlp_forward(x.float().numpy(), cw.float().numpy(), np.ascontiguousarray(dn.float().numpy().T),
                                     "relu", False)
    assert_close(out.float().cpu().numpy(), want, "float16", "out")
    assert_close(parent[:, :n].float().cpu().numpy(), wantc[:, :n], "float16", "combined view")


@pytest.mark.parametrize("B,H,I,n,dtype,gated", [
    (17, 4096, 11000, 11000, "float16", False), (24, 4096, 14336, 3500, "bfloat16", True), (31, 3840, 10240, 9001, "float16", True),
    (32, 3072, 11000, 10999, "bfloat16", True), (24, 3072, 11000, 8200, "float16", False),
])
def test_17_to_32_rows_of_large_matrices(B, H, I, n, dtype, gated):
    """17 to 32 rows where n * H passes 32 Mi: `combined` as a column slice gets act(gate) * up, the raw up projection behind it
    when gated, and nothing is written outside the slice; the same bits with the count from the host or from the device.
    Against float64 on weights that keep the intermediate of order one."""
    td = getattr(torch, dtype)
    g = torch.Generator().manual_seed(B + H + n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * H ** -0.5).to(td).to(DEV) for _ in range(3))
    x = torch.randn(B, H, generator=g).to(td).to(DEV)
    u = x.double() @ up[:n].double().t()
    h = torch.nn.functional.silu(x.double() @ gate[:n].double().t()) * u if gated else torch.nn.functional.silu(u)
    want, wantc = h @ dn[:n].double(), torch.cat([h, u], 1) if gated else h
    first = None
    for cap, n_dev in ((n, None), (I, torch.tensor([n], dtype=torch.int32, device=DEV))):
        cols = (2 if gated else 1) * cap
        parent = torch.full((B, (cols + 263) // 8 * 8), 7.0, dtype=td, device=DEV)
        out = torch.empty(B, H, dtype=td, device=DEV)
        mlp_forward_rows(x, gate if gated else None, up, dn, cap, n_dev, out, parent[:, :cols], "silu", gated)
        torch.cuda.synchronize()
        assert bool((parent[:, cols:] == 7.0).all()), "columns outside the view were written"
        assert_close(out.float().cpu().numpy(), want.cpu().numpy(), dtype, "out")
        assert_close(parent[:, :wantc.size(1)].float().cpu().numpy(), wantc.cpu().numpy(), dtype, "combined")
        first = out if first is None else first
        assert torch.equal(first, out)


# ---- MFMA batch kernels (3 <= B <= 32, fp16 / bf16, hidden sizes that are multiples of 256) ----
@pytest.mark.parametrize("name,B,H,n,dtype,act,has_gate", [
    ("llama-3b bf16, 4 rows", 4, 3072, 4620, "bfloat16", "silu", True),
    ("llama-3b bf16, 16 rows", 16, 3072, 7660, "bfloat16", "silu", True),
    ("mistral-7b bf16, 8 rows", 8, 4096, 3584, "bfloat16", "silu", True),
    ("4096-wide fp16, 4 rows, ungated relu", 4, 4096, 1100, "float16", "relu", False),
    ("two passes of 16 + ragged tail", 19, 2048, 1237, "float16", "gelu_pytorch_tanh", True),
    ("31 rows, fewer active rows than blocks", 31, 3072, 97, "bfloat16", "sigmoid", True),
    ("32 rows: two full passes", 32, 3072, 2867, "float16", "silu", True),
    ("one active row", 5, 2048, 1, "float16", "silu", True),
    ("33 rows per block (two tiles)", 3, 2048, 8450, "float16", "silu", False),
    # hidden sizes without a kernel instantiated for them (run-time K loop; x from LDS up to 4096 columns, from memory beyond)
    ("qwen2-7b width 3584, 8 rows", 8, 3584, 2500, "bfloat16", "silu", True),
    ("width 5120, 4 rows (x straight from memory)", 4, 5120, 1800, "float16", "silu", True),
    ("opt-125m width 768, 16 rows, ungated relu", 16, 768, 1111, "float16", "relu", False),
    ("qwen2-1.5b width 1536, 20 rows (two passes of 16 + 4)", 20, 1536, 3000, "bfloat16", "silu", True),
    ("width 8192, 3 rows, ragged tiles", 3, 8192, 1031, "float16", "gelu_pytorch_tanh", True),
    ("width 256, 5 rows: a single k-step per wave", 5, 256, 300, "float16", "silu", True),
])
def test_batch_mfma_vs_oracle(name, B, H, n, dtype, act, has_gate):
    x, cw, dn = _case(4242 + B + n, B, H, n, dtype, has_gate)
    out, db, cb = _run(x, cw, dn, act, has_gate)
    want, wantc = oracle.mlp_forward(x.float().numpy(), cw.float().numpy(), dn.float().numpy().T, act, has_gate)
    assert tuple(out.shape) == (B, H) and tuple(cb.shape) == (B, cw.shape[0])
    assert_close(out.float().cpu().numpy(), want, dtype, name)
    assert_close(cb.float().cpu().numpy(), wantc, dtype, name + " combined")


@pytest.mark.parametrize("B,H,I,n,dtype,gated", [
    (3, 64, 40, 1, "float32", True), (8, 128, 300, 257, "float32", False), (17, 1424, 700, 511, "float32", True),
    (5, 2816, 5000, 4113, "float32", True), (33, 912, 4500, 4097, "float32", True), (70, 8192, 300, 299, "float32", False),
    (3, 64, 40, 16, "float16", True), (16, 192, 17000, 16385, "bfloat16", False), (17, 128, 33, 17, "float16", True),
    (9, 1664, 6144, 1230, "bfloat16", True), (32, 896, 4500, 4096, "float16", True), (25, 1152, 9000, 8200, "bfloat16", True),
    (32, 1600, 5000, 4095, "float16", False), (31, 3200, 2000, 1999, "bfloat16", True), (12, 4736, 700, 333, "float16", True),
    (22, 16384, 100, 97, "bfloat16", False), (40, 1216, 3000, 2900, "float16", True),
    (9, 48, 300, 257, "float32", False), (9, 16, 40, 1, "float32", True), (5, 64, 40, 16, "float16", True),
])
def test_batch_any_width(B, H, I, n, dtype, gated):
    """The batch kernels for any width whose rows are multiples of 64 bytes, and fp32: remainders of the steps per wave, both
    forms of x (LDS, registers), one and two subtiles per tile, several passes of 32 rows; the count comes from the device, rows
    past it are NaN and the last active row of the down weights holds an infinity, which must meet nothing but its own
    intermediate.  Against float64; fp32 sums of at most 16384 products in another order: within 1e-5 of the largest value."""
    td = getattr(torch, dtype)
    g = torch.Generator().manual_seed(B * H + n)
    gate, up, dn = ((torch.randn(I, H, generator=g) * H ** -0.5).to(td).to(DEV) for _ in range(3))
    x = torch.randn(B, H, generator=g).to(td).to(DEV)
    dn[n - 1, H // 2] = float("inf")
    hu = x.double() @ up[:n].double().t()
    hh = (x.double() @ gate[:n].double().t()) if gated else hu
    h = torch.nn.functional.silu(hh) * (hu if gated else 1.0)
    fin = dn[:n].double()
    fin[n - 1, H // 2] = 0.0
    want = h @ fin
    for t in (gate, up, dn):
        t[n:] = float("nan")
    comb = torch.full((B, 2 * n if gated else n), float("nan"), dtype=td, device=DEV)
    outs = []
    for cap, n_dev, c in ((I, torch.tensor([n], dtype=torch.int32, device=DEV), None), (n, None, comb)):
        out = torch.full((B, H), float("nan"), dtype=td, device=DEV)
        mlp_forward_rows(x, gate if gated else None, up, dn, cap, n_dev, out, c, "silu", gated)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])                       # the form does not depend on where the count comes from
    inf_col = outs[0][:, H // 2].double()
    assert torch.equal(inf_col, h[:, n - 1].sign() * float("inf"))
    outs[0][:, H // 2], want[:, H // 2] = 0, 0
    assert_close(outs[0].float().cpu().numpy(), want.cpu().numpy(), dtype, "out")
    assert_close(comb[:, :n].float().cpu().numpy(), h.cpu().numpy(), dtype, "combined, h")
    if gated and not (B == 32 and H % 128 == 0 and H % 256 != 0):   # (32 rows at such widths take the GEMM kernels, which leave it out)
        assert_close(comb[:, n:].float().cpu().numpy(), hu.cpu().numpy(), dtype, "combined, up")


@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("B,H,n", [(5, 896, 700), (9, 960, 500), (16, 1152, 1111), (31, 1152, 2000), (12, 2048, 300)])
def test_batch_rows_do_not_meet(B, H, n, dtype):
    """A row's result has the same bits whatever the other rows of its tile hold: rows up to 2^20 larger, of zeros, with an infinity."""
    td = getattr(torch, dtype)
    g = torch.Generator().manual_seed(B + H)
    gate, up, dn = ((torch.randn(n, H, generator=g) * H ** -0.5).to(td).to(DEV) for _ in range(3))
    x = (torch.randn(B, H, generator=g) * 2.0 ** -7).to(td).to(DEV)
    y = x.clone()
    y[0] *= 2.0 ** 20 if dtype != "float16" else 2.0 ** 15
    y[2] = 0.0
    y[B - 1, 3] = float("inf")
    outs = []
    for v in (x, y):
        out = torch.empty(B, H, dtype=td, device=DEV)
        mlp_forward_rows(v, gate, up, dn, n, None, out, None, "silu", True)
        torch.cuda.synchronize()
        outs.append(out)
    same = [b for b in range(B) if b not in (0, 2, B - 1)]
    assert torch.equal(outs[0][same], outs[1][same])
    assert not outs[1][2].any()


def test_batch_mfma_device_count_and_determinism():
    """The batch kernels take the active count from device memory (rows past it may hold anything, here NaN),
    and repeat bit-identically."""
    B, H, I, n = 8, 3072, 2000, 1333
    x, cw, dn = _case(99, B, H, I, "float16", True)
    gate, up = cw[:I].clone(), cw[I:].clone()
    gate[n:], up[n:], dn[n:] = float("nan"), float("nan"), float("nan")
    xg, gg, ug, dg = x.to(DEV), gate.to(DEV), up.to(DEV), dn.to(DEV)
    n_dev = torch.tensor([n], dtype=torch.int32, device=DEV)
    outs = []
    for _ in range(3):
        out = torch.full((B, H), float("nan"), dtype=torch.float16, device=DEV)
        mlp_forward_rows(xg, gg, ug, dg, I, n_dev, out, None, "silu", True)
        torch.cuda.synchronize()
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    want, _ = oracle.mlp_forward(x.float().numpy(), torch.cat([gate[:n], up[:n]]).float().numpy(),
                                 dn[:n].float().numpy().T, "silu", True)
    assert_close(outs[0].float().numpy(), want, "float16", "device count")
    # an empty active set gives zeros
    n_dev.zero_()
    out = torch.full((B, H), float("nan"), dtype=torch.float16, device=DEV)
    mlp_forward_rows(xg, gg, ug, dg, I, n_dev, out, None, "silu", True)
    torch.cuda.synchronize()
    assert torch.count_nonzero(out).item() == 0


def test_batch_mfma_agrees_with_streaming_kernel():
    """Same inputs through the MFMA batch kernels (4 rows at once) and the streaming kernel (row by row)."""
    H, n = 3072, 2867
    x, cw, dn = _case(7, 4, H, n, "bfloat16", True)
    out4, _, _ = _run(x, cw, dn, "silu", True)
    ref = torch.cat([_run(x[i:i + 1], cw, dn, "silu", True)[0].clone() for i in range(4)]).float().cpu().numpy()
    assert_close(out4.float().cpu().numpy(), ref, "bfloat16", "batch vs streaming")


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("B,H,n", [(1, 64, 3), (4, 4096, 40), (16, 1024, 700), (17, 1024, 900), (32, 576, 1000), (9, 2048, 5000),
                                   (31, 4160, 800), (3, 8192, 900), (100, 256, 6000), (100, 1152, 9000), (128, 2048, 4000)])
def test_sums_of_splits(B, H, n, dtype):
    """Every number of row splits the kernels behind a K split sum (two to sixteen by the width, twice that for narrow ones), with as
    many results as make full blocks or not, into an output off its alignment.  Against float64, as above."""
    td = getattr(torch, dtype)
    g = torch.Generator().manual_seed(B + H + n)
    gate, up, dn = ((torch.randn(n, H, generator=g) * H ** -0.5).to(td).to(DEV) for _ in range(3))
    x = torch.randn(B, H, generator=g).to(td).to(DEV)
    h = torch.nn.functional.silu(x.double() @ gate.double().t()) * (x.double() @ up.double().t())
    store = torch.full((B * H + 1,), float("nan"), dtype=td, device=DEV)
    out = store[1:].view(B, H)
    mlp_forward_rows(x, gate, up, dn, n, None, out, None, "silu", True)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), (h @ dn.double()).cpu().numpy(), dtype, "out")
    assert bool(torch.isnan(store[0]))


def test_batch_kernels_can_be_switched_off():
    """ST_MLP_BATCH_MIN above 32: no row count takes the batch kernels or their workspace (the variable is read once per process)."""
    script = """
import ctypes as C, torch
from sparse_transformers_amd import _lib
from sparse_transformers_amd.ops import mlp_forward_rows
L = _lib.lib()
for dtype, B, H in ((torch.float32, 33, 256), (torch.float32, 6, 2048), (torch.float16, 40, 192), (torch.float16, 16, 2048), (torch.float16, 40, 256)):
    w = [torch.randn(300, H, device="cuda").to(dtype) * 0.05 for _ in range(3)]
    x = torch.randn(B, H, device="cuda").to(dtype)
    kinds, ms = (C.c_int32 * 64)(), (C.c_float * 64)()
    _lib.check(L.st_profile_enable(64), "st_profile_enable")
    mlp_forward_rows(x, *w, 300, None, torch.empty_like(x), None, "silu", True)
    torch.cuda.synchronize()
    names = {_lib.KERNEL_KINDS[kinds[i]] for i in range(L.st_profile_collect(kinds, ms, 64))}
    L.st_profile_disable()
    print("CALL", any("batch" in n for n in names), any("prefill" in n for n in names), L.st_mlp_workspace_bytes(40, 64, 16384))
"""
    lines = {}
    for value in ("33", "40", "3"):
        p = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=100,
                           env={**os.environ, "ST_MLP_BATCH_MIN": value, "PYTHONPATH": ROOT}, cwd=ROOT)
        assert p.returncode == 0, p.stderr[-2000:]
        lines[value] = [l.split()[1:] for l in p.stdout.splitlines() if l.startswith("CALL")]
    for value in ("33", "40"):
        assert [l[:2] for l in lines[value]] == [["False", "False"]] * 4 + [["False", "True"]], lines
        assert lines[value][0][2] < lines["3"][0][2]
    assert [l[0] for l in lines["3"]] == ["True"] * 4 + ["False"], lines
