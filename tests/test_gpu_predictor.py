"""LoRA predictor + threshold mask + batch union on the GPU vs the oracle.  Scores are floating point
(tolerance); masks are bits and must be exact, so thresholds are placed in a gap between scores that is
much wider than the rounding difference between the two implementations (the guard band is asserted)."""
import numpy as np
import pytest
import torch

import oracle
import sparse_transformers_amd as st
from sparse_transformers_amd import synthetic as syn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _weights(seed, B, H, r, I, dtype):
    g = torch.Generator().manual_seed(seed)
    tdt = getattr(torch, dtype)
    A = (torch.randn(r, H, generator=g) * 0.02).to(tdt)
    Bm = (torch.randn(I, r, generator=g) * 0.02).to(tdt)
    x = torch.randn(B, H, generator=g).to(tdt)
    return x, A, Bm


@pytest.mark.parametrize("B,H,r,I,dtype,frac", [
    (1, 2048, 64, 8192, "float32", 0.30),      # Llama-3.2-1B layer, fp32
    (1, 3072, 128, 8192, "float16", 0.35),     # Llama-3.2-3B layer, fp16
    (8, 4096, 256, 14336, "bfloat16", 0.25),   # Mistral-7B layer, bf16, batch union
    (1, 4096, 440, 11008, "float16", 0.10),    # ReLU-Llama-7B layer: rank int(0.04 * I), 55 chunks per row
    (16, 3072, 128, 8192, "bfloat16", 0.30),   # Llama-3.2-3B layer, bf16, decode batch 16
    (3, 128, 8, 50, "float16", 0.5),           # tiny / ragged
    (2, 64, 4, 17, "float32", 0.5),
    (1, 1024, 1024, 300, "float16", 0.4),      # rank rows longer than one pass of the wave
    (150, 1024, 64, 2048, "float16", 0.02),    # more rows than one pass takes (64): three passes, mask bytes accumulate
    (70, 512, 256, 1024, "bfloat16", 0.02),    # rank 256: a pass takes 56 rows
])
def test_scores_and_mask(B, H, r, I, dtype, frac):
    x, A, Bm = _weights(B * 7 + r, B, H, r, I, dtype)
    s_ref = oracle.predictor_scores(x.float().numpy(), A.float().numpy(), Bm.float().numpy())
    m, s = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), 0.0, True, return_scores=True)
    s = s.cpu().numpy()
    scale = np.abs(s_ref).max()
    assert np.abs(s - s_ref).max() <= 2e-6 * scale + 1e-9           # fp32 accumulation on both sides
    guard = 8e-6 * scale
    thr = syn.threshold_for_fraction(s_ref.max(0) if B > 1 else s_ref, frac, guard=0.0)
    near = np.abs(s_ref - thr) < guard
    for ge in (True, False):
        want = oracle.mask_threshold(s_ref, thr, ge)
        got = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), thr, ge).cpu().numpy()
        diff = got != want
        assert not (diff & ~near.any(0)).any(), "mask bit differs outside the guard band"
        assert diff.sum() <= near.any(0).sum()
    assert near.sum() <= 3, f"guard band population {near.sum()}"      # expected 0, reported if not


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,H,r,I", [
    (9, 64, 8, 17),          # one tile of everything, none of them full; the fewest rows these kernels take
    (16, 72, 40, 50),        # H is not a multiple of a k step
    (17, 1024, 128, 2048),   # one row into the second tile of rows
    (33, 512, 136, 1000),    # ranks one chunk into the next register form: 128, 256, 384
    (64, 768, 264, 1024),
    (65, 768, 392, 777),
    (130, 3072, 512, 4096),  # the largest rank of these kernels
    (300, 640, 24, 333),
    (515, 2048, 128, 8192),
])
def test_matrix_core_predictor(B, H, r, I, dtype):
    """Several rows of x: fp32 accuracy of the scores although the rank-r intermediate goes through 16-bit operands,
    also for rows of very different magnitude."""
    x, A, Bm = _weights(B + r, B, H, r, I, dtype)
    mag = torch.logspace(-3, 3, B)[:, None]
    x = (x.float() * mag).to(x.dtype)
    s_ref = oracle.predictor_scores(x.float().numpy(), A.float().numpy(), Bm.float().numpy())
    m, s = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), 0.0, True, return_scores=True)
    scale = np.abs(s_ref).max(1, keepdims=True)                     # per row: each has its own magnitude
    assert (np.abs(s.cpu().numpy() - s_ref) <= 2e-6 * scale + 1e-12).all()   # (the bound of test_scores_and_mask, per row)
    # a cut that only a few indices pass in any row, so that every row decides some of them
    thr = float(np.sort(s_ref.max(0))[-max(1, I // 3)]) * (1 - 1e-4)
    near = (np.abs(s_ref - thr) < 8e-6 * scale).any(0)
    for ge in (True, False):
        got = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), thr, ge).cpu().numpy()
        assert np.array_equal(got[~near], oracle.mask_threshold(s_ref, thr, ge)[~near])
    assert near.mean() < 0.01 + 2.0 / I
    assert np.array_equal(m.cpu().numpy(), (s.cpu().numpy() >= 0).any(0))   # mask and scores come from the same sums


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,H,r", [(9, 64, 8), (40, 3072, 128), (100, 512, 392)])
def test_matrix_core_predictor_keeps_every_bit_of_the_intermediate(dtype, B, H, r):
    """With a unit matrix as the second map the scores are the fp32 intermediate, all 24 bits of it: 16-bit parts of it that
    sum to less would show.  (fp16 parts reach down to 2^-24 on a scale where a row's largest element is at least 2^13: what
    lies below that, at most 2^-25 of 2^13, may be lost.)"""
    x, A, _ = _weights(B, B, H, r, r, dtype)
    t_ws = torch.empty(B, r, dtype=torch.float32, device=DEV)
    _, s = st.predictor_mask(x.to(DEV), A.to(DEV), torch.eye(r, dtype=x.dtype, device=DEV), 0.0, True, t_ws=t_ws,
                             return_scores=True)
    want = x.double() @ A.double().t()                               # (and the intermediate is the first map's)
    assert (t_ws.cpu() - want).abs().max() <= 2e-6 * want.abs().max()
    lost = 2.0 ** -38 * t_ws.abs().amax(1, keepdim=True) if dtype == "float16" else 0.0
    assert ((s - t_ws).abs() <= lost).all(), ((s != t_ws).float().mean(), ((s - t_ws) / t_ws).abs().max())


def test_matrix_core_predictor_reads_beyond_4_gib():
    """x and Bm of more than 4 GiB: the last row of either decides the mask (byte offsets of 32 bits would wrap)."""
    H, r, I, B = 4096, 16, 64, 600_000                              # x: 4.9 GB
    g = torch.Generator(device=DEV).manual_seed(3)
    A, Bm = (torch.randn(a, b, generator=g, device=DEV).half() * 0.05 for a, b in ((r, H), (I, r)))
    x = torch.zeros(B, H, dtype=torch.float16, device=DEV)
    x[-1] = torch.randn(H, generator=g, device=DEV).half()
    s = (x[-1:].float() @ A.float().t() @ Bm.float().t())[0]
    hi = s.sort().values[I // 2:]
    at = int((hi[1:] - hi[:-1]).argmax())
    thr = float(hi[at] + hi[at + 1]) / 2
    assert thr > 0 and torch.equal(st.predictor_mask(x, A, Bm, thr, True), s >= thr)
    del x
    H, r, I, B = 64, 136, 1 << 24, 9                                # Bm: 4.6 GB
    A = torch.full((r, H), 0.125, dtype=torch.float16, device=DEV)
    Bm = torch.zeros(I, r, dtype=torch.float16, device=DEV)
    Bm[-1] = 0.125
    x = torch.ones(B, H, dtype=torch.float16, device=DEV)
    assert st.predictor_mask(x, A, Bm, 1.0, True).nonzero().flatten().tolist() == [I - 1]


def test_matrix_core_predictor_rows_beyond_32_bit_offsets():
    """Enough rows of x for tiles of 64, so wide that 64 of them are more than 4 GiB (H a little above 2^25): products of the
    first and last columns only, so that a row read for another would show.  fp32 sums of 32 products: 1e-6 of the largest."""
    H, r, I, B = (1 << 25) + 8, 512, 64, 705
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 100 GB of device memory")
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.zeros(B, H, dtype=torch.float16, device=DEV)          # 47 GB
    A = torch.zeros(r, H, dtype=torch.float16, device=DEV)          # 34 GB
    for t in (x, A):
        for cols in (slice(0, 16), slice(H - 16, H)):
            t[:, cols] = torch.randn(t.size(0), 16, generator=g, device=DEV).half()
    edge = lambda t: torch.cat([t[:, :16], t[:, -16:]], 1).double()
    t_ws = torch.empty(B, r, dtype=torch.float32, device=DEV)
    st.predictor_mask(x, A, torch.zeros(I, r, dtype=torch.float16, device=DEV), t_ws=t_ws)
    want = edge(x) @ edge(A).t()
    assert (t_ws - want).abs().max() <= 1e-6 * want.abs().max()
    del x, A
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("where", ["x", "A", "Bm"])
@pytest.mark.parametrize("round_to_storage", [False, True])
def test_matrix_core_predictor_infinities_and_nan(dtype, where, round_to_storage):
    """Infinities, NaN and the largest finite values: every score is of the kind (NaN, either infinity, finite) that the
    kernels for fewer rows of x, which multiply in fp32, give for the same row."""
    B, H, r, I = 24, 256, 40, 300
    x, A, Bm = (t.to(DEV) for t in _weights(11, B, H, r, I, dtype))
    inf, nan, big = float("inf"), float("nan"), torch.finfo(x.dtype).max
    x[7] = 0.0                                                   # 0 * inf
    if where == "x":
        x[2, 9], x[5, 200], x[19, 255] = inf, -inf, nan
        x[11, :16] = big
        A[8, 9], Bm[8] = 0.0, 0.0                                # inf * 0, once in either map
        if dtype == "bfloat16":   # an element of the intermediate that is finite and would round to an infinity in 16 bits
            A[30] = 0.0
            A[30, 0] = A[30, 1] = 1.0
            x[13] = 0.0
            x[13, 0], x[13, 1] = big, 0.75 * 2.0 ** 120
    elif where == "A":
        A[3] = 0.0
        A[20, 0], A[21, 255], A[22, 17] = inf, -inf, inf
        Bm[10:, 20:23] = 0.0
        x[12, 0] = x[12, 255] = 0.0
    else:
        Bm[3, 5], Bm[4, 6], Bm[5, 7] = inf, -inf, nan
        Bm[6, 0], Bm[6, 1], Bm[7] = inf, -inf, inf
        Bm[8], Bm[9, 39] = 0.0, big
        A[3] = 0.0
        Bm[11, 3] = inf                                          # meets t = 0
        A[0, 0], A[38], x[15] = 6e4, 0.0, 0.0                    # meets an element 2^-60 of its row's largest one
        x[15, 0], x[15, 1], A[38, 1], Bm[12, 38] = 6e4, 2.0 ** -14, 2.0 ** -14, inf
    few = torch.cat([st.predictor_scores(x[b:b + 8].contiguous(), A, Bm, round_to_storage) for b in range(0, B, 8)])
    m, s = st.predictor_mask(x, A, Bm, 0.5, True, return_scores=True, round_to_storage=round_to_storage)
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(s), kind(few)), (kind.__name__, (kind(s) != kind(few)).nonzero()[:8].tolist())
    assert torch.isnan(s).any() and (where == "x" or torch.isposinf(s).any() and torch.isneginf(s).any())
    assert torch.equal(m, (s >= 0.5).any(0))
    near = torch.isfinite(few) & ((few - 0.5).abs() < 1e-4 + (1e-2 if round_to_storage else 0.0))
    assert torch.equal(m[~near.any(0)], (few >= 0.5).any(0)[~near.any(0)])


@pytest.mark.parametrize("dtype,r", [("float32", 12), ("float16", 40), ("bfloat16", 72), ("float16", 512), ("float32", 264)])
@pytest.mark.parametrize("B", [1, 2, 8])
def test_infinite_intermediate_decides_by_sign(dtype, r, B):
    """Ranks that leave lanes of a group without a part of the row: an infinity at either end of the intermediate gives
    infinities of the weights' signs, not NaN."""
    H, I = 64, 200
    x, A, Bm = (t.to(DEV) for t in _weights(r, B, H, r, I, dtype))
    x[:, 3] = 1.0
    for at in (0, 7, r - 1):
        Ai = A.clone()
        Ai[at, 3] = float("inf")
        m, s = st.predictor_mask(x, Ai, Bm, 0.0, True, return_scores=True)
        assert torch.equal(s, torch.where(Bm[:, at] > 0, float("inf"), -float("inf")).expand(B, I)), (at, s[0, :4])
        assert torch.equal(m, Bm[:, at] > 0)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,H,r,I", [
    (5, 520, 136, 26600), (8, 1000, 256, 14336), (6, 264, 232, 7192),                         # the second map alone (bf16)
    (9, 64, 16, 200), (20, 1000, 128, 8192), (33, 520, 200, 5001), (64, 256, 256, 1000),      # four waves, 4 / 2 / 1 groups
    (77, 520, 104, 5001), (130, 128, 384, 777), (300, 264, 440, 8191), (257, 64, 512, 640),   # eight (four above rank 384)
    (2100, 200, 200, 5001), (2100, 1000, 224, 1000),                                         # 64 x 32 tiles of the intermediate
    (200, 520, 48, 1000), (160, 264, 320, 1000), (400, 264, 320, 1000), (530, 136, 512, 640),   # tiles of x first; of the rank: x smaller, an uneven number
])
def test_matrix_core_mask_without_scores(dtype, B, H, r, I):
    """Masks decided in registers against the scores the same kernels write: every rank and group form, thresholds that are a
    score (>= and > differ there), infinities and NaN; and the scores against float64 (fp32 sums: 4e-6 of the largest)."""
    x, A, Bm = (t.to(DEV) for t in _weights(r + B, B, H, r, I, dtype))
    s = st.predictor_scores(x, A, Bm)
    want = (x.double() @ A.double().t()) @ Bm.double().t()
    assert (s.double() - want).abs().max() <= 4e-6 * want.abs().max()
    cases = [(x, Bm, s)]
    Bi, xi = Bm.clone(), x.clone()
    Bi[3, 5], Bi[4, 6], Bi[5, 7], Bi[I - 1] = float("inf"), float("-inf"), float("nan"), float("inf")
    cases.append((x, Bi, st.predictor_scores(x, A, Bi)))
    xi[B - 1, 0], xi[0, 1] = float("inf"), float("nan")
    cases.append((xi, Bm, st.predictor_scores(xi, A, Bm)))
    for xc, Bc, sc in cases:
        top = torch.where(torch.isnan(sc), -float("inf"), sc).amax(0)       # a NaN never passes
        for thr in (0.0, float(top.sort().values[I // 2]), float("inf"), float("-inf"), float("nan")):
            for ge in (True, False):
                got = st.predictor_mask(xc, A, Bc, thr, ge)
                assert torch.equal(got, ((sc >= thr) if ge else (sc > thr)).any(0)), (thr, ge)


def test_naive_threshold_is_score_ge_zero():
    x, A, Bm = _weights(1, 2, 256, 16, 512, "float32")
    # make some scores exactly zero: a zero row of Bm gives score 0 for every input row
    Bm[5] = 0.0
    Bm[77] = 0.0
    m_ge = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), 0.0, True).cpu().numpy()
    m_gt = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), 0.0, False).cpu().numpy()
    assert m_ge[5] and m_ge[77] and not m_gt[5] and not m_gt[77]     # >= vs > on an exact tie
    s = oracle.predictor_scores(x.numpy(), A.numpy(), Bm.numpy())
    safe = np.abs(s).min(0) > 1e-6
    assert np.array_equal(m_ge[safe], (s >= 0).any(0)[safe])


@pytest.mark.parametrize("method", ["naive", "topk", "statistical_topk"])
def test_mask_methods_of_the_reference(method):
    """The three sparsity methods of SkipDecoderLayer._compute_binary_mask, union over rows included."""
    B, H, r, I = 4, 512, 32, 2048
    x, A, Bm = _weights(3, B, H, r, I, "float32")
    pred = st.FastLoRAProjection(A.to(DEV), Bm.to(DEV))
    s_ref = oracle.predictor_scores(x.numpy(), A.numpy(), Bm.numpy())
    if method == "naive":
        got = pred.mask(x.to(DEV), "naive").cpu().numpy()
        want, margin = oracle.mask_threshold(s_ref, 0.0, True), np.abs(s_ref).min(0)
    elif method == "topk":
        k = 300
        got = pred.mask(x.to(DEV), "topk", k=k).cpu().numpy()
        want = oracle.mask_topk(s_ref, k)
        kth = np.sort(s_ref, axis=1)[:, -k][:, None]
        margin = np.abs(s_ref - kth).min(0)
    else:
        z = float(torch.distributions.normal.Normal(0, 1).icdf(torch.tensor(0.7)))
        got = pred.mask(x.to(DEV), "statistical_topk", std_multiplier=z).cpu().numpy()
        want, cut = oracle.mask_statistical(s_ref, z)
        margin = np.abs(s_ref - cut[:, None]).min(0)
    safe = margin > 1e-5 * np.abs(s_ref).max()
    assert safe.mean() > 0.99
    assert np.array_equal(got[safe], want[safe])


def test_predictor_argument_errors():
    x, A, Bm = _weights(0, 1, 64, 8, 32, "float32")
    with pytest.raises(ValueError):
        st.predictor_mask(x.to(DEV), A.to(DEV)[:, :32], Bm.to(DEV))
    with pytest.raises(TypeError):
        st.predictor_mask(x.to(DEV), A.to(DEV).half(), Bm.to(DEV))
    with pytest.raises(ValueError):
        st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), out=torch.zeros(31, dtype=torch.bool, device=DEV))
    sd = {"down.weight": A, "up.weight": Bm}
    p = st.FastLoRAProjection.from_state_dict(sd, device=DEV, dtype=torch.float32)   # the reference's checkpoint keys
    assert p.lora_size == 8 and p.intermediate_size == 32


def test_loaded_checkpoints_drive_the_hip_predictor(tmp_path):
    """Predictor files as the reference's trainer writes them (fp32 state dicts with keys down.weight [r,H] and
    up.weight [I,r] under final_predictor_layer_{i}_lora_{pct}pct.pt, src/trainer.py:569-585), loaded the way
    benchmark.py:460-468 consumes them, here onto the GPU in fp16: the loaded predictors' scores and masks against
    the oracle on the same (fp16-rounded) weights."""
    H, I = 3072, 8192
    r = int(I * 0.016)          # the trainer's sizing rule int(I * pct / 100) at 1.6 % -> 131 -> not a multiple of 8
    r = (r // 8) * 8            # 128: rank rows must be 16-byte multiples in fp16
    g = torch.Generator().manual_seed(21)
    want = []
    for layer in range(2):
        sd = {"down.weight": torch.randn(r, H, generator=g) * 0.02, "up.weight": torch.randn(I, r, generator=g) * 0.02}
        torch.save(sd, tmp_path / st.FastLoRAProjection.checkpoint_name(layer, 1.6))
        want.append(sd)
    preds = st.load_predictors(str(tmp_path), 2, 1.6, device=DEV, dtype=torch.float16)
    x = torch.randn(2, H, generator=g).half()
    for p, sd in zip(preds, want):
        assert p.down_weight.is_cuda and p.down_weight.dtype == torch.float16 and p.lora_size == r
        A, Bm = sd["down.weight"].half().float().numpy(), sd["up.weight"].half().float().numpy()
        s_ref = oracle.predictor_scores(x.float().numpy(), A, Bm)
        s = p(x.to(DEV)).cpu().numpy()
        scale = np.abs(s_ref).max()
        assert np.abs(s - s_ref).max() <= 2e-6 * scale
        thr = syn.threshold_for_fraction(s_ref.max(0), 0.35)
        near = (np.abs(s_ref - thr) < 8e-6 * scale).any(0)
        got = p.mask(x.to(DEV), "threshold", thr=thr).cpu().numpy()
        assert np.array_equal(got[~near], oracle.mask_threshold(s_ref, thr, True)[~near]) and near.sum() <= 3
        got_naive = p.mask(x.to(DEV), "naive").cpu().numpy()
        safe = np.abs(s_ref).min(0) > 8e-6 * scale
        assert np.array_equal(got_naive[safe], oracle.mask_threshold(s_ref, 0.0, True)[safe]) and safe.mean() > 0.999


@pytest.mark.parametrize("dtype,B,H,r,I", [("float16", 1, 3072, 128, 8192), ("bfloat16", 4, 4096, 256, 14336)])
def test_scores_rounded_to_the_storage_type(dtype, B, H, r, I):
    """round_to_storage: the rank-r intermediate and the scores as two half-precision modules hand them on
    (FastLoRAProjection in an fp16 / bf16 model, src/modeling_skip.py:52-53) against the oracle's restatement of that;
    and how many mask bits that moves against the fp32 scores at the benchmark's active fraction."""
    x, A, Bm = _weights(5, B, H, r, I, dtype)
    xs, As, Bs = x.float().numpy(), A.float().numpy(), Bm.float().numpy()
    want = oracle.predictor_scores(xs, As, Bs, storage=dtype)
    got = st.predictor_scores(x.to(DEV), A.to(DEV), Bm.to(DEV), round_to_storage=True).cpu().numpy()
    # every score is a value of the storage type
    tdt = getattr(torch, dtype)
    assert np.array_equal(torch.from_numpy(got).to(tdt).float().numpy(), got)
    # equal to the oracle's except where an fp32 sum sat within rounding distance of a tie between two storage values:
    # a score is then one step of the storage type off, or -- when it was an entry of the intermediate -- a few
    ulp = np.abs(want) * (2.0 ** -10 if dtype == "float16" else 2.0 ** -7) + 1e-30
    diff = np.abs(got - want)
    assert (diff <= 8 * ulp + 1e-3 * np.abs(want).max()).all() and (diff > 0).mean() < 0.02, \
        ((diff > 0).mean(), (diff / ulp).max())
    # masks: exact wherever the two implementations' scores agree; and the count of bits the rounding itself moves
    s32 = oracle.predictor_scores(xs, As, Bs)
    thr = syn.threshold_for_fraction(s32.max(0), 0.35)
    m_round = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), thr, True, round_to_storage=True).cpu().numpy()
    agree = (diff == 0).all(0)
    assert np.array_equal(m_round[agree], oracle.mask_threshold(want, thr, True)[agree])
    m_fp32 = st.predictor_mask(x.to(DEV), A.to(DEV), Bm.to(DEV), thr, True).cpu().numpy()
    moved = int((m_round != m_fp32).sum())
    print(f"{dtype}: {moved} of {I} mask bits differ between scores kept in fp32 and scores rounded to {dtype}")
    assert moved <= (40 if dtype == "float16" else 300)
    # fp32 storage: the flag changes nothing
    x32, A32, B32 = _weights(6, 1, 256, 16, 512, "float32")
    a = st.predictor_scores(x32.to(DEV), A32.to(DEV), B32.to(DEV), round_to_storage=True)
    b = st.predictor_scores(x32.to(DEV), A32.to(DEV), B32.to(DEV))
    assert torch.equal(a, b)


@pytest.mark.parametrize("B,H,r,I,dtype", [(8, 1000, 256, 14336, "bfloat16"), (5, 520, 136, 26600, "float16"), (3, 512, 128, 4096, "float16"),
                                           (20, 512, 200, 5001, "bfloat16")])
def test_layers_together_give_the_masks_of_one(B, H, r, I, dtype):
    """What a stack's layers share is the launch: masks and intermediate equal the single-layer calls', bit for bit."""
    L = 3
    ws = [tuple(t.to(DEV) for t in _weights(10 * l + B, B, H, r, I, dtype)) for l in range(L)]
    x = torch.stack([w[0] for w in ws])
    t_all, masks = torch.empty(L * B * r, dtype=torch.float32, device=DEV), [torch.ones(I, dtype=torch.bool, device=DEV) for _ in range(L)]
    thrs = []
    for _, A, Bm in ws:
        thrs.append(float(st.predictor_scores(x[len(thrs)], A, Bm).amax(0).sort().values[I // 2]))   # a score: a tie
    st.ops.predictor_mask_layers(x, [(A, Bm, m, thr, l % 2 == 0) for l, ((_, A, Bm), m, thr) in enumerate(zip(ws, masks, thrs))], t_all)
    for l, (_, A, Bm) in enumerate(ws):
        t = torch.empty(B * r, dtype=torch.float32, device=DEV)
        assert torch.equal(masks[l], st.predictor_mask(x[l], A, Bm, thrs[l], l % 2 == 0, t_ws=t))
        assert torch.equal(t_all[l * B * r:(l + 1) * B * r], t)
