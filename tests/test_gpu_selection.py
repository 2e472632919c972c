"""GPU parity of the other KV-selection cases of the reference (RoCo, SnapKV, Corm, KeyFormer) and of the selection ops
around them (pooling, KV-cache compaction), against the CPU oracle on identical seeded inputs."""
import numpy as np
import pytest
import torch

from conftest import assert_close, progress
from deepgengraph_amd import _lib
from deepgengraph_amd import attention as A
from deepgengraph_amd.compile import compile as dgg_compile
from oracle import attention as oa
from oracle import cases as ocases
from oracle import selection as osel

pytestmark = pytest.mark.gpu

TOL_F16 = (1e-2, 5e-3)


def _qkv(S, H, D, seed, dtype=torch.float16, sinks=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(1, S, H, D, generator=g)
    k = torch.randn(1, S, H, D, generator=g)
    v = torch.randn(1, S, H, D, generator=g)
    if sinks:
        k[:, torch.randperm(S, generator=g)[:sinks]] *= 4.0
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _corm_check(hit, q, k, v, thr, what):
    """Booleans must equal the oracle's; a differing key is accepted only when its deciding comparison is a
    tie to within 2e-6 relative (max_i (p - thr) / thr ~ 0), where fp32 rounding order decides."""
    _, ref, _ = oa.corm(q, k, v, thr)
    diff = hit.cpu() != ref
    if diff.any():
        rows, _, _ = oa._causal_probs(q, k, v, 256)
        rel = torch.full(ref.shape, float("-inf"))
        for i0, n, probs in rows:
            t = thr[i0:i0 + n]
            rel = torch.maximum(rel, ((probs - t) / t).amax(dim=2))
        assert (rel[diff].abs() < 2e-6).all(), f"{what}: {int(diff.sum())} keys differ away from a tie"
    return int(diff.sum())


@pytest.mark.parametrize("S,H,D", [(300, 2, 128), (1000, 4, 128), (257, 2, 64)])
def test_roco_matches_oracle(gpu, S, H, D):
    progress(f"roco S{S} H{H} D{D}")
    q, k, v = _qkv(S, H, D, S + D, sinks=4)
    ref_out, ref_s1, ref_s2, _ = oa.roco(q, k, v)
    out, s1, s2 = A.roco_attention(q.to(gpu), k.to(gpu), v.to(gpu))
    what = f"roco S{S} H{H} D{D}"
    assert_close(out.cpu().float(), ref_out.float(), *TOL_F16, what + " out")
    assert_close(s1.cpu(), ref_s1, 1e-6, 1e-3, what + " roco_score")
    assert_close(s2.cpu(), ref_s2, 1e-6, 1e-3, what + " roco_sq_score")
    assert_close(s1.sum(-1).cpu(), torch.full((1, H), float(S)), 0, 1e-4, what + " sum of colsums = q_len")


@pytest.mark.parametrize("S,H,D,ks", [(300, 2, 128, 5), (777, 2, 128, 3), (257, 2, 64, 5)])
def test_snapkv_matches_oracle(gpu, S, H, D, ks):
    progress(f"snapkv S{S} H{H} D{D} k{ks}")
    q, k, v = _qkv(S, H, D, 2 * S + D)
    ref_out, ref_score, _ = oa.snapkv(q, k, v, kernel_size=ks)
    out, score = A.snapkv_attention(q.to(gpu), k.to(gpu), v.to(gpu), kernel_size=ks)
    assert_close(out.cpu().float(), ref_out.float(), *TOL_F16, "snapkv out")
    assert_close(score.cpu(), ref_score, 1e-6, 1e-3, "snapkv_score")


@pytest.mark.parametrize("S,H,D", [(300, 2, 128), (1000, 2, 128), (257, 2, 64)])
def test_corm_matches_oracle(gpu, S, H, D):
    progress(f"corm S{S} H{H} D{D}")
    q, k, v = _qkv(S, H, D, 3 * S + D, sinks=3)
    thr = oa.corm_mask(S, S)
    out, hit = A.corm_attention(q.to(gpu), k.to(gpu), v.to(gpu), thr.to(gpu))
    assert hit.dtype == torch.bool and hit.shape == (1, H, S)
    ref_out, ref_hit, _ = oa.corm(q, k, v, thr)
    assert_close(out.cpu().float(), ref_out.float(), *TOL_F16, "corm out")
    _corm_check(hit, q, k, v, thr, f"corm S{S} H{H} D{D}")
    assert hit[..., 0].all()  # row 0 attends key 0 with p = 1 >= 1
    # q = 0: every visible p equals its threshold 1/(i+1) exactly, so every key is selected
    _, hit0 = A.corm_attention(torch.zeros_like(q).to(gpu), k.to(gpu), v.to(gpu), thr.to(gpu))
    assert hit0.all()


@pytest.mark.parametrize("S,H,D,aligned", [(300, 2, 128, True), (1000, 2, 128, True), (257, 2, 64, True),
                                            (301, 2, 128, False)])
def test_keyformer_matches_oracle(gpu, S, H, D, aligned):
    progress(f"keyformer S{S} H{H} D{D} aligned={aligned}")
    q, k, v = _qkv(S, H, D, 4 * S + D, sinks=4)
    g = torch.Generator().manual_seed(S)
    er = oa.exp_rand(1, H, S, S, g)
    if aligned:
        er_dev = er.to(gpu)
    else:  # rows of S + 1 floats from an offset of one element: the unaligned (4-byte load) path
        big = torch.ones(1, H, S, S + 2)
        big[..., 1:S + 1] = er
        er_dev = big.to(gpu)[..., 1:S + 1]
    out, score = A.keyformer_attention(q.to(gpu), k.to(gpu), v.to(gpu), er_dev, tau=1.5)
    ref_out, ref_score, _ = oa.keyformer(q, k, v, er, tau=1.5)
    what = f"keyformer S{S} H{H} D{D}"
    assert_close(out.cpu().float(), ref_out.float(), *TOL_F16, what + " out")
    assert_close(score.cpu(), ref_score, 1e-6, 1e-3, what + " kf_score")
    assert_close(score.sum(-1).cpu(), torch.full((1, H), float(S)), 0, 1e-4, what + " sum of kf scores = q_len")


def test_keyformer_wide_exp_rand_rows(gpu):
    # exp_rand rows 4.1M floats apart: the column pass's 32-bit tile offsets do not fit, every tile takes the
    # general addressing (a 4.2 GB device buffer of which the [256, 256] corner is used)
    S, H, D = 256, 1, 128
    progress("keyformer wide exp_rand rows")
    q, k, v = _qkv(S, H, D, 77, sinks=2)
    er = oa.exp_rand(1, H, S, S, torch.Generator().manual_seed(78))
    wide = 4_100_000
    buf = torch.empty(S, wide, dtype=torch.float32, device=gpu)
    buf[:, :S] = er[0, 0].to(gpu)
    er_dev = buf[:, :S].view(1, 1, S, S)
    out, score = A.keyformer_attention(q.to(gpu), k.to(gpu), v.to(gpu), er_dev, tau=1.5)
    ref_out, ref_score, _ = oa.keyformer(q, k, v, er, tau=1.5)
    assert_close(out.cpu().float(), ref_out.float(), *TOL_F16, "keyformer wide out")
    assert_close(score.cpu(), ref_score, 1e-6, 1e-3, "keyformer wide kf_score")
    del buf


@pytest.mark.parametrize("kind", ["never", "some_keys", "late_rows", "zero", "nan_inf"])
def test_corm_thresholds_that_decide_late_or_never(gpu, kind):
    # The head_dim-128 Corm column pass stops a workgroup once every key of every wave is flagged. These
    # thresholds keep keys undecided for the whole pass (never: p <= 1 < 2), for some key ranges only, until the
    # last rows, or decide them at once (zero); NaN never selects, -inf always does.
    S, H, D = 1100, 2, 128
    q, k, v = _qkv(S, H, D, 5 * S + len(kind), sinks=4)
    g = torch.Generator().manual_seed(17)
    thr = oa.corm_mask(S, S).clone()
    if kind == "never":
        thr.fill_(2.0)
    elif kind == "some_keys":
        thr[:, 300:700] = 2.0  # keys of these columns never pass; the others decide as usual
    elif kind == "late_rows":
        thr[: S - 40] = 2.0    # only the last 40 rows can flag anything
    elif kind == "zero":
        thr.zero_()            # p >= 0 everywhere, masked pairs included
    else:
        thr = torch.rand(S, S, generator=g)
        thr[torch.rand(S, S, generator=g) < 0.3] = float("nan")
        thr[torch.rand(S, S, generator=g) < 0.01] = float("-inf")
    progress(f"corm thresholds {kind}")
    _, hit = A.corm_attention(q.to(gpu), k.to(gpu), v.to(gpu), thr.to(gpu))
    n = _corm_check(hit, q, k, v, thr, f"corm thresholds {kind}")
    if kind == "never":
        assert not hit.any()
    if kind == "zero":
        assert hit.all()
    if kind == "some_keys":
        assert not hit[..., 300:700].any() and n == 0


def _corm_reference(q, k, thr, causal, window):
    """corm.py:35-37 over every query row: probs >= thr with the reference's probabilities (scores rounded in the
    input dtype, masked pairs -inf, so p = 0 there and NaN on rows that see no key), any over the rows. Also
    returns the float64 probabilities for the tie check."""
    B, Sq, H, D = q.shape
    Sk = k.shape[1]
    s = oa._scores(q.transpose(1, 2), k.transpose(1, 2).transpose(-2, -1), D).float()
    m = oa._mask(0, Sq, Sq, Sk, causal, window or None)
    if m is not None:
        s = s.masked_fill(m, float("-inf"))
    probs = torch.softmax(s, -1)
    return (probs >= thr).any(dim=2), probs.double()


@pytest.mark.parametrize("D,dtype,Sq,Sk,causal,window", [
    (128, torch.float16, 600, 600, True, 0),
    (128, torch.float16, 700, 400, True, 0),      # Sq > Sk: the first 300 rows see no key (NaN probabilities)
    (128, torch.bfloat16, 500, 500, True, 97),    # causal + window: masked pairs on both sides
    (128, torch.float16, 300, 450, False, 80),    # window without causal
    (64, torch.float16, 400, 300, True, 0),       # the generic column kernel
    (256, torch.bfloat16, 300, 300, True, 50),
    (128, torch.float32, 300, 200, True, 0),      # the fp32 column kernel
])
def test_corm_masked_pairs_and_empty_rows(gpu, D, dtype, Sq, Sk, causal, window):
    # thresholds 2 (never passed) except: <= 0 at random masked pairs, and at every pair of the rows that see
    # no key; plus random positive thresholds on a band so that visible pairs flag some keys too
    g = torch.Generator().manual_seed(D + Sq + Sk + window)
    q = torch.randn(1, Sq, 2, D, generator=g).to(dtype)
    k = torch.randn(1, Sk, 2, D, generator=g).to(dtype)
    v = torch.randn(1, Sk, 2, D, generator=g).to(dtype)
    thr = torch.full((Sq, Sk), 2.0)
    hidden = oa._mask(0, Sq, Sq, Sk, causal, window or None)
    pick = torch.rand(Sq, Sk, generator=g) < 0.002
    thr[hidden & pick] = torch.tensor([0.0, -0.0, -1.0, float("-inf")])[torch.randint(0, 4, (int((hidden & pick).sum()),),
                                                                                      generator=g)]
    if Sq > Sk and causal:
        thr[: Sq - Sk] = -1.0  # rows that see no key: NaN >= -1 is False, they flag nothing
    band = torch.rand(Sq, Sk, generator=g) < 0.05
    thr[band & ~hidden] = 0.02
    progress(f"corm masked pairs D{D} {dtype} Sq{Sq} Sk{Sk} causal={causal} w={window}")
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    _, lse = A.attention(qg, kg, vg, causal=causal, window=window, return_lse=True, ref_rounding=True, lse_base2=True)
    hit = A.attention_colscore(qg, kg, lse, epilogue=_lib.COL_ANY_GE, thr=thr.to(gpu), causal=causal, window=window,
                               lse_base2=True).cpu()
    ref, probs = _corm_reference(q, k, thr, causal, window)
    diff = hit != ref
    if diff.any():  # only a visible pair whose p ties its threshold to fp32 rounding may differ
        b, h, j = diff.nonzero()[0].tolist()
        col_p, col_t = probs[b, h, :, j], thr[:, j].double()
        assert ((col_p - col_t).abs() / col_t.abs() < 2e-6).any(), f"key {j} head {h} differs away from a tie"
    assert hit.any() and not hit.all()


def test_colscore_thresholds_and_strides(gpu):
    # a strided threshold view and an arbitrary threshold: any(p >= t) with t = 0.05 everywhere
    S, H, D = 200, 2, 128
    q, k, v = _qkv(S, H, D, 91)
    big = torch.full((S, S + 40), 0.05, dtype=torch.float32)
    thr = big[:, 8:8 + S]
    out, hit = A.corm_attention(q.to(gpu), k.to(gpu), v.to(gpu), big.to(gpu)[:, 8:8 + S])
    _corm_check(hit, q, k, v, thr.contiguous(), "corm strided threshold")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_kv_gather_matches_oracle(gpu, dtype):
    g = torch.Generator().manual_seed(5)
    B, S, H, D, n = 2, 500, 4, 128, 64
    k = torch.randn(B, S, H, D, generator=g).to(dtype)
    v = torch.randn(B, S, H, D, generator=g).to(dtype)
    idx = torch.stack([torch.stack([torch.sort(torch.randperm(S, generator=g)[:n])[0] for _ in range(H)])
                       for _ in range(B)]).contiguous()
    got = A.kv_gather(k.to(gpu), v.to(gpu), idx.to(gpu)).cpu()
    assert torch.equal(got, osel.kv_gather(k, v, idx))
    # strided k/v views (the fused QKV activation), and indices outside [0, S) -> zero rows
    kv = torch.randn(B, S, H, 3 * D, generator=g).to(dtype)
    kview, vview = kv[..., :D], kv[..., D:2 * D]
    bad = idx.clone()
    bad[0, 1, 3] = -1
    bad[1, 2, 7] = S
    got = A.kv_gather(kview.to(gpu), vview.to(gpu), bad.to(gpu)).cpu()
    want = osel.kv_gather(kview.contiguous(), vview.contiguous(), bad.clamp(0, S - 1))
    want[0, :, 3, 1] = 0
    want[1, :, 7, 2] = 0
    assert torch.equal(got, want)


@pytest.mark.parametrize("shape,density", [((1, 32, 4096), 0.02), ((2, 3, 1000), 0.5), ((5,), 0.6),
                                           ((3, 2, 2, 300), 1.0), ((4, 700), 0.0), ((3, 0), 0.5)])
def test_nonzero_matches_oracle(gpu, shape, density):
    g = torch.Generator().manual_seed(len(shape) * 7 + int(density * 10))
    x = torch.rand(*shape, generator=g) < density
    got = A.nonzero(x.to(gpu))
    want = osel.nonzero(x)
    assert got.dtype == torch.int64 and got.shape == want.shape, (got.shape, want.shape)
    assert torch.equal(got.cpu(), want)
    if x.numel():
        assert torch.equal(A.nonzero(x.to(torch.uint8).to(gpu)).cpu(), want)  # uint8 input


def test_corm_selection_nonzero(gpu):
    # models/corm.py:45-55: the keys Corm flags, as coordinates (b, h, j) in row-major order
    S, H, D = 500, 3, 128
    q, k, v = _qkv(S, H, D, 17, sinks=3)
    thr = oa.corm_mask(S, S)
    _, hit = A.corm_attention(q.to(gpu), k.to(gpu), v.to(gpu), thr.to(gpu))
    sel = A.nonzero(hit)
    assert torch.equal(sel.cpu(), torch.nonzero(hit.cpu()))
    assert sel.shape[1] == 3 and (sel[:, 2] == 0).sum().item() == H  # key 0 is flagged in every head


def test_avg_pool1d_matches_oracle(gpu):
    x = torch.randn(6, 1000, generator=torch.Generator().manual_seed(2))
    for ks in (1, 3, 5, 9):
        assert_close(A.avg_pool1d(x.to(gpu), ks).cpu(), osel.avg_pool1d(x, ks), 1e-6, 1e-6, f"pool k={ks}")


@pytest.mark.parametrize("case_cls", [ocases.RoCo, ocases.SnapKV, ocases.Corm, ocases.KeyFormer])
def test_compile_drop_in_selection_cases(gpu, case_cls):
    # run_kernel.py:44-78 flow for the other selection cases
    model = case_cls(kv_head_num=4, head_num=4, head_dim=128).eval()
    specs = model.prepare(q_len=384, kv_len=384, dtype=torch.float16, seed=11)
    names = list(specs["input"].keys())
    inputs = [specs["input"][n] for n in names]
    f = dgg_compile(model=model, input_names=names, inputs=inputs, output_names=specs["output"], system="mi355x")
    outs = f(*[t.to(gpu) for t in inputs])
    refs = model(*inputs)
    assert isinstance(outs, tuple) and len(outs) == len(refs) == len(specs["output"])
    assert_close(outs[0].cpu().float(), refs[0].float(), *TOL_F16, f"{case_cls.__name__} out")
    for o, r in zip(outs[1:], refs[1:]):
        assert o.shape == r.shape and o.dtype == r.dtype
        if r.dtype == torch.bool:
            _corm_check(o, *[t for t in inputs[:3]], inputs[3], "compiled corm")
        else:
            assert_close(o.cpu(), r, 1e-6, 1e-3, f"{case_cls.__name__} score")


def test_selection_full_size_heads(gpu):
    # config-4 shapes (fp16, S = 4096, D = 128) on two heads: RoCo sums and Corm flags against the oracle,
    # then the top-256 selection and the compaction of the selected rows
    S, H, D = 4096, 2, 128
    progress("selection full size: oracle")
    q, k, v = _qkv(S, H, D, 4096, sinks=16)
    _, ref_s1, ref_s2, _ = oa.roco(q, k, v, q_chunk=512)
    progress("selection full size: gpu")
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    out, s1, s2 = A.roco_attention(qg, kg, vg)
    assert_close(s1.cpu(), ref_s1, 1e-6, 1e-3, "roco_score full")
    assert_close(s2.cpu(), ref_s2, 1e-6, 1e-3, "roco_sq_score full")
    idx = A.topk_indices(s1, 256)
    np.testing.assert_array_equal(idx.cpu().numpy(), osel.topk_indices(ref_s1.numpy(), 256))
    kv = A.kv_gather(kg, vg, idx).cpu()
    assert torch.equal(kv, osel.kv_gather(k, v, idx.cpu()))
    thr = oa.corm_mask(S, S)
    _, hit = A.corm_attention(qg, kg, vg, thr.to(gpu))
    n = _corm_check(hit, q, k, v, thr, "corm full")
    progress(f"corm full: {n} tie-decided keys")
    progress("keyformer full size")
    er = oa.exp_rand(1, H, S, S, torch.Generator().manual_seed(4))
    _, ref_kf, _ = oa.keyformer(q, k, v, er, q_chunk=512)
    _, kf = A.keyformer_attention(qg, kg, vg, er.to(gpu))
    assert_close(kf.cpu(), ref_kf, 1e-6, 1e-3, "kf_score full")
    np.testing.assert_array_equal(A.topk_indices(kf, 256).cpu().numpy(), osel.topk_indices(ref_kf.numpy(), 256))


@pytest.mark.parametrize("S", [448, 577])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_column_forms_agree(gpu, S, dtype):
    """The column passes of large launches (128 keys per workgroup in two row groups, from more than 768 workgroups of 64
    keys) against those of small ones (64 keys, four groups), which the oracle tests cover: 112 heads in one call and
    three of them in a call of their own. The same fp32 terms in another order: 577 of them, each sum within
    577 * 2^-24 = 3.4e-5 of exact in the worst case (twice that for the two together)."""
    H, hs = 112, [0, 50, 111]
    q, k, v = (t.to(gpu) for t in _qkv(S, H, 128, S, dtype=dtype, sinks=4))
    er = 1.0 + torch.randn(1, H, S, S, generator=torch.Generator(device=gpu).manual_seed(S), device=gpu).abs()
    some = [t[:, :, hs].contiguous() for t in (q, k, v)]
    for ref_rounding in (True, False):
        big = A.roco_attention(q, k, v, ref_rounding=ref_rounding)
        few = A.roco_attention(*some, ref_rounding=ref_rounding)
        # the forward picks its form by the launch's size too: its row lse may differ in the last bits
        for b, f, what in zip(big[1:], few[1:], ("sum", "sum of squares")):
            assert_close(b[:, hs].cpu(), f.cpu(), 1e-7, 7e-5, f"roco {what} S{S} {dtype} ref={ref_rounding}")
        big = A.keyformer_attention(q, k, v, er, ref_rounding=ref_rounding)[1]
        few = A.keyformer_attention(*some, er[:, hs].contiguous(), ref_rounding=ref_rounding)[1]
        assert_close(big[:, hs].cpu(), few.cpu(), 1e-7, 7e-5, f"keyformer S{S} {dtype} ref={ref_rounding}")


@pytest.mark.parametrize("largest", [True, False])
@pytest.mark.parametrize("n", [14335, 14336, 15360, 15361, 16383, 16384, 16385, 40000, 65536])
def test_topk_two_stages_by_choice(gpu, n, largest):
    """Rows around and above the length from which topk_indices splits a row over several workgroups, against the
    one-workgroup form: exact, with ties across the chunks, NaN and infinities, k at the limits of the prefilter."""
    g = torch.Generator(device=gpu).manual_seed(n)
    x = torch.randint(0, 3000, (5, n), generator=g, device=gpu).float()
    x[1] = torch.randn(n, generator=g, device=gpu)
    x[2] = 1.0
    x[3, ::7] = float("nan")
    x[3, 5::11] = float("inf")
    x[3, 6::11] = -float("inf")
    x[4] = torch.arange(n, device=gpu).float()
    lib = _lib.load()
    for k in (1, 512, 513, 2048):
        want = torch.empty(5, k, dtype=torch.int64, device=gpu)
        assert lib.dgg_topk_select(_lib.ptr(x), 5, n, k, int(largest), _lib.ptr(want), _lib.stream_handle(gpu)) == 0
        got = A.topk_indices(x, k, largest=largest)
        assert torch.equal(got, want), f"n {n} k {k} largest {largest}"


@pytest.mark.parametrize("n", [16384, 65536])
def test_topk_select_ws_leaves_the_workspace_of_short_rows_alone(gpu, n):
    """dgg_topk_select_ws ignores its workspace for rows of up to 65,536 keys (a caller may have it in use elsewhere),
    whatever its size; the result is dgg_topk_select's."""
    lib = _lib.load()
    x = torch.randn(3, n, generator=torch.Generator(device=gpu).manual_seed(n), device=gpu)
    ws = torch.full((lib.dgg_select_workspace_bytes(3, 1 << 17),), 0xA5, dtype=torch.uint8, device=gpu)
    got, want = (torch.empty(3, 100, dtype=torch.int64, device=gpu) for _ in range(2))
    stream = _lib.stream_handle(gpu)
    assert lib.dgg_topk_select(_lib.ptr(x), 3, n, 100, 1, _lib.ptr(want), stream) == 0
    assert lib.dgg_topk_select_ws(_lib.ptr(x), 3, n, 100, 1, _lib.ptr(got), _lib.ptr(ws), ws.numel(), stream) == 0
    assert torch.equal(got, want) and bool((ws == 0xA5).all())


@pytest.mark.parametrize("n,k", [(5120, 256), (6144, 512), (7736, 64), (7744, 64), (7928, 512), (7936, 512), (16385, 256),
                                 (17000, 16), (27647, 64), (27648, 64), (40000, 512)])
def test_selection_around_the_prefilters_line(gpu, n, k):
    """Rows and counts on either side of the lines from which the one-workgroup selections run the prefilter (threads with
    keys in the last wave; keys per thread; RoCo's own line beyond 16): exact, with ties, against the oracle."""
    g = torch.Generator().manual_seed(n + k)
    x = torch.stack([torch.randn(n, generator=g), torch.randint(0, 50, (n,), generator=g).float()])
    lib = _lib.load()
    xg, got = x.to(gpu), torch.empty(2, k, dtype=torch.int64, device=gpu)
    assert lib.dgg_topk_select(_lib.ptr(xg), 2, n, k, 1, _lib.ptr(got), _lib.stream_handle(gpu)) == 0
    np.testing.assert_array_equal(got.cpu().numpy(), osel.topk_indices(x.numpy(), k))
    s1 = torch.rand(2, n, generator=g) * 100
    s1[1] = torch.randint(1, 60, (n,), generator=g).float()
    s2 = s1 * s1 / n + torch.rand(2, n, generator=g)
    rec = A.roco_select(s1.to(gpu), s2.to(gpu), n, 64, k).cpu().numpy()
    np.testing.assert_array_equal(rec, osel.roco_select(s1.numpy(), s2.numpy(), n, 64, k))


@pytest.mark.parametrize("D,Sq,Sk,Hq,Hkv,causal,window,dtype,row_pad", [
    (128, 200, 512, 4, 4, 1, 0, torch.float16, 0),      # Sq < Sk
    (128, 300, 164, 4, 4, 1, 0, torch.bfloat16, 0),     # Sq > Sk: 136 rows see no key; 36 keys in the last tile
    (128, 640, 640, 4, 4, 1, 70, torch.float16, 0),     # a window that starts past tile 0, tiles in rotated order
    (128, 260, 700, 4, 4, 0, 90, torch.bfloat16, 0),    # a window without a causal mask
    (128, 130, 260, 8, 2, 0, 0, torch.float16, 0),      # no mask, grouped heads, 4 keys in the last tile
    (128, 129, 96, 4, 1, 1, 0, torch.bfloat16, 12),     # 32 keys in the last tile, exp_rand rows longer than the keys
    (128, 33, 4, 2, 2, 1, 0, torch.float16, 0),         # one chunk of keys
    (128, 200, 333, 4, 2, 1, 0, torch.float16, 3),      # keys and rows off 16 bytes (the register-staged kernel)
    (128, 130, 200, 1, 1, 1, 0, torch.float16, 4100000),  # exp_rand rows too far apart for 32-bit lane offsets
    (64, 200, 512, 4, 2, 1, 100, torch.bfloat16, 0),
])
def test_keyformer_row_pass(gpu, D, Sq, Sk, Hq, Hkv, causal, window, dtype, row_pad):
    """dgg_attn_kf_rowlse by itself, over what the entry point accepts beyond the KeyFormer case (kf.py:36-39 is causal with
    Sq == Sk), against the log-sum-exp in 64 bits. fp32 scores: the sums of up to 700 terms and exponents of a size of 10 are
    within 700 * 2^-24 + 10 * 2^-23 < 5e-5 of exact (base-2 logarithm)."""
    B, tau = 2 if row_pad < 1000 else 1, 1.5
    g = torch.Generator(device=gpu).manual_seed(Sq + Sk)
    q = torch.randn(B, Sq, Hq, D, generator=g, device=gpu).to(dtype)
    k = torch.randn(B, Sk, Hkv, D, generator=g, device=gpu).to(dtype)
    rs = Sk + row_pad
    er = torch.empty(B * Hq * Sq * rs, device=gpu).as_strided((B, Hq, Sq, Sk), (Hq * Sq * rs, Sq * rs, rs, 1))
    er.copy_(1.0 + torch.randn(B, Hq, Sq, Sk, generator=g, device=gpu).abs())
    lse2 = torch.full((B, Hq, Sq), float("nan"), device=gpu)
    strides = _lib.int64_array([*q.stride()[:3], *k.stride()[:3]])
    _lib.call("dgg_attn_kf_rowlse", _lib.ptr(q), _lib.ptr(k), _lib.ptr(er), _lib.int64_array(er.stride()[:3]),
              _lib.ptr(lse2), B, Sq, Sk, Hq, Hkv, D, strides, D ** -0.5, tau, window, causal, _lib.dtype_code(dtype),
              _lib.stream_handle(gpu))
    qc, kc = q.double().cpu().transpose(1, 2), k.double().cpu().transpose(1, 2).repeat_interleave(Hq // Hkv, dim=1)
    y = (torch.matmul(qc, kc.transpose(2, 3).contiguous()) * D ** -0.5 - er.double().cpu().log()) / tau
    rel = torch.arange(Sq).unsqueeze(1) + (Sk - Sq) - torch.arange(Sk)
    hidden = torch.zeros(Sq, Sk, dtype=torch.bool)
    if causal:
        hidden |= rel < 0
    if window:
        hidden |= rel >= window
    ref = torch.logsumexp(y.masked_fill(hidden, float("-inf")), dim=-1) / np.log(2.0)
    out = lse2.double().cpu()
    assert torch.equal(torch.isinf(out), torch.isinf(ref)) and not torch.isnan(out).any()
    fin = torch.isfinite(ref)
    assert (out[fin] - ref[fin]).abs().max().item() < 5e-5
