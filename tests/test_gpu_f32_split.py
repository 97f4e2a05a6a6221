"""f32 attention whose products go through bf16 matrix instructions, every value as three bf16 parts (f32_split.h): the edges of its tiles
of 64 keys and blocks of 64 rows, values at the ends of f32's range, infinities, and its error against 64 bits."""
import numpy as np
import pytest

from incin_amd import capi, host
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def inputs(seed, B, H, Sq, Skv, D):
    r = np.random.Generator(np.random.PCG64(seed))
    return [r.standard_normal((B, H, n, D), dtype=np.float32) for n in (Sq, Skv, Skv)]


@pytest.mark.parametrize("D", [4, 64, 72, 96, 100, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 1), (33, 31), (64, 64), (63, 65), (65, 33), (127, 129), (130, 200)])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(gpu, D, Sq, Skv, causal):
    """One key, blocks and tiles with one row or key more or less than full, a tile whose second block is empty; the causal edge in each."""
    if causal and Skv < Sq:
        pytest.skip("rows without keys: test_gpu_parity has those")
    q, k, v = inputs(Sq * 7 + Skv + D, 2, 3, Sq, Skv, D)
    got, info = host.sdpa(q, k, v, capi.F32, causal=causal, impl=capi.IMPL_MFMA, return_info=True)
    assert info["impl"] == capi.IMPL_MFMA
    assert np.max(np.abs(got - O.sdpa(q, k, v, causal=causal))) <= 1e-5


@pytest.mark.parametrize("D", [64, 96, 128])
def test_values_that_are_not_finite(gpu, D):
    """What an infinity or a NaN reaches is what the IEEE products give: against the generic kernel (f32 multiply-adds), for an infinite
    value of V (its column), of K (rows whose score is +inf are NaN, those of -inf do without the key) and a NaN in Q (its row)."""
    q, k, v = inputs(5, 1, 2, 70, 90, D)
    for what, t, at, x in (("v", v, (0, 0, 40, 3), np.inf), ("v", v, (0, 1, 89, D - 1), -np.inf), ("k", k, (0, 0, 11, 5), np.inf), ("q", q, (0, 1, 69, 0), np.nan)):
        was = t[at]
        t[at] = x
        with np.errstate(invalid="ignore"):
            got = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA)
            ref = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_GENERIC)
        t[at] = was
        assert np.array_equal(np.isnan(got), np.isnan(ref)), what
        assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref)), what
        fin = np.isfinite(ref)
        assert fin.any() and not fin.all() and np.max(np.abs(got[fin] - ref[fin])) <= 1e-5, what


@pytest.mark.parametrize("D", [64, 96])
@pytest.mark.parametrize("how", ["causal", "limits", "window"])
def test_hidden_blocks_may_hold_anything(gpu, D, how):
    """A NaN in V reaches the rows whose block of 32 sees any of its block of 32 keys, and no other: under the causal flag, the same mask as a tensor
    (through its row limits) and a mask of values with a hidden block inside a tile that is not hidden as a whole."""
    H, S = 96, 192      # (enough workgroups that the planner hands the mask's limits to this kernel)
    q, k, v = inputs(13, 1, H, S, S, D)
    mask = np.zeros((S, S), np.float32)
    if how == "window":
        mask += np.random.Generator(np.random.PCG64(2)).standard_normal((S, S), dtype=np.float32)
        mask[:32, 32:96] = mask[96:, 64:96] = -np.inf
    else:
        mask += np.triu(np.full((S, S), -np.inf, np.float32), 1)
    ref = O.sdpa(q, k, v, mask=mask[None, None])
    hit = [63, 70] + [191] * (how != "window")
    v[0, :, hit, 5] = np.nan
    if how == "causal":
        got = host.sdpa(q, k, v, capi.F32, causal=True, impl=capi.IMPL_MFMA)
    else:
        got = host.sdpa(q, k, v, capi.F32, mask=mask[None, None], impl=capi.IMPL_AUTO if how == "limits" else capi.IMPL_MFMA)
    seen = (mask > -np.inf).reshape(S // 32, 32, S // 32, 32).any(axis=(1, 3))
    bad = np.repeat(seen[:, [x // 32 for x in hit]].any(axis=1), 32)
    assert bad.any() and not bad.all()
    want = ref.copy()
    want[..., bad, 5] = np.nan
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.nanmax(np.abs(got - want)) <= 1e-5


@pytest.mark.parametrize("B,H,S", [(3, 11, 512), (1, 152, 192), (9, 8, 250), (7, 9, 500), (2, 32, 450)])
def test_one_round_of_uneven_blocks_is_paired(gpu, B, H, S):
    """264, 456, 288, 504 and 512 blocks under a causal flag: the part of an XCD's list that goes in reverse is part of it, or all of the second half."""
    q, k, v = inputs(S, B, H, S, S, 64)
    assert np.max(np.abs(host.sdpa(q, k, v, capi.F32, causal=True, impl=capi.IMPL_MFMA) - O.sdpa(q, k, v, causal=True))) <= 1e-5


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,rows64", [
    (48, 1, 1, 143, 402, 64, False, False), (80, 1, 1, 65, 314, 128, False, False), (24, 1, 1, 384, 384, 64, False, True), (48, 1, 1, 192, 192, 64, True, True),
    (24, 4, 4, 152, 300, 64, True, False), (17, 8, 8, 78, 200, 64, False, False), (24, 8, 8, 92, 200, 64, False, True),
    (8, 12, 12, 130, 260, 96, True, False), (25, 8, 8, 70, 300, 96, False, False), (8, 4, 4, 568, 568, 80, True, False), (6, 8, 8, 512, 512, 80, True, True),
    (15, 8, 8, 173, 600, 128, True, False), (11, 6, 6, 350, 900, 128, True, True),
], ids=str)
def test_which_launches_take_64_rows_per_workgroup(gpu, B, Hq, Hkv, Sq, Skv, D, causal, rows64):
    """Both sides of the rule's lines (they were measured on 256 compute units): what AUTO takes gives the bits of the prefill kernel, or others; both are right."""
    if capi.device_info(0).compute_units != 256:
        pytest.skip("the lines are by compute units")
    r = np.random.Generator(np.random.PCG64(Sq + Skv))
    q, k, v = (r.standard_normal(s, dtype=np.float32) for s in ((B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    got, info = host.sdpa(q, k, v, capi.F32, causal=causal, return_info=True)
    assert info["impl"] == capi.IMPL_SPLITKV_MFMA and info["splits"] == 1
    ref = host.sdpa(q, k, v, capi.F32, causal=causal, impl=capi.IMPL_MFMA)
    assert np.array_equal(got, ref) == rows64 and np.max(np.abs(got - ref)) <= 1e-5


@pytest.mark.parametrize("B,H,S,D", [(8, 4, 568, 128), (12, 8, 144, 64), (6, 8, 150, 64), (1, 8, 300, 64)], ids=str)
def test_mask_tensors_that_take_64_rows_per_workgroup(gpu, B, H, S, D):
    """The causal mask as a tensor, on both sides of the lines of the flag (the last one fills no device and goes 32 rows per workgroup): the bits of the prefill kernel
    under the flag where its blocks take the mask's limits, others elsewhere."""
    if capi.device_info(0).compute_units != 256:
        pytest.skip("the lines are by compute units")
    q, k, v = inputs(S + D, B, H, S, S, D)
    mask = np.triu(np.full((S, S), -np.inf, np.float32), 1)[None, None]
    got, flag = host.sdpa(q, k, v, capi.F32, mask=mask), host.sdpa(q, k, v, capi.F32, causal=True, impl=capi.IMPL_MFMA)
    assert np.array_equal(got, flag) == (B > 1) and np.max(np.abs(got - flag)) <= 1e-5


def test_split_launch_without_a_workspace(gpu):
    """An f32 launch whose keys the planner splits runs without a workspace too, unsplit and 64 rows per workgroup - and so where its partial results exceed
    the static buffer."""
    for B, Hq, Hkv, Sq, Skv, D, fits in ((36, 4, 1, 43, 4096, 32, True), (18, 8, 8, 64, 5120, 128, True), (18, 8, 8, 64, 5120, 128, False)):
        r = np.random.Generator(np.random.PCG64(17))
        q, k, v = (r.standard_normal(s, dtype=np.float32) for s in ((B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
        tq, tk, tv = (host.DeviceTensor.from_f32(x, capi.F32) for x in (q, k, v))
        to = host.DeviceTensor(q.shape, capi.F32)
        d = host.make_desc(tq, tk, tv, to)
        need, splits, _ = capi.sdpa_workspace(d)
        assert need > 0 and splits > 1
        if fits:
            capi.sdpa_fwd(d)
        else:
            assert need > capi.STATIC_SCRATCH_BYTES
            capi.sdpa_fwd_static(d)
        capi.sync()
        assert np.array_equal(to.to_f32(), host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA, num_splits=1))


@pytest.mark.parametrize("D", [64, 96])
@pytest.mark.parametrize("bias", [False, True])
def test_padding_rows_may_hold_anything(gpu, D, bias):
    """NaN in the query rows behind a sequence's count, and in their mask rows, changes no bit of the rows before it: a block that is partly filled does not go
    through its keys a second time for them (the second walk's products, and so its last bits, are others)."""
    q, k, v = inputs(31, 3, 4, 200, 200, D)
    lens = np.array([100, 137, 64], np.int32)
    mask = np.random.Generator(np.random.PCG64(4)).standard_normal((3, 4, 200, 200), dtype=np.float32) if bias else None
    run = lambda: host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA, kv_lens=lens, q_lens=lens, mask=mask)
    clean = run()
    for b, n in enumerate(lens):
        q[b, :, n:] = np.nan
        if bias:
            mask[b, :, n:] = np.nan
    got = run()
    for b, n in enumerate(lens):
        assert np.isfinite(clean[b, :, :n]).all() and np.array_equal(got[b, :, :n], clean[b, :, :n])


@pytest.mark.parametrize("exponent", [-60, -20, 20, 60, 120])
def test_values_of_any_size(gpu, exponent):
    """Values far from 1 keep their 24 bits: Q large where K is small, V of any size; and values that round to infinity in bf16."""
    q, k, v = inputs(9, 1, 2, 100, 100, 64)
    s = np.float32(2.0 ** (exponent / 2))
    ref = O.sdpa(q, k, v)
    got = host.sdpa(q * s, k / s, v * np.float32(2.0 ** exponent), capi.F32, impl=capi.IMPL_MFMA)
    assert np.max(np.abs(got.astype(np.float64) * 2.0 ** -exponent - ref)) <= 1e-5
    if exponent == 120:      # (the largest finite value: its first bf16 part would be infinite)
        v[0, 0, 7, 5] = np.finfo(np.float32).max
        got, gen = (host.sdpa(q, k, v, capi.F32, impl=i) for i in (capi.IMPL_MFMA, capi.IMPL_GENERIC))
        assert np.isfinite(got).all() and np.max(np.abs(got - gen) / np.maximum(np.abs(gen), 1)) <= 1e-5


def exact(q, k, v):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(q.shape[-1])
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v


@pytest.mark.parametrize("D,splits", [(64, 0), (96, 0), (128, 0), (40, 0), (64, 2)])
@pytest.mark.parametrize("what", ["v", "v column", "q", "k"])
@pytest.mark.parametrize("exponent", [-104, -112, -118, -123])
def test_values_whose_last_bits_no_part_holds(gpu, D, splits, what, exponent):
    """Below 2^-110 the third bf16 part loses bits; f32 does not down to 2^-126.  V as small as that, or one of its columns beside ordinary ones, Q under
    a K as large as Q is small, K under such a Q: each column within 1e-6 of 64 bits (the IEEE products: 3e-7; a column at 2^-125, whose values lie 2^-149 apart, 6e-8 more)."""
    q, k, v = inputs(21, 1, 2, 70, 200, D)
    small, large = np.float32(2.0 ** exponent), np.float32(2.0 ** -exponent)
    if what == "v":
        v *= small
    elif what == "v column":
        v[..., 3] *= small
    else:
        q, k = (q * small, k * large) if what == "q" else (q * large, k * small)
    got, ref = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA, num_splits=splits), exact(q, k, v)
    off = np.linalg.norm(got - ref, axis=2) / np.linalg.norm(ref, axis=2)
    assert np.max(off) <= 1e-6


@pytest.mark.parametrize("D,Dv", [(64, 64), (40, 36), (80, 68), (128, 100)])
@pytest.mark.parametrize("what", ["small", "large", "zeros"])
def test_results_at_the_ends_of_the_range_that_is_taken_at_once(gpu, D, Dv, what):
    """Results of 2^-50 to 2^-30, V of 2^45 to 2^55, and a V of zeros but for one value too small for three parts; with and without columns of padding: each column
    within 1e-6 of 64 bits, as above, and zeros where V is zero."""
    q, k, v = inputs(23, 1, 2, 70, 100, D)
    v = v[..., :Dv].copy()
    if what == "zeros":
        v[:] = 0.0
        v[..., 7, 3] = np.float32(1.37 * 2.0 ** -118)
    else:
        v *= (2.0 ** (np.linspace(-50, -30, Dv) if what == "small" else np.linspace(45, 55, Dv))).astype(np.float32)
    got, ref = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA), exact(q, k, v)
    norm = np.linalg.norm(ref, axis=2)
    assert np.max(np.linalg.norm(got - ref, axis=2)[norm > 0] / norm[norm > 0]) <= 1e-6 and np.all(got[ref == 0] == 0)


def test_small_weights_of_large_values(gpu):
    """A weight of 2^-121.5 whose value is 2^120 and makes up the result: what scores of that size leave (2^-23 of them, in the exponent)."""
    q, k, v = inputs(22, 1, 2, 40, 200, 64)
    q[:], k[:] = 0.0, 0.0
    q[..., 0], k[..., 150, 0] = 1.0, -121.5 * np.log(2.0) * 8.0
    big = np.sign(v[..., 150, :]) * 2.0 ** 120
    v[:] = 0.0
    v[..., 150, :] = big
    got, ref = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA), exact(q, k, v)
    assert np.max(np.abs(got / ref - 1)) <= 122 * np.log(2.0) * 3 * 2.0 ** -24


@pytest.mark.parametrize("D,splits", [(64, 0), (96, 0), (128, 0), (64, 2)])
def test_large_values_under_a_late_maximum(gpu, D, splits):
    """A key of a later tile 2^7 times as probable as the first ones, and V near the largest finite value there: 2^7 V overflows, the result does
    not (weights of a row are at most one against its maximum).  Bound: the 24 bits of a weighted mean of V."""
    q, k, v = inputs(7, 1, 2, 40, 640, D)
    q[:], k[:] = 0.0, 0.0
    q[..., 0], k[..., 600, 0] = 1.0, 7.0 * np.log(2.0) * np.sqrt(D)
    v[..., :600, :] *= 1e-3
    v[..., 600, :] = np.sign(v[..., 600, :]) * 2e38
    got = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA, num_splits=splits)
    assert np.isfinite(got).all() and np.max(np.abs(got / exact(q, k, v) - 1)) <= 2e-6


@pytest.mark.parametrize("S,D,causal", [(1024, 64, False), (512, 96, True), (700, 128, False)])
def test_error_against_64_bits(gpu, S, D, causal):
    """No larger than that of IEEE-f32 products: those leave 2.2e-7 - 3.5e-7 of the 2-norm here, this kernel 1.2e-7 - 2.0e-7.  The bound is the
    rounding of P and O in f32 (2^-24 each) and of a sum of S / 32 steps (2^-25 sqrt(S / 32) at most), together below 2.5e-7."""
    q, k, v = inputs(S + D, 1, 4, S, S, D)
    q64, k64, v64 = (x.astype(np.float64) for x in (q, k, v))
    s = q64 @ k64.transpose(0, 1, 3, 2) / np.sqrt(D)
    if causal:
        s += np.triu(np.full((S, S), -np.inf), 1)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v64
    got = host.sdpa(q, k, v, capi.F32, causal=causal, impl=capi.IMPL_MFMA)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2.5e-7


def test_scores_take_the_scale_unrounded(gpu):
    """One key and one column: a row's normaliser is its score, q c k with c = scale log2 e, times log 2.  Rounded as IEEE products round it (q c, times k, times
    log 2) its error is 4.33e-8 in the mean square over 40000 rows (1 % by chance); the parts of q c before it is rounded leave 4.19e-8, those of a rounded one 4.84e-8."""
    r = np.random.Generator(np.random.PCG64(8))
    q, k, v = np.zeros((10, 8, 500, 4), np.float32), np.zeros((10, 8, 1, 4), np.float32), np.ones((10, 8, 1, 4), np.float32)
    q[..., 0], k[..., 0] = r.uniform(1, 2, q.shape[:3]), r.uniform(1, 2, k.shape[:3])
    scale, ln2 = np.float32(0.7), np.float32(0.6931471805599453)
    _, lse = host.sdpa(q, k, v, capi.F32, scale=float(scale), impl=capi.IMPL_MFMA, return_lse=True)
    c = np.float32(scale * np.float32(1.4426950408889634))
    true = q[..., 0].astype(np.float64) * float(c) * k[..., 0] * float(ln2)
    off = lambda x: np.sqrt(np.mean((x.astype(np.float64) / true - 1) ** 2))
    assert off(lse) < 1.01 * off(((q[..., 0] * c) * k[..., 0]) * ln2)


# ---- backward -----------------------------------------------------------------------------------------------------------

BWD = [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, mask: launches that the split kernel takes, with the edges of its tiles (64 rows) and blocks (128)
    (3, 16, 16, 129, 127, 64, 64, False, None, None),
    (4, 12, 12, 128, 193, 64, 32, True, None, None),
    (2, 24, 24, 200, 256, 40, 64, True, None, None),
    (4, 16, 16, 100, 100, 4, 4, True, (100, 65, 64, 1), None),
    (4, 24, 12, 194, 194, 64, 64, True, (194, 1, 0, 129), None),
    (50, 1, 1, 33, 31, 64, 64, False, None, None),
    (2, 24, 24, 150, 150, 64, 64, False, None, "bias"),
    (3, 16, 16, 129, 200, 64, 64, False, None, "window"),
    (2, 32, 16, 160, 161, 64, 64, False, None, "rows"),
]


def bwd_case(shape, seed=3):
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, mk = shape
    r = np.random.Generator(np.random.PCG64(seed))
    q, k, v, go = (r.standard_normal(s, dtype=np.float32) for s in ((B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, Dv), (B, Hq, Sq, Dv)))
    far = (np.arange(Sq)[:, None] + Skv - Sq - np.arange(Skv)[None]).astype(np.float32)
    mask = None
    if mk == "bias":
        mask = np.where(far >= 0, -far[None] * 0.5 ** np.arange(1, Hq + 1, dtype=np.float32)[:, None, None], -np.inf)[None]
    elif mk == "window":
        mask = np.where(np.abs(far) < 40, 0.0, -np.inf)[None, None]
    elif mk == "rows":
        mask = r.standard_normal((1, 1, 1, Skv))
    return q, k, v, go, None if mask is None else mask.astype(np.float32), None if lens is None else np.asarray(lens, np.int32)


def f64_gradients(q, k, v, go, causal, mask, lens):
    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1:3]
    G = Hq // Hkv
    q, k, v, go = (x.astype(np.float64) for x in (q, k, v, go))
    k, v = (np.repeat(x, G, 1) for x in (k, v))
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(D)
    if mask is not None:
        s = s + mask
    if causal:
        s = np.where(np.arange(Skv)[None] > np.arange(Sq)[:, None] + Skv - Sq, -np.inf, s)
    if lens is not None:
        s = np.where(np.arange(Skv) >= lens[:, None, None, None], -np.inf, s)
    m = s.max(-1, keepdims=True)
    p = np.exp(s - np.where(np.isinf(m), 0, m))
    p = p / np.maximum(p.sum(-1, keepdims=True), 1e-300)
    o = p @ v
    ds = p * (go @ v.transpose(0, 1, 3, 2) - (go * o).sum(-1, keepdims=True))
    per = lambda x: x.reshape(B, Hkv, G, Skv, -1).sum(2)
    return ds @ k / np.sqrt(D), per(ds.transpose(0, 1, 3, 2) @ q / np.sqrt(D)), per(p.transpose(0, 1, 3, 2) @ go)


@pytest.mark.parametrize("shape", BWD, ids=lambda s: "x".join(map(str, s[:7])) + ("" if s[9] is None else s[9]))
def test_backward_tile_edges(gpu, shape, monkeypatch):
    """Gradients at the edges of tiles and blocks, key counts down to none, grouped queries, masks as tensors: against 64 bits at 1e-5 of the largest
    gradient, and never further off (2-norm, all three together, 2 % for ties) than the kernel of IEEE-f32 products, which forced parts call."""
    q, k, v, go, mask, lens = bwd_case(shape)
    kw = dict(causal=shape[7], kv_lens=lens, mask=mask)
    ref = f64_gradients(q, k, v, go, shape[7], mask, lens)
    _, *got = host.sdpa_backward(q, k, v, go, capi.F32, **kw)
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", "1")
    _, *ieee = host.sdpa_backward(q, k, v, go, capi.F32, **kw)
    assert any(not np.array_equal(a, b) for a, b in zip(got, ieee)), "the same kernel"
    off = [0.0, 0.0]
    for name, a, b, r in zip(("dq", "dk", "dv"), got, ieee, ref):
        assert np.max(np.abs(a - r)) <= 1e-5 * max(np.max(np.abs(r)), 1e-3), name
        off[0] += np.sum((a - r) ** 2) / np.sum(r ** 2)
        off[1] += np.sum((b - r) ** 2) / np.sum(r ** 2)
    assert off[0] <= 1.04 * off[1]


def test_backward_values_that_are_not_finite(gpu, monkeypatch):
    """An infinite value of dO and a NaN in K reach what they reach in the kernel of IEEE-f32 products, and a dO whose first bf16 part would be
    infinite stays finite."""
    shape = (3, 16, 16, 129, 150, 64, 64, False, None, None)
    q, k, v, go, _, _ = bwd_case(shape)
    v[2, 0, :, 0] *= 0.01      # (so that dO V and dO O do not overflow where dO is the largest finite value)
    for t, at, x in ((go, (0, 3, 128, 5), np.inf), (k, (1, 2, 149, 0), np.nan), (go, (2, 0, 0, 0), np.finfo(np.float32).max)):
        was = t[at]
        t[at] = x
        with np.errstate(invalid="ignore", over="ignore"):
            _, *got = host.sdpa_backward(q, k, v, go, capi.F32)
            monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", "1")
            _, *ieee = host.sdpa_backward(q, k, v, go, capi.F32)
            monkeypatch.delenv("INCIN_ROCM_BWD_PARTS")
        t[at] = was
        for name, a, b in zip(("dq", "dk", "dv"), got, ieee):
            assert np.array_equal(np.isfinite(a), np.isfinite(b)) and np.array_equal(np.isnan(a), np.isnan(b)), (name, x)
            for h in np.ndindex(a.shape[:2]):      # 1e-5 of a head's largest gradient, as above
                fin = np.isfinite(b[h])
                if fin.any():
                    assert np.max(np.abs(a[h][fin] - b[h][fin])) <= 1e-5 * max(np.max(np.abs(b[h][fin])), 1), (name, x, h)


@pytest.mark.parametrize("what", ["go", "go column", "q", "k", "v", "go and v", "go and q"])
@pytest.mark.parametrize("exponent", [-104, -112, -118, -122])
def test_backward_values_whose_last_bits_no_part_holds(gpu, what, exponent):
    """As forward: dO below 2^-110, a column of it, Q or K as small under the other as large, V under such a dO, and two ordinary operands whose product is that
    small.  Gradients, each column, within 3e-6 of 64 bits (the IEEE products: 1.3e-6) where they are not below f32's normal range."""
    q, k, v, go, _, _ = bwd_case((3, 16, 16, 129, 127, 64, 64, False, None, None))
    small, large, half = np.float32(2.0 ** exponent), np.float32(2.0 ** -exponent), np.float32(2.0 ** (exponent // 2))
    if what == "go":
        go *= small
    elif what == "go column":
        go[..., 3] *= small
    elif what in "qk":
        q, k = (q * small, k * large) if what == "q" else (q * large, k * small)
    elif what == "v":
        v, go = v * small, go * large
    elif what == "go and v":
        go, v = go * half, v * half
    else:
        go, q, k = go * half, q * half, k / half
    _, *got = host.sdpa_backward(q, k, v, go, capi.F32)
    for name, a, r in zip(("dq", "dk", "dv"), got, f64_gradients(q, k, v, go, False, None, None)):
        norm = np.linalg.norm(r, axis=2)
        normal = norm / np.sqrt(r.shape[2]) >= 2.0 ** -125
        off = np.linalg.norm(a - r, axis=2) / norm
        assert not normal.any() or np.max(off[normal]) <= 3e-6, name


def test_backward_hidden_blocks_may_hold_anything(gpu):
    """A NaN in a row of dO or K reaches the gradients of what sees it, by blocks of 32 x 32, and no other: the causal flag, and the same mask as a
    tensor, whose hidden blocks lie inside the range that the walk trims to."""
    shape = (2, 24, 24, 256, 256, 64, 64, True, None, None)
    q, k, v, go, _, _ = bwd_case(shape)
    tri = np.triu(np.full((256, 256), -np.inf, np.float32), 1)[None, None]
    rdq, rdk, rdv = f64_gradients(q, k, v, go, True, None, None)
    blocks = np.arange(256) // 32
    go[1, :, 70, 3], k[0, :, 200, 2] = np.nan, np.nan
    for kw in (dict(causal=True), dict(mask=tri)):
        _, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, **kw)
        assert np.isnan(dv[1, :, blocks == 2, 3]).any() and np.isnan(dq[0, :, blocks == 7]).any()
        for name, got, ref, clean in (("dk", dk[1], rdk[1], blocks > 2), ("dv", dv[1], rdv[1], blocks > 2), ("dq", dq[0], rdq[0], blocks < 6)):
            assert np.max(np.abs(got[:, clean] - ref[:, clean])) <= 1e-5 * np.max(np.abs(ref)), (name, kw)


def test_backward_padding_rows_may_hold_anything(gpu):
    """NaN in the query rows behind a sequence's count - Q, dO, O, the row normalisers and the mask - changes no bit of any gradient: no block is done over for
    them."""
    B, H, S = 4, 16, 160
    q, k, v, go, _, _ = bwd_case((B, H, H, S, S, 64, 64, False, None, None))
    lens = np.array([100, 137, 64, 160], np.int32)
    mask = np.random.Generator(np.random.PCG64(6)).standard_normal((B, H, S, S), dtype=np.float32)
    run = lambda: host.sdpa_backward(q, k, v, go, capi.F32, q_lens=lens, mask=mask, poison_padding=True)[1:]
    clean = run()
    for b, n in enumerate(lens):
        q[b, :, n:] = go[b, :, n:] = mask[b, :, n:] = np.nan
    for name, a, c in zip(("dq", "dk", "dv"), run(), clean):
        assert np.isfinite(c).all() and np.array_equal(a, c), name
