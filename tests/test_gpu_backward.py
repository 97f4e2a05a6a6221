"""Attention backward through the C ABI against the backward oracle (the gradients the reference's tape walk
gives, oracle/sdpa_backward.py): dq, dk, dv for f16 / bf16 operands, D = 128, grouped queries, causal masks with
Sq != Skv, ragged key counts.  Tolerance: 2e-2 relative to the largest magnitude of the gradient tensor compared
(bf16 / f16 inputs, bf16 / f16 probabilities and dS as matrix operands, f32 accumulation)."""
import sys

import numpy as np
import pytest

from incin_amd import capi, dtypes, host
from oracle import sdpa_backward as BW

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, file=sys.stderr, flush=True)


def make(seed, B, Hq, Hkv, Sq, Skv, D, dtype):
    r = np.random.Generator(np.random.PCG64(seed))
    mk = lambda *s: dtypes.round_to(r.standard_normal(s, dtype=np.float32), dtype)
    return mk(B, Hq, Sq, D), mk(B, Hkv, Skv, D), mk(B, Hkv, Skv, D), mk(B, Hq, Sq, D)


def compare(name, got, ref, tol=2e-2):
    ref = np.asarray(ref, np.float64)
    scale = float(np.abs(ref).max()) or 1.0
    err = float(np.abs(got - ref).max()) / scale
    say("   %s: max-abs err / max|ref| = %.3e (max|ref| %.3g)" % (name, err, scale))
    assert not np.isnan(got).any(), name
    assert err <= tol, "%s: %.3e" % (name, err)


@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, causal, kv_lens
    (1, 1, 1, 32, 32, False, None),
    (1, 1, 1, 128, 128, True, None),
    (2, 4, 4, 200, 333, False, None),
    (2, 4, 2, 300, 300, True, None),
    (1, 8, 2, 130, 450, True, None),                  # Sq < Skv: causal alignment, grouped queries
    (3, 2, 2, 257, 257, True, [257, 100, 31]),
    (2, 2, 1, 64, 700, False, [700, 1]),
], ids=["tiny", "one_tile_causal", "rect", "gqa_causal", "gqa_rect_causal", "ragged_causal", "ragged"])
@pytest.mark.parametrize("D", [128, 64])
def test_backward_against_the_oracle(gpu, dtype, shape, D):
    B, Hq, Hkv, Sq, Skv, causal, lens = shape
    G = Hq // Hkv
    say("backward: %s D=%d dtype %d" % (shape, D, dtype))
    q, k, v, go = make(11, B, Hq, Hkv, Sq, Skv, D, dtype)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, causal=causal, kv_lens=lens_a)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D),
                                  causal=causal, kv_lens=None if lens is None else lens_a.reshape(B, 1, 1))
    compare("dq", dq, rq.reshape(B, Hq, Sq, D))
    compare("dk", dk, rk.reshape(B, Hkv, Skv, D))
    compare("dv", dv, rv.reshape(B, Hkv, Skv, D))
    if lens is not None:
        for b in range(B):
            assert not dk[b, :, lens[b]:].any() and not dv[b, :, lens[b]:].any()      # padded keys: exactly zero


def test_backward_random_cases(gpu):
    """Seeded random shapes: batch, heads, group size, lengths on either side of the 64-row tiles and the 128-key
    workgroups, causal alignment with Sq <= Skv, ragged key counts >= 1 (every query row keeps a visible key, so the
    oracle has no NaN), scales.  Each case is printed before it runs."""
    r = np.random.Generator(np.random.PCG64(2026))
    for case in range(28):
        D = 128 if case % 3 else 64
        B, Hkv, G = int(r.integers(1, 4)), int(r.integers(1, 4)), int(r.choice([1, 2, 4]))
        Skv = int(r.choice([r.integers(1, 70), r.integers(60, 140), r.integers(120, 420)]))
        causal = bool(r.integers(0, 2))
        Sq = int(r.integers(1, Skv + 1)) if causal else int(r.integers(1, 300))
        lens = None
        if r.integers(0, 2):
            lens = r.integers(1, Skv + 1, B).astype(np.int32)      # (row 0 sees key 0 whenever Sq <= Skv and the count is >= 1)
        dtype = capi.BF16 if case % 2 else capi.F16
        scale = float(r.choice([0.0883883461356163, 0.05, 0.2]))
        Hq = Hkv * G
        say("backward random case %d: B=%d Hq=%d Hkv=%d Sq=%d Skv=%d causal=%s lens=%s dtype=%d scale=%g"
            % (case, B, Hq, Hkv, Sq, Skv, causal, None if lens is None else lens.tolist(), dtype, scale))
        q, k, v, go = make(100 + case, B, Hq, Hkv, Sq, Skv, D, dtype)
        out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, scale=scale, causal=causal, kv_lens=lens)
        rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D),
                                      scale=scale, causal=causal, kv_lens=None if lens is None else lens.reshape(B, 1, 1))
        rq, rk, rv = rq.reshape(B, Hq, Sq, D), rk.reshape(B, Hkv, Skv, D), rv.reshape(B, Hkv, Skv, D)
        assert not np.isnan(rq).any(), "case construction: a row without keys"
        compare("dq", dq, rq)
        compare("dk", dk, rk)
        compare("dv", dv, rv)


def test_backward_random_cases_f32(gpu):
    """The same draw in f32 over longer sequences: key and query counts up to 1600, where a call this small has the walks of
    its blocks dealt to 2 or 4 workgroups and its dQ kernel on a second stream - by the library's own rule, nothing forced.
    1e-5 of the largest gradient magnitude against the f64 oracle."""
    r = np.random.Generator(np.random.PCG64(2027))
    for case in range(18):
        D = 128 if case % 3 else 64
        B, Hkv, G = int(r.integers(1, 3)), int(r.integers(1, 4)), int(r.choice([1, 2, 4]))
        Skv = int(r.choice([r.integers(1, 140), r.integers(120, 700), r.integers(500, 1600), r.integers(1000, 1600)]))
        causal = bool(r.integers(0, 2))
        Sq = int(r.integers(1, Skv + 1)) if causal else int(r.choice([r.integers(1, 300), r.integers(500, 1300)]))
        lens = None
        if r.integers(0, 2):
            lens = r.integers(1, Skv + 1, B).astype(np.int32)
        scale = float(r.choice([1.0 / np.sqrt(D), 0.05, 0.2]))
        Hq = Hkv * G
        say("backward random case %d (f32): B=%d Hq=%d Hkv=%d Sq=%d Skv=%d D=%d causal=%s lens=%s scale=%g"
            % (case, B, Hq, Hkv, Sq, Skv, D, causal, None if lens is None else lens.tolist(), scale))
        q, k, v, go = make(300 + case, B, Hq, Hkv, Sq, Skv, D, capi.F32)
        out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, scale=scale, causal=causal, kv_lens=lens)
        rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D),
                                      scale=scale, causal=causal, kv_lens=None if lens is None else lens.reshape(B, 1, 1))
        rq, rk, rv = rq.reshape(B, Hq, Sq, D), rk.reshape(B, Hkv, Skv, D), rv.reshape(B, Hkv, Skv, D)
        assert not np.isnan(rq).any(), "case construction: a row without keys"
        compare("dq", dq, rq, tol=1e-5)
        compare("dk", dk, rk, tol=1e-5)
        compare("dv", dv, rv, tol=1e-5)


def test_rows_without_visible_keys_get_zero_gradients(gpu):
    # Sq > Skv under causal alignment: the first Sq - Skv rows see nothing (NaN in the forward).  They get a zero dq
    # and contribute nothing to dk, dv; the other rows are what the oracle gives for them alone.
    B, H, Sq, Skv, D = 1, 2, 96, 40, 128
    q, k, v, go = make(12, B, H, H, Sq, Skv, D, capi.BF16)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.BF16, causal=True)
    dead = Sq - Skv
    assert np.isnan(out[:, :, :dead]).all() and not np.isnan(out[:, :, dead:]).any()
    assert not dq[:, :, :dead].any()
    rq, rk, rv = BW.sdpa_backward(q[:, :, dead:], k, v, go[:, :, dead:], causal=True)
    compare("dq (live rows)", dq[:, :, dead:], rq)
    compare("dk", dk, rk)
    compare("dv", dv, rv)
    # a sequence with no keys at all: zero gradients everywhere for it
    lens = np.array([0], np.int32)
    out, dq, dk, dv = host.sdpa_backward(q[:, :, :40], k, v, go[:, :, :40], capi.BF16, kv_lens=lens)
    assert not dq.any() and not dk.any() and not dv.any()


@pytest.mark.parametrize("D", [128, 64])
def test_backward_at_a_few_thousand_tokens(gpu, D):
    B, Hq, Hkv, S = 1, 4, 2, 2048
    q, k, v, go = make(13, B, Hq, Hkv, S, S, D, capi.BF16)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.BF16, causal=True)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, 2, S, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, 2, S, D), causal=True)
    compare("dq", dq, rq.reshape(B, Hq, S, D))
    compare("dk", dk, rk.reshape(B, Hkv, S, D))
    compare("dv", dv, rv.reshape(B, Hkv, S, D))


def make_d(seed, B, Hq, Hkv, Sq, Skv, D, Dv, dtype):
    r = np.random.Generator(np.random.PCG64(seed))
    mk = lambda *s: dtypes.round_to(r.standard_normal(s, dtype=np.float32), dtype)
    return mk(B, Hq, Sq, D), mk(B, Hkv, Skv, D), mk(B, Hkv, Skv, Dv), mk(B, Hq, Sq, Dv)


@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, mask kind
    (2, 2, 2, 4, 4, 8, 8, False, None, None),                    # the reference's smoke shape (shape_ops.rs:1575-1591)
    (1, 3, 3, 33, 65, 16, 24, False, None, None),                # D != Dv, lengths off the 32-wide tiles
    (2, 4, 2, 70, 70, 64, 64, True, None, None),
    (2, 4, 1, 50, 90, 40, 40, True, [90, 37], None),             # grouped queries, causal alignment, ragged keys
    (2, 2, 2, 45, 61, 32, 32, False, None, "full"),              # dense additive mask with -inf holes
    (2, 3, 3, 40, 40, 128, 128, False, None, "row"),             # [1, 1, 1, Skv] mask: broadcast over batch, head, row
    (1, 2, 2, 20, 30, 256, 200, True, None, "head"),             # the widest heads, [1, H, Sq, Skv] mask on top of causal
], ids=["ref_smoke", "d_ne_dv", "causal", "gqa_ragged", "mask_full", "mask_row", "wide_mask_head"])
def test_generic_backward_f32_against_the_oracle(gpu, shape):
    """The reference's own dtype through the generic kernels: 1e-5 of the largest gradient magnitude against the f64 oracle
    (f32 products and sums in a different order than the reference's tape; measured about 1e-6)."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, mk = shape
    G = Hq // Hkv
    say("generic backward f32: %s" % (shape,))
    q, k, v, go = make_d(21, B, Hq, Hkv, Sq, Skv, D, Dv, capi.F32)
    r = np.random.Generator(np.random.PCG64(22))
    mask = None
    if mk is not None:
        mshape = {"full": (B, Hq, Sq, Skv), "row": (1, 1, 1, Skv), "head": (1, Hq, Sq, Skv)}[mk]
        mask = r.standard_normal(mshape, dtype=np.float32)
        mask[r.random(mshape) < 0.25] = -np.inf
        mask[..., 0] = 0.0                                       # every row keeps a visible key
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, causal=causal, kv_lens=lens_a, mask=mask, impl=capi.IMPL_GENERIC)
    m5 = None if mask is None else np.broadcast_to(mask, (B, Hq, Sq, Skv)).reshape(B, Hkv, G, Sq, Skv)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, Dv),
                                  mask=m5, causal=causal, kv_lens=None if lens is None else lens_a.reshape(B, 1, 1))
    compare("dq", dq, rq.reshape(B, Hq, Sq, D), tol=1e-5)
    compare("dk", dk, rk.reshape(B, Hkv, Skv, D), tol=1e-5)
    compare("dv", dv, rv.reshape(B, Hkv, Skv, Dv), tol=1e-5)


@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16, capi.F32], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, mask kind
    (2, 2, 2, 150, 200, 128, 128, False, None, "full"),            # values with -inf holes, a mask of its own per batch entry and head
    (2, 4, 2, 130, 130, 64, 64, True, None, "head"),               # grouped queries: [1, Hq, Sq, Skv] on top of the causal flag
    (2, 3, 3, 100, 260, 128, 128, False, [260, 90], "row"),        # [1, 1, 1, Skv]: one row for everybody, with key counts
    (1, 2, 2, 200, 200, 96, 72, False, None, "causal_tensor"),     # the causal mask as a tensor (no flag), padded head dimensions
    (2, 2, 1, 70, 333, 128, 128, False, None, "batch"),            # [B, 1, Sq, Skv]; 333 keys: rows of the mask are not 8-byte aligned
    (1, 4, 2, 330, 400, 128, 128, False, None, "causal_bias"),     # per-head distance bias under the causal triangle: blocks of all kinds
    (2, 2, 2, 300, 304, 64, 64, False, None, "window"),            # a band of 70 keys: hidden blocks on both sides, zeros between
    (1, 2, 1, 257, 296, 128, 128, True, None, "blocks"),           # random 32 x 32 blocks hidden / zero / values, under the causal flag
], ids=["full", "gqa_head_causal", "row_lens", "causal_tensor", "batch_unaligned", "causal_bias", "window", "blocks"])
def test_matrix_core_backward_with_a_dense_mask(gpu, dtype, shape):
    """Gradients with a dense additive mask run on the matrix-core kernels, 16-bit and f32 (instances that add the mask's values
    to the scores before the exponential): against the f64 oracle, AUTO picks them, and the generic kernels agree."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, mk = shape
    G = Hq // Hkv
    say("matrix-core backward with a mask: %s %s" % (dtypes.NAMES[dtype], shape))
    q, k, v, go = make_d(71 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    r = np.random.Generator(np.random.PCG64(72))
    if mk == "causal_tensor":
        mask = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq).reshape(1, 1, Sq, Skv)
    elif mk == "causal_bias":
        dist = (np.arange(Sq)[:, None] + (Skv - Sq) - np.arange(Skv)[None, :]).astype(np.float32)
        mask = np.where(dist >= 0, -dist[None] * (0.5 ** np.arange(1, Hq + 1, dtype=np.float32))[:, None, None], -np.inf)[None].astype(np.float32)
    elif mk == "window":
        dist = np.arange(Sq)[:, None] + (Skv - Sq) - np.arange(Skv)[None, :]
        mask = np.where((dist >= 0) & (dist < 70), 0.0, -np.inf).astype(np.float32).reshape(1, 1, Sq, Skv)
    elif mk == "blocks":
        kinds = r.integers(0, 3, size=(B, Hq, (Sq + 31) // 32, (Skv + 31) // 32))
        kinds[..., 0] = 1                                        # every row keeps visible keys
        big = np.repeat(np.repeat(kinds, 32, axis=2), 32, axis=3)[:, :, :Sq, :Skv]
        mask = np.where(big == 0, -np.inf, np.where(big == 1, 0.0, r.standard_normal((B, Hq, Sq, Skv), dtype=np.float32))).astype(np.float32)
    else:
        mshape = {"full": (B, Hq, Sq, Skv), "row": (1, 1, 1, Skv), "head": (1, Hq, Sq, Skv), "batch": (B, 1, Sq, Skv)}[mk]
        mask = r.standard_normal(mshape, dtype=np.float32)
        mask[r.random(mshape) < 0.25] = -np.inf
        mask[..., 0] = 0.0                                       # every row keeps a visible key
    mask = dtypes.round_to(mask, dtype)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    kw = dict(causal=causal, kv_lens=lens_a, mask=mask)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_MFMA, **kw)
    auto = host.sdpa_backward(q, k, v, go, dtype, **kw)
    gen = host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_GENERIC, **kw)
    m5 = np.broadcast_to(mask, (B, Hq, Sq, Skv)).reshape(B, Hkv, G, Sq, Skv)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, Dv),
                                  mask=m5, causal=causal, kv_lens=None if lens is None else lens_a.reshape(B, 1, 1))
    f32 = dtype == capi.F32
    for name, x, a, gx, r_ in zip(("dq", "dk", "dv"), (dq, dk, dv), auto[1:], gen[1:],
                                  (rq.reshape(B, Hq, Sq, D), rk.reshape(B, Hkv, Skv, D), rv.reshape(B, Hkv, Skv, Dv))):
        compare(name, x, r_, tol=1e-5 if f32 else 2e-2)
        if f32:       # (AUTO's forward of an f32 launch this small may be another kernel: last-bit differences in O and lse)
            compare(name + " AUTO vs pinned", a, x, tol=2e-6)
        else:
            assert np.array_equal(x, a), name + ": AUTO takes the same kernels"
        compare(name + " generic vs matrix-core", gx, x, tol=1e-5 if f32 else 1e-2)


@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16, capi.F32], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, causal, mask kind
    (1, 4, 2, 1100, 1400, 128, True, "blocks"),
    (1, 2, 2, 1300, 1304, 64, False, "band"),
    (2, 2, 1, 900, 1600, 128, False, "values"),
    (1, 2, 2, 1027, 1501, 64, True, "blocks"),          # rows of the mask that cannot be copied 16 bytes at a time
], ids=["blocks_gqa128", "band64", "values128", "blocks_unaligned64"])
def test_matrix_core_backward_with_a_dense_mask_over_many_tiles(gpu, dtype, shape):
    """Masks over 14 - 25 tiles of keys and of query rows, where the kernels' look-ahead (flags two tiles ahead, values or their
    copies into LDS one ahead, tile ranges trimmed by the flags) runs at length: random blocks of 32 x 32 that are hidden, zero or
    valued (runs of each), a band of values around the diagonal with -inf away from it, values with holes everywhere."""
    B, Hq, Hkv, Sq, Skv, D, causal, mk = shape
    G = Hq // Hkv
    say("matrix-core backward with a mask over many tiles: %s %s" % (dtypes.NAMES[dtype], shape))
    q, k, v, go = make(81 + Sq, B, Hq, Hkv, Sq, Skv, D, dtype)
    r = np.random.Generator(np.random.PCG64(82))
    if mk == "blocks":
        kinds = r.integers(0, 3, size=(1, Hq, (Sq + 31) // 32, (Skv + 31) // 32))
        kinds[..., 0] = 1                                        # every row keeps visible keys
        big = np.repeat(np.repeat(kinds, 32, axis=2), 32, axis=3)[:, :, :Sq, :Skv]
        mask = np.where(big == 0, -np.inf, np.where(big == 1, 0.0, r.standard_normal((1, Hq, Sq, Skv), dtype=np.float32))).astype(np.float32)
    elif mk == "band":
        dist = np.abs(np.arange(Sq)[:, None] - np.arange(Skv)[None, :])
        mask = np.where(dist > 300, -np.inf, np.where(dist < 100, r.standard_normal((Sq, Skv)), 0.0)).astype(np.float32).reshape(1, 1, Sq, Skv)
    else:
        mask = r.standard_normal((B, 1, Sq, Skv), dtype=np.float32)
        mask[r.random(mask.shape) < 0.25] = -np.inf
        mask[..., 0] = 0.0
    mask = dtypes.round_to(mask, dtype)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, causal=causal, mask=mask)
    m5 = np.broadcast_to(mask, (B, Hq, Sq, Skv)).reshape(B, Hkv, G, Sq, Skv)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D), mask=m5, causal=causal)
    assert not np.isnan(rq).any(), "case construction: a row without keys"
    tol = 1e-5 if dtype == capi.F32 else 2e-2
    compare("dq", dq, rq.reshape(B, Hq, Sq, D), tol=tol)
    compare("dk", dk, rk.reshape(B, Hkv, Skv, D), tol=tol)
    compare("dv", dv, rv.reshape(B, Hkv, Skv, D), tol=tol)


def test_backward_random_cases_with_a_dense_mask(gpu):
    """Seeded random shapes with a mask tensor on the matrix-core backward kernels, all three dtypes: values with holes, blocks
    of 32 x 32 hidden / zero / valued at random, a band; any leading axis of the mask broadcast; lengths on either side of the
    tiles; with and without the causal flag and key counts.  Column 0 of every mask row stays visible (and row 0 sees key 0
    under the causal alignment with Sq <= Skv), so the oracle has no NaN.  Each case is printed before it runs."""
    r = np.random.Generator(np.random.PCG64(2027))
    for case in range(30):
        dtype = (capi.BF16, capi.F16, capi.F32)[case % 3]
        D = 128 if case % 2 else 64
        B, Hkv, G = int(r.integers(1, 3)), int(r.integers(1, 3)), int(r.choice([1, 2, 4]))
        Skv = int(r.choice([r.integers(1, 70), r.integers(60, 140), r.integers(120, 420)]))
        if case % 4 < 2:
            Skv = (Skv + 7) // 8 * 8          # (rows the 16-bit dK/dV kernel can copy into LDS)
        causal = bool(r.integers(0, 2))
        Sq = int(r.integers(1, Skv + 1)) if causal else int(r.integers(1, 300))
        lens = r.integers(1, Skv + 1, B).astype(np.int32) if r.integers(0, 2) else None
        Hq = Hkv * G
        shp = [B if r.random() < 0.5 else 1, Hq if r.random() < 0.5 else 1, Sq if r.random() < 0.8 else 1, Skv]
        kind = str(r.choice(["holes", "blocks", "band"]))
        mask = r.standard_normal(shp, dtype=np.float32)
        if kind == "holes":
            mask[r.random(shp) < 0.25] = -np.inf
        elif kind == "blocks":
            kinds = r.integers(0, 3, size=(shp[0], shp[1], (shp[2] + 31) // 32, (Skv + 31) // 32))
            big = np.repeat(np.repeat(kinds, 32, axis=2), 32, axis=3)[:, :, :shp[2], :Skv]
            mask = np.where(big == 0, -np.inf, np.where(big == 1, 0.0, mask)).astype(np.float32)
        elif shp[2] > 1:
            dist = np.arange(Sq)[:, None] + (Skv - Sq) - np.arange(Skv)[None, :]
            mask = np.where((np.abs(dist) <= int(r.integers(8, 120)))[None, None], 0.1 * mask, -np.inf).astype(np.float32)
        mask[..., 0] = 0.0
        mask = dtypes.round_to(mask, dtype)
        say("masked backward random case %d: dtype=%d D=%d B=%d Hq=%d Hkv=%d Sq=%d Skv=%d causal=%s lens=%s mask %s %r"
            % (case, dtype, D, B, Hq, Hkv, Sq, Skv, causal, None if lens is None else lens.tolist(), kind, tuple(shp)))
        q, k, v, go = make(300 + case, B, Hq, Hkv, Sq, Skv, D, dtype)
        out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, causal=causal, kv_lens=lens, mask=mask, impl=capi.IMPL_MFMA)
        m5 = np.broadcast_to(mask, (B, Hq, Sq, Skv)).reshape(B, Hkv, G, Sq, Skv)
        rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D),
                                      mask=m5, causal=causal, kv_lens=None if lens is None else lens.reshape(B, 1, 1))
        assert not np.isnan(rq).any(), "case construction: a row without keys"
        tol = 1e-5 if dtype == capi.F32 else 2e-2
        compare("dq", dq, rq.reshape(B, Hq, Sq, D), tol=tol)
        compare("dk", dk, rk.reshape(B, Hkv, Skv, D), tol=tol)
        compare("dv", dv, rv.reshape(B, Hkv, Skv, D), tol=tol)


@pytest.mark.parametrize("dtype,dims", [(capi.BF16, (96, 96)), (capi.BF16, (40, 72)), (capi.F16, (128, 64)), (capi.BF16, (8, 8)), (capi.F16, (80, 80)),
                                        (capi.F32, (96, 96)), (capi.F32, (20, 36)), (capi.F32, (128, 64)), (capi.F32, (4, 4))],
                         ids=lambda x: dtypes.NAMES[x] if isinstance(x, int) else "D%d_Dv%d" % x)
def test_matrix_core_backward_with_padded_head_dimensions(gpu, dtype, dims):
    """Head dimensions up to 128 in whole 16-byte vectors, D and Dv not necessarily equal, through the matrix-core backward
    kernels (pinned, and AUTO must pick them): zero-padded into the 64 / 128 instances, gradient stores cut at D and Dv."""
    D, Dv = dims
    tol = 1e-5 if dtype == capi.F32 else 2e-2
    for B, Hq, Hkv, Sq, Skv, causal, lens in ((2, 4, 2, 150, 200, True, [200, 77]), (1, 2, 2, 70, 70, False, None)):
        G = Hq // Hkv
        say("padded backward: %s D=%d Dv=%d %r" % (dtypes.NAMES[dtype], D, Dv, (B, Hq, Hkv, Sq, Skv)))
        q, k, v, go = make_d(61 + D, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
        lens_a = None if lens is None else np.asarray(lens, np.int32)
        out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, causal=causal, kv_lens=lens_a, impl=capi.IMPL_MFMA)
        auto = host.sdpa_backward(q, k, v, go, dtype, causal=causal, kv_lens=lens_a)
        rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, Dv),
                                      causal=causal, kv_lens=None if lens is None else lens_a.reshape(B, 1, 1))
        for name, x, a, r_ in zip(("dq", "dk", "dv"), (dq, dk, dv), auto[1:], (rq.reshape(B, Hq, Sq, D), rk.reshape(B, Hkv, Skv, D), rv.reshape(B, Hkv, Skv, Dv))):
            compare(name, x, r_, tol=tol)
            if dtype == capi.F32:       # (AUTO's forward of an f32 launch this small is the split-KV kernel: last-bit differences in O and lse)
                compare(name + " AUTO vs pinned", a, x, tol=2e-6)
            else:
                assert np.array_equal(x, a), name + ": AUTO takes the same kernels"


@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, causal, kv_lens, scale
    (1, 1, 1, 32, 32, 64, False, None, None),
    (1, 1, 1, 32, 32, 128, True, None, None),
    (2, 3, 3, 128, 128, 64, True, None, None),                   # the reference's bench head shape, causal
    (2, 4, 4, 200, 333, 64, False, None, 0.3),
    (2, 4, 2, 300, 300, 128, True, None, None),
    (1, 8, 2, 130, 450, 64, True, None, None),                   # Sq < Skv: causal alignment, grouped queries
    (3, 2, 2, 257, 257, 64, True, [257, 100, 31], None),
    (2, 2, 1, 64, 700, 128, False, [700, 2], None),
    (1, 2, 2, 513, 129, 64, False, None, -0.125),                # a negative scale is a scale like any other in f32
    (8, 2, 1, 77, 140, 128, True, [140, 70, 64, 65, 128, 129, 100, 96], None),      # (batch, KV head) pairs dealt over the XCDs
], ids=["tiny64", "tiny128_causal", "bench_head", "rect", "gqa_causal128", "gqa_rect_causal", "ragged_causal", "ragged128",
        "negative_scale", "dealt_pairs"])
def test_matrix_core_backward_f32_against_the_oracle(gpu, shape):
    """f32 through the f32 matrix-core kernels (D = 64 and 128), picked by AUTO and pinned: 1e-5 of the largest
    gradient magnitude against the f64 oracle, and the generic f32 kernels within the same distance."""
    B, Hq, Hkv, Sq, Skv, D, causal, lens, scale = shape
    G = Hq // Hkv
    say("matrix-core backward f32: %s" % (shape,))
    q, k, v, go = make(41, B, Hq, Hkv, Sq, Skv, D, capi.F32)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    kw = dict(causal=causal, kv_lens=lens_a, scale=scale)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, impl=capi.IMPL_MFMA, **kw)
    auto = host.sdpa_backward(q, k, v, go, capi.F32, **kw)
    gen = host.sdpa_backward(q, k, v, go, capi.F32, impl=capi.IMPL_GENERIC, **kw)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D),
                                  scale=scale, causal=causal, kv_lens=None if lens is None else lens_a.reshape(B, 1, 1))
    refs = (rq.reshape(B, Hq, Sq, D), rk.reshape(B, Hkv, Skv, D), rv.reshape(B, Hkv, Skv, D))
    for name, x, a, g_, r_ in zip(("dq", "dk", "dv"), (dq, dk, dv), auto[1:], gen[1:], refs):
        compare(name, x, r_, tol=1e-5)
        # (AUTO's forward of launches this small is the f32 split-KV kernel: O and the row normalisers differ in the last bits)
        compare(name + " AUTO vs pinned", a, x, tol=2e-6)
        compare(name + " generic vs matrix-core", g_, x, tol=2e-5)
    if lens is not None:
        for b in range(B):
            assert not dk[b, :, lens[b]:].any() and not dv[b, :, lens[b]:].any()      # padded keys: exactly zero


@pytest.mark.parametrize("parts", ["1", "2", "4"])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, q_lens, mask
    (1, 4, 4, 1024, 1024, 64, 64, True, None, None, None),
    (2, 4, 2, 600, 1100, 128, 128, True, [1100, 300], None, None),           # a sequence whose keys end inside the first part
    (1, 2, 2, 1030, 520, 64, 32, False, None, None, None),                  # D != Dv: planes of different widths
    (1, 8, 2, 520, 1500, 128, 128, True, None, None, "window"),             # a mask whose block flags trim the walk before it is dealt
    (2, 2, 2, 1024, 1024, 64, 64, True, [1024, 700], [1024, 700], None),    # padding rows: zero in every plane
    (1, 2, 1, 300, 2100, 64, 64, False, None, None, "values"),
], ids=["causal", "ragged_gqa128", "rect_d_dv", "window_gqa128", "padded", "values"])
def test_matrix_core_backward_f32_in_parts(gpu, monkeypatch, parts, shape):
    """The f32 matrix-core kernels with the tiles of a block dealt to 1, 2 and 4 workgroups whose sums meet in planes of the
    workspace (what a call that does not fill the device gets by itself; INCIN_ROCM_BWD_PARTS forces it): 1e-5 of the largest
    gradient magnitude against the f64 oracle each, exact zeros where padding is."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, qlens, mk = shape
    G = Hq // Hkv
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    say("matrix-core backward f32 in %s parts: %s" % (parts, shape))
    q, k, v, go = make_d(91 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, capi.F32)
    r = np.random.Generator(np.random.PCG64(92))
    mask = None
    if mk == "window":
        dist = np.arange(Sq)[:, None] + (Skv - Sq) - np.arange(Skv)[None, :]
        mask = np.where((dist >= 0) & (dist < 400), 0.0, -np.inf).astype(np.float32).reshape(1, 1, Sq, Skv)
    elif mk == "values":
        mask = r.standard_normal((1, Hq, Sq, Skv), dtype=np.float32)
        mask[r.random(mask.shape) < 0.25] = -np.inf
        mask[..., 0] = 0.0
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    qlens_a = None if qlens is None else np.asarray(qlens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens_a, q_lens=qlens_a, mask=mask,
                                         poison_padding=qlens is not None)
    for b in range(B):
        nq = Sq if qlens is None else int(qlens[b])
        nk = Skv if lens is None else int(lens[b])
        m5 = None if mask is None else np.broadcast_to(mask, (B, Hq, Sq, Skv))[b:b + 1, :, :nq, :nk].reshape(1, Hkv, G, nq, nk)
        # (a sequence cut to its lengths: the causal diagonal is anchored at the full extents)
        if causal and (nq != Sq or nk != Skv) and nk - nq != Skv - Sq:
            tri = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)[:nq, :nk].reshape(1, 1, 1, nq, nk)
            m5 = tri if m5 is None else m5 + tri
            cz = False
        else:
            cz = causal
        rq, rk, rv = BW.sdpa_backward(q[b:b + 1, :, :nq].reshape(1, Hkv, G, nq, D), k[b:b + 1, :, None, :nk], v[b:b + 1, :, None, :nk],
                                      go[b:b + 1, :, :nq].reshape(1, Hkv, G, nq, Dv), mask=m5, causal=cz)
        compare("dq[%d]" % b, dq[b:b + 1, :, :nq], rq.reshape(1, Hq, nq, D), tol=1e-5)
        compare("dk[%d]" % b, dk[b:b + 1, :, :nk], rk.reshape(1, Hkv, nk, D), tol=1e-5)
        compare("dv[%d]" % b, dv[b:b + 1, :, :nk], rv.reshape(1, Hkv, nk, Dv), tol=1e-5)
        assert not dq[b, :, nq:].any() and not dk[b, :, nk:].any() and not dv[b, :, nk:].any()


@pytest.mark.parametrize("parts", ["1", "2", "4", "8"])
@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, q_lens, mask
    (1, 8, 1, 1024, 1024, 128, 128, True, None, None, None),                # eight query heads walking one KV head's key blocks
    (2, 4, 2, 600, 1100, 64, 64, True, [1100, 300], None, None),
    (1, 2, 2, 2100, 520, 128, 64, False, None, None, None),                 # D != Dv: planes of different widths
    (1, 8, 2, 520, 1504, 128, 128, True, None, None, "window"),             # a mask whose values go through LDS; its flags trim the walk before it is dealt
    (2, 2, 2, 1024, 1024, 64, 64, True, [1024, 700], [1024, 700], None),    # padding rows and keys: zero in every plane
    (1, 4, 1, 700, 333, 128, 128, False, None, None, "values"),             # a mask whose rows cannot be copied
], ids=["gqa8", "ragged_gqa64", "rect_d_dv", "window_gqa", "padded", "values_unaligned"])
def test_matrix_core_backward_16bit_in_parts(gpu, monkeypatch, parts, dtype, shape):
    """The 16-bit dK/dV kernel with the walk of a key block - the query tiles of every head of its group - dealt to 1, 2, 4 and 8
    workgroups whose sums meet as f32 in planes of the workspace (what a call with few key blocks gets by itself;
    INCIN_ROCM_BWD_PARTS forces it): against the f64 oracle each, exact zeros where padding is."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, qlens, mk = shape
    G = Hq // Hkv
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    say("matrix-core backward %s in %s parts: %s" % (dtypes.NAMES[dtype], parts, shape))
    q, k, v, go = make_d(95 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    r = np.random.Generator(np.random.PCG64(96))
    mask = None
    if mk == "window":
        dist = np.arange(Sq)[:, None] + (Skv - Sq) - np.arange(Skv)[None, :]
        mask = np.where((dist >= 0) & (dist < 400), -0.01 * dist, -np.inf).astype(np.float32).reshape(1, 1, Sq, Skv)
    elif mk == "values":
        mask = r.standard_normal((1, Hq, Sq, Skv), dtype=np.float32)
        mask[r.random(mask.shape) < 0.25] = -np.inf
        mask[..., 0] = 0.0
    if mask is not None:
        mask = dtypes.round_to(mask, dtype)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    qlens_a = None if qlens is None else np.asarray(qlens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens_a, q_lens=qlens_a, mask=mask,
                                         poison_padding=qlens is not None)
    for b in range(B):
        nq = Sq if qlens is None else int(qlens[b])
        nk = Skv if lens is None else int(lens[b])
        m5 = None if mask is None else np.broadcast_to(mask, (B, Hq, Sq, Skv))[b:b + 1, :, :nq, :nk].reshape(1, Hkv, G, nq, nk)
        if causal and nk - nq != Skv - Sq:      # (a sequence cut to its lengths: the causal diagonal stays anchored at the full extents)
            tri = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)[:nq, :nk].reshape(1, 1, 1, nq, nk)
            m5 = tri if m5 is None else m5 + tri
            cz = False
        else:
            cz = causal
        rq, rk, rv = BW.sdpa_backward(q[b:b + 1, :, :nq].reshape(1, Hkv, G, nq, D), k[b:b + 1, :, None, :nk], v[b:b + 1, :, None, :nk],
                                      go[b:b + 1, :, :nq].reshape(1, Hkv, G, nq, Dv), mask=m5, causal=cz)
        compare("dq[%d]" % b, dq[b:b + 1, :, :nq], rq.reshape(1, Hq, nq, D))
        compare("dk[%d]" % b, dk[b:b + 1, :, :nk], rk.reshape(1, Hkv, nk, D))
        compare("dv[%d]" % b, dv[b:b + 1, :, :nk], rv.reshape(1, Hkv, nk, Dv))
        assert not dq[b, :, nq:].any() and not dk[b, :, nk:].any() and not dv[b, :, nk:].any()


def test_matrix_core_backward_f32_rows_without_keys(gpu):
    # Sq > Skv under causal alignment: the first Sq - Skv rows see nothing; they get a zero dq and add nothing to dk, dv
    B, H, Sq, Skv, D = 1, 2, 96, 40, 64
    q, k, v, go = make(42, B, H, H, Sq, Skv, D, capi.F32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, causal=True, impl=capi.IMPL_MFMA)
    dead = Sq - Skv
    assert np.isnan(out[:, :, :dead]).all() and not dq[:, :, :dead].any()
    rq, rk, rv = BW.sdpa_backward(q[:, :, dead:], k, v, go[:, :, dead:], causal=True)
    compare("dq (live rows)", dq[:, :, dead:], rq, tol=1e-5)
    compare("dk", dk, rk, tol=1e-5)
    compare("dv", dv, rv, tol=1e-5)
    lens = np.array([0], np.int32)
    out, dq, dk, dv = host.sdpa_backward(q[:, :, :40], k, v, go[:, :, :40], capi.F32, kv_lens=lens, impl=capi.IMPL_MFMA)
    assert not dq.any() and not dk.any() and not dv.any()


def test_matrix_core_backward_f32_single_key(gpu):
    """One visible key: P = 1, dS = dP - D = 0 and dq = dk = 0 in real arithmetic.  The reference's tape subtracts dP from
    itself there (cpu/ops/elementwise.rs:1062-1077: the sum over one element) and gets an exact zero; the kernels subtract
    D_i = dO_i . O_i from dP_i0 = dO_i . V_0, two f32 evaluations of one sum of D products, each off by the rounding of its
    partial sums (of the order of sqrt(D) half units in the last place).  What reaches the gradients is bounded by that:
    2 sqrt(D) 2^-24 max|dP| per dS, times |scale| sum_i |Q_id| for dk and |scale| |K_0d| for dq; dv is the plain column sum
    of dO."""
    B, Hq, Hkv, Sq, Skv, D = 1, 2, 1, 64, 70, 128
    q, k, v, go = make(44, B, Hq, Hkv, Sq, Skv, D, capi.F32)
    lens = np.array([1], np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, kv_lens=lens, impl=capi.IMPL_MFMA)
    s = 1.0 / np.sqrt(D)
    eps_ds = 2.0 * np.sqrt(D) * 2.0 ** -24 * float(np.abs(go.astype(np.float64) @ v[0, 0, 0].astype(np.float64)).max())
    say("   single key: max|dq| %.3e max|dk| %.3e, dS rounding level %.3e" % (np.abs(dq).max(), np.abs(dk).max(), eps_ds))
    assert np.abs(dq).max() <= eps_ds * s * np.abs(k[0, 0, 0]).max()
    assert np.abs(dk[0, 0, 0]).max() <= eps_ds * s * np.abs(q).sum(axis=(1, 2)).max()
    assert not dk[0, 0, 1:].any() and not dv[0, 0, 1:].any()
    compare("dv", dv[0, 0, 0], go.astype(np.float64).sum(axis=(0, 1, 2)), tol=1e-5)


def test_matrix_core_backward_f32_at_a_few_thousand_tokens(gpu):
    B, Hq, Hkv, S, D = 1, 4, 2, 2048, 128
    q, k, v, go = make(43, B, Hq, Hkv, S, S, D, capi.F32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, causal=True, impl=capi.IMPL_MFMA)
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, 2, S, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, 2, S, D), causal=True)
    compare("dq", dq, rq.reshape(B, Hq, S, D), tol=1e-5)
    compare("dk", dk, rk.reshape(B, Hkv, S, D), tol=1e-5)
    compare("dv", dv, rv.reshape(B, Hkv, S, D), tol=1e-5)


@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16])
@pytest.mark.parametrize("D", [128, 64])
def test_generic_and_matrix_core_backward_agree(gpu, dtype, D):
    """The same 16-bit problem through both sets of kernels: each within tolerance of the oracle, and of each other."""
    B, Hq, Hkv, S = 2, 4, 2, 200
    q, k, v, go = make(31, B, Hq, Hkv, S, S, D, dtype)
    lens = np.array([200, 77], np.int32)
    a = host.sdpa_backward(q, k, v, go, dtype, causal=True, kv_lens=lens, impl=capi.IMPL_GENERIC)
    b = host.sdpa_backward(q, k, v, go, dtype, causal=True, kv_lens=lens, impl=capi.IMPL_MFMA)
    ref = BW.sdpa_backward(q.reshape(B, Hkv, 2, S, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, 2, S, D),
                           causal=True, kv_lens=lens.reshape(B, 1, 1))
    shapes = [(B, Hq, S, D), (B, Hkv, S, D), (B, Hkv, S, D)]
    for name, x, y, r_, shp in zip(("dq", "dk", "dv"), a[1:], b[1:], ref, shapes):
        compare(name + " generic", x, r_.reshape(shp))
        compare(name + " mfma", y, r_.reshape(shp))
        compare(name + " generic vs mfma", x, y)


def test_backward_refuses_what_it_does_not_cover(gpu):
    q, k, v, go = make(14, 1, 1, 1, 32, 32, 36, capi.BF16)
    with pytest.raises(capi.RocmError) as e:                     # the matrix-core kernels, pinned, outside their domain (72-byte rows)
        host.sdpa_backward(q, k, v, go, capi.BF16, impl=capi.IMPL_MFMA)
    assert e.value.code == capi.EUNSUPPORTED
    q, k, v, go = make(14, 1, 1, 1, 8, 8, 320, capi.F32)         # wider than any kernel
    with pytest.raises(capi.RocmError) as e:
        host.sdpa_backward(q, k, v, go, capi.F32)
    assert e.value.code == capi.EUNSUPPORTED


@pytest.mark.parametrize("dtype", [capi.BF16, capi.F32])
def test_no_keys_gives_a_zero_query_gradient(gpu, dtype):
    """Queries but no keys: the output is zeros whatever q holds, so dq is zeros (the reference's tape gives zeros), and
    the entry point promises to overwrite it; dk and dv have no elements."""
    say("backward with an empty key axis, dtype %d" % dtype)
    B, H, Sq, D = 2, 3, 50, 128
    q, _, _, go = make(5, B, H, H, Sq, 1, D, dtype)
    empty = np.zeros((B, H, 0, D), np.float32)
    tq, tg = host.DeviceTensor.from_f32(q, dtype), host.DeviceTensor.from_f32(go, dtype)
    tk, tv, tdk, tdv = (host.DeviceTensor.from_f32(empty, dtype) for _ in range(4))
    to, tdq = host.DeviceTensor((B, H, Sq, D), dtype), host.DeviceTensor((B, H, Sq, D), dtype)
    capi.check(capi.load().incin_rocm_memset(0, tdq.ptr, 0x7f, tdq.buf.nbytes))          # what an allocator may leave behind
    lse = capi.DeviceBuffer(B * H * Sq * 4)
    bd = capi.SdpaBwdDesc()
    bd.fwd = host.make_desc(tq, tk, tv, to, lse=lse)
    for name, t in (("d_o", tg), ("d_q", tdq), ("d_k", tdk), ("d_v", tdv)):
        setattr(bd, name, t.ptr)
        for i, s in enumerate(host._strides3(t.shape)):
            getattr(bd, name + "_stride")[i] = s
    assert capi.sdpa_bwd_workspace(bd) == 0
    capi.sdpa_fwd(bd.fwd)
    capi.sdpa_bwd(bd)
    capi.sync()
    assert not to.to_f32().any() and not tdq.to_f32().any()


@pytest.mark.parametrize("case", [
    # dtype, impl, D
    (capi.BF16, capi.IMPL_AUTO, 128), (capi.F16, capi.IMPL_MFMA, 64), (capi.F32, capi.IMPL_AUTO, 64), (capi.F32, capi.IMPL_MFMA, 128),
    (capi.F32, capi.IMPL_GENERIC, 80), (capi.BF16, capi.IMPL_GENERIC, 128),
], ids=["bf16_auto", "f16_mfma_d64", "f32_auto_d64", "f32_mfma", "f32_generic_d80", "bf16_generic"])
def test_backward_of_a_padded_batch(gpu, case):
    """A padded self-attention batch: sequence b has lens[b] real positions, the rest of its rows and keys are padding
    (q_lens = kv_lens = lens).  The forward leaves the padding rows of O and lse unspecified - here they are overwritten
    with NaN, and the padding rows of dO hold NaN too - and the backward must give, per sequence, the gradients of that
    sequence alone: dQ, dK, dV of the truncated problem inside the lengths, exact zeros outside."""
    dtype, impl, D = case
    B, Hq, Hkv, S = 3, 4, 2, 300
    G = Hq // Hkv
    lens = np.array([300, 131, 64], np.int32)
    q, k, v, go = make(71, B, Hq, Hkv, S, S, D, dtype)
    for b in range(B):
        go[b, :, lens[b]:] = np.nan
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, causal=True, kv_lens=lens, q_lens=lens, impl=impl, poison_padding=True)
    tol = 1e-5 if dtype == capi.F32 else 2e-2
    for b in range(B):
        n = int(lens[b])
        rq, rk, rv = BW.sdpa_backward(q[b:b + 1, :, :n].reshape(1, Hkv, G, n, D), k[b:b + 1, :, None, :n], v[b:b + 1, :, None, :n],
                                      go[b:b + 1, :, :n].reshape(1, Hkv, G, n, D), causal=True)
        compare("dq[%d]" % b, dq[b:b + 1, :, :n], rq.reshape(1, Hq, n, D), tol)
        compare("dk[%d]" % b, dk[b:b + 1, :, :n], rk.reshape(1, Hkv, n, D), tol)
        compare("dv[%d]" % b, dv[b:b + 1, :, :n], rv.reshape(1, Hkv, n, D), tol)
        assert not dq[b, :, n:].any() and not dk[b, :, n:].any() and not dv[b, :, n:].any()


@pytest.mark.parametrize("parts", ["1", "4"])
@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, q_lens, scale
    (1, 1, 1, 1, 1, 256, 256, True, None, None, None),                      # one query, one key
    (1, 2, 1, 33, 31, 136, 144, False, None, None, None),                   # a row past and a row short of a tile; the narrowest heads
    (2, 4, 2, 127, 129, 256, 256, True, None, None, None),                  # a row short of and a row past a block
    (1, 2, 2, 161, 97, 192, 128, True, None, None, None),                   # more queries than keys: rows that see none; D != Dv
    (3, 4, 1, 300, 420, 160, 256, True, [420, 131, 0], None, None),         # key counts, one sequence without keys
    (2, 2, 2, 300, 300, 256, 192, True, [300, 70], [300, 70], None),        # a padded batch
    (1, 8, 2, 260, 520, 256, 256, False, None, None, -0.05),                # a negative scale
    (1, 2, 1, 1057, 1057, 256, 256, True, None, None, None),                # many tiles: every stage of the ring, four parts by themselves
], ids=["one", "narrow", "block_edges", "rect", "ragged", "padded", "negative_scale", "long"])
def test_matrix_core_backward_above_128(gpu, monkeypatch, parts, dtype, shape):
    """Head dimensions above 128 on the matrix cores, with the walks of the dK and dV blocks whole and dealt to four workgroups.  P
    and dS enter their products as two 16-bit values, so what is left is the rounding of the results (half a step of the storage
    type, 2^-9 and 2^-12, of values up to the largest) and of the forward's O and normalisers: 4 times that half step of the largest magnitude.
    (That these kernels run, and that both values count: test_backward_above_128_has_the_precision_of_f32_arithmetic.)"""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, qlens, scale = shape
    G = Hq // Hkv
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    say("matrix-core backward above 128, %s in %s parts: %s" % (dtypes.NAMES[dtype], parts, shape))
    q, k, v, go = make_d(131 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    qlens_a = None if qlens is None else np.asarray(qlens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_AUTO, causal=causal, kv_lens=lens_a, q_lens=qlens_a, scale=scale,
                                         poison_padding=qlens is not None)
    tol = 2.0 ** -7 if dtype == capi.BF16 else 2.0 ** -10
    for b in range(B):
        nq = Sq if qlens is None else int(qlens[b])
        nk = Skv if lens is None else int(lens[b])
        if nk > 0:
            tri = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)[:nq, :nk].reshape(1, 1, 1, nq, nk) if causal else None
            rows = np.isfinite(tri).any(axis=-1).reshape(nq) if causal else np.ones(nq, bool)      # (rows that see a key: the others have zero gradients here)
            sel = lambda x: x[b:b + 1, :, :nq][:, :, rows]
            tri = None if tri is None else tri[:, :, :, rows]
            n = int(rows.sum())
            rq, rk, rv = BW.sdpa_backward(sel(q).reshape(1, Hkv, G, n, D), k[b:b + 1, :, None, :nk], v[b:b + 1, :, None, :nk],
                                          sel(go).reshape(1, Hkv, G, n, Dv), mask=tri, scale=scale)
            compare("dq[%d]" % b, sel(dq), rq.reshape(1, Hq, n, D), tol=tol)
            compare("dk[%d]" % b, dk[b:b + 1, :, :nk], rk.reshape(1, Hkv, nk, D), tol=tol)
            compare("dv[%d]" % b, dv[b:b + 1, :, :nk], rv.reshape(1, Hkv, nk, Dv), tol=tol)
            assert not dq[b, :, :nq][:, ~rows].any()
        else:
            assert not dq[b].any()
        assert not dq[b, :, nq:].any() and not dk[b, :, nk:].any() and not dv[b, :, nk:].any()


@pytest.mark.parametrize("parts", ["1", "4"])
@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, q_lens
    (2, 130, 130, 1, 33, 64, 64, True, None, None),                         # enough blocks without groups: one query, a key past a 32-key share
    (1, 260, 260, 65, 31, 64, 64, False, None, None),                       # a row past a tile, a key short of a share
    (2, 6, 3, 200, 333, 64, 48, True, [333, 70], None),                     # grouped queries, D != Dv, a count inside the first block
    (1, 8, 1, 1030, 640, 40, 64, False, None, None),                        # many tiles of eight heads
    (1, 4, 2, 700, 260, 64, 64, True, None, None),                          # rows that see no key
    (3, 4, 2, 300, 300, 64, 64, True, [300, 131, 0], [300, 131, 1]),        # a padded batch, a sequence without keys
    (2, 130, 130, 1, 33, 96, 96, True, None, None),                         # the same edges in the instance for 65 - 96
    (1, 260, 260, 65, 31, 80, 72, False, None, None),
    (2, 6, 3, 200, 333, 72, 96, True, [333, 70], None),
    (1, 8, 1, 1030, 640, 96, 40, False, None, None),
    (1, 4, 2, 700, 260, 40, 96, True, None, None),
    (3, 4, 2, 300, 300, 96, 80, True, [300, 131, 0], [300, 131, 1]),
    (1, 4, 2, 200, 200, 96, 104, True, None, None),                         # past its edge: the paired kernel
], ids=["one_row", "rect", "ragged", "gqa8", "no_keys_seen", "padded", "one_row_96", "rect_96", "ragged_96", "gqa8_96", "no_keys_seen_96", "padded_96", "edge_104"])
def test_matrix_core_backward_narrow_heads(gpu, monkeypatch, parts, dtype, shape):
    """The dK/dV kernel for head dimensions up to 64, or 96 (one wavefront per 32 keys) against the f64 oracle, walks whole and dealt to
    four workgroups; and the same call with the row dots computed inside the dQ kernel (one stream) bit-identical to the
    call that has a kernel for them and the dQ kernel beside (where the rule takes a second stream)."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, qlens = shape
    G = Hq // Hkv
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    say("matrix-core backward, narrow heads, %s in %s parts: %s" % (dtypes.NAMES[dtype], parts, shape))
    q, k, v, go = make_d(141 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    qlens_a = None if qlens is None else np.asarray(qlens, np.int32)
    res = []
    for streams in (None, "1"):
        if streams:
            monkeypatch.setenv("INCIN_ROCM_BWD_STREAMS", streams)
        res.append(host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens_a, q_lens=qlens_a,
                                      poison_padding=qlens is not None))
    for a, b in zip(res[0][1:], res[1][1:]):
        assert np.array_equal(a, b)
    out, dq, dk, dv = res[0]
    for b in range(B):
        nq = Sq if qlens is None else int(qlens[b])
        nk = Skv if lens is None else int(lens[b])
        if nk > 0:
            tri = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)[:nq, :nk] if causal else np.zeros((nq, nk), np.float32)
            rows = np.isfinite(tri).any(axis=-1)                            # (rows that see a key: the others have zero gradients here)
            sel = lambda x: x[b:b + 1, :, :nq][:, :, rows]
            n = int(rows.sum())
            rq, rk, rv = BW.sdpa_backward(sel(q).reshape(1, Hkv, G, n, D), k[b:b + 1, :, None, :nk], v[b:b + 1, :, None, :nk],
                                          sel(go).reshape(1, Hkv, G, n, Dv), mask=tri[rows].reshape(1, 1, 1, n, nk))
            compare("dq[%d]" % b, sel(dq), rq.reshape(1, Hq, n, D))
            compare("dk[%d]" % b, dk[b:b + 1, :, :nk], rk.reshape(1, Hkv, nk, D))
            compare("dv[%d]" % b, dv[b:b + 1, :, :nk], rv.reshape(1, Hkv, nk, Dv))
            assert not dq[b, :, :nq][:, ~rows].any()
        else:
            assert not dq[b].any()
        assert not dq[b, :, nq:].any() and not dk[b, :, nk:].any() and not dv[b, :, nk:].any()


@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, kv_lens, q_lens, mask
    (1, 1, 1, 1, 1, 64, 64, False, None, None, False),                      # four wavefronts to a walk of one row
    (2, 3, 3, 33, 129, 64, 32, True, [129, 97], None, False),               # ... a tile of 128 rows and one more
    (1, 4, 2, 260, 131, 64, 64, True, None, None, False),                   # ... rows that see no key, grouped queries
    (1, 2, 2, 161, 300, 40, 64, False, None, None, True),                   # ... a mask of values
    (3, 4, 4, 193, 193, 64, 64, True, [193, 64, 0], [193, 64, 1], False),   # ... a padded batch, a sequence without keys
    (4, 20, 20, 97, 95, 64, 64, True, None, None, True),                    # two: more blocks of 32 than compute units
    (8, 36, 36, 450, 450, 64, 64, True, None, None, False),                 # one: many rounds of blocks
    (1, 2, 1, 65, 63, 80, 80, True, None, None, False),                     # 96 of 128 columns: a row past and a key short of a tile
    (2, 4, 2, 127, 200, 96, 68, False, [200, 33], None, True),
    (1, 3, 3, 130, 97, 100, 96, True, None, None, False),                   # ... and past their edge
    (3, 4, 4, 193, 193, 128, 128, True, [193, 64, 0], [193, 64, 1], False),
    (2, 8, 8, 1464, 1464, 80, 80, False, None, None, False),                # dealt to two workgroups because a round would be left part empty
], ids=lambda s: "x".join(str(x) for x in s[:7]))
def test_matrix_core_backward_f32_walks_shared(gpu, shape):
    """The f32 backward launch with 1, 2 and 4 wavefronts of a workgroup to a block's walk, as the sizes choose: 1e-5 of the largest
    gradient magnitude against the f64 oracle (sampled batch entries of the large ones), exact zeros where padding is."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, qlens, values = shape
    G = Hq // Hkv
    say("matrix-core backward f32, walks shared: %s" % (shape,))
    q, k, v, go = make_d(171 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, capi.F32)
    r = np.random.Generator(np.random.PCG64(172))
    mask = None
    if values:
        mask = r.standard_normal((1, Hq, Sq, Skv), dtype=np.float32)
        mask[r.random(mask.shape) < 0.25] = -np.inf
        mask[..., 0] = 0.0
    lens_a = None if lens is None else np.asarray(lens, np.int32)
    qlens_a = None if qlens is None else np.asarray(qlens, np.int32)
    out, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.F32, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens_a, q_lens=qlens_a, mask=mask,
                                         poison_padding=qlens is not None)
    for b in (range(B) if B * Hq < 200 else (0, B - 1)):
        nq = Sq if qlens is None else int(qlens[b])
        nk = Skv if lens is None else int(lens[b])
        if nk > 0:
            m = np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)[:nq, :nk] if causal else np.zeros((nq, nk), np.float32)
            rows = np.isfinite(m).any(axis=-1)                              # (rows that see a key: the others have zero gradients here)
            n = int(rows.sum())
            sel = lambda x: x[b:b + 1, :, :nq][:, :, rows]
            m5 = m[rows].reshape(1, 1, 1, n, nk)
            if values:
                m5 = m5 + mask[:, :, :nq, :nk][:, :, rows].reshape(1, Hkv, G, n, nk)
            rq, rk, rv = BW.sdpa_backward(sel(q).reshape(1, Hkv, G, n, D), k[b:b + 1, :, None, :nk], v[b:b + 1, :, None, :nk],
                                          sel(go).reshape(1, Hkv, G, n, Dv), mask=m5)
            # (one visible key leaves dS = 0, and what f32 leaves of it is the rounding of dP - D: measured on dP's scale instead)
            for name, x, y in (("dq", sel(dq), rq.reshape(1, Hq, n, D)), ("dk", dk[b:b + 1, :, :nk], rk.reshape(1, Hkv, nk, D)),
                               ("dv", dv[b:b + 1, :, :nk], rv.reshape(1, Hkv, nk, Dv))):
                if nk == 1 and name != "dv":
                    assert np.abs(x).max() <= 1e-5 * float(np.abs(v).max() * np.abs(go).max() * Dv)
                else:
                    compare("%s[%d]" % (name, b), x, y, tol=1e-5)
            assert not dq[b, :, :nq][:, ~rows].any()
        else:
            assert not dq[b].any()
        assert not dq[b, :, nq:].any() and not dk[b, :, nk:].any() and not dv[b, :, nk:].any()


@pytest.mark.parametrize("case", [
    # dtype, B, Hq, Hkv, S, D, planes of dQ and of dK, dV that the smallest workspace has room for (256 compute units)
    (capi.BF16, 1, 8, 1, 1024, 256, 0, 0),
    (capi.BF16, 1, 8, 2, 512, 64, 0, 0),
    (capi.F16, 1, 4, 1, 512, 96, 0, 0),
    (capi.F32, 1, 2, 2, 192, 64, 0, 0),
    (capi.F32, 1, 16, 2, 2048, 64, 1, 3),           # (dealt to four workgroups each when there is room)
], ids=["wide", "narrow64", "narrow96", "f32_undivided", "f32"])
def test_backward_with_the_smallest_workspace(gpu, case):
    """A call whose workspace holds the per-row floats but not the planes of the walks that it would divide by itself: the same gradients
    (planes change the order of f32 sums and nothing else: one rounding step of the storage type of the largest magnitude); a byte less is refused."""
    dtype, B, Hq, Hkv, S, D, planes_q, planes_kv = case
    say("backward, smallest workspace: %s" % (case,))
    q, k, v, go = make(173 + D, B, Hq, Hkv, S, S, D, dtype)
    tq, tk, tv, tg = (host.DeviceTensor.from_f32(x, dtype) for x in (q, k, v, go))
    to, tdq, tdk, tdv = (host.DeviceTensor(t.shape, dtype) for t in (tq, tq, tk, tv))
    lse = capi.DeviceBuffer(B * Hq * S * 4)
    bd = capi.SdpaBwdDesc()
    bd.fwd = host.make_desc(tq, tk, tv, to, causal=True, lse=lse)
    fneed = capi.sdpa_workspace(bd.fwd)[0]
    fws = capi.DeviceBuffer(max(fneed, 256))
    bd.fwd.workspace, bd.fwd.workspace_bytes = fws.ptr, fneed
    for name, t in (("d_o", tg), ("d_q", tdq), ("d_k", tdk), ("d_v", tdv)):
        setattr(bd, name, t.ptr)
        for i, s in enumerate(host._strides3(t.shape)):
            getattr(bd, name + "_stride")[i] = s
    capi.sdpa_fwd(bd.fwd)
    least, full = (2 * B * Hq * S + planes_q * B * Hq * S * D + planes_kv * 2 * B * Hkv * S * D) * 4, capi.sdpa_bwd_workspace(bd)
    assert full > least or (dtype == capi.F32 and S < 1024 and full == least)
    ws = capi.DeviceBuffer(full)
    got = []
    for given in (full, least):
        bd.workspace, bd.workspace_bytes = ws.ptr, given
        capi.sdpa_bwd(bd)
        capi.sync()
        got.append([t.to_f32() for t in (tdq, tdk, tdv)])
    step = {capi.BF16: 2.0 ** -8, capi.F16: 2.0 ** -11, capi.F32: 1e-5}[dtype]
    for name, a, b in zip(("dq", "dk", "dv"), *got):
        compare(name, b, a, tol=step)
    bd.workspace_bytes = least - 1
    with pytest.raises(capi.RocmError) as e:
        capi.sdpa_bwd(bd)
    assert e.value.code == capi.EWORKSPACE


class Gradients:
    """One forward with row normalisers, and backward calls on what it left, by whichever kernels a call names."""

    def __init__(self, q, k, v, go, dtype, **kw):
        self.dtype = dtype
        self.t = {n: host.DeviceTensor.from_f32(x, dtype) for n, x in (("q", q), ("k", k), ("v", v), ("d_o", go))}
        self.t["o"] = host.DeviceTensor(go.shape, dtype)
        for n in ("q", "k", "v"):
            self.t["d_" + n] = host.DeviceTensor(self.t[n].shape, dtype)
        self.lens = {n: capi.DeviceBuffer.from_numpy(np.asarray(kw.pop(n), np.int32)) for n in ("kv_lens", "q_lens") if kw.get(n) is not None}
        self.lse = capi.DeviceBuffer(int(np.prod(go.shape[:3])) * 4)
        self.bd = bd = capi.SdpaBwdDesc()
        bd.fwd = host.make_desc(self.t["q"], self.t["k"], self.t["v"], self.t["o"], lse=self.lse, **{**kw, **self.lens})
        self.fws = capi.DeviceBuffer(max(capi.sdpa_workspace(bd.fwd)[0], 256))
        bd.fwd.workspace, bd.fwd.workspace_bytes = self.fws.ptr, self.fws.nbytes
        for n in ("d_o", "d_q", "d_k", "d_v"):
            setattr(bd, n, self.t[n].ptr)
            for a, s in enumerate(host._strides3(self.t[n].shape)):
                getattr(bd, n + "_stride")[a] = s
        capi.sdpa_fwd(bd.fwd)
        capi.sync()

    def workspace(self, impl):
        self.bd.fwd.impl = impl
        return capi.sdpa_bwd_workspace(self.bd)

    def run(self, impl):
        ws = capi.DeviceBuffer(self.workspace(impl))
        self.bd.workspace, self.bd.workspace_bytes = ws.ptr, ws.nbytes
        capi.sdpa_bwd(self.bd)
        capi.sync()
        ws.free()
        return [self.t[n].to_f32() for n in ("d_q", "d_k", "d_v")]


def step_of(x, dtype):
    """The distance between neighbouring values of the storage type at magnitude x."""
    bits, least = (11, -24) if dtype == capi.F16 else (8, -133)
    return 2.0 ** np.maximum(np.floor(np.log2(np.maximum(np.abs(x), 2.0 ** -140))) + 1 - bits, least)


def assert_same_but_for_the_last_rounding(name, got, ref, dtype):
    """Both rounded from sums whose terms are exact to 16 bits (bf16) or 22 (f16) at least, where the storage type has 8 and 11: a result
    is the neighbouring value where the two sums lie on either side of a rounding border, about one in 2^8 of them; with terms
    rounded to the storage type once, one in three or four.  (A result far below its row's others is looked at in their steps.)"""
    rms = np.sqrt((ref.astype(np.float64) ** 2).mean(-1, keepdims=True))
    assert np.isfinite(got).all() and np.isfinite(ref).all(), name
    steps = np.abs(got.astype(np.float64) - ref) / step_of(np.maximum(np.abs(ref), rms), dtype)
    say("   %s: %.2e of the results differ, by %.2f steps at most" % (name, (got != ref).mean(), steps.max()))
    assert steps.max() <= 1.0, name
    assert (got != ref).mean() <= 2.0 ** -5, name


@pytest.mark.parametrize("parts", ["1", "4"])
@pytest.mark.parametrize("dtype", [capi.BF16, capi.F16], ids=lambda x: dtypes.NAMES[x])
@pytest.mark.parametrize("magnitudes", ["one", "small", "rising", "falling", "opposed_pair"])
def test_backward_above_128_has_the_precision_of_f32_arithmetic(gpu, monkeypatch, parts, dtype, magnitudes):
    """Head dimensions above 128 on the matrix cores against the generic kernels' f32 arithmetic on the same forward: gradients of any
    magnitude that the storage type holds.  small: an unscaled mean loss; rising, falling: the rows of dO and V over a
    factor of 2^16, so that in either walk what a row has to hold grows again and again, or only shrinks; opposed_pair: two keys with equal
    scores and opposed values under a scaled loss, whose dS pass what f16 holds while the gradients do not come near it."""
    say("backward above 128 against f32 arithmetic: %s, %s, %s parts" % (magnitudes, dtypes.NAMES[dtype], parts))
    if magnitudes == "opposed_pair":
        B, Hq, Hkv, Sq, Skv, D, Dv, causal = 1, 2, 1, 50, 2, 256, 256, False
    else:
        B, Hq, Hkv, Sq, Skv, D, Dv, causal = 2, 4, 2, 333, 420, 256, 192, True
    q, k, v, go = make_d(241, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    if magnitudes == "small":
        go *= 2.0 ** -10
    elif magnitudes in ("rising", "falling"):
        up = lambda n: (2.0 ** np.linspace(-8, 8, n)[:: 1 if magnitudes == "rising" else -1]).astype(np.float32)[:, None]
        go, v = go * up(Sq) / 16, v * up(Skv) / 16
    elif magnitudes == "opposed_pair":
        q, go = q / 64, np.full_like(go, 512.0)
        v[:, :, 0], v[:, :, 1] = 1.0, -1.0
    q, go, v = (dtypes.round_to(x, dtype) for x in (q, go, v))
    g = Gradients(q, k, v, go, dtype, causal=causal)
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", "4")
    if magnitudes != "opposed_pair":      # (the matrix-core kernels have planes of f32 sums then, the generic kernels have none)
        assert g.workspace(capi.IMPL_AUTO) > g.workspace(capi.IMPL_GENERIC)
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    for name, a, b in zip(("dq", "dk", "dv"), g.run(capi.IMPL_AUTO), g.run(capi.IMPL_GENERIC)):
        assert_same_but_for_the_last_rounding(name, a, b, dtype)


@pytest.mark.parametrize("case", [
    # dtype, B, heads, D: one query over one key; more blocks of all gradients together than one launch takes, though not of any one
    (capi.BF16, 60000, 48, 256),
    (capi.F32, 60000, 150, 68),
], ids=["wide", "f32"])
def test_backward_of_more_heads_than_one_launch_takes(gpu, case):
    """Heads of one query and one key, the inputs the same in every batch entry (strides of 0): P = 1, so dV is dO (P to 1e-5: in bf16
    the same or the neighbouring value) and dQ, dK are what rounding leaves of dP - D = 0."""
    dtype, B, H, D = case
    say("backward of %d x %d heads, %s, D = %d" % (B, H, dtypes.NAMES[dtype], D))
    r = np.random.Generator(np.random.PCG64(251))
    q, k, v, go = (dtypes.round_to(r.standard_normal((1, H, 1, D), dtype=np.float32), dtype) for _ in range(4))
    scale = host.resolve_scale(None, D)
    lse = np.broadcast_to((q.astype(np.float64) * k).sum(-1).reshape(1, H) * scale, (B, H)).astype(np.float32)
    ins = [host.DeviceTensor.from_f32(x, dtype) for x in (q, k, v, v, go)]      # (O is V)
    size = dtypes.ITEMSIZE[dtype]
    grads = [capi.DeviceBuffer(B * H * D * size) for _ in range(3)]
    for g in grads:
        capi.check(capi.load().incin_rocm_memset(0, g.ptr, 0x7f, g.nbytes))
    tl = capi.DeviceBuffer.from_numpy(np.ascontiguousarray(lse))
    bd = capi.SdpaBwdDesc()
    bd.fwd = host.make_desc(*ins[:4], lse=tl)
    bd.fwd.B = B
    for name in ("q_stride", "k_stride", "v_stride", "o_stride"):
        getattr(bd.fwd, name)[0] = 0
    bd.d_o = ins[4].ptr
    bd.d_q, bd.d_k, bd.d_v = (g.ptr for g in grads)
    for name in ("d_o", "d_q", "d_k", "d_v"):
        for a, s in enumerate((0 if name == "d_o" else H * D, D, D)):
            getattr(bd, name + "_stride")[a] = s
    ws = capi.DeviceBuffer(capi.sdpa_bwd_workspace(bd))
    bd.workspace, bd.workspace_bytes = ws.ptr, ws.nbytes
    capi.sdpa_bwd(bd)
    capi.sync()
    most = float(np.abs(v).max() * np.abs(go).max() * D)
    for b in list(range(0, B, 997)) + [B - 1]:
        for g, name in zip(grads, ("dq", "dk", "dv")):
            raw = np.empty((H, D), dtypes.storage_numpy_dtype(dtype))
            capi.check(capi.load().incin_rocm_memcpy_d2h(0, raw.ctypes.data, g.ptr + b * raw.nbytes, raw.nbytes))
            x, ref = dtypes.decode(raw, dtype), go[0, :, 0] if name == "dv" else 0.0
            assert np.isfinite(x).all() and (np.abs(x - ref) <= (np.abs(ref) * (2.0 ** -7 if dtype == capi.BF16 else 1e-5) if name == "dv" else 1e-5 * most)).all(), (b, name)
    for x in grads:
        x.free()


def in_view(x, dtype, layout):
    """x [B, H, S, D] in a wider buffer whose other places hold NaN: (the buffer's values, element strides of B, H, S, element offset)."""
    B, H, S, D = x.shape
    pad = 16 // dtypes.ITEMSIZE[dtype]
    if layout == 0:          # positions outside heads, as a projection leaves them
        w = np.full((B, S, H, D), np.nan, np.float32)
        at, strides = w.transpose(0, 2, 1, 3), (S * H * D, D, H * D)
    elif layout == 1:        # rows with padding behind them, a head and a row more than there are
        w = np.full((B, H + 1, S + 1, D + pad), np.nan, np.float32)
        at, strides = w[:, :H, :S, :D], ((H + 1) * (S + 1) * (D + pad), (S + 1) * (D + pad), D + pad)
    else:                    # one of three tensors side by side in a row; batch innermost but for that
        w = np.full((S, B, 3, H, D), np.nan, np.float32)
        at, strides = w[:, :, 1].transpose(1, 2, 0, 3), (3 * H * D, D, B * 3 * H * D)
    at[...] = x
    return w, strides, H * D if layout == 2 else 0


@pytest.mark.parametrize("parts", ["1", "4"])
@pytest.mark.parametrize("case", [
    # dtype, B, Hq, Hkv, Sq, Skv, D, Dv, causal
    (capi.BF16, 2, 4, 2, 200, 530, 256, 192, True),         # above 128
    (capi.F16, 2, 4, 2, 333, 200, 64, 48, True),            # the kernel for narrow heads; a forward with all keys in LDS
    (capi.BF16, 2, 4, 2, 600, 120, 96, 80, False),
    (capi.F16, 3, 5, 5, 31, 30, 128, 64, True),             # ... a pair of wavefronts per head
    (capi.BF16, 2, 4, 2, 300, 300, 128, 128, True),         # the paired kernel, row dots in the dQ kernel
    (capi.F32, 2, 4, 2, 333, 260, 64, 40, True),
    (capi.F32, 2, 4, 2, 300, 333, 80, 96, False),
    (capi.F32, 2, 4, 2, 300, 333, 128, 128, True),
], ids=["wide", "narrow64", "narrow96", "few_keys", "paired", "f32_d64", "f32_d96", "f32_d128"])
def test_training_step_on_views(gpu, monkeypatch, parts, case):
    """Forward and backward on operands and results in views of wider buffers, neighbours in layouts of their own, against contiguous ones: the same
    values to the bit, and nothing written beside the results."""
    dtype, B, Hq, Hkv, Sq, Skv, D, Dv, causal = case
    monkeypatch.setenv("INCIN_ROCM_BWD_PARTS", parts)
    say("training step on views: %s" % (case,))
    q, k, v, go = make_d(307 + Sq + Skv, B, Hq, Hkv, Sq, Skv, D, Dv, dtype)
    lens = np.asarray([Skv - 7 * b for b in range(B)], np.int32)
    values = dict(q=q, k=k, v=v, o=np.zeros_like(go), d_o=go, d_q=np.zeros_like(q), d_k=np.zeros_like(k), d_v=np.zeros_like(v))
    g = Gradients(q, k, v, go, dtype, causal=causal, kv_lens=lens)
    expect = dict(zip(("d_q", "d_k", "d_v"), g.run(capi.IMPL_AUTO)), o=g.t["o"].to_f32(), lse=g.lse.to_numpy(np.float32, (B, Hq, Sq)))
    size = dtypes.ITEMSIZE[dtype]
    for turn in range(3):
        views = {n: in_view(x, dtype, (i + i // 3 + turn) % 3) for i, (n, x) in enumerate(values.items())}
        bufs = {n: capi.DeviceBuffer.from_numpy(dtypes.encode(w, dtype)) for n, (w, _, _) in views.items()}
        for n, (w, strides, offset) in views.items():
            at = bufs[n].ptr + offset * size
            setattr(g.bd if n.startswith("d_") else g.bd.fwd, n, at)
            for a in range(3):
                getattr(g.bd if n.startswith("d_") else g.bd.fwd, n + "_stride")[a] = strides[a]
        capi.check(capi.load().incin_rocm_memset(0, g.lse.ptr, 0, g.lse.nbytes))
        capi.sdpa_fwd(g.bd.fwd)
        ws = capi.DeviceBuffer(capi.sdpa_bwd_workspace(g.bd))
        g.bd.workspace, g.bd.workspace_bytes = ws.ptr, ws.nbytes
        capi.sdpa_bwd(g.bd)
        capi.sync()
        ws.free()
        assert np.array_equal(g.lse.to_numpy(np.float32, (B, Hq, Sq)), expect["lse"]), turn
        for n in ("o", "d_q", "d_k", "d_v"):
            i = list(values).index(n)
            ref = in_view(expect[n], dtype, (i + i // 3 + turn) % 3)[0]
            got = dtypes.decode(bufs[n].to_numpy(dtypes.storage_numpy_dtype(dtype), ref.shape), dtype)
            assert np.array_equal(got, ref, equal_nan=True), (n, turn)
        for x in bufs.values():
            x.free()


@pytest.mark.parametrize("case", [
    # B, Hq, Hkv, Sq, Skv, D, Dv, causal, key counts, mask
    (4, 66, 66, 65, 65, 128, 128, True, None, False),           # a row past a tile
    (4, 66, 66, 65, 70, 80, 72, False, None, True),
    (4, 66, 66, 96, 96, 128, 128, True, None, True),            # whole tiles, a mask of values
    (3, 90, 90, 200, 97, 128, 100, False, [97, 33, 0], False),  # two blocks of rows, the second not full; a sequence without keys
    (3, 32, 8, 384, 384, 128, 128, False, None, False),         # grouped queries: dK / dV walks dealt to two workgroups
    (4, 70, 70, 65, 65, 40, 64, False, None, False),
    (4, 70, 70, 96, 70, 64, 48, True, None, True),
], ids=lambda c: "x".join(str(x) for x in c[:7]))
def test_matrix_core_backward_f32_of_many_short_heads(gpu, case):
    """Launches in which a wavefront walks its block of 32 alone because that issues fewer products (on 256 compute units): many heads of 65 - 96
    positions, and blocks of 128 that fill the device, against the generic kernels on the same forward."""
    B, Hq, Hkv, Sq, Skv, D, Dv, causal, lens, masked = case
    say("f32 backward of many short heads: %s" % (case,))
    q, k, v, go = make_d(331 + Sq, B, Hq, Hkv, Sq, Skv, D, Dv, capi.F32)
    kw = {}
    if masked:
        r = np.random.Generator(np.random.PCG64(337))
        m = r.standard_normal((1, 1, Sq, Skv), dtype=np.float32)
        m[..., 1:][r.random((1, 1, Sq, Skv - 1)) < 0.3] = -np.inf
        m[..., :32, 32:64] = -np.inf
        tm = capi.DeviceBuffer.from_numpy(m)
        kw = dict(mask=tm, mask_strides=host.mask_strides_for(m.shape, B, Hq, Sq, Skv))
    g = Gradients(q, k, v, go, capi.F32, causal=causal, kv_lens=lens, **kw)
    got, ref = g.run(capi.IMPL_MFMA), g.run(capi.IMPL_GENERIC)
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        compare(name, a, b, tol=1e-5)
