"""The work lists of the matrix-core prefill and dQ kernels (work_order in sdpa_mfma_common.h): every block of query rows of every head is
computed once, whatever the order - one list per XCD, eighths of one list, one list dealt item by item in groups of pairs of which the
last takes what is left.  All rows against numpy in float64; tolerances as in the parity tests of these kernels (16-bit: inputs, P and the result
rounded; f32: 1e-5)."""
import numpy as np
import pytest

from incin_amd import capi, dtypes, host
from oracle import sdpa_backward as BW
from tests.test_gpu_backward import compare, say

pytestmark = pytest.mark.gpu

SHAPES = [
    # B, Hq, Hkv, Sq, Skv, causal, key counts from - to, query counts too
    (1, 12, 12, 256, 256, False, None, False),          # eighths
    (3, 5, 5, 300, 300, False, None, False),            # a list that does not divide by 8
    (3, 12, 12, 300, 300, True, None, False),           # dealt, one group
    (5, 128, 4, 500, 500, True, None, False),           # dealt, groups of eight and twelve
    (40, 4, 1, 500, 130, False, (1, 130), False),       # key counts, the query heads of a pair innermost, one group
    (35, 8, 1, 1000, 130, False, (1, 130), False),      # likewise, two groups
    (9, 32, 2, 513, 513, True, (100, 513), True),       # a padded batch
    (7, 3, 3, 260, 260, True, (1, 260), True),          # without grouped queries
]


def operands(seed, dtype, B, Hq, Hkv, Sq, Skv, D):
    r = np.random.Generator(np.random.PCG64(seed))
    mk = lambda *s: dtypes.round_to(r.standard_normal(s, dtype=np.float32), dtype)
    return mk(B, Hq, Sq, D), mk(B, Hkv, Skv, D), mk(B, Hkv, Skv, D), mk(B, Hq, Sq, D)


@pytest.mark.parametrize("dtype,D,tol", [(capi.BF16, 128, 2e-2), (capi.F16, 64, 4e-3), (capi.F32, 64, 1e-5), (capi.BF16, 256, 2e-2)], ids=["bf16_128", "f16_64", "f32_64", "bf16_256"])
@pytest.mark.parametrize("shape", SHAPES)
def test_every_query_block_is_computed_once(gpu, monkeypatch, dtype, D, tol, shape):
    B, Hq, Hkv, Sq, Skv, causal, counts, padded = shape
    monkeypatch.setenv("INCIN_ROCM_PREFILL_BLOCK_ROWS", "128")
    D = min(D, 32) if dtype == capi.F32 else D      # (a host that counts: the instance is the same)
    say("prefill work list %s %s" % (dtypes.NAMES[dtype], shape))
    q, k, v, _ = operands(5 + Sq, dtype, B, Hq, Hkv, Sq, Skv, D)
    lens = None if counts is None else np.linspace(counts[0], counts[1], B).astype(np.int32)
    got = host.sdpa(q, k, v, dtype, causal=causal, kv_lens=lens, q_lens=lens if padded else None, impl=capi.IMPL_MFMA)
    tri = np.triu(np.full((Sq, Skv), -np.inf), 1 + Skv - Sq) if causal else np.zeros((Sq, Skv))
    G = Hq // Hkv
    worst = 0.0
    for b in range(B):
        nk = Skv if lens is None else int(lens[b])
        nq = nk if padded else Sq
        for h in range(Hq):
            s = q[b, h, :nq].astype(np.float64) @ k[b, h // G, :nk].astype(np.float64).T / np.sqrt(D) + tri[:nq, :nk]
            p = np.exp(s - s.max(axis=-1, keepdims=True))
            ref = p @ v[b, h // G, :nk].astype(np.float64) / p.sum(axis=-1, keepdims=True)
            worst = max(worst, float(np.abs(got[b, h, :nq] - ref).max()))
    say("   max-abs err %.3e" % worst)
    assert worst <= tol


@pytest.mark.parametrize("dtype,D", [(capi.BF16, 128), (capi.F16, 64), (capi.F32, 64), (capi.F32, 96)], ids=["bf16_128", "f16_64", "f32_64", "f32_96"])
@pytest.mark.parametrize("shape", [(3, 12, 12, 300, 300, True, None), (40, 4, 1, 500, 130, False, (1, 130)), (3, 44, 4, 200, 200, True, None)])
def test_every_dq_block_is_computed_once(gpu, dtype, D, shape):
    B, Hq, Hkv, Sq, Skv, causal, counts = shape
    q, k, v, go = operands(7 + Sq, dtype, B, Hq, Hkv, Sq, Skv, D)
    lens = None if counts is None else np.linspace(counts[0], counts[1], B).astype(np.int32)
    say("dQ work list %s %s" % (dtypes.NAMES[dtype], shape))
    _, dq, dk, dv = host.sdpa_backward(q, k, v, go, dtype, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens)
    mask = np.zeros((B, 1, 1, Sq, Skv), np.float32)
    if causal:
        mask += np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)
    for b in range(B if lens is not None else 0):
        mask[b, ..., lens[b]:] = -np.inf
    G = Hq // Hkv
    rq, rk, rv = BW.sdpa_backward(q.reshape(B, Hkv, G, Sq, D), k[:, :, None], v[:, :, None], go.reshape(B, Hkv, G, Sq, D), mask=mask)
    tol = 1e-5 if dtype == capi.F32 else 2e-2
    compare("dq", dq, rq.reshape(B, Hq, Sq, D), tol)
    compare("dk", dk, rk.reshape(B, Hkv, Skv, D), tol)
    compare("dv", dv, rv.reshape(B, Hkv, Skv, D), tol)
