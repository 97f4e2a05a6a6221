"""The work lists of the 16-bit dK/dV kernels: every key block of every (batch, KV head) pair is computed once, whatever the groups of
pairs that share the list (key_groups in sdpa_bwd_mfma.hip): one group, several, a last one that takes what is left, pairs that do and do not divide by
the eight XCDs.  All heads against the float64 oracle; tolerance as in test_gpu_backward.py (16-bit inputs, P and dS, f32 sums)."""
import numpy as np
import pytest

from incin_amd import capi, host
from oracle import sdpa_backward as BW
from tests.test_gpu_backward import compare, make, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, Sq, Skv, D, causal, key counts from - to
    (8, 9, 9, 33, 1100, 128, True, None),          # paired kernel, 9 pairs per XCD: groups of four and five
    (8, 1, 1, 70, 300, 128, True, None),           # one pair per XCD
    (3, 44, 44, 33, 1100, 128, True, None),        # 132 pairs over all XCDs: groups of 64 and 68
    (1, 6, 3, 100, 520, 128, True, None),          # fewer pairs than XCDs, grouped queries
    (24, 3, 3, 33, 1100, 128, False, (1, 1100)),   # key counts: groups of four and five
    (8, 44, 44, 33, 1100, 64, True, None),         # a wavefront per 32 keys, 44 pairs per XCD: two groups of 22
    (68, 2, 2, 40, 300, 64, False, (1, 300)),      # with key counts, 17 pairs per XCD: groups of eight and nine
    (31, 1, 1, 40, 300, 96, False, (0, 300)),      # 31 pairs over all XCDs, a sequence without keys
])
def test_every_key_block_is_computed_once(gpu, shape):
    B, Hq, Hkv, Sq, Skv, D, causal, counts = shape
    say("dK/dV work list: %s" % (shape,))
    q, k, v, go = make(31 + B + Skv, B, Hq, Hkv, Sq, Skv, D, capi.BF16)
    lens = None if counts is None else np.linspace(counts[0], counts[1], B).astype(np.int32)
    _, dq, dk, dv = host.sdpa_backward(q, k, v, go, capi.BF16, impl=capi.IMPL_MFMA, causal=causal, kv_lens=lens)
    mask = np.zeros((B, 1, 1, Sq, Skv), np.float32)
    if causal:
        mask += np.triu(np.full((Sq, Skv), -np.inf, np.float32), 1 + Skv - Sq)
    for b in range(B if lens is not None else 0):
        mask[b, ..., lens[b]:] = -np.inf
    live = np.arange(B) if lens is None else np.flatnonzero(lens)
    G = Hq // Hkv
    rq, rk, rv = BW.sdpa_backward(q[live].reshape(-1, Hkv, G, Sq, D), k[live][:, :, None], v[live][:, :, None], go[live].reshape(-1, Hkv, G, Sq, D), mask=mask[live])
    compare("dq", dq[live], rq.reshape(-1, Hq, Sq, D))
    compare("dk", dk[live], rk.reshape(-1, Hkv, Skv, D))
    compare("dv", dv[live], rv.reshape(-1, Hkv, Skv, D))
    dead = np.setdiff1d(np.arange(B), live)
    assert not dq[dead].any() and not dk[dead].any() and not dv[dead].any()
