"""The work that a user of this library has it do, as cases with sizes: what a time or a gain is quoted on.

Every case goes through a public entry point: the C ABI's forward and backward calls by their ctypes binding (`incin_amd.capi`),
with descriptors that a program makes once and keeps, or the rank-generic operator (`incin_amd.rocm_backend`), which the
reference's caller knows.  A case is a dict of plain values:

  path     "forward" (one launch of the forward), "train" (the forward with its row normalisers, then the backward) or
           "operator" (the operator on storages; `grad`: with the gradients)
  dtype    "bf16", "f16" or "f32"
  B Hq Hkv Sq Skv D   batch, query heads, key / value heads, query positions, key positions (the capacity of a cache), head dimension
  causal   the causal flag
  len_lo len_hi   key counts per sequence, spread evenly from one to the other and dealt to the batch by the seed (0, 0: all keys)
  pad_q    query rows beyond a sequence's count are padding too (a padded batch)
  mask     operator only: "none", "causal" (0 / -inf triangle as a tensor) or "bias" (a distance bias per head under that triangle)
"""
import collections
import math

import torch

from incin_amd import capi, host
from incin_amd import rocm_backend as RB

_TAG = {"f32": capi.F32, "f16": capi.F16, "bf16": capi.BF16}
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_Tensor = collections.namedtuple("_Tensor", "shape dtype dev ptr nbytes")

_FIELDS = ("path", "dtype", "B", "Hq", "Hkv", "Sq", "Skv", "D", "causal", "len_lo", "len_hi", "pad_q", "mask", "grad")


def _case(path, dtype, B, Hq, Hkv, Sq, Skv, D, causal=False, len_lo=0, len_hi=0, pad_q=False, mask="none", grad=False):
    return dict(zip(_FIELDS, (path, dtype, B, Hq, Hkv, Sq, Skv, D, causal, len_lo, len_hi, pad_q, mask, grad)))


def listed():
    return [
        # one user's chat: a token of one sequence, grouped heads, a cache with room left - latency and launches
        dict(_case("forward", "bf16", 1, 32, 8, 1, 4096, 128, len_lo=2085, len_hi=2085), name="decode_one_sequence"),
        # a serving batch in mid-flight: grouped heads, every sequence at a length of its own
        dict(_case("forward", "bf16", 32, 32, 8, 1, 8192, 128, len_lo=1031, len_hi=8192), name="decode_batch_grouped"),
        # a full batch without grouped heads: the decode benchmark
        dict(_case("forward", "bf16", 32, 32, 32, 1, 8192, 128), name="decode_batch_full"),
        # a prompt batch, or the forward of a training step: the prefill benchmark
        dict(_case("forward", "bf16", 8, 16, 16, 4096, 4096, 128, causal=True), name="prefill"),
        # long prompts of different lengths in one padded batch, grouped heads
        dict(_case("forward", "bf16", 4, 32, 8, 16384, 16384, 128, causal=True, len_lo=2048, len_hi=16384, pad_q=True), name="prefill_ragged"),
        # the next chunk of one long prompt over what is cached of it
        dict(_case("forward", "bf16", 1, 32, 8, 512, 32768, 128, causal=True), name="prefill_chunk"),
        # an encoder over image patches: many short sequences of an odd length, nothing masked
        dict(_case("forward", "f16", 64, 12, 12, 197, 197, 64), name="encoder_short"),
        # the operator as the reference's caller states it: f32, the causal mask as a tensor
        dict(_case("operator", "f32", 4, 8, 8, 1024, 1024, 64, mask="causal"), name="operator_f32"),
        # a training step's attention: the forward with row normalisers and the gradients
        dict(_case("train", "bf16", 8, 16, 16, 4096, 4096, 128, causal=True), name="train"),
        # the same in the dtype the reference trains in, at its size
        dict(_case("train", "f32", 4, 8, 8, 1024, 1024, 64, causal=True), name="train_f32"),
        # an encoder's training step: padded sentences, key counts
        dict(_case("train", "bf16", 32, 12, 12, 512, 512, 64, len_lo=61, len_hi=512), name="train_encoder"),
        # a training step with wide heads, grouped
        dict(_case("train", "bf16", 2, 16, 8, 1024, 1024, 256, causal=True), name="train_wide_heads"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(("decode", "decode", "prefill", "prefill_ragged", "chunk", "encoder", "operator", "train", "train", "train_f32", "train_encoder", "train_wide"))
    half = rng.choice(("bf16", "bf16", "f16"))
    hkv, group = rng.choice((1, 2, 4, 8, 8, 16, 32)), rng.choice((1, 1, 2, 4, 4, 8))
    group = min(group, 64 // hkv)
    while True:
        if kind == "decode":
            dtype, D = rng.choice((half, half, half, "f32")), rng.choice((64, 128, 128, 128, 256))
            B, cap = _log(rng, 1, 64), _log(rng, 256, 65536)
            if rng.random() < 0.3:      # a short run of positions checked at once
                c = _case("forward", dtype, B, hkv * group, hkv, rng.choice((2, 4, 5, 8)), cap, D, causal=True)
            else:
                hi = rng.randint(max(1, cap // 2), cap)
                c = _case("forward", dtype, B, hkv * group, hkv, 1, cap, D, len_lo=rng.randint(max(1, hi // 8), hi), len_hi=hi)
        elif kind == "prefill":
            S = _log(rng, 64, 8192)
            c = _case("forward", half, _log(rng, 1, 16), hkv * group, hkv, S, S, rng.choice((64, 80, 96, 128, 128, 128, 256)), causal=rng.random() < 0.8)
        elif kind == "prefill_ragged":
            S = _log(rng, 256, 16384)
            c = _case("forward", half, _log(rng, 2, 16), hkv * group, hkv, S, S, rng.choice((64, 128, 128)), causal=True,
                      len_lo=rng.randint(S // 8, S), len_hi=S, pad_q=True)
        elif kind == "chunk":
            c = _case("forward", half, _log(rng, 1, 4), hkv * group, hkv, _log(rng, 96, 1024), _log(rng, 4096, 65536), rng.choice((64, 128, 128, 256)), causal=True)
        elif kind == "encoder":
            S, h = _log(rng, 16, 1024), rng.choice((8, 12, 16))
            c = _case("forward", half, _log(rng, 8, 256), h, h, S, S, rng.choice((64, 64, 80, 128)))
        elif kind == "operator":
            S, h = _log(rng, 32, 1024), rng.choice((1, 2, 8, 12))
            c = _case("operator", rng.choice(("f32", "f32", half)), _log(rng, 1, 8), h, h, S, S, rng.choice((64, 64, 128)),
                      mask=rng.choice(("none", "causal", "bias")), grad=rng.random() < 0.5)
        elif kind == "train":
            S = _log(rng, 128, 8192)
            c = _case("train", half, _log(rng, 1, 16), hkv * group, hkv, S, S, rng.choice((64, 96, 128, 128)), causal=True)
        elif kind == "train_f32":
            S, h = _log(rng, 64, 2048), rng.choice((4, 8, 12))
            c = _case("train", "f32", _log(rng, 1, 8), h, h, S, S, rng.choice((64, 64, 80, 128)), causal=rng.random() < 0.7)
        elif kind == "train_encoder":
            S, h = _log(rng, 32, 1024), rng.choice((8, 12, 16))
            c = _case("train", half, _log(rng, 4, 128), h, h, S, S, rng.choice((64, 64, 80)), len_lo=rng.randint(max(1, S // 8), S), len_hi=S)
        else:
            S = _log(rng, 128, 4096)
            c = _case("train", half, _log(rng, 1, 8), rng.choice((1, 2, 8)) * group, 1, S, S, rng.choice((160, 192, 256, 256)), causal=rng.random() < 0.8)
            c["Hkv"] = c["Hq"] // group
        w = work(c)
        # none larger than the largest listed of its kind of kernel
        most = 2.5e11 if c["dtype"] == "f32" else 5.5e10 if kind == "train_wide" else 4.2e12 if kind == "prefill_ragged" else 2.0e12
        if w["flops"] <= most and w["bytes"] <= 4.4e9:
            return c


def _lengths(case):
    """Key counts of the batch, before they are dealt: evenly spread."""
    B, lo, hi = case["B"], case["len_lo"], case["len_hi"]
    return [hi if B == 1 else lo + (hi - lo) * b // (B - 1) for b in range(B)] if hi else None


def _gpu(t):
    return _Tensor(tuple(t.shape), {torch.float32: capi.F32, torch.float16: capi.F16, torch.bfloat16: capi.BF16}.get(t.dtype), 0, t.data_ptr(),
                   t.numel() * t.element_size())


def prepare(case, seed):
    if case["path"] == "operator":
        return _prepare_operator(case, seed)
    B, Hq, Hkv, Sq, Skv, D = (case[k] for k in ("B", "Hq", "Hkv", "Sq", "Skv", "D"))
    dt = _TORCH[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):      # what projections of normalised activations look like
        return torch.randn(*shape, generator=g, device="cuda", dtype=dt)

    q, k, v = normal(B, Hq, Sq, D), normal(B, Hkv, Skv, D), normal(B, Hkv, Skv, D)
    o = torch.zeros_like(q)
    st = {"case": case, "q": q, "k": k, "v": v, "o": o, "stream": torch.cuda.current_stream().cuda_stream or None}
    lens = _lengths(case)
    if lens:
        order = torch.randperm(B, generator=torch.Generator().manual_seed(seed)).tolist()
        st["lens"] = torch.tensor([lens[i] for i in order], dtype=torch.int32, device="cuda")
    lens = _gpu(st["lens"]) if lens else None
    train = case["path"] == "train"
    if train:
        st["lse"] = torch.zeros(B, Hq, Sq, device="cuda", dtype=torch.float32)
    fwd = host.make_desc(_gpu(q), _gpu(k), _gpu(v), _gpu(o), causal=case["causal"], kv_lens=lens, q_lens=lens if case["pad_q"] else None,
                         lse=_gpu(st["lse"]) if train else None)
    need = capi.sdpa_workspace(fwd)[0]
    if need:
        st["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
        fwd.workspace, fwd.workspace_bytes = st["workspace"].data_ptr(), need
    st["fwd"] = fwd
    if train:
        bwd = capi.SdpaBwdDesc()
        bwd.fwd = fwd
        st["d_o"] = normal(B, Hq, Sq, D)
        st["d_q"], st["d_k"], st["d_v"] = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for name in ("d_o", "d_q", "d_k", "d_v"):
            setattr(bwd, name, st[name].data_ptr())
            for a in range(3):
                getattr(bwd, name + "_stride")[a] = st[name].stride(a)
        need = capi.sdpa_bwd_workspace(bwd)
        if need:
            st["bwd_workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
            bwd.workspace, bwd.workspace_bytes = st["bwd_workspace"].data_ptr(), need
        st["bwd"] = bwd
    return st


def _prepare_operator(case, seed):
    B, H, S, D = case["B"], case["Hq"], case["Sq"], case["D"]
    dt, tag = _TORCH[case["dtype"]], _TAG[case["dtype"]]
    g = torch.Generator().manual_seed(seed)

    def upload(t):
        t = t.to(dt).contiguous()
        raw = (t if dt == torch.float32 else t.view(torch.int16)).numpy().tobytes()
        return RB.RocmStorage.from_bytes(raw, tuple(t.shape), tag)

    st = {"case": case, "q": None, "k": None, "v": None, "d_o": None}
    for name in ("q", "k", "v", "d_o") if case["grad"] else ("q", "k", "v"):
        st[name] = upload(torch.randn(B, H, S, D, generator=g))
    st["mask"] = None
    if case["mask"] != "none":
        i = torch.arange(S, dtype=torch.float32)
        far = i[:, None] - i[None, :]
        m = torch.zeros(1, 1, S, S) if case["mask"] == "causal" else -far.abs() * (2.0 ** -torch.arange(1.0, H + 1.0)).reshape(1, H, 1, 1)
        st["mask"] = upload(m.masked_fill(far < 0, float("-inf")))
    RB.set_stream(torch.cuda.current_stream().cuda_stream or None)
    return st


class _Kept:
    """A storage of the backend as an array that torch can look at without a copy."""

    def __init__(self, storage, dtype):
        self.storage = storage
        self.__cuda_array_interface__ = {"shape": storage.shape, "typestr": "<f4" if dtype == "f32" else "<i2", "data": (storage.data_ptr, False), "version": 2}


def _seen(storage, dtype):
    t = torch.as_tensor(_Kept(storage, dtype), device="cuda")
    return t if dtype == "f32" else t.view(_TORCH[dtype])


def run(st):
    case = st["case"]
    if case["path"] == "operator":
        if case["grad"]:
            got = RB.attention_backward(st["q"], st["k"], st["v"], st["d_o"], mask=st["mask"])
        else:
            got = (RB.scaled_dot_product_attention(st["q"], st["k"], st["v"], mask=st["mask"]),)
        return [_seen(x, case["dtype"]) for x in got]
    capi.sdpa_fwd(st["fwd"], st["stream"])
    if case["path"] == "forward":
        return st["o"]
    capi.sdpa_bwd(st["bwd"], st["stream"])
    return {name: st[name] for name in ("o", "d_q", "d_k", "d_v")}


def work(case):
    """Each input read once, each output written once; 4 D operations forward and 10 D backward per visible (query, key) pair."""
    B, Hq, Hkv, Sq, Skv, D = (case[k] for k in ("B", "Hq", "Hkv", "Sq", "Skv", "D"))
    size = 4 if case["dtype"] == "f32" else 2
    pairs = rows = keys = 0
    for n in _lengths(case) or [Skv] * B:
        r = min(Sq, n) if case["pad_q"] else Sq
        rows += r
        keys += n
        if case["causal"] or case["mask"] in ("causal", "bias"):
            off = Skv - Sq      # row i sees keys up to i + off
            full = max(0, min(r, n - 1 - off))      # rows that do not reach the last key
            pairs += full * off + full * (full + 1) // 2 + (r - full) * n
        else:
            pairs += r * n
    grad = case["path"] == "train" or case["grad"]
    q, kv = rows * Hq * D * size, keys * Hkv * D * size
    mask = {"none": 0, "causal": 1, "bias": Hq}[case["mask"]] * Sq * Skv * size
    nbytes = 2 * q + 2 * kv + mask
    if grad:      # and dO in, dQ, dK, dV out
        nbytes += 2 * q + 2 * kv
    return {"bytes": nbytes, "flops": (14 if grad else 4) * D * pairs * Hq}


def tolerance(case):
    """About four times what output and gradients were seen to be off from the same formulas in 64 bits on the same stored inputs
    (bf16 2.8e-3 and 3.1e-3 of the 2-norm, f16 3.5e-4 and 4.1e-4, f32 3.1e-7 and 1.4e-6; single values of bf16 gradients 0.09,
    of f16 0.012, of f32 1.9e-5)."""
    if case["dtype"] == "f32":
        return {"rel": 5.5e-6, "max": 8e-5}
    grad = case["path"] == "train" or case["grad"]
    return {"bf16": {"rel": 1.2e-2 if grad else 1.1e-2, "max": 0.35}, "f16": {"rel": 1.6e-3 if grad else 1.4e-3, "max": 0.05}}[case["dtype"]]
