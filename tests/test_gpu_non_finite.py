"""Infinite and NaN scores through ``sageattn``: keys masked through a channel of K (-inf, or bf16's lowest value against
a query entry of 2, whose product overflows in fp32).  A masked key has weight 0 wherever it lies: whole key tiles, the
first tiles that a wave, a key group or a key split reads, whole splits, all keys (output 0, LSE -inf).  A row whose scores
are NaN gives a NaN output and a NaN LSE, with and without key splits.

References: softmax attention in 64 bits over the same values (direct path), or the same call on the live keys alone
(INT8 path; the masked ranges are whole scale groups, so the live keys quantise alike).  Tolerance: the parity tests'.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
TOL = {"fp16": (2e-3, 4e-3), "bf16": (4e-3, 1.6e-2)}
THRESHOLDS = ["SAGEATTN_DIRECT_THRESHOLD_" + n for n in ("D64", "D64_CAUSAL", "D64_CROSS", "D128", "D128_CROSS")]


def set_path(monkeypatch, direct, splits=None):
    for name in THRESHOLDS:
        monkeypatch.setenv(name, "100000" if direct else "-1")
    if splits is None:
        monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    else:
        monkeypatch.setenv("SAGEATTN_KV_SPLITS", str(splits))


def inputs(B, Hq, Hkv, Sq, Sk, D, dtype, low, seed=3):
    """Small scores; channel 0 masks (q = 2 there, k = 0 for a live key), channel 1 shifts every score by -60 if low."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, h, s, D, generator=g) for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    q[..., :2], k[..., 0], k[..., 1] = torch.tensor([2.0, 1.0]), 0.0, -60.0 if low else 0.0
    q[..., 2:] *= 0.3
    return [x.to(DTYPES[dtype]).cuda() for x in (q, k, v)]


def lowest(dtype):
    return float("-inf") if dtype == "fp16" else torch.finfo(torch.bfloat16).min


def exact(q, k, v, causal, scale=1.0):
    """(output, LSE) in 64 bits; scores past fp32's range are infinite, a row without a live key gives 0 and -inf."""
    B, Hq, Sq, D = q.shape
    Sk, group = k.shape[2], Hq // k.shape[1]
    out = torch.empty(B, Hq, Sq, D, dtype=torch.float64, device="cuda")
    lse = torch.empty(B, Hq, Sq, dtype=torch.float64, device="cuda")
    dead = torch.arange(Sk, device="cuda")[None] > torch.arange(Sq, device="cuda")[:, None]
    for b in range(B):
        for h in range(Hq):
            s = (q[b, h].double() @ k[b, h // group].double().T * scale).float().double()
            if causal:
                s.masked_fill_(dead, float("-inf"))
            m = s.amax(1, keepdim=True).clamp_min(torch.finfo(torch.float32).min)
            p = (s - m).exp()
            total = p.sum(1, keepdim=True)
            out[b, h] = p @ v[b, h // group].half().double() / torch.where(total > 0, total, 1.0)
            lse[b, h] = (m + total.log()).squeeze(1)
    return out, lse


def assert_close(got, want, dtype):
    (o, lse), (w, wl) = got, want
    atol, rtol = TOL[dtype]
    assert torch.equal(torch.isnan(o), torch.isnan(w)) and torch.equal(torch.isnan(lse), torch.isnan(wl))
    assert torch.allclose(o.double(), w.double(), atol=atol, rtol=rtol, equal_nan=True)
    assert torch.allclose(lse.double(), wl.double(), atol=2e-4, rtol=2e-6, equal_nan=True)


@pytest.mark.parametrize("low", [False, True])
@pytest.mark.parametrize("masked", [(0, 40), (0, 129), (2048, 4096), (0, 4096)], ids=lambda m: f"keys{m[0]}-{m[1]}")
@pytest.mark.parametrize("Sq", [4, 32], ids=["one_row_tile", "two_row_tiles"])
@pytest.mark.parametrize("D,dtype", [(64, "fp16"), (64, "bf16"), (128, "fp16"), (128, "bf16")])
def test_few_queries_masked_keys(D, dtype, Sq, masked, low, monkeypatch):
    """The few-queries kernel: a wave's first tile, every wave's first tile, whole key splits, every key."""
    from sageattention import sageattn

    set_path(monkeypatch, direct=True)
    q, k, v = inputs(1, 2, 1, Sq, 4096, D, dtype, low)
    k[:, :, masked[0]:masked[1], 0] = lowest(dtype)
    assert_close(sageattn(q, k, v, sm_scale=1.0, return_lse=True), exact(q, k, v, False), dtype)


@pytest.mark.parametrize("D", [64, 128])
def test_few_queries_masked_keys_int8(D, monkeypatch):
    """INT8 scores overflow to -inf where the K scale is large enough (bf16 only)."""
    from sageattention import sageattn

    set_path(monkeypatch, direct=False)
    q, k, v = inputs(1, 2, 1, 4, 4096, D, "bf16", False)
    q[..., 0] = 20.0
    want = sageattn(q, k[:, :, 64:], v[:, :, 64:], sm_scale=1.0, return_lse=True)
    k[:, :, :64, 0] = lowest("bf16")
    assert_close(sageattn(q, k, v, sm_scale=1.0, return_lse=True), want, "bf16")


# block shapes of the general kernel: 128-row blocks in two key groups (17 key tiles), 128-row blocks (8), 256-row blocks,
# causal 128-row blocks in two key groups, causal 128-row blocks of few key tiles
SHAPES = [(3, 300, 1088, 64, False), (5, 600, 512, 64, False), (3, 300, 700, 128, False), (3, 500, 500, 64, True),
          (3, 500, 500, 128, True), (3, 300, 300, 64, True), (3, 300, 300, 128, True)]


@pytest.mark.parametrize("low", [False, True])
@pytest.mark.parametrize("masked", [(0, 64), (64, 128), (0, 200)], ids=lambda m: f"keys{m[0]}-{m[1]}")
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("H,Sq,Sk,D,causal", SHAPES)
def test_masked_keys(H, Sq, Sk, D, causal, dtype, masked, low, monkeypatch):
    """The general kernel: the first key tile of the item, of its second key group, of both."""
    from sageattention import sageattn

    set_path(monkeypatch, direct=True)
    q, k, v = inputs(1, H, H, Sq, Sk, D, dtype, low)
    k[:, :, masked[0]:masked[1], 0] = lowest(dtype)
    assert_close(sageattn(q, k, v, is_causal=causal, sm_scale=1.0, return_lse=True), exact(q, k, v, causal), dtype)


@pytest.mark.parametrize("masked", [(0, 64), (64, 128)], ids=lambda m: f"keys{m[0]}-{m[1]}")
@pytest.mark.parametrize("H,Sq,Sk,D", [(3, 300, 1088, 64), (5, 600, 512, 64), (3, 300, 700, 128)])
def test_masked_keys_int8(H, Sq, Sk, D, masked, monkeypatch):
    from sageattention import sageattn

    set_path(monkeypatch, direct=False)
    q, k, v = inputs(1, H, H, Sq, Sk, D, "bf16", False)
    q[..., 0] = 20.0
    live = [torch.cat([x[:, :, :masked[0]], x[:, :, masked[1]:]], 2) for x in (k, v)]
    want = sageattn(q, *live, sm_scale=1.0, return_lse=True)
    k[:, :, masked[0]:masked[1], 0] = lowest("bf16")
    assert_close(sageattn(q, k, v, sm_scale=1.0, return_lse=True), want, "bf16")


# (Hq, Hkv, Sq, Sk, D, causal, key splits): few queries with and without key splits, the general kernel unsplit and
# split, causal
NAN_CASES = [(4, 2, 3, 4096, 64, False, None), (4, 2, 3, 4096, 128, False, None), (4, 2, 3, 90, 128, False, None),
             (4, 2, 3, 90, 64, False, None), (4, 2, 300, 1088, 64, False, 1), (4, 2, 300, 1088, 64, False, 3),
             (4, 2, 300, 700, 128, False, 1), (4, 2, 300, 700, 128, False, 3), (4, 2, 300, 300, 128, True, None),
             (4, 2, 300, 300, 64, True, None), (4, 2, 600, 600, 128, True, None), (4, 2, 600, 600, 64, True, None)]
NAN_IDS = [f"H{c[0]}q{c[2]}kv{c[3]}D{c[4]}{'_c' if c[5] else ''}_s{c[6]}" for c in NAN_CASES]


@pytest.mark.parametrize("direct", [True, False])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,Sq,Sk,D,causal,splits", NAN_CASES, ids=NAN_IDS)
def test_nan_query(Hq, Hkv, Sq, Sk, D, causal, splits, dtype, direct, monkeypatch):
    """A query without a defined result stays visible: NaN output and NaN LSE, never the zeros of a row without keys.
    Direct: one NaN in the query.  INT8: an infinite entry (infinite scale of its 32-token group: 0 * inf scores)."""
    from sageattention import sageattn

    set_path(monkeypatch, direct, splits)
    q, k, v = inputs(1, Hq, Hkv, Sq, Sk, D, dtype, False)
    o, lse = (x.clone() for x in sageattn(q, k, v, is_causal=causal, sm_scale=0.3, return_lse=True))
    q[0, 1, 1, 5] = float("nan") if direct else float("inf")
    rows = slice(1, 2) if direct else slice(0, min(Sq, 32))
    o[0, 1, rows], lse[0, 1, rows] = float("nan"), float("nan")
    assert_close(sageattn(q, k, v, is_causal=causal, sm_scale=0.3, return_lse=True), (o, lse), dtype)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,Sq,Sk,D,causal,splits", NAN_CASES, ids=NAN_IDS)
def test_nan_key(Hq, Hkv, Sq, Sk, D, causal, splits, dtype, monkeypatch):
    """A NaN in one key of the direct path reaches the output and the LSE of every row that reads the key."""
    from sageattention import sageattn

    set_path(monkeypatch, True, splits)
    q, k, v = inputs(1, Hq, Hkv, Sq, Sk, D, dtype, False)
    o, lse = (x.clone() for x in sageattn(q, k, v, is_causal=causal, sm_scale=0.3, return_lse=True))
    k[0, 1, 70, 5] = float("nan")
    first = 70 if causal else 0
    o[0, Hq // 2:, first:], lse[0, Hq // 2:, first:] = float("nan"), float("nan")
    assert_close(sageattn(q, k, v, is_causal=causal, sm_scale=0.3, return_lse=True), (o, lse), dtype)
