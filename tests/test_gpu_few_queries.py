"""The few-queries kernel (one pass over K and V in place, the rows of all query heads of a kv head together) through
``sageattn`` against the oracle, at the sizes where it can go wrong: one query; one, two and three 32-column tiles of
rows; units that leave columns empty (5 or 20 queries), fill a tile exactly (32) or run past it (33); one key, a key
range of one tile, a last tile of one key, fewer key tiles than waves, waves with no tile; both row paths (direct and
INT8), both head dims, dtypes and layouts; key splits up to many per head; head counts that are no power of two.
"""
import numpy as np
import pytest
import torch

from _helpers import Config, make_inputs
from test_gpu_random_shapes import test_random_shape_through_sageattn as check

pytestmark = pytest.mark.gpu


def case(i, B, Hq, Hkv, Sq, S, D, dtype):
    return Config(f"r{i:02d}_B{B}H{Hq}k{Hkv}q{Sq}kv{S}D{D}_{dtype}", B, Hq, Hkv, S, D, dtype, "NHD" if i % 2 else "HND",
                  False, False, Sq=None if Sq == S else Sq)


# (config, INT8 path forced)
CASES = [
    (case(0, 1, 1, 1, 1, 1, 128, "bf16"), True),
    (case(1, 1, 2, 1, 1, 31, 64, "fp16"), True),
    (case(2, 2, 3, 3, 1, 33, 128, "fp16"), False),
    (case(3, 1, 8, 1, 1, 97, 64, "bf16"), False),
    (case(4, 3, 4, 2, 5, 129, 128, "bf16"), True),
    (case(5, 1, 12, 3, 7, 1000, 128, "fp16"), True),
    (case(6, 1, 5, 5, 20, 1025, 64, "bf16"), True),
    (case(7, 1, 6, 3, 20, 640, 128, "bf16"), False),
    (case(8, 1, 2, 2, 32, 2048, 128, "bf16"), True),
    (case(9, 1, 4, 2, 33, 2049, 64, "fp16"), True),
    (case(10, 1, 2, 1, 33, 2049, 128, "fp16"), False),
    (case(11, 2, 2, 2, 64, 1500, 64, "fp16"), False),
    (case(12, 1, 32, 4, 1, 4500, 128, "fp16"), True),
    (case(13, 1, 1, 1, 3, 20000, 128, "bf16"), True),
    (case(14, 1, 1, 1, 1, 20011, 64, "bf16"), True),
    (case(15, 1, 7, 7, 17, 4097, 128, "fp16"), False),
]


@pytest.mark.parametrize("cfg,force_i8", CASES, ids=[c[0].name for c in CASES])
def test_few_queries_against_oracle(cfg, force_i8, monkeypatch):
    monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    check(cfg, force_i8, monkeypatch)


@pytest.mark.parametrize("force_i8", [True, False])
@pytest.mark.parametrize("D", [64, 128])
def test_few_queries_strided_views_and_growing_scores(D, force_i8, monkeypatch):
    """Slices of a packed K/V cache (row pitch above the row), a negative scale, and keys whose scores grow along the
    range (the reference max moves on most tiles), against the general path (the same call with key splits forced,
    which the few-queries kernel does not take): both round P and the output, so 2^-9 + 2^-10 of the value each."""
    from sageattention import sageattn

    for name in ("SAGEATTN_DIRECT_THRESHOLD_D64_CROSS", "SAGEATTN_DIRECT_THRESHOLD_D128_CROSS"):
        monkeypatch.setenv(name, "-1" if force_i8 else "100000")
    cfg = Config("few", 2, 4, 2, 3000, D, "fp16", "HND", False, False, Sq=6)
    q, k, v = make_inputs(cfg, seed=5)
    ramp = torch.linspace(0.1, 6.0, cfg.S)[None, None, :, None]
    cache = torch.zeros(2, 2, 3100, 3 * D, dtype=torch.float16)
    cache[:, :, 50:3050, :D] = (k.float() * ramp).half()
    cache[:, :, 50:3050, 2 * D:] = v
    cache = cache.cuda()
    kk, vv = cache[:, :, 50:3050, :D], cache[:, :, 50:3050, 2 * D:]
    for scale in (D ** -0.5, -0.3):
        monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
        o, lse = sageattn(q.cuda(), kk, vv, sm_scale=scale, return_lse=True)
        monkeypatch.setenv("SAGEATTN_KV_SPLITS", "1")
        w, wl = sageattn(q.cuda(), kk, vv, sm_scale=scale, return_lse=True)
        o, w = o.float().cpu().numpy(), w.float().cpu().numpy()
        assert np.all(np.abs(o - w) <= 2e-3 + 4e-3 * np.abs(w))
        assert torch.allclose(lse, wl, rtol=2e-6, atol=2e-4)


@pytest.mark.parametrize("force_i8", [True, False])
def test_few_queries_graph_capture_and_replay(force_i8, monkeypatch):
    """The launches (attention, merge of the key splits) and the workspace in a HIP graph: every replay, with eager
    work between, gives the eager call's bits."""
    from sageattention import sageattn

    monkeypatch.setenv("SAGEATTN_DIRECT_THRESHOLD_D128_CROSS", "-1" if force_i8 else "100000")
    q, k, v = (t.cuda() for t in make_inputs(Config("few", 2, 8, 2, 6000, 128, "bf16", "HND", False, False, Sq=3), seed=9))
    ref = sageattn(q, k, v)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        sageattn(q, k, v)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sageattn(q, k, v)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        assert torch.equal(sageattn(q, k, v), ref)


@pytest.mark.parametrize("B,H,Sq,Sk,D,dtype,direct", [
    (2, 2, 64, 1500, 64, torch.float16, True),     # few heads, long keys, two row tiles
    (1, 1, 1, 20011, 64, torch.bfloat16, False),   # little K and V in all: many key splits
    (20, 16, 96, 64, 64, torch.bfloat16, True),    # a batch of windows: more blocks than CUs, waves without a tile
    (20, 16, 49, 49, 128, torch.float16, True),
])
def test_few_queries_entry_where_the_general_kernel_is_faster(B, H, Sq, Sk, D, dtype, direct, monkeypatch):
    """Shapes that ``sageattn`` leaves to the general kernel, through the C entry, against ``sageattn``: both round P and
    the output, so 2^-9 + 2^-10 (bf16: 2^-7) of the value each."""
    from sageattention import _capi, ops, sageattn

    for name in ("D64", "D64_CROSS", "D128", "D128_CROSS"):
        monkeypatch.setenv("SAGEATTN_DIRECT_THRESHOLD_" + name, "100000" if direct else "-1")
    monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    g = torch.Generator().manual_seed(Sk)
    q, k, v = (torch.randn(B, H, s, D, generator=g).to(dtype).cuda() for s in (Sq, Sk, Sk))
    w, wl = sageattn(q, k, v, return_lse=True)
    o, lse = torch.full_like(q, float("nan")), torch.full_like(wl, float("nan"))
    ws_bytes = _capi.query("sage_attn_few_workspace_bytes", B, H, H, Sq, Sk, D)
    ws = torch.empty(max(ws_bytes, 16), device="cuda", dtype=torch.uint8)
    strides = [x.stride(i) for x in (q, k, v, o) for i in range(3)]
    _capi.call("sage_attn_few_fwd", 0 if direct else 1, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
               lse.data_ptr(), 1 if dtype == torch.bfloat16 else 0, B, H, H, Sq, Sk, D, *strides, D ** -0.5,
               ws.data_ptr() if ws_bytes else None, ws_bytes, ops._stream(q))
    rtol = 1.6e-2 if dtype == torch.bfloat16 else 4e-3
    assert torch.allclose(o.float(), w.float(), atol=2e-3, rtol=rtol)
    assert torch.allclose(lse, wl, rtol=2e-6, atol=2e-4)
