"""Scores far larger than their differences: the kernels take a score relative to the row's reference max with one
rounding (an FMA of the exact integer dot product), so P is as exact as for small scores.

Integer-valued Q and K whose dot products (about 2^20 to 2^21, partial sums included) are exact in fp32; the keys of a
row differ by a few units.  A score rounded before the max is taken off is off by up to 2^-4 here, and P by 4%.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direct", [True, False])
@pytest.mark.parametrize("Sq", [1, 5, 400], ids=["few1", "few5", "general"])
@pytest.mark.parametrize("Sk", [8, 40, 700])
@pytest.mark.parametrize("D,dtype", [(64, "fp16"), (128, "bf16")])
def test_large_scores(D, dtype, Sk, Sq, direct, monkeypatch):
    from sageattention import sageattn

    for n in ("D64", "D64_CAUSAL", "D64_CROSS", "D128", "D128_CROSS"):
        monkeypatch.setenv("SAGEATTN_DIRECT_THRESHOLD_" + n, "100000" if direct else "-1")
    monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    g = torch.Generator().manual_seed(Sk + Sq)
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    q = torch.full((1, 2, Sq, D), 127.0)
    q[..., D - 1] = 1.0
    k = torch.full((1, 2, Sk, D), 127.0)
    k[..., D - 1] = -torch.randint(0, 9, (1, 2, Sk), generator=g).float()
    v = torch.rand(1, 2, Sk, D, generator=g) * 2 - 1
    sm = 0.6
    o = sageattn(q.to(dt).cuda(), k.to(dt).cuda(), v.to(dt).cuda(), sm_scale=sm)
    # the scale of a score in log2 units; INT8: q_scale * k_scale with k_scale 1 and q_scale = absmax / 127, all in fp32
    sc = torch.tensor(sm, dtype=torch.float32) * torch.tensor(1.4426950408889634, dtype=torch.float32)
    if not direct:
        sc = sc * 127 / 127
    p = torch.exp2(k[..., D - 1].double() * sc.double())  # the common part of the scores cancels
    want = (p[:, :, None] @ v.to(dt).half().double()) / p.sum(-1)[..., None, None]
    # |v| <= 1: P to fp16 (2^-11 of each weight, in the sum of weights too) and the output to its dtype
    tol = 2 * 2.0 ** -11 + (2.0 ** -11 if dtype == "fp16" else 2.0 ** -9)
    err = (o.double().cpu() - want).abs().max().item()
    assert err <= tol, f"max error {err:.2e} > {tol:.2e}"
