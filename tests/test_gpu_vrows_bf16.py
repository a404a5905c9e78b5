"""bf16 V read in place (converted to fp16 in LDS) by the direct kernel against the V_T path, bit for bit, through the
C ABI: the three block shapes (256-row, 128-row, two key groups), ring depths, ragged ends, one tile, key
splits, causal and not, grouped heads, a strided V; values that overflow fp16 (in one column of one head, so that the
rest of the output stays comparable) become infinite on both paths."""
import pytest
import torch

from _helpers import Config, make_inputs

pytestmark = pytest.mark.gpu


def case(B, Hq, Hkv, Sq, S, D, layout, causal):
    return Config(f"B{B}H{Hq}k{Hkv}q{Sq}kv{S}D{D}_{layout}{'_c' if causal else ''}", B, Hq, Hkv, S, D, "bf16", layout,
                  causal, False, Sq=None if Sq == S else Sq)


CASES = [
    case(1, 2, 2, 40, 1, 128, "HND", False),
    case(1, 3, 1, 100, 65, 64, "NHD", False),
    case(1, 4, 2, 300, 513, 128, "NHD", False),
    case(1, 10, 10, 700, 154, 64, "NHD", False),
    case(1, 5, 5, 900, 1100, 64, "HND", False),
    case(2, 20, 20, 1000, 700, 64, "HND", False),
    case(1, 6, 3, 777, 777, 128, "HND", True),
    case(1, 3, 3, 130, 2000, 128, "NHD", True),
    case(1, 7, 7, 1021, 1021, 64, "NHD", True),
    case(1, 34, 34, 2300, 2300, 128, "HND", True),
    case(1, 33, 33, 2100, 1300, 128, "HND", False),
]


def both_paths(cfg, splits, overflow):
    """(o, lse) in place and by way of V_T."""
    from sageattention import _capi, ops

    print(f"[bf16 v rows] {cfg.name} splits={splits} overflow={overflow}", flush=True)
    q, k, v = (t.cuda() for t in make_inputs(cfg, seed=11))
    lay = ops.HND if cfg.layout == "HND" else ops.NHD
    if overflow:
        (v if lay == ops.HND else v.transpose(1, 2))[0, -1, ::7, 3] = 1e6  # past fp16's range
    wide = torch.zeros(v.shape[:-1] + (2 * cfg.D,), device="cuda", dtype=v.dtype)
    wide[..., 8: 8 + cfg.D] = v
    v = wide[..., 8: 8 + cfg.D]
    causal, sm = int(cfg.causal), cfg.D ** -0.5
    vt = torch.empty(cfg.B, cfg.Hkv, cfg.D, (cfg.S + 63) // 64 * 64, device="cuda", dtype=torch.float16)
    ops.v_transpose(v, vt, lay)
    o_ref, o = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    lse_ref = torch.full((cfg.B, cfg.Hq, cfg.q_len), float("nan"), device="cuda")
    lse = torch.full_like(lse_ref, float("nan"))
    sq, sk, sv, so = ([x.stride(0)] + ([x.stride(1), x.stride(2)] if lay == ops.HND else [x.stride(2), x.stride(1)])
                      for x in (q, k, v, o))
    ws_bytes = 0 if cfg.causal else _capi.query("sage_attn_workspace_bytes", 0, cfg.B, cfg.Hq, cfg.q_len,
                                                cfg.S, cfg.D, 0, splits)
    ws = torch.empty(max(ws_bytes, 16), device="cuda", dtype=torch.uint8)
    sizes = (cfg.B, cfg.Hq, cfg.Hkv, cfg.q_len, cfg.S, cfg.D)
    tail = (causal, sm, splits, ws.data_ptr() if ws_bytes else None, ws_bytes, ops._stream(q))
    ops.bf16_attn_t(q, k, vt, o_ref, lay, causal, sm, 0, lse=lse_ref, num_splits=splits)
    _capi.call("sage_attn_direct_fwd_vrows_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
               lse.data_ptr(), *sizes, *sq, *sk, *sv, *so, *tail)
    torch.cuda.synchronize()
    return o, lse, o_ref, lse_ref


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("cfg", CASES, ids=lambda c: c.name)
def test_bf16_v_in_place_equals_vt_path(cfg, splits):
    o, lse, o_ref, lse_ref = both_paths(cfg, splits, False)
    assert torch.isfinite(o_ref).all() and torch.isfinite(lse_ref).all()
    assert torch.equal(o, o_ref) and torch.equal(lse, lse_ref)


@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("cfg", CASES, ids=lambda c: c.name)
def test_bf16_v_in_place_overflow(cfg, splits):
    o, lse, o_ref, lse_ref = both_paths(cfg, splits, True)
    # one column of the query heads of one kv head of the first batch is infinite (NaN where P is 0 there)
    bad = ~torch.isfinite(o_ref)
    share = (cfg.Hq // cfg.Hkv) / (cfg.B * cfg.Hq * cfg.D)
    assert 0 < bad.float().mean().item() <= share * (1 + 1e-6)
    assert torch.equal(torch.isnan(o), torch.isnan(o_ref))
    assert torch.equal(torch.nan_to_num(o.float()), torch.nan_to_num(o_ref.float()))
    assert torch.equal(lse, lse_ref)


@pytest.mark.parametrize("causal", [False, True])
def test_sageattn_across_the_in_place_line(causal, monkeypatch):
    """``sageattn`` on a launch that takes the V_T pass against the entry that reads V in place: the same bits."""
    from sageattention import _capi, core, ops, sageattn

    for name in ("D64", "D64_CAUSAL", "D64_CROSS"):
        monkeypatch.delenv("SAGEATTN_DIRECT_THRESHOLD_" + name, raising=False)
    monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    B, Hq, Hkv, Sq, Sk, D = (1, 16, 1, 4001 if causal else 2700, 4001 if causal else 3000, 64)
    assert not core._host().bf16_v_in_place(B, Hq, Hkv, Sq, Sk, D, causal)
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(B, h, s, D, generator=g).bfloat16().cuda() for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    ref, lse_ref = sageattn(q, k, v, is_causal=causal, return_lse=True)
    o, lse = torch.full_like(q, float("nan")), torch.full_like(lse_ref, float("nan"))
    ws_bytes = 0 if causal else _capi.query("sage_attn_workspace_bytes", 0, B, Hq, Sq, Sk, D, 0, 0)
    ws = torch.empty(max(ws_bytes, 16), device="cuda", dtype=torch.uint8)
    strides = [x.stride(i) for x in (q, k, v, o) for i in range(3)]
    _capi.call("sage_attn_direct_fwd_vrows_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
               B, Hq, Hkv, Sq, Sk, D, *strides, int(causal), D ** -0.5, 0, ws.data_ptr() if ws_bytes else None, ws_bytes,
               ops._stream(q))
    assert torch.equal(o, ref) and torch.equal(lse, lse_ref)
