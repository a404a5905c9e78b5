"""Host validation of the few-queries entry points and of the bf16 in-place-V one: every refusal comes back as a status
with its message before anything is launched, sizes past the kernel's limits included; no work is OK."""
import ctypes

import pytest
import torch

from sageattention import _capi

FAKE, ODD, NULL = ctypes.c_void_p(0x10000), ctypes.c_void_p(0x10001), ctypes.c_void_p(0)  # never dereferenced


@pytest.fixture(scope="module")
def lib():
    return _capi.load()


def few(lib, **kw):
    a = dict(quant=1, q=FAKE, k=FAKE, v=FAKE, o=FAKE, lse=NULL, dtype=0, B=1, Hq=4, Hkv=2, Sq=2, Sk=64, D=128, qsb=1024,
             qsh=256, qsn=128, ksb=16384, ksh=8192, ksn=128, vsb=16384, vsh=8192, vsn=128, osb=1024, osh=256, osn=128,
             sm=0.1, ws=NULL, wsb=0)
    a.update(kw)
    return lib.sage_attn_few_fwd(*a.values(), NULL)


@pytest.mark.parametrize("kw,code,msg", [
    (dict(dtype=2), _capi.ERR_INVALID_ARG, "dtype"),
    (dict(D=96), _capi.ERR_UNSUPPORTED, "head_dim"),
    (dict(Hkv=3), _capi.ERR_INVALID_ARG, "multiple of kv_heads"),
    (dict(Hkv=0), _capi.ERR_INVALID_ARG, "size"),
    (dict(Sk=0), _capi.ERR_INVALID_ARG, "size"),
    (dict(B=-1), _capi.ERR_INVALID_ARG, "size"),
    (dict(k=NULL), _capi.ERR_INVALID_ARG, "null pointer"),
    (dict(v=ODD), _capi.ERR_ALIGNMENT, "aligned"),
    (dict(lse=ODD), _capi.ERR_ALIGNMENT, "aligned"),
    (dict(qsn=132), _capi.ERR_ALIGNMENT, "strides"),
    (dict(osh=-256), _capi.ERR_INVALID_ARG, "strides"),
    (dict(ksn=64), _capi.ERR_INVALID_ARG, "overlap"),
    (dict(vsn=64), _capi.ERR_INVALID_ARG, "overlap"),
    (dict(Sq=5000), _capi.ERR_UNSUPPORTED, "limits"),
    (dict(Sk=2 ** 24, ksn=128), _capi.ERR_UNSUPPORTED, "limits"),
    (dict(Sk=2 ** 31 - 1, ksn=128), _capi.ERR_UNSUPPORTED, "limits"),
    (dict(B=2 ** 20, Hq=4), _capi.ERR_UNSUPPORTED, "limits"),
    (dict(Sk=65536), _capi.ERR_INVALID_ARG, "workspace"),
])
def test_few_validation(lib, kw, code, msg):
    assert few(lib, **kw) == code
    assert msg in lib.sage_last_error().decode()


def test_few_zero_work_is_ok(lib):
    assert few(lib, B=0) == _capi.OK
    assert few(lib, Sq=0) == _capi.OK


def test_few_workspace(lib):
    ws = lib.sage_attn_few_workspace_bytes
    assert ws(1, 4, 2, 1, 64, 128) == 0          # too short to split
    assert ws(0, 4, 2, 1, 8192, 128) == ws(1, 4, 2, 0, 8192, 128) == ws(1, 4, 2, 1, 0, 128) == 0
    assert ws(1, 4, 3, 1, 64, 128) == _capi.ERR_INVALID_ARG
    assert ws(1, 4, 2, 1, 64, 32) == _capi.ERR_UNSUPPORTED


@pytest.mark.skipif(torch.cuda.is_available(), reason="key splits depend on the device's CU count")
def test_few_workspace_for_256_cus(lib):
    """Without a device the plan assumes MI355X's 256 CUs: 64 kv heads take 4 key splits of one 32-row tile."""
    assert lib.sage_attn_few_workspace_bytes(8, 32, 8, 1, 8192, 128) == 64 * 4 * 32 * 129 * 4


@pytest.mark.parametrize("kw,code,msg", [
    (dict(q=NULL), _capi.ERR_INVALID_ARG, "null pointer"),
    (dict(v=ODD), _capi.ERR_ALIGNMENT, "value"),
    (dict(vsn=32), _capi.ERR_INVALID_ARG, "V rows must not overlap"),
    (dict(vsn=132), _capi.ERR_ALIGNMENT, "value strides"),
    (dict(D=80), _capi.ERR_UNSUPPORTED, "head_dim"),
    (dict(Sk=2 ** 25), _capi.ERR_UNSUPPORTED, "32-bit"),
])
def test_direct_vrows_bf16_validation(lib, kw, code, msg):
    a = dict(q=FAKE, k=FAKE, v=FAKE, o=FAKE, lse=NULL, B=1, Hq=4, Hkv=2, Sq=64, Sk=64, D=64, qsb=16384, qsh=4096, qsn=64,
             ksb=8192, ksh=4096, ksn=64, vsb=8192, vsh=4096, vsn=64, osb=16384, osh=4096, osn=64, causal=0, sm=0.1,
             splits=1, ws=NULL, wsb=0)
    a.update(kw)
    assert lib.sage_attn_direct_fwd_vrows_bf16(*a.values(), NULL) == code
    assert msg in lib.sage_last_error().decode()
