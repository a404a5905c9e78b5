"""The compiled host layer's dispatch (default thresholds) equals core.use_direct_path over both head dims, layouts,
causality and lengths around every threshold."""
import itertools


def test_compiled_dispatch_equals_python(monkeypatch):
    from sageattention import core

    for name in ("D64", "D64_CAUSAL", "D64_CROSS", "D128", "D128_CROSS"):
        monkeypatch.delenv("SAGEATTN_DIRECT_THRESHOLD_" + name, raising=False)
    host = core._host()
    lens = [0, 1, 77, 1023, 1024, 1025, 2047, 2048, 2049, 3071, 3072, 3073, 4095, 4096, 4097, 6143, 6144, 6145, 20000]
    for d, sq, sk, causal, layout in itertools.product((64, 128), lens, lens, (False, True), ("HND", "NHD")):
        want = core.use_direct_path(d, sq, sk, causal, layout)
        assert host.default_direct(d, sq, sk, causal, layout == "HND") == want, (d, sq, sk, causal, layout)
