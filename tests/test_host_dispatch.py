"""The compiled host layer's dispatch: its direct / INT8 choice (default thresholds) equals core.use_direct_path over both
head dims, layouts, causality and lengths around every threshold; which calls take the few-queries kernel
and which bf16 ones read V in place."""
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


def test_few_queries_rule():
    """Calls on both sides of the few-queries rule's lines: decode and short cross-attention take the kernel, batches
    of many short windows (whose blocks it would run in several times the general kernel's rounds), windows of one key
    tile and few heads against long keys do not."""
    from sageattention import core

    few = core._host().few_pays
    takes = [  # batch, q_heads, kv_heads, q_len, kv_len, head_dim, direct
        (8, 32, 8, 1, 8192, 128, False), (4, 32, 4, 8, 16384, 128, False), (4, 16, 16, 128, 4096, 128, False),
        (1, 8, 8, 256, 8192, 128, False), (1, 8, 8, 1, 16384, 64, False), (1, 8, 8, 1, 5000, 64, False),
        (1, 64, 8, 1, 8192, 64, False),
        (16, 16, 16, 1, 256, 64, True), (16, 16, 16, 32, 77, 64, True), (64, 16, 16, 16, 64, 128, True),
        (4, 16, 16, 64, 256, 128, True), (4, 16, 16, 96, 256, 64, True),
        (1, 32, 8, 1, 4096, 64, True), (2, 32, 8, 40, 3000, 128, True), (1, 16, 16, 1, 1, 128, True),
    ]
    general = [
        # windows: many blocks, few keys
        (64, 16, 16, 64, 64, 64, True), (64, 16, 16, 96, 96, 64, True), (64, 16, 16, 49, 49, 64, True),
        (64, 16, 16, 1, 1024, 64, True), (256, 16, 16, 16, 16, 64, True), (64, 16, 16, 96, 96, 128, True),
        (64, 16, 4, 48, 64, 64, True),
        # several row tiles against one key tile
        (4, 16, 16, 64, 64, 64, True), (4, 16, 16, 64, 64, 128, True),
        # few heads, long keys
        (1, 8, 8, 1, 4096, 64, True), (1, 8, 8, 64, 1024, 64, True), (1, 8, 8, 64, 4096, 128, True),
        (1, 4, 4, 1, 8192, 64, False), (1, 4, 4, 128, 8192, 64, False),
        # INT8: four row groups
        (8, 16, 16, 256, 8192, 128, False), (4, 16, 16, 256, 8192, 128, False), (16, 32, 32, 128, 8192, 64, False),
        # too many rows, no work
        (1, 16, 16, 257, 8192, 128, False), (1, 16, 16, 128, 1024, 128, True), (1, 4, 4, 0, 100, 64, True),
        (1, 4, 4, 1, 0, 64, True),
    ]
    for args in takes:
        assert few(*args), args
    for args in general:
        assert not few(*args), args


def test_bf16_v_in_place_rule():
    """Direct path, bf16: V in place on short and causal launches, through the V_T pass where the conversion of the V
    tiles by every query block costs more than the pass."""
    from sageattention import core

    rule = core._host().bf16_v_in_place
    for args in [(1, 16, 16, 4096, 512, 128, False), (1, 32, 32, 2048, 2048, 128, True), (1, 20, 20, 1024, 1024, 64, False),
                 (1, 32, 32, 4096, 4096, 64, True), (1, 1, 1, 1, 1, 64, False), (1, 10, 10, 4096, 77, 64, False),
                 (1, 4, 4, 100, 6144, 64, True), (1, 4, 4, 100, 0, 64, False)]:
        assert rule(*args), args
    for args in [(1, 32, 32, 5529, 6144, 64, False), (1, 32, 8, 5529, 6144, 64, False), (1, 32, 8, 5000, 5000, 64, True),
                 (2, 32, 4, 8192, 2048, 64, False), (2, 32, 4, 8192, 2048, 128, False)]:
        assert not rule(*args), args
