"""Launch shapes of the decode projections (``qwen_hip.ops``): host arithmetic only."""

import copy
import json
import os
import pickle

import pytest

from qwen_hip import _lib, ops

needs_lib = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libqwen_hip.so not built")

QKV, O, GU, DOWN = (6144, 2560, False), (2560, 4096, False), (19456, 2560, True), (2560, 9728, False)


@pytest.mark.parametrize("M", range(1, 33))
def test_choice_by_value_is_the_general_launch(M):
    """By value a shape is always ``(ntw, waves, ksplit)`` or ``(ntw, waves, gn, gk)`` of the general launches, in
    the table's M classes, whether or not the stream is the faster launch."""
    i = 0 if M <= 16 else (1 if M <= 24 else 2)
    want = {QKV: ((2, 8, 1), (2, 4, 1), (4, 4, 2))[i], O: ((1, 8, 1), (2, 8, 3), (2, 4, 3))[i],
            GU: ((2, 8, 1), (2, 16, 256, 1), (2, 16, 256, 1))[i], DOWN: (2, 4, 3) if M > 1 else (1, 16, 1)}
    for (N, K, pair), shape in want.items():
        cfg = ops.gemm_config(M, N, K, pair)
        assert cfg == shape and tuple(cfg) == shape and len(cfg) == len(shape)
        assert isinstance(cfg, ops.StreamShape) == (M >= 3 and (N, K, pair) != DOWN)


def test_stream_shape_survives_copies():
    cfg = ops.gemm_config(20, *GU)
    for c in (copy.copy(cfg), copy.deepcopy(cfg), pickle.loads(pickle.dumps(cfg))):
        assert isinstance(c, ops.StreamShape) and c == cfg and c.nt == cfg.nt == 6
    assert repr(cfg) == "StreamShape(6, (2, 16, 256, 1))"


def test_kernel_names_of_every_form():
    name = ops.gemm_kernel_name
    assert name(8, ops.gemm_config(8, *GU), True, ops.EPI_SWIGLU) == "decode_gemm_kernel<1, 6, 4, 2, 4, true, 2>"
    assert name(20, (6,), True, ops.EPI_SWIGLU) == "decode_gemm_kernel<2, 6, 4, 2, 3, true, 2>"
    assert name(20, (1,), False, ops.EPI_RES) == "decode_gemm_kernel<2, 1, 8, 1, 5, false, 1>"
    assert name(32, tuple(ops.gemm_config(32, *GU)), True, ops.EPI_SWIGLU) == "rect_gemm_kernel<2, 2, 16, true, 2>"
    assert name(32, ops.gemm_config(32, *DOWN), False, ops.EPI_RES) == "skinny_gemm_kernel<2, 2, 4, false, 1>"
    assert name(4, (1, 8, 0), False, ops.EPI_STORE) == "sk_gemm_kernel<1, 1, false, 0>"


@needs_lib
def test_workspace_of_every_form():
    for M in (3, 16, 20, 32):
        for N, K, pair in (QKV, O, GU, DOWN):
            cfg = ops.gemm_config(M, N, K, pair)
            assert ops.gemm_workspace_bytes(M, N, cfg) == ops.gemm_workspace_bytes(M, N, tuple(cfg))
    assert ops.gemm_workspace_bytes(32, 6144, ops.gemm_config(32, *QKV)) > 0
    assert ops.gemm_workspace_bytes(32, 6144, (2,)) == 0


def test_measured_traffic_is_of_the_launches_that_run():
    """``bench.py`` looks measured HBM bytes up by the kernel's name: the committed names are those that the
    MFMA projections launch now (M = sequences x tokens per step; the other entries are GEMVs and attention)."""
    import bench
    with open(bench.TRAFFIC_FILE) as f:
        traffic = json.load(f)
    roles = {"gu": (GU, True, ops.EPI_SWIGLU), "o": (O, False, ops.EPI_RES), "qkv": (QKV, True, ops.EPI_STORE),
             "down": (DOWN, False, ops.EPI_RES)}
    rows = {"c3": 8, "c4": 32, "c5": 4 * bench.SPEC_T}
    seen = 0
    for key, entry in traffic.items():
        config, _, role = key.partition("_")
        if config not in rows or key == "c4":   # (c4's own entry is the attention's)
            continue
        shape, norm, epi = roles[role or "gu"]
        M = rows[config]
        name = ops.gemm_kernel_name(M, ops.gemm_config(M, *shape), norm, epi)
        assert entry["kernel"] == name, key
        assert bench.measured_traffic(key, name) == entry["bytes_per_launch"]
        seen += 1
    assert seen == 6
