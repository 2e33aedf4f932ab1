"""The weight-stream projections (``qwen_linear_stream``): every row count around its 16-row tiles, n-tile counts
that fill and do not fill the last workgroup, fewer and more k stages than the LDS ring holds.

Bar: an fp32 product of the same (normed, rounded) rows. One bf16 rounding (2^-8 relative) of a sum whose fp32
error is at most K 2^-24 times the sum of the products' magnitudes; where the sum is rounded before SwiGLU or
the residual add, an fp32 difference can flip that rounding by a whole ulp, 2^-7 of the part.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
DEV = "cuda:0"
EPS = 1e-6


@pytest.fixture(scope="module")
def qops():
    from qwen_hip import ops
    return ops


def _case(qops, M, N, K, kind, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.03).to(BF16)
    gain = (1 + 0.2 * torch.randn(K, generator=g, device=DEV)).to(BF16)
    res = torch.randn(M, N, generator=g, device=DEV).to(BF16)
    xn = qops.rms_norm(x, gain, EPS) if kind in ("norm", "silu") else x
    acc = xn.float() @ w.float().T
    err = K * 2.0 ** -24 * (xn.float().abs() @ w.float().abs().T)
    if kind in ("norm", "silu"):
        # the kernel's sum of squares is ordered otherwise than rms_norm's: an element may round to its neighbour
        err = err + 2.0 ** -8 * (xn.float().abs() @ w.float().abs().T) / K ** 0.5
    if kind == "silu":
        gate, up = acc.to(BF16).float().chunk(2, dim=1)
        want = torch.nn.functional.silu(gate).to(BF16).float() * up
        eg, eu = (err + 2.0 ** -7 * acc.abs()).chunk(2, dim=1)
        bar = 2.0 ** -7 * want.abs() + (1.2 * eg + 2.0 ** -8 * gate.abs()) * up.abs() + gate.abs() * eu + 1e-5
    elif kind == "res":
        want = res.float() + acc.to(BF16).float()
        bar = 2.0 ** -8 * want.abs() + err + 2.0 ** -7 * acc.abs()
    else:
        want, bar = acc, 2.0 ** -8 * acc.abs() + err
    t = qops.tile_weight(w, pair=kind == "silu")
    return x, t, gain, res, want, bar


def _run(qops, x, t, gain, res, kind, nt):
    out = torch.full((x.shape[0] + 2, t.N // 2 if kind == "silu" else t.N), 5.0, dtype=BF16, device=DEV)
    psq = torch.full((x.shape[0], t.N // 16), -1.0, device=DEV) if kind == "res" else None
    o = out[:x.shape[0]]
    if kind == "res":
        o.copy_(res)
    qops.fused_linear(x, t, (nt,), norm_w=gain if kind in ("norm", "silu") else None, eps=EPS,
                      residual=o if kind == "res" else None, silu_pair=kind == "silu", out=o, psq_out=psq)
    assert bool((out[x.shape[0]:] == 5.0).all()), "rows past M were written"
    return o, psq


@pytest.mark.parametrize("M", [1, 3, 8, 15, 16, 17, 20, 31, 32])
@pytest.mark.parametrize("kind,N,K,nt", [
    ("norm", 6144, 2560, 2), ("res", 2560, 4096, 1), ("silu", 19456, 2560, 6),     # the Qwen3-4B projections
    ("plain", 208, 256, 6), ("silu", 224, 512, 6), ("norm", 48, 2304, 2),           # a last workgroup of 1, 2, 1 tiles
    ("plain", 48, 8192, 1), ("res", 192, 1280, 6), ("silu", 64, 256, 2),
])
def test_stream_matches_fp32(qops, M, kind, N, K, nt):
    x, t, gain, res, want, bar = _case(qops, M, N, K, kind, seed=M + N + K)
    got, psq = _run(qops, x, t, gain, res, kind, nt)
    assert bool(((got.float() - want).abs() <= bar).all()), float(((got.float() - want).abs() - bar).max())
    if kind == "res":   # the next norm's statistics: of the rounded rows, 16 columns each
        sq = got.float().pow(2).view(M, -1, 16).sum(-1)
        assert torch.allclose(psq, sq, rtol=16 * 2.0 ** -23, atol=0)


def test_stream_residual_off_a_4_byte_boundary(qops):
    """A residual (and output) whose rows start at odd multiples of 2 bytes."""
    M, N, K = 20, 256, 512
    x, t, gain, res, want, bar = _case(qops, M, N, K, "res", seed=7)
    base, _ = _run(qops, x, t, gain, res, "res", 1)
    odd = torch.empty(M * N + 1, dtype=BF16, device=DEV)[1:].view(M, N)
    odd.copy_(res)
    assert odd.data_ptr() % 4 == 2
    got = qops.fused_linear(x, t, (1,), residual=odd, out=odd)
    assert torch.equal(got, base)


def test_stream_is_the_choice_for_qwen_projections(qops):
    for M in (3, 20, 32):
        for N, K, pair, nt in ((6144, 2560, False, 2), (2560, 4096, False, 1), (19456, 2560, True, 6)):
            cfg = qops.gemm_config(M, N, K, pair)
            assert isinstance(cfg, qops.StreamShape) and cfg.nt == nt
        down = qops.gemm_config(M, 2560, 9728)
        assert len(down) == 3 and not isinstance(down, qops.StreamShape)


@pytest.mark.parametrize("M", [8, 20, 32])
@pytest.mark.parametrize("kind,N,K", [("norm", 6144, 2560), ("res", 2560, 4096), ("silu", 19456, 2560)])
def test_plain_copy_of_the_choice(qops, M, kind, N, K):
    """A plain tuple with the values of the chosen shape is the general launch of the same projection, and
    ``gemm_workspace_bytes`` of the chosen shape is enough for it."""
    x, t, gain, res, want, bar = _case(qops, M, N, K, kind, seed=M + K)
    cfg = qops.gemm_config(M, N, K, kind == "silu")
    ws = qops.linear_workspace(qops.gemm_workspace_bytes(M, N, cfg), DEV)
    for c in (cfg, tuple(cfg)):
        got = qops.fused_linear(x, t, c, norm_w=gain if kind in ("norm", "silu") else None, eps=EPS,
                                residual=res if kind == "res" else None, silu_pair=kind == "silu", workspace=ws)
        assert bool(((got.float() - want).abs() <= bar).all()), (c, float(((got.float() - want).abs() - bar).max()))


@pytest.mark.parametrize("kind,N,K,nt", [("plain", 64, 320, 1), ("res", 64, 256, 6), ("silu", 64, 256, 1),
                                         ("norm", 64, 8448, 1), ("plain", 64, 256, 3)])
def test_stream_rejects_unfit_shapes(qops, kind, N, K, nt):
    x, t, gain, res, _, _ = _case(qops, 4, N, K, "silu" if kind == "silu" else "plain", seed=1)
    with pytest.raises(RuntimeError):
        _run(qops, x, t, gain, res, kind, nt)


@pytest.mark.parametrize("off", [1, 2, 4, 7])
@pytest.mark.parametrize("kind,N,K,nt", [("norm", 512, 1280, 2), ("res", 256, 512, 1), ("silu", 384, 256, 6)])
@pytest.mark.parametrize("M", [3, 20])
def test_stream_operands_off_a_16_byte_boundary(qops, M, kind, N, K, nt, off):
    """Rows and weights that start at any bf16 element: the stream hands these on, the result is held to the same bar."""
    x, t, gain, res, want, bar = _case(qops, M, N, K, kind, seed=M + off)

    def shifted(v):
        flat = torch.empty(v.numel() + off, dtype=BF16, device=DEV)[off:]
        assert flat.data_ptr() % 16 == 2 * off
        return flat.view(v.shape).copy_(v)

    ts = qops.TiledWeight(shifted(t.data), N, K, t.pair)
    for xx, tt in ((shifted(x), t), (x, ts), (shifted(x), ts)):
        got, _ = _run(qops, xx, tt, gain, res, kind, nt)
        assert bool(((got.float() - want).abs() <= bar).all()), float(((got.float() - want).abs() - bar).max())
