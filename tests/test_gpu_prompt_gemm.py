"""The prompt GEMM's output tiles (``qwen_gemm`` picks one by M, N and K): every row count around the tile
edges against a launch of many rows.

An output element accumulates its k range in the same order in every tile, so the first M rows of a launch
do not depend on M: bit for bit the same. The many-row result itself is held to an fp32 product: one
bf16 rounding (2^-8 relative) of a sum whose fp32 error is at most K 2^-24 times the sum of the
products' magnitudes. SwiGLU and the residual work on sums that are rounded first: an fp32 difference can
flip such a rounding by a whole ulp, 2^-7 of the part.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
DEV = "cuda:0"
ROWS = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 255, 256, 257, 384, 511, 513, 769, 1024, 1025, 1500]


@pytest.fixture(scope="module")
def qops():
    from qwen_hip import ops
    return ops


def _inputs(N, K, M, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.03).to(BF16)
    res = torch.randn(M, N, generator=g, device=DEV).to(BF16)
    return x, w, res


def _bar(x, w, res, kind):
    """The fp32 product of the operands and what a correct launch may differ from it by."""
    acc = x.float() @ w.float().T
    err = x.shape[1] * 2.0 ** -24 * (x.float().abs() @ w.float().abs().T)
    if kind == "silu":
        gate, up = acc.to(BF16).float().chunk(2, dim=1)
        want = (torch.nn.functional.silu(gate).to(BF16).float() * up)
        eg, eu = (err + 2.0 ** -7 * acc.abs()).chunk(2, dim=1)
        bar = 2.0 ** -7 * want.abs() + (1.2 * eg + 2.0 ** -8 * gate.abs()) * up.abs() + gate.abs() * eu + 1e-5
    elif kind == "res":
        want = res.float() + acc.to(BF16).float()
        bar = 2.0 ** -8 * want.abs() + err + 2.0 ** -7 * acc.abs()
    else:
        want, bar = acc, 2.0 ** -8 * acc.abs() + err
    return want, bar


# Qwen3-4B widths; K of one 64-step, an odd number of them, and one that is not a multiple of 128; N that
# only the 128-, 64- or 32-column tiles divide
@pytest.mark.parametrize("kind,N,K", [("plain", 6144, 2560), ("res", 2560, 4096), ("res", 2560, 9728),
                                      ("silu", 19456, 2560), ("plain", 256, 64), ("res", 512, 192),
                                      ("silu", 1024, 1088), ("plain", 384, 640), ("silu", 640, 128)])
def test_rows_do_not_depend_on_the_tile(qops, kind, N, K):
    top = 2113
    x, w, res = _inputs(N, K, top, seed=N + K)
    t = qops.tile_weight(w, pair=kind == "silu")

    def call(m, out=None):
        return qops.gemm(x[:m], t, residual=res[:m] if kind == "res" else None, silu_pair=kind == "silu", out=out)

    many = call(top)
    want, bar = _bar(x, w, res, kind)
    assert bool(((many.float() - want).abs() <= bar).all()), float(((many.float() - want).abs() - bar).max())
    ncols = many.shape[1]
    for m in ROWS:
        buf = torch.full((m + 3, ncols), 7.0, dtype=BF16, device=DEV)
        call(m, out=buf[:m])
        assert torch.equal(buf[:m], many[:m]), f"{kind} N={N} K={K}: {m} rows differ from the same rows of {top}"
        assert bool((buf[m:] == 7.0).all()), f"rows past {m} were written"


# A persistent workgroup goes from one output tile to the next with the next one's loads already in flight, and the
# residual loads and the stores of the epilogue fall between them. (kind, N, K, rows, tile, tiles of the busiest
# workgroup), on 256 CUs.
ROUNDS = [("res", 2560, 4096, 3100, (128, 128), 2), ("res", 2560, 4096, 3300, (256, 256), 1),
          ("res", 2560, 4096, 6450, (128, 128), 4), ("res", 2560, 4096, 6600, (256, 128), 3),
          ("res", 2560, 4096, 9800, (256, 256), 2), ("res", 2560, 9728, 3073, (128, 128), 2),
          ("res", 2560, 9728, 6529, (256, 128), 3), ("res", 2560, 9728, 10241, (256, 256), 2),
          ("plain", 6144, 2560, 2600, (128, 128), 4), ("plain", 6144, 2560, 2700, (256, 128), 3),
          ("plain", 6144, 2560, 4100, (256, 256), 2), ("silu", 19456, 2560, 300, (128, 128), 2),
          ("silu", 19456, 2560, 800, (256, 128), 3), ("silu", 19456, 2560, 1600, (256, 256), 3),
          ("res", 16384, 128, 256, (64, 128), 2), ("res", 16384, 192, 3000, (256, 256), 3),
          ("res", 32896, 4096, 11, (32, 64), 3), ("res", 65536, 4096, 11, (32, 128), 2)]


@pytest.mark.parametrize("kind,N,K,M,tile,rounds", ROUNDS)
def test_several_tiles_of_a_workgroup(qops, kind, N, K, M, tile, rounds):
    """Every element against an fp32 product, and bit for bit against launches of at most 512 of the rows; the residual
    in place and from a tensor of its own."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert qops.gemm_tile(M, N, K) == tile, "the tile choice changed: choose rows that reach this tile again"
        run = -(-(-(-M // tile[0]) * (N // tile[1])) // 8)
        assert -(-run // 32) == rounds
    x, w, res = _inputs(N, K, M, seed=M + N)
    t = qops.tile_weight(w, pair=kind == "silu")

    def call(rows, out=None, r=res):
        return qops.gemm(x[rows], t, residual=r[rows] if kind == "res" else None, silu_pair=kind == "silu", out=out)

    got = call(slice(0, M))
    want, bar = _bar(x, w, res, kind)
    assert bool(((got.float() - want).abs() <= bar).all()), float(((got.float() - want).abs() - bar).max())
    for r in range(0, M, 512):
        rows = slice(r, min(M, r + 512))
        assert torch.equal(got[rows], call(rows)), f"rows {r}.. differ from a launch of their own"
    if kind == "res":
        inplace = res.clone()
        call(slice(0, M), out=inplace, r=inplace)
        assert torch.equal(inplace, got)


def test_k_of_more_than_2_to_22(qops):
    """Weight offsets past 2^32 bytes. Small whole numbers: every partial sum is exact."""
    M, N, K = 3, 128, (1 << 22) + 64
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randint(-1, 2, (M, K), generator=g, device=DEV).to(BF16)
    w = torch.randint(-3, 4, (N, K), generator=g, device=DEV).to(BF16)
    want = torch.zeros(M, N, dtype=torch.float64, device=DEV)
    for k in range(0, K, 1 << 19):
        want += x[:, k:k + (1 << 19)].double() @ w[:, k:k + (1 << 19)].double().T
    assert torch.equal(qops.gemm(x, qops.tile_weight(w)), want.to(torch.float32).to(BF16))


@pytest.mark.parametrize("M", [5, 100, 600])
@pytest.mark.parametrize("kind", ["plain", "res", "silu"])
def test_output_at_8_byte_alignment(qops, M, kind):
    """An output (and residual) that starts 8 bytes off a 16-byte boundary: same bits."""
    N, K = 512, 256
    x, w, res = _inputs(N, K, M, seed=M)
    t = qops.tile_weight(w, pair=kind == "silu")
    ncols = N // 2 if kind == "silu" else N
    want = qops.gemm(x, t, residual=res if kind == "res" else None, silu_pair=kind == "silu")
    store = torch.empty(M * ncols + 4, dtype=BF16, device=DEV)
    out = store[4:].view(M, ncols)
    assert out.data_ptr() % 16 == 8
    if kind == "res":
        out.copy_(res)
    got = qops.gemm(x, t, residual=out if kind == "res" else None, silu_pair=kind == "silu", out=out)
    assert torch.equal(got, want)


@pytest.mark.parametrize("which,off", [("x", 1), ("x", 2), ("x", 4), ("w", 1), ("w", 4), ("xw", 5)])
@pytest.mark.parametrize("kind,N,K,M", [("plain", 384, 640, 5), ("res", 512, 192, 129), ("silu", 640, 128, 300),
                                        ("plain", 128, 64, 1), ("res", 128, 64, 257), ("silu", 256, 1088, 64),
                                        ("plain", 6144, 128, 1100), ("silu", 6144, 448, 700),
                                        ("res", 6144, 320, 2200)])
def test_operands_off_a_16_byte_boundary(qops, which, off, kind, N, K, M):
    """Rows and weights that start at any bf16 element, with fewer k stages than LDS slots and more, in both tiles
    (the large one past 256 small ones: N = 6144), and with several tiles of a workgroup (2,200 rows): the same bits
    as from aligned operands."""
    from qwen_hip import _lib
    x, w, res = _inputs(N, K, M, seed=M + off)
    t = qops.tile_weight(w, pair=kind == "silu")

    def shifted(v):
        flat = torch.empty(v.numel() + off, dtype=BF16, device=DEV)[off:]
        assert flat.data_ptr() % 16 == 2 * off
        return flat.view(v.shape).copy_(v)

    def entry(x, t):   # without ops.gemm's aligned copy of x
        out = torch.empty((M, N // 2 if kind == "silu" else N), dtype=BF16, device=DEV)
        _lib.call("qwen_gemm", x.data_ptr(), t.data.data_ptr(), out.data_ptr(), M, N, K, out.shape[1],
                  res.data_ptr() if kind == "res" else None, {"plain": 0, "res": 1, "silu": 2}[kind],
                  torch.cuda.current_stream().cuda_stream)
        return out

    def call(x, t):
        return qops.gemm(x, t, residual=res if kind == "res" else None, silu_pair=kind == "silu")

    want = call(x, t)
    ts = qops.TiledWeight(shifted(t.data), N, K, t.pair) if "w" in which else t
    xs = shifted(x) if "x" in which else x
    assert torch.equal(entry(xs, ts), want)
    assert torch.equal(call(xs, ts), want)
