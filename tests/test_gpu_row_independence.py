"""Rows of a projection do not meet: a row of infinities (one sequence of a batch that overflowed) leaves every other
row's bits as they are, in every launch form, also where k does not divide evenly among wavefronts, splits and stages."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
DEV = "cuda:0"


@pytest.fixture(scope="module")
def qops():
    from qwen_hip import ops
    return ops


def _others_unchanged(call, M, K, bad, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    want = call(x).clone()
    x[bad] = float("inf")
    got = call(x)
    keep = [m for m in range(M) if m != bad]
    assert bool(torch.isfinite(want.float()).all())
    assert torch.equal(got[keep], want[keep])
    assert not bool(torch.isfinite(got[bad].float()).any())


# launch form, N, K, most rows that the form is built for
FORMS = [((1, 8, 1), 256, 1600, 32), ((1, 4, 1), 256, 416, 32), ((2, 8, 1), 256, 1632, 32), ((2, 4, 3), 256, 2080, 32),
         ((4, 8, 1), 512, 1600, 32), ((1, 16, 1), 256, 2208, 16), ((8, 4, 1), 512, 1056, 32), ((1, 8, 0), 2560, 1600, 32),
         ((1,), 256, 1280, 32), ((2,), 256, 512, 32), ((6,), 384, 1792, 32), ((1, 8, 2, 1), 128, 256, 16),
         ((2, 4, 3), 2560, 9728, 32)]


@pytest.mark.parametrize("M,cfg,N,K", [(M, c, N, K) for c, N, K, most in FORMS for M in (2, 8, 20, 32) if M <= most])
def test_decode_forms(qops, M, cfg, N, K):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    t = qops.tile_weight((torch.randn(N, K, generator=g, device=DEV) * 0.03).to(BF16))
    for bad in (0, M - 1):
        _others_unchanged(lambda x: qops.fused_linear(x, t, cfg), M, K, bad, seed=M)


@pytest.mark.parametrize("M", [2, 17, 33, 70, 300])
@pytest.mark.parametrize("K", [64, 192, 1600])
def test_prompt_gemm(qops, M, K):
    g = torch.Generator(device=DEV).manual_seed(K)
    t = qops.tile_weight((torch.randn(384, K, generator=g, device=DEV) * 0.03).to(BF16))
    for bad in (0, M - 1):
        _others_unchanged(lambda x: qops.gemm(x, t), M, K, bad, seed=M)
