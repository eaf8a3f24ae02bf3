"""Token rows of unusual strides in the kernels that rebuild keys: expanded (stride 0), overlapping, and on both sides of the line for 32-bit row offsets."""
import pytest
import torch

import oracle
from util import check_out, check_scores, f32, gen

pytestmark = pytest.mark.gpu

from kernel_collections_amd import ops  # noqa: E402

BF = torch.bfloat16


def rows(dev, L, r, stride, seed):
    """[1, L, r] whose rows lie `stride` elements apart."""
    if stride >= r:
        return torch.empty((L - 1) * stride + r, dtype=BF, device=dev).as_strided((1, L, r), (0, stride, 1)).copy_(gen((1, L, r), seed=seed))
    return gen(((L - 1) * stride + r,), seed=seed).to(dev).as_strided((1, L, r), (0, stride, 1))


@pytest.mark.parametrize("r", [512, 384, 256])
@pytest.mark.parametrize("L,stride", [(70, 0), (70, 8), (70, 264), (9, (1 << 25) - 8), (9, 1 << 25)])
def test_one_basis(dev, r, L, stride):
    b, hq, hkv = 1, 8, 2
    q, kB, vB = gen((b, hq, 128), std=0.4, seed=1), gen((b, hkv, r, 128), std=r ** -0.5, seed=3), gen((b, hkv, r, 128), std=r ** -0.5, seed=5)
    A = rows(dev, L, r, stride, 2)
    cos, sin = oracle.rope_cos_sin(torch.arange(L), 128, 5e5)
    inv = ops.rope_inv_freq(128, 5e5, A.device)
    qd, kBd = q.to(dev), kB.to(dev)
    part, lse = torch.empty((b, hq, 2, r), device=dev), torch.empty((b, hq, 2), device=dev)
    ops.recon_stage1(qd, A, kBd, A, part, lse, None, None, None, b, hq, hkv, L, 2, 128 ** -0.5, True, inv, 0, None)
    o = ops.merge_stage2(part, lse, torch.empty((b, hq, 128), device=dev), vB.to(dev), None, None, b, hq, hkv, L, 2)
    Ac = A.cpu()
    check_out(o, oracle.gqa_factorized_rope(*f32(q.unsqueeze(2), Ac, kB, Ac, vB), cos, sin, sm_scale=128 ** -0.5)[:, :, 0])
    s = torch.empty((b, hq, 1, L), device=dev)
    ops.recon_stage1(qd, A, kBd, None, None, None, s, None, None, b, hq, hkv, L, 2, 0.25, True, inv, 0, None)
    check_scores(s, 0.25 * oracle.qab_rope(*f32(q.unsqueeze(2), Ac, kB), cos, sin))


@pytest.mark.parametrize("rk,rv", [(512, 512), (256, 256)])
@pytest.mark.parametrize("stride,vstride", [(0, 512), (512, 0), (264, 512), (512, 8)])
def test_two_bases(dev, rk, rv, stride, vstride):
    """Rows of either basis that overlap: the two-basis kernel's offsets from row to row are unsigned, the call is not for it."""
    b, hq, hkv, L = 1, 8, 2, 70
    q, kB, vB = gen((b, hq, 128), std=0.4, seed=1), gen((b, hkv, rk, 128), std=rk ** -0.5, seed=3), gen((b, hkv, rv, 128), std=rv ** -0.5, seed=5)
    A, V = rows(dev, L, rk, stride, 2), rows(dev, L, rv, vstride, 4)
    cos, sin = oracle.rope_cos_sin(torch.arange(L), 128, 5e5)
    part, lse = torch.empty((b, hq, 2, rv), device=dev), torch.empty((b, hq, 2), device=dev)
    ops.recon_stage1(q.to(dev), A, kB.to(dev), V, part, lse, None, None, None, b, hq, hkv, L, 2, 128 ** -0.5, True, ops.rope_inv_freq(128, 5e5, A.device), 0, None)
    o = ops.merge_stage2(part, lse, torch.empty((b, hq, 128), device=dev), vB.to(dev), None, None, b, hq, hkv, L, 2)
    check_out(o, oracle.gqa_factorized_rope(*f32(q.unsqueeze(2), A.cpu(), kB, V.cpu(), vB), cos, sin, sm_scale=128 ** -0.5)[:, :, 0])
