"""Kernels chosen by a rule on sizes, at the sizes where the rule or the tiling can go wrong, against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle as orc
from gpu_util import qspec, rel_err, to_np
from strixite_amd import moe

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print("[shapes]", *a, flush=True)


def _bf16(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(DEV).view(torch.bfloat16)


def _weight(bits, N, K, G, seed):
    q, s, m = orc.gen_q(bits, orc.tensor_key(seed, "gu_q"), orc.tensor_key(seed, "gu_s"), N, K, G)
    return moe.QWeight.from_host(bits, q, s, m, N, K, G)


# the served model's K (gate_up 2560: ten streaming waves; down 640: five groups a row, the swizzle of odd group counts)
# at one token, at the most tokens of the decode form, and gathered above it; one slot has an invalid id
@pytest.mark.parametrize("M,A,E,H,I", [(1, 3, 8, 2560, 640), (16, 4, 24, 2560, 640), (17, 4, 9, 2560, 640),
                                       (90, 3, 5, 2560, 640)])
def test_streamed_experts_at_the_served_widths(M, A, E, H, I):
    say("streamed experts", M, A, E, H, I)
    gu, dn = _weight(4, E * 2 * I, H, 128, 31), _weight(4, E * H, I, 128, 32)
    x = orc.gen_bf16_normal(orc.tensor_key(8, "x"), 1.0, (M, H))
    ids = np.stack([np.random.default_rng(500 + m).permutation(E)[:A] for m in range(M)]).astype(np.int32)
    ids[M // 2, A - 1] = E
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    ex = moe.MOE_MATH_WMMA_BF16
    h = to_np(moe.experts_gather_grouped_swiglu(_bf16(x), gu, E, ws, M, A, math=ex))
    bad = np.array([M // 2 * A + A - 1])
    good = np.setdiff1d(np.arange(M * A), bad)
    assert np.all(np.isnan(orc.bf16_to_f32(h[bad]))) and not np.isnan(orc.bf16_to_f32(h[good])).any()
    ok_ids = np.where(ids >= E, 0, ids).astype(np.int32)
    b, q, s, m, G = qspec(gu)
    href = orc.experts_gate_up_swiglu(x, orc.qview(b, q, s, m, gu.N, H, G), E, ok_ids)
    assert rel_err(h[good], href[good]) < 1e-2  # h is BF16: one rounding apart, 2^-8 of a value
    hz = h.copy()
    hz[bad] = 0
    pt = torch.full((M * A, H), 7.0, dtype=torch.float32, device=DEV)
    coef = torch.full((M, A), 0.25, device=DEV)
    moe.experts_combine_grouped(_bf16(hz), dn, E, tid, coef, ws, M, A, partial=pt, math=ex)
    p = pt.cpu().numpy()
    assert np.all(np.isnan(p[bad]))
    b, q, s, m, G = qspec(dn)
    pref = orc.experts_down(hz, orc.qview(b, q, s, m, dn.N, I, G), E, ok_ids)
    assert rel_err(p[good], pref[good]) < 1e-4  # FP32 sums of 640 products in another order
