"""GPU parity of the split-K decode's merge on both sides of the head count
and of the number of records (32 at D = 256, 64 at D = 128: splits of 128 rows)
where it changes from several workgroups per head (64 dims each) to one,
against the CPU oracle (AttentionOps.cpp:73-166). bf16 outputs within 1e-2 of
the tensor maximum."""
import numpy as np
import pytest

import oracle
from aila_amd import datagen as dg

pytestmark = pytest.mark.gpu


def _t(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(torch.bfloat16).cuda()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,Hq,Hkv", [(1, 1, 1), (1, 16, 4), (4, 8, 4), (11, 3, 1), (9, 8, 2)])
def test_merge_either_side_of_32_heads(B, Hq, Hkv, D):
    import torch
    import aila_amd
    for L in (257, 1100, 4096, 4097, 8192, 8193):
        seed = 7100 + 31 * B + D + L
        q = dg.normal_bf16(seed, 0, (B, Hq, D))
        k, v = (dg.normal_bf16(seed, i, (B, Hkv, L, D)) for i in (1, 2))
        print(f"decode merge B={B} Hq={Hq} D={D} L={L}", flush=True)
        ws = torch.full((aila_amd.gqa_decode_workspace_size(B, Hq, D) // 4,), float("nan"), device="cuda")
        out = aila_amd.gqa_decode(_t(q), _t(k), _t(v), L, workspace=ws.view(torch.uint8))
        torch.cuda.synchronize()
        got = dg.bf16_to_f32(out.view(torch.int16).cpu().numpy().view(np.uint16))
        want = dg.bf16_to_f32(oracle.attention_decode_baseline(q, k, v, B, Hq, Hkv, D, L, L))
        assert float(np.max(np.abs(got - want))) <= 1e-2 * float(np.max(np.abs(want)))
