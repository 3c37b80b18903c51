"""GPU parity of the decode at every query-head tile and of groups above 8 that
are shared unevenly (9 = 5 + 4, 13 = 7 + 6, 17 = 6 + 6 + 5), contiguous, paged and
windowed, against the CPU oracle (AttentionOps.cpp:73-166, 533-551). bf16 outputs
within 1e-2 of the tensor maximum."""
import numpy as np
import pytest

import oracle
from aila_amd import datagen as dg

pytestmark = pytest.mark.gpu


def _t(x):
    import torch
    if x.dtype == np.uint16:
        return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(torch.bfloat16).cuda()
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("G", [3, 5, 6, 7, 9, 13, 17])
def test_every_tile(G, D):
    import torch
    import aila_amd
    B, Hkv, page, max_pages = 2, 2, 64, 12
    L, max_seq = page * max_pages - 37, page * max_pages
    Hq, seed = Hkv * G, 7300 + 16 * G + D
    q = dg.normal_bf16(seed, 0, (B, Hq, D), std=2.0)
    k, v = (dg.normal_bf16(seed, i, (B, Hkv, max_seq, D)) for i in (1, 2))
    k[:, :, L:] = v[:, :, L:] = 0x7FC0   # rows past the length are never read
    table = np.random.default_rng(seed).permutation(B * max_pages).astype(np.int32).reshape(B, max_pages)
    kp, vp = (np.empty((B * max_pages, Hkv, page, D), np.uint16) for _ in range(2))
    for pool, rows in ((kp, k), (vp, v)):
        pool[table] = rows.reshape(B, Hkv, max_pages, page, D).transpose(0, 2, 1, 3, 4)
    want = oracle.attention_decode_baseline(q, k, v, B, Hq, Hkv, D, max_seq, L)
    wwant = oracle.attention_decode_window(q, k, v, B, Hq, Hkv, D, max_seq, L, 400, 300, 5)
    lens = _t(np.full(B, L, np.int32))
    for split in (True, False):
        n = aila_amd.gqa_decode_workspace_size(B, Hq, D) // 4
        ws = torch.full((n,), float("nan"), device="cuda").view(torch.uint8) if split else None
        for name, ref, run in (
                ("plain", want, lambda: aila_amd.gqa_decode(_t(q), _t(k), _t(v), L, workspace=ws)),
                ("paged", want, lambda: aila_amd.gqa_decode_paged(_t(q), _t(kp), _t(vp), _t(table), lens, L,
                                                                  workspace=ws)),
                ("window", wwant, lambda: aila_amd.gqa_decode(_t(q), _t(k), _t(v), L, workspace=ws,
                                                              window=(400, 300, 5)))):
            print(f"decode tile G={G} D={D} {name} split={split}", flush=True)
            out = run()
            torch.cuda.synchronize()
            got, r = (dg.bf16_to_f32(x) for x in (out.view(torch.int16).cpu().numpy().view(np.uint16), ref))
            assert float(np.max(np.abs(got - r))) <= 1e-2 * float(np.max(np.abs(r))), (name, split)
