"""GPU parity of the D = 256 prefill whose two wave groups share one K/V tile
stream: sizes that its dispatch takes (128-row blocks that fill the device's
rounds; key-split turns with an even number of 64-row blocks), with an odd
number of blocks, ragged last blocks and tiles, and over a cached prefix not
aligned to either. Rows are checked against the oracle's decode of that row over
the rows it attends (AttentionOps.cpp:73-166 against :649-842, :2308-2507);
bf16 outputs within 1e-2 of the row's maximum. Rows are also checked to be
bitwise the same when a V row outside their reach is not finite."""
import numpy as np
import pytest

import oracle
from aila_amd import datagen as dg

pytestmark = pytest.mark.gpu
D = 256


def _t(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(torch.bfloat16).cuda()


def _np(t):
    import torch
    return t.detach().view(torch.int16).cpu().numpy().view(np.uint16)


def _check(q, kc, vc, got, S, base, Hq, Hkv, max_seq):
    assert np.isfinite(got).all()
    for r in sorted({0, 1, 15, 31, 32, 63, 64, 127, 128, S // 2, S // 2 + 1, S - 33, S - 2, S - 1} & set(range(S))):
        want = dg.bf16_to_f32(oracle.attention_decode_baseline(q[r].reshape(1, Hq, D), kc[None], vc[None], 1, Hq, Hkv, D,
                                                               max_seq, base + r + 1))[0].reshape(-1)
        assert float(np.max(np.abs(got[r] - want))) <= 1e-2 * float(np.max(np.abs(want))), r


@pytest.mark.parametrize("S,Hq,Hkv,scale", [(1985, 32, 8, 1.0), (2048, 32, 4, 1.0), (3456, 16, 4, 1.0), (2047, 32, 8, 8.0)])
def test_shared_prefill(S, Hq, Hkv, scale):
    import torch
    import aila_amd
    print(f"shared prefill S={S} Hq={Hq} scale={scale}", flush=True)
    seed, max_seq = 9100 + S, S + 5
    q = dg.normal_bf16(seed, 0, (S, Hq * D), std=scale)
    k, v = (dg.normal_bf16(seed, i, (S, Hkv * D)) for i in (1, 2))
    kc, vc = (torch.full((Hkv, max_seq, D), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    out = aila_amd.gqa_prefill(_t(q), _t(k), _t(v), Hq, Hkv, k_cache=kc, v_cache=vc, cache_pos=2)
    torch.cuda.synchronize()
    ck, cv = _np(kc), _np(vc)
    assert np.array_equal(ck[:, 2:2 + S], k.reshape(S, Hkv, D).transpose(1, 0, 2))
    assert np.array_equal(cv[:, 2:2 + S], v.reshape(S, Hkv, D).transpose(1, 0, 2))
    seven = dg.f32_to_bf16(np.float32([7.0]))[0]
    for c in (ck, cv):
        assert (c[:, :2] == seven).all() and (c[:, 2 + S:] == seven).all()
    _check(q, np.ascontiguousarray(ck[:, 2:]), np.ascontiguousarray(cv[:, 2:]), dg.bf16_to_f32(_np(out)), S, 0, Hq, Hkv,
           max_seq - 2)


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("S,start", [(65, 777), (128, 3000), (250, 2051), (500, 5003), (710, 250), (711, 250), (2048, 101)])
def test_shared_turn(S, start, split):
    """Turns over a cached prefix with the key split (S = 2048: none planned) and
    without; 710 and 711 tokens over 250 rows lie on both sides of three times the
    first block's keys; NaN past the rows any query attends."""
    import torch
    import aila_amd
    Hq, Hkv = (32, 4) if S == 2048 else (16, 4)
    print(f"shared turn S={S} start={start} split={split}", flush=True)
    seed, max_seq = 9300 + S, start + S + 7
    q = dg.normal_bf16(seed, 0, (S, Hq * D))
    k, v = (dg.normal_bf16(seed, i, (Hkv, max_seq, D)) for i in (1, 2))
    k[:, start + S:] = 0x7FC0
    v[:, start + S:] = 0x7FC0
    need = aila_amd.gqa_prefill_cached_workspace_size(S, start, Hq, Hkv, D)
    ws = torch.full((need // 4,), float("nan"), device="cuda").view(torch.uint8) if split and need else None
    out = aila_amd.gqa_prefill_cached(_t(q), _t(k), _t(v), start, Hq, workspace=ws)
    torch.cuda.synchronize()
    _check(q, k, v, dg.bf16_to_f32(_np(out)), S, start, Hq, Hkv, max_seq)


@pytest.mark.parametrize("S,start,Hq,row", [(3456, 0, 16, 100), (3456, 0, 16, 3455), (2047, 0, 32, 1100), (250, 2051, 16, 100),
                                            (250, 2051, 16, 249), (500, 5003, 16, 70), (128, 3000, 16, 127)])
def test_not_finite_v_row(S, start, Hq, row):
    """A wave (16 query rows) reads no key block (32 rows) that lies wholly past
    its last row, so one V row of infinities leaves every such row's bits as
    they are without it. The rows that attend it are checked to be spoiled, so
    that the poison is known to be read."""
    import torch
    import aila_amd
    print(f"shared V row S={S} start={start} Hq={Hq} row={row}", flush=True)
    Hkv, seed = 4, 9500 + S + row
    q = _t(dg.normal_bf16(seed, 0, (S, Hq * D)))
    if start:
        n = start + S
        k, v = (dg.normal_bf16(seed, i, (Hkv, n, D)) for i in (1, 2))
        bad = v.copy()
        bad[:, start + row] = 0x7F80
        need = aila_amd.gqa_prefill_cached_workspace_size(S, start, Hq, Hkv, D)
        assert need > 0, "planned with a key split"
        run = lambda x: aila_amd.gqa_prefill_cached(q, _t(k), _t(x), start, Hq,  # noqa: E731
                                                    workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))
    else:
        k, v = (dg.normal_bf16(seed, i, (S, Hkv * D)) for i in (1, 2))
        bad = v.copy()
        bad[row] = 0x7F80
        run = lambda x: aila_amd.gqa_prefill(q, _t(k), _t(x), Hq, Hkv)  # noqa: E731
    clean, got = _np(run(v)), _np(run(bad))
    reach = (start + row) // 32 * 32                        # first key of the poisoned block
    free = [r for r in range(S) if start + r // 16 * 16 + 15 < reach]
    assert free and free[-1] >= row - 48
    assert np.array_equal(got[free], clean[free])
    assert not np.isfinite(dg.bf16_to_f32(got[row:])).any()
