"""GPU parity of the decode entry points for any query/KV head ratio
(the reference maps query head h to KV head h / (Hq / Hkv),
AttentionOps.cpp:100): ratios up to 8 run on a query-head tile of their
size, ratios above 8 on several workgroups per KV head. Qwen3-14B (40 q / 8 kv heads) has ratio 5.

Tolerance: bf16 outputs within max relative error 1e-2 of the fp32 oracle.
"""
import numpy as np
import pytest

import oracle
from aila_amd import datagen as dg

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _t(x):
    import torch
    if x.dtype == np.uint16:
        return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(torch.bfloat16).cuda()
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _np(t):
    return t.detach().view(__import__("torch").int16).cpu().numpy().view(np.uint16)


def _rel(a, r):
    a = dg.bf16_to_f32(a).astype(np.float64)
    r = dg.bf16_to_f32(r).astype(np.float64)
    return float(np.max(np.abs(a - r)) / max(float(np.max(np.abs(r))), 1e-30))


def _ws(B, Hq, D):
    import torch
    import aila_amd
    return torch.full((aila_amd.gqa_decode_workspace_size(B, Hq, D) // 4,), float("nan"), device="cuda").view(
        torch.uint8)


@pytest.mark.parametrize("G,Hkv,D,B,L,split", [
    (5, 8, 128, 2, 1500, True),     # Qwen3-14B: 40 q / 8 kv heads
    (5, 8, 128, 1, 700, False),
    (3, 2, 256, 2, 2000, True),
    (6, 2, 64, 3, 333, True),
    (7, 1, 128, 2, 100, True),      # short context: single pass with a workspace
    (12, 2, 128, 2, 1500, True),    # two workgroups per KV head (6 + 6 heads)
    (16, 4, 256, 2, 3000, True),    # 64 q / 4 kv heads
    (16, 1, 128, 1, 900, False),
    (16, 4, 128, 9, 399, True),     # splits of 64 rows: 504 workgroups, at once
    (14, 8, 128, 6, 352, True),     # of 128: 576 of 64 would not run at once
    (12, 4, 128, 1, 3000, True),    # of 128: 192 workgroups, one to a CU
])
def test_decode_any_group(G, Hkv, D, B, L, split):
    import torch
    import aila_amd
    Hq, max_seq = Hkv * G, L + 40
    print(f"decode group G={G} Hkv={Hkv} D={D} B={B} L={L} split={split}", flush=True)
    seed = 0x6A0 + G * 7 + D
    q = dg.normal_bf16(seed, 0, (B, Hq, D), std=2.0)
    kc = dg.normal_bf16(seed, 1, (B, Hkv, max_seq, D))
    vc = dg.normal_bf16(seed, 2, (B, Hkv, max_seq, D))
    kc[:, :, L:] = 0x7FC0   # rows past the length are never read
    vc[:, :, L:] = 0x7FC0
    want = oracle.attention_decode_baseline(q, kc, vc, B, Hq, Hkv, D, max_seq, L)
    out = aila_amd.gqa_decode(_t(q), _t(kc), _t(vc), L, workspace=_ws(B, Hq, D) if split else None)
    torch.cuda.synchronize()
    got = _np(out)
    assert np.isfinite(dg.bf16_to_f32(got)).all()
    assert _rel(got, want) <= TOL


@pytest.mark.parametrize("G,Hkv,D", [(5, 2, 128), (12, 1, 256)])
def test_decode_any_group_device_lengths_and_append(G, Hkv, D):
    """Append at device positions plus decode (ElementwiseOps.cpp:105-216
    cache write, then AttentionOps.cpp:499-643)."""
    import torch
    import aila_amd
    B, max_seq = 3, 2100
    Hq = Hkv * G
    print(f"decode group append G={G} Hkv={Hkv} D={D}", flush=True)
    seed = 0x6B0 + G + D
    q = dg.normal_bf16(seed, 0, (B, Hq, D), std=2.0)
    k = dg.normal_bf16(seed, 1, (B, Hkv, D), std=2.0)
    v = dg.normal_bf16(seed, 2, (B, Hkv, D))
    kc = dg.normal_bf16(seed, 3, (B, Hkv, max_seq, D))
    vc = dg.normal_bf16(seed, 4, (B, Hkv, max_seq, D))
    pos = np.array([2047, 5, 700], np.int32)
    kw, vw = kc.copy(), vc.copy()
    for b in range(B):
        kw[b, :, pos[b]] = k[b]
        vw[b, :, pos[b]] = v[b]
    out = aila_amd.gqa_decode_append(_t(q), _t(k), _t(v), _t(kc), _t(vc), int(pos.max()), workspace=_ws(B, Hq, D),
                                     positions=_t(pos))
    torch.cuda.synchronize()
    got = _np(out)
    for b in range(B):
        want = oracle.attention_decode_baseline(q[b:b + 1], kw[b:b + 1], vw[b:b + 1], 1, Hq, Hkv, D, max_seq,
                                                int(pos[b]) + 1)[0]
        assert _rel(got[b], want) <= TOL, f"sequence {b}"


@pytest.mark.parametrize("G,Hkv,D,rot,gate,split", [(5, 8, 128, 128, True, True), (10, 2, 256, 64, False, True),
                                                     (3, 4, 128, 32, True, False)]
                         # tiles 6 and 7, a tile of 8 with 7 heads (D = 128), and 13 heads as 7 + 6
                         + [(G, 2, D, D, split, split) for G in (6, 7, 13) for D in (64, 128, 256)
                            for split in (True, False)])
def test_fused_prepare_append_any_group(G, Hkv, D, rot, gate, split):
    """QK-norm + RoPE + append + decode in one launch (ElementwiseOps.cpp:
    555-863 then AttentionOps.cpp:499-643) for ratios outside 1, 2, 4, 8."""
    import torch
    import aila_amd
    B, max_seq, theta, eps = 2, 2048, 1e6, 1e-6
    Hq = Hkv * G
    print(f"fused prep group G={G} Hkv={Hkv} D={D} rot={rot} gate={gate} split={split}", flush=True)
    seed = 0x6C0 + G + D
    q = dg.normal_bf16(seed, 0, (B, Hq, 2 * D), std=2.0)
    k = dg.normal_bf16(seed, 1, (B, Hkv, D), std=2.0)
    v = dg.normal_bf16(seed, 2, (B, Hkv, D))
    qw = dg.normal_bf16(seed, 3, (D,))
    kw = dg.normal_bf16(seed, 4, (D,))
    kc = dg.normal_bf16(seed, 5, (B, Hkv, max_seq, D))
    vc = dg.normal_bf16(seed, 6, (B, Hkv, max_seq, D))
    pos = np.array([1500, 17], np.int32)
    kx, vx = kc.copy(), vc.copy()
    qo, gw, _ = oracle.decode_prepare(q, k, v, qw, kw, kx, vx, pos, B, Hq, Hkv, D, max_seq, rot, theta, eps,
                                      packed=True)
    res = aila_amd.gqa_decode_prepare_append(_t(q), _t(k), _t(v), _t(kc), _t(vc), int(pos.max()), q_norm_w=_t(qw),
                                             k_norm_w=_t(kw), rotary_dim=rot, theta=theta, eps=eps,
                                             packed_gate=True, apply_gate=gate, positions=_t(pos),
                                             workspace=_ws(B, Hq, D) if split else None)
    torch.cuda.synchronize()
    got = _np(res if gate else res[0])
    for b in range(B):
        att = oracle.attention_decode_baseline(qo[b:b + 1], kx[b:b + 1], vx[b:b + 1], 1, Hq, Hkv, D, max_seq,
                                               int(pos[b]) + 1)[0]
        want = oracle.sigmoid_mul(att, gw[b]) if gate else att
        assert _rel(got[b], want) <= TOL, f"sequence {b}"
    if not gate:
        assert np.array_equal(_np(res[1]), q[:, :, D:])   # the gate half, copied through


def test_decode_window_any_group():
    """Decode window with sinks (AttentionOps.cpp:533-551, 598-616) at ratio 6."""
    import torch
    import aila_amd
    B, Hkv, G, D, L, max_seq = 2, 2, 6, 128, 3000, 3072
    Hq = Hkv * G
    q = dg.normal_bf16(0x6D0, 0, (B, Hq, D), std=2.0)
    kc = dg.normal_bf16(0x6D0, 1, (B, Hkv, max_seq, D))
    vc = dg.normal_bf16(0x6D0, 2, (B, Hkv, max_seq, D))
    want = oracle.attention_decode_window(q, kc, vc, B, Hq, Hkv, D, max_seq, L, 1000, 512, 4)
    out = aila_amd.gqa_decode(_t(q), _t(kc), _t(vc), L, workspace=_ws(B, Hq, D), window=(1000, 512, 4))
    torch.cuda.synchronize()
    assert _rel(_np(out), want) <= TOL


def test_paged_decode_any_group():
    """Paged decode over a shuffled pool at ratio 5 (and 16) against the
    oracle on the rows the pages hold."""
    import torch
    import aila_amd
    for G, Hkv, D, page in ((5, 2, 128, 64), (16, 1, 256, 256)):
        B, L = 2, 1501
        Hq = Hkv * G
        max_pages = (L + page - 1) // page
        seed = 0x6E0 + G
        q = dg.normal_bf16(seed, 0, (B, Hq, D), std=2.0)
        kc = dg.normal_bf16(seed, 1, (B, Hkv, max_pages * page, D))
        vc = dg.normal_bf16(seed, 2, (B, Hkv, max_pages * page, D))
        table = np.random.default_rng(seed).permutation(B * max_pages).astype(np.int32).reshape(B, max_pages)
        kp = np.zeros((B * max_pages, Hkv, page, D), np.uint16)
        vp = np.zeros_like(kp)
        for b in range(B):
            for j in range(max_pages):
                kp[table[b, j]] = kc[b, :, j * page:(j + 1) * page]
                vp[table[b, j]] = vc[b, :, j * page:(j + 1) * page]
        want = oracle.attention_decode_baseline(q, kc, vc, B, Hq, Hkv, D, max_pages * page, L)
        out = aila_amd.gqa_decode_paged(_t(q), _t(kp), _t(vp), _t(table), _t(np.full(B, L, np.int32)), L,
                                        workspace=_ws(B, Hq, D))
        torch.cuda.synchronize()
        assert _rel(_np(out), want) <= TOL, (G, D)
