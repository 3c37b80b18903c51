"""GPU parity of the chunked DeltaNet prefill over the forms its dispatch
distinguishes: value heads per key head (one prep workgroup forms 1-4 of them
at a time, more in passes; on small grids several share a key head, two value
heads each), column slabs of the scan (16, 32 or 64 columns by
the number of heads) and chunk counts around its two- and three-chunk
rotations, against the sequential oracle recurrence
(run_linear_delta_host, Qwen35HybridTextBackend.cpp:1640-1798).

Tolerances as for the other prefill tests: bf16 outputs within 1e-2 of the
tensor maximum (one bf16 rounding is 2^-9), fp32 states within 1e-3.
"""
import numpy as np
import pytest

import oracle
from aila_amd import datagen as dg

pytestmark = pytest.mark.gpu
OUT_TOL, STATE_TOL = 1e-2, 1e-3
D = 128


def _t(x):
    import torch
    if x.dtype == np.uint16:
        return torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).view(torch.bfloat16).cuda()
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _bf(t):
    import torch
    return dg.bf16_to_f32(t.detach().view(torch.int16).cpu().numpy().view(np.uint16))


def _rel(a, r):
    return float(np.max(np.abs(a - r)) / max(float(np.max(np.abs(r))), 1e-30))


# (B, Hk, Hv): heads per key head 1, 2, 3, 4, 5, 8 and B * Hv on both sides of
# 32 and 64, where the scan's slabs widen
SHAPES = [(1, 2, 2), (2, 2, 4), (1, 2, 6), (1, 1, 4), (1, 1, 5), (1, 1, 8), (1, 16, 32), (3, 11, 11), (2, 16, 32),
          (5, 13, 13), (2, 12, 36)]


@pytest.mark.parametrize("T", [1, 64, 65, 129, 257])
@pytest.mark.parametrize("B,Hk,Hv", SHAPES)
def test_recurrence_matches_oracle(B, Hk, Hv, T):
    import torch
    import aila_amd
    print(f"deltanet_prefill B={B} T={T} Hk={Hk} Hv={Hv}", flush=True)
    seed = 41000 + 97 * Hv + T
    q, k = (dg.normal_bf16(seed, i, (B, T, Hk, D)) for i in (0, 1))
    v = dg.normal_bf16(seed, 2, (B, T, Hv, D))
    a, b = (dg.normal_bf16(seed, i, (B, T, Hv)) for i in (3, 4))
    S0 = dg.normal(seed, 5, B * Hv * D * D, std=0.1).reshape(B, Hv, D, D)
    st = _t(S0)
    out = aila_amd.deltanet_prefill(_t(q), _t(k), _t(v), _t(a), _t(b), st)
    torch.cuda.synchronize()
    _, want_o, want_S = oracle.deltanet_recurrent(q, k, v, a, b, S0, B, T, Hk, Hv, D, D, fast=True)
    assert _rel(st.cpu().numpy(), want_S) <= STATE_TOL
    assert _rel(_bf(out), dg.bf16_to_f32(want_o)) <= OUT_TOL


@pytest.mark.parametrize("T", [2, 63, 64, 66, 129, 200])
@pytest.mark.parametrize("B,Hk,Hv", SHAPES)
def test_layer_matches_oracle(B, Hk, Hv, T):
    import torch
    import aila_amd
    print(f"deltanet_layer_prefill B={B} T={T} Hk={Hk} Hv={Hv}", flush=True)
    seed, ch, head = 42000 + 89 * Hv + T, 2 * Hk * D + Hv * D, T % 3
    qkv, z = dg.normal_bf16(seed, 0, (B, T, ch)), dg.normal_bf16(seed, 1, (B, T, Hv * D))
    a, b = (dg.normal_bf16(seed, i, (B, T, Hv)) for i in (2, 3))
    w = dg.normal_bf16(seed, 4, (ch, 4), std=0.5)
    ring = dg.normal(seed, 5, B * 3 * ch).reshape(B, 3, ch)
    S0 = dg.normal(seed, 6, B * Hv * D * D, std=0.1).reshape(B, Hv, D, D)
    norm = 1.0 + dg.normal(seed, 7, D, std=0.1)
    st, cs = _t(S0), _t(ring)
    out = aila_amd.deltanet_layer_prefill(_t(qkv), _t(z), _t(a), _t(b), _t(w), cs, head, _t(norm), st, Hk)
    torch.cuda.synchronize()
    want_o, want_S, want_cs = oracle.deltanet_layer(qkv, z, a, b, w, ring, head, norm, S0, B, T, Hk, Hv, D, D,
                                                   fast=True)
    assert _rel(st.cpu().numpy(), want_S) <= STATE_TOL
    assert _rel(_bf(out), dg.bf16_to_f32(want_o)) <= OUT_TOL
    assert np.array_equal(cs.cpu().numpy(), want_cs)


@pytest.mark.parametrize("B,G", [(64, 3), (65, 3), (64, 4), (65, 4), (79, 5), (80, 5), (79, 8), (80, 8)])
def test_prep_either_side_of_its_rule(B, G):
    # two chunks a sequence: shares of two value heads up to 256 workgroups (more than
    # four heads: below 160 of whole key heads), the last one ragged; then whole key heads
    test_recurrence_matches_oracle(B, 1, G, 65)
    test_layer_matches_oracle(B, 1, G, 65)


@pytest.mark.parametrize("B,Hk,Hv,T", [(1, 1, 1, 1), (2, 2, 4, 129), (1, 1, 8, 300), (3, 11, 33, 65)])
def test_calls_stay_inside_their_workspace(B, Hk, Hv, T):
    import torch
    import aila_amd
    seed, ch = 44000 + T, 2 * Hk * D + Hv * D
    q, k = (_t(dg.normal_bf16(seed, i, (B, T, Hk, D))) for i in (0, 1))
    v, z = (_t(dg.normal_bf16(seed, i, (B, T, Hv, D))) for i in (2, 3))
    a, b = (_t(dg.normal_bf16(seed, i, (B, T, Hv))) for i in (4, 5))
    qkv, w = _t(dg.normal_bf16(seed, 6, (B, T, ch))), _t(dg.normal_bf16(seed, 7, (ch, 4), std=0.5))
    for need, run in (
            (aila_amd.deltanet_prefill_workspace_size(B, T, Hv, D, D),
             lambda ws, st: aila_amd.deltanet_prefill(q, k, v, a, b, st, workspace=ws)),
            (aila_amd.deltanet_layer_prefill_workspace_size(B, T, Hk, Hv),
             lambda ws, st: aila_amd.deltanet_layer_prefill(qkv, z.view(B, T, Hv * D), a, b, w,
                                                            torch.zeros((B, 3, ch), device="cuda"), 0,
                                                            torch.ones(D, device="cuda"), st, Hk, workspace=ws))):
        print(f"workspace B={B} Hk={Hk} Hv={Hv} T={T} bytes={need}", flush=True)
        buf = torch.full((need + 65536,), 0xA5, dtype=torch.uint8, device="cuda")
        st, st2 = (torch.zeros((B, Hv, D, D), device="cuda") for _ in range(2))
        out = run(buf[:need], st)
        assert (buf[need:] == 0xA5).all().item()
        assert torch.equal(out, run(None, st2)) and torch.equal(st, st2)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("B,Hk", [(1, 1), (3, 2), (8, 16)])
def test_layer_decode_three_value_heads(B, Hk, wide):
    """Whole-layer decode steps with three value heads to a key head; an
    arrivals array is ignored, whatever it holds."""
    import torch
    import aila_amd
    Hv, T, head = 3 * Hk, 5, 2
    seed, ch = 43000 + B, 2 * Hk * D + 3 * Hk * D
    qkv, z = dg.normal_bf16(seed, 0, (B, T, ch)), dg.normal_bf16(seed, 1, (B, T, Hv * D))
    a, b = (dg.normal_bf16(seed, i, (B, T, Hv)) for i in (2, 3))
    w = dg.normal_bf16(seed, 4, (ch, 4), std=0.5)
    ring = dg.normal(seed, 5, B * 3 * ch).reshape(B, 3, ch)
    S0 = dg.normal(seed, 6, B * Hv * D * D, std=0.1).reshape(B, Hv, D, D)
    norm = 1.0 + dg.normal(seed, 7, D, std=0.1)
    st, cs, wt, nw = _t(S0), _t(ring), _t(w), _t(norm)
    x = [_t(v) for v in (qkv, z, a, b)]
    arr = torch.full((B * Hk,), 7, dtype=torch.int32, device="cuda") if wide else None
    print(f"deltanet_layer_decode B={B} Hk={Hk} Hv={Hv} wide={wide}", flush=True)
    outs = [aila_amd.deltanet_layer_decode(*(v[:, t] for v in x), wt, cs, (head + t) % 3, nw, st, Hk, arrivals=arr)
            for t in range(T)]
    torch.cuda.synchronize()
    want_o, want_S, want_cs = oracle.deltanet_layer(qkv, z, a, b, w, ring, head, norm, S0, B, T, Hk, Hv, D, D, fast=True)
    assert _rel(st.cpu().numpy(), want_S) <= STATE_TOL
    assert _rel(np.stack([_bf(o) for o in outs], axis=1), dg.bf16_to_f32(want_o)) <= OUT_TOL
    assert np.array_equal(cs.cpu().numpy(), want_cs)
    assert arr is None or (arr == 7).all().item()


def _three_heads(B, Hk, pad):
    """One layer step with three value heads to a key head; z rows `pad` elements apart."""
    Hv, seed = 3 * Hk, 43500 + B
    ch = 2 * Hk * D + Hv * D
    x = dict(qkv=dg.normal_bf16(seed, 0, (B, 1, ch)), z=dg.normal_bf16(seed, 1, (B, 1, Hv * D)),
             a=dg.normal_bf16(seed, 2, (B, 1, Hv)), b=dg.normal_bf16(seed, 3, (B, 1, Hv)),
             w=dg.normal_bf16(seed, 4, (ch, 4), std=0.5), ring=dg.normal(seed, 5, B * 3 * ch).reshape(B, 3, ch),
             norm=1.0 + dg.normal(seed, 7, D, std=0.1), S0=dg.normal(seed, 6, B * Hv * D * D, std=0.1).reshape(B, Hv, D, D))
    zw = np.zeros((B, Hv * D + pad), np.uint16)
    zw[:, :Hv * D] = x["z"][:, 0]
    return x, Hv, ch, _t(zw)[:, :Hv * D]


def test_layer_decode_three_value_heads_unaligned_z_rows():
    """z rows a number of elements apart that is no multiple of 4: the general
    kernel takes the call."""
    import torch
    import aila_amd
    B, Hk = 3, 2
    x, Hv, _, z = _three_heads(B, Hk, 2)
    assert z.stride(0) % 4 == 2
    print("deltanet_layer_decode three value heads, unaligned z rows", flush=True)
    st, cs = _t(x["S0"]), _t(x["ring"])
    out = aila_amd.deltanet_layer_decode(_t(x["qkv"][:, 0]), z, _t(x["a"][:, 0]), _t(x["b"][:, 0]), _t(x["w"]), cs, 1,
                                         _t(x["norm"]), st, Hk)
    torch.cuda.synchronize()
    want_o, want_S, want_cs = oracle.deltanet_layer(x["qkv"], x["z"], x["a"], x["b"], x["w"], x["ring"], 1, x["norm"],
                                                   x["S0"], B, 1, Hk, Hv, D, D, fast=True)
    assert _rel(st.cpu().numpy(), want_S) <= STATE_TOL
    assert _rel(_bf(out), dg.bf16_to_f32(want_o)[:, 0]) <= OUT_TOL
    assert np.array_equal(cs.cpu().numpy(), want_cs)


def test_layer_decode_three_value_heads_ignores_arrivals_address():
    """The array is ignored for this ratio, its alignment too: the same kernel
    runs, so the same bits come out."""
    import torch
    import aila_amd
    B, Hk = 2, 2
    x, Hv, ch, z = _three_heads(B, Hk, 0)
    t = {k: _t(x[k][:, 0]) for k in ("qkv", "a", "b")}
    w, norm = _t(x["w"]), _t(x["norm"])
    arr = torch.full((4 * B * Hk + 4,), 7, dtype=torch.uint8, device="cuda")
    res = []
    for address in (None, arr.data_ptr() + 1):
        print(f"deltanet_layer_decode three value heads, arrivals at {address}", flush=True)
        st, cs, out = _t(x["S0"]), _t(x["ring"]), torch.empty((B, Hv * D), dtype=torch.bfloat16, device="cuda")
        rc = aila_amd.lib().aila_hip_deltanet_layer_decode(
            t["qkv"].data_ptr(), ch, z.data_ptr(), Hv * D, t["a"].data_ptr(), t["b"].data_ptr(), Hv, w.data_ptr(),
            cs.data_ptr(), 0, None, None, None, norm.data_ptr(), st.data_ptr(), out.data_ptr(), B, Hk, Hv, D, D, 4, 1e-6,
            D ** -0.5, address, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == 0
        res.append((st, cs, out))
    assert all(torch.equal(a, b) for a, b in zip(*res))
    assert (arr == 7).all().item()
