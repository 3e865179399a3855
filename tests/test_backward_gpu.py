"""Parity of the HIP backward (mvpa_backward through the FlashMVPA autograd function) with
reverse-mode differentiation of the oracle's closed-form MVPA in float64.

The oracle forward is pinned in tests/test_oracle.py; its gradient is what torch.autograd derives
from it (and tests/test_oracle.py::test_direct_gradcheck checks that derivation against finite
differences).  Tolerances: fp32 inputs max-abs <= 2e-5 + 1e-4 * max|ref| per gradient; bf16
inputs rel-L2 <= 2e-2 per gradient (inputs rounded to bf16 on both sides, gradients returned in
bf16)."""
import math
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (os.path.join(ROOT, "multi-variate-parallel-transformer_amd"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)

from oracle import mvpa_oracle as O  # noqa: E402
from mvpa_hip.synthetic import make_mvpa_inputs  # noqa: E402

pytestmark = pytest.mark.gpu

NAMES = ("q", "u", "vb", "z", "k", "k_time", "k_chan", "v")


def _oracle_grads(inp, d_out, window, chan_valid=None, time_bias=True, chan_bias=True):
    leaves = {n: getattr(inp, n).double().clone().requires_grad_(True) for n in NAMES}
    k_time = leaves["k_time"] if time_bias else leaves["k_time"] * 0
    k_chan = leaves["k_chan"] if chan_bias else leaves["k_chan"] * 0
    vb = leaves["vb"] if time_bias else leaves["vb"] * 0
    z = leaves["z"] if chan_bias else leaves["z"] * 0
    out = O.mvpa_direct(leaves["q"], leaves["k"], leaves["v"], leaves["u"], vb, z, k_time, k_chan,
                        window=window, chan_valid=chan_valid)
    grads = torch.autograd.grad((out * d_out.double()).sum(), [leaves[n] for n in NAMES],
                                allow_unused=True)
    return out.detach(), {n: (g if g is not None else torch.zeros_like(leaves[n])) for n, g in zip(NAMES, grads)}


def _gpu_grads(inp, d_out, window, dtype, chan_valid=None, time_bias=True, chan_bias=True):
    from attentions import flashmvpa
    hkv, dh = inp.u.shape
    t_len, c_len = inp.k_time.shape[1], inp.k_chan.shape[1]
    leaves = {n: getattr(inp, n).to(dtype).cuda().requires_grad_(True) for n in NAMES}
    out = flashmvpa(leaves["q"], leaves["u"].view(1, hkv, 1, dh), leaves["vb"].view(1, hkv, 1, dh),
                    leaves["z"].view(1, hkv, 1, dh), leaves["k"],
                    leaves["k_time"].view(1, hkv, t_len, dh), leaves["k_chan"].view(1, hkv, c_len, dh),
                    leaves["v"], True, 1.0 / math.sqrt(dh), window_size=window,
                    rel_bias_time=time_bias, rel_bias_chan=chan_bias,
                    chan_valid=chan_valid.cuda() if chan_valid is not None else None)
    out.backward(d_out.to(dtype).cuda())
    return out.detach().float().cpu(), {n: (leaves[n].grad.float().cpu() if leaves[n].grad is not None
                                            else torch.zeros_like(getattr(inp, n))) for n in NAMES}


CASES = [
    dict(B=2, C=8, T=32, H=4, Hkv=4, Dh=32, window=10),     # the reference's CPU-runnable size
    dict(B=1, C=3, T=13, H=4, Hkv=2, Dh=16, window=10),     # GQA, window active
    dict(B=2, C=5, T=7, H=2, Hkv=1, Dh=64, window=10),      # window vacuous, ragged C
    dict(B=1, C=4, T=14, H=2, Hkv=2, Dh=32, window=3),      # narrow window
    dict(B=1, C=6, T=9, H=2, Hkv=2, Dh=128, window=0),      # content everywhere
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{B}C{C}T{T}H{H}g{Hkv}D{Dh}w{window}".format(**c))
def test_backward_fp32_matches_oracle_autograd(case):
    cfg = dict(case)
    window = cfg.pop("window")
    inp = make_mvpa_inputs(seed=3, qkv_unit=True, **cfg)
    g = torch.Generator().manual_seed(11)
    d_out = torch.randn(inp.q.shape, generator=g)
    ref_out, ref = _oracle_grads(inp, d_out, window)
    out, got = _gpu_grads(inp, d_out, window, torch.float32)
    assert (out.double() - ref_out).abs().max().item() <= 1e-5
    for n in NAMES:
        err = (got[n].double() - ref[n]).abs().max().item()
        assert err <= 2e-5 + 1e-4 * ref[n].abs().max().item(), (n, err)


def test_backward_with_channel_validity():
    inp = make_mvpa_inputs(B=2, C=6, T=12, H=2, Hkv=2, Dh=32, seed=5, qkv_unit=True)
    valid = torch.tensor([[1, 1, 0, 1, 1, 0], [0, 1, 1, 1, 1, 1]], dtype=torch.bool)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(2))
    _, ref = _oracle_grads(inp, d_out, 10, chan_valid=valid)
    _, got = _gpu_grads(inp, d_out, 10, torch.float32, chan_valid=valid)
    for n in NAMES:
        err = (got[n].double() - ref[n]).abs().max().item()
        assert err <= 2e-5 + 1e-4 * ref[n].abs().max().item(), (n, err)
    # keys of absent channels receive no gradient at all
    absent = (~valid)[:, None, None, :].expand(2, 2, 12, 6).reshape(2, 2, 72)
    assert got["k"][absent].abs().max().item() == 0.0
    assert got["v"][absent].abs().max().item() == 0.0


def test_backward_bf16_within_tolerance():
    inp = make_mvpa_inputs(B=1, C=16, T=24, H=4, Hkv=2, Dh=64, seed=9, qkv_unit=True).round_to(torch.bfloat16)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(4)).bfloat16().float()
    _, ref = _oracle_grads(inp, d_out, 10)
    _, got = _gpu_grads(inp, d_out, 10, torch.bfloat16)
    for n in NAMES:
        rel = (got[n].double() - ref[n]).norm().item() / max(ref[n].norm().item(), 1e-30)
        assert rel <= 2e-2, (n, rel)


BF16_CASES = [
    dict(B=1, C=64, T=12, H=2, Hkv=2, Dh=64, window=10),      # two waves per time step
    dict(B=1, C=40, T=37, H=2, Hkv=1, Dh=64, window=10),      # ragged channels, two 32-step slabs, GQA
    dict(B=2, C=8, T=70, H=1, Hkv=1, Dh=64, window=4),        # three slabs, narrow window
    dict(B=1, C=33, T=9, H=2, Hkv=2, Dh=64, window=0),        # content everywhere; odd C (workspace rows padded to 36)
    dict(B=1, C=117, T=9, H=2, Hkv=1, Dh=64, window=2),       # two channel parts (64 + 53), four launches per pass, GQA
    dict(B=1, C=128, T=6, H=1, Hkv=1, Dh=64, window=10),      # two full channel parts
    dict(B=2, C=65, T=35, H=2, Hkv=2, Dh=64, window=3),       # second part of one channel; two slabs
    dict(B=1, C=36, T=9, H=2, Hkv=2, Dh=64, window=0),        # content everywhere, ragged second channel tile
    dict(B=1, C=32, T=21, H=2, Hkv=1, Dh=64, window=3),       # one channel tile, four key steps per workgroup, GQA
    dict(B=2, C=20, T=40, H=2, Hkv=2, Dh=64, window=5),       # one ragged channel tile, two slabs
    dict(B=1, C=64, T=45, H=1, Hkv=1, Dh=64, window=2),       # odd T: the last key pair of a workgroup is half empty
    # head dim 128: rows of 256 bytes in the LDS tiles
    dict(B=1, C=32, T=21, H=2, Hkv=1, Dh=128, window=3),      # one channel tile, GQA
    dict(B=2, C=20, T=40, H=2, Hkv=2, Dh=128, window=5),      # one ragged channel tile, two slabs
    dict(B=1, C=64, T=12, H=2, Hkv=2, Dh=128, window=10),     # two channel tiles per query step
    dict(B=1, C=40, T=37, H=2, Hkv=1, Dh=128, window=10),     # ragged second tile, two slabs, GQA
    dict(B=1, C=117, T=9, H=2, Hkv=1, Dh=128, window=2),      # two channel parts: 4 launches of either pass
    dict(B=1, C=128, T=6, H=1, Hkv=1, Dh=128, window=10),     # two full channel parts
    dict(B=2, C=65, T=35, H=2, Hkv=2, Dh=128, window=3),      # second part of one channel; two slabs
    dict(B=1, C=33, T=9, H=2, Hkv=2, Dh=128, window=0),       # content everywhere; odd C
]


@pytest.mark.parametrize("case", BF16_CASES, ids=lambda c: "B{B}C{C}T{T}H{H}g{Hkv}D{Dh}w{window}".format(**c))
def test_backward_bf16_mfma_query_pass(case):
    """bf16, Dh = 64 or 128, C <= 128 takes the MFMA passes (dq, dk, dv, bias-table gradients)."""
    cfg = dict(case)
    window = cfg.pop("window")
    inp = make_mvpa_inputs(seed=13, qkv_unit=True, **cfg).round_to(torch.bfloat16)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(6)).bfloat16().float()
    valid = None
    if cfg["C"] in (40, 20, 117):
        valid = torch.ones(cfg["B"], cfg["C"], dtype=torch.bool)
        valid[:, [3, 17, cfg["C"] - 1]] = False
    _, ref = _oracle_grads(inp, d_out, window, chan_valid=valid)
    _, got = _gpu_grads(inp, d_out, window, torch.bfloat16, chan_valid=valid)
    for n in NAMES:
        rel = (got[n].double() - ref[n]).norm().item() / max(ref[n].norm().item(), 1e-30)
        assert rel <= 2e-2, (n, rel)


@pytest.mark.parametrize("cfg", [
    dict(B=1, C=5, T=130, H=2, Hkv=1, Dh=64, window=4),       # a second tile of 2 time-table rows; GQA
    dict(B=2, C=4, T=129, H=1, Hkv=1, Dh=128, window=10),     # one row in it; rows of 516 bytes (no 16-byte loads)
    # one ragged step of everything.  Not fewer rows: delta = rowsum(d_o o) takes o in bf16 and is off by up to
    # 2^-9 sum |d_o o| ~ 2^-9 * 64 * 0.6 = 0.08, a fiftieth of a row's dP - delta (~ 4 for unit inputs) before
    # rows average out; T = 2, C = 1 read 2.05e-2
    dict(B=1, C=3, T=4, H=1, Hkv=1, Dh=64, window=0),
], ids=lambda c: "B{B}C{C}T{T}H{H}g{Hkv}D{Dh}".format(**c))
def test_backward_finish_tile_edges(cfg):
    """Tiles of 128 table rows and 128 query rows, 64 columns a step; the bound is the file's for bf16."""
    cfg = dict(cfg)
    window = cfg.pop("window")
    inp = make_mvpa_inputs(seed=17, qkv_unit=True, **cfg).round_to(torch.bfloat16)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(8)).bfloat16().float()
    _, ref = _oracle_grads(inp, d_out, window)
    _, got = _gpu_grads(inp, d_out, window, torch.bfloat16)
    for n in NAMES:
        rel = (got[n].double() - ref[n]).norm().item() / max(ref[n].norm().item(), 1e-30)
        assert rel <= 2e-2, (n, rel)


def test_backward_rows_are_causal():
    """do confined to the first time steps must leave dk/dv of later keys exactly zero."""
    inp = make_mvpa_inputs(B=1, C=4, T=10, H=2, Hkv=2, Dh=32, seed=1, qkv_unit=True)
    d_out = torch.zeros(inp.q.shape)
    d_out[:, :, : 3 * 4] = torch.randn(1, 2, 12, 32, generator=torch.Generator().manual_seed(8))
    _, got = _gpu_grads(inp, d_out, 10, torch.float32)
    assert got["k"][:, :, 3 * 4:].abs().max().item() == 0.0
    assert got["v"][:, :, 3 * 4:].abs().max().item() == 0.0
    assert got["q"][:, :, 3 * 4:].abs().max().item() == 0.0


@pytest.mark.parametrize("flags", [dict(time_bias=False), dict(chan_bias=False)],
                         ids=lambda f: "+".join(sorted(f)))
def test_backward_bf16_mfma_bias_flags(flags):
    """The matrix-core passes with a bias term switched off: its parameters get zero gradient."""
    inp = make_mvpa_inputs(B=1, C=64, T=20, H=2, Hkv=2, Dh=64, seed=21, qkv_unit=True).round_to(torch.bfloat16)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(3)).bfloat16().float()
    _, ref = _oracle_grads(inp, d_out, 4, **flags)
    _, got = _gpu_grads(inp, d_out, 4, torch.bfloat16, **flags)
    for n in NAMES:
        if ref[n].abs().max().item() == 0.0:
            assert got[n].abs().max().item() == 0.0, n
            continue
        rel = (got[n].double() - ref[n]).norm().item() / max(ref[n].norm().item(), 1e-30)
        assert rel <= 2e-2, (n, rel)


def test_backward_bf16_mfma_rows_are_causal():
    """As test_backward_rows_are_causal, on the matrix-core passes."""
    inp = make_mvpa_inputs(B=1, C=32, T=10, H=2, Hkv=2, Dh=64, seed=1, qkv_unit=True)
    d_out = torch.zeros(inp.q.shape)
    d_out[:, :, : 3 * 32] = torch.randn(1, 2, 96, 64, generator=torch.Generator().manual_seed(8))
    _, got = _gpu_grads(inp, d_out, 10, torch.bfloat16)
    assert got["k"][:, :, 3 * 32:].abs().max().item() == 0.0
    assert got["v"][:, :, 3 * 32:].abs().max().item() == 0.0
    assert got["q"][:, :, 3 * 32:].abs().max().item() == 0.0


@pytest.mark.parametrize("cfg", [dict(B=4, C=64, T=128, H=16, Hkv=16, Dh=64),
                                 dict(B=1, C=128, T=128, H=4, Hkv=2, Dh=128)],
                         ids=["c2", "C128-Dh128-GQA"])
def test_backward_bf16_full_size_invariants(cfg):
    """At the benchmark shape (B4 C64 T128 H16 Dh64, too large for the float64 oracle) and at the
    base model's channels, head dim and head grouping (C128 Dh128, two query heads per kv head) the
    gradients must satisfy what the softmax fixes for ANY d_o:
      * dS rows sum to zero, so every row of dbias_time and of dbias_chan sums to zero
        (up to the bf16 rounding of the probabilities: <= 1e-2 of the absolute sum of the row of
        dbias_chan, which stands for sum_keys |dS|);
      * with d_o = 1 the columns of dv are the column sums of P, so dv summed over the keys of a
        (batch, kv head) equals the number of queries of the group's heads, N * H/Hkv."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=0, **cfg).to("cuda", torch.bfloat16)
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan,
                                     return_lse=True)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).bfloat16()
    dq, dk, dv, dbt, dbc = mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, d_o, lse, inp.u, inp.vb, inp.z,
                                                  inp.k_time, inp.k_chan)
    for t in (dq, dk, dv, dbt, dbc):
        assert torch.isfinite(t).all()
    scale = dbc.abs().sum(-1)                          # ~ sum_keys |dS| of the row (measured: ratio <= 3.4e-3)
    for g in (dbt, dbc):
        rows = g.sum(-1).abs()
        assert (rows <= 1e-2 * scale).all(), (rows / scale).max().item()
    # the two tables hold the same dS, summed differently
    assert torch.allclose(dbt.sum(-1), dbc.sum(-1), atol=1e-4, rtol=0)
    ones = torch.ones_like(out)
    _, _, dv1, _, _ = mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, ones, lse, inp.u, inp.vb, inp.z,
                                             inp.k_time, inp.k_chan)
    n_q = cfg["T"] * cfg["C"] * (cfg["H"] // cfg["Hkv"])
    tot = dv1.sum(2)                                  # [B,Hkv,Dh]
    assert (tot / n_q - 1).abs().max().item() <= 2e-3, (tot / n_q - 1).abs().max().item()


def test_backward_bf16_strided_inputs_match_contiguous():
    """q, k, v, o, d_o as head-interleaved views ([B,N,H,Dh] buffers, the layout the layer's fused
    projection produces): the same gradients, bit for bit, as from contiguous copies."""
    import mvpa_hip
    cfg = dict(B=2, C=48, T=20, H=4, Hkv=2, Dh=64)
    inp = make_mvpa_inputs(seed=4, qkv_unit=True, **cfg).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, *tabs, return_lse=True)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).bfloat16()
    ref = mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, d_o, lse, *tabs)

    def interleave(t):                      # [B,h,N,Dh] -> view of a [B,N,h,Dh] buffer
        return t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    q, k, v, o, g = (interleave(t) for t in (inp.q, inp.k, inp.v, out, d_o))
    assert not q.is_contiguous() and q.stride(-1) == 1
    got = mvpa_hip.mvpa_backward(q, k, v, o, g, lse, *tabs)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,C,T,H,Hkv,Dh,window,masked", [
    (48, 33, 21, 8, 4, 64, 3, True),       # 384 workgroups of 16 key steps, the second holds 5; one live channel in tile 2
    (32, 64, 33, 4, 4, 64, 1, False),      # a third group of one key step; whole tiles
    (24, 65, 40, 16, 8, 64, 20, True),     # four launches, parts of 64 and 1 channels; the far steps end inside a group
    (32, 40, 13, 2, 2, 128, 3, True),      # 128 workgroups of 8 key steps, the second has no far step
    (8, 100, 25, 8, 4, 128, 10, False),    # parts of 64 and 36 channels, GQA
    (4, 33, 268, 2, 1, 128, 10, True),     # 256 far steps: two launches of the query pass; 136 workgroups
])
def test_far_steps_in_their_own_kernel(B, C, T, H, Hkv, Dh, window, masked):
    """A batch whose far query steps get a kernel of their own against its samples one at a time, which do
    not: the same sums in another order (fp32), rounded to bf16 once on either side."""
    from attentions import flashmvpa
    g = torch.Generator(device="cuda").manual_seed(C * T)

    def rn(*s, std=1.0):
        return (torch.randn(s, generator=g, device="cuda") * std).bfloat16()
    q, k, v, d = rn(B, H, T * C, Dh), rn(B, Hkv, T * C, Dh, std=Dh ** -0.5), rn(B, Hkv, T * C, Dh), rn(B, H, T * C, Dh)
    tabs = [rn(1, Hkv, 1, Dh, std=0.1) for _ in range(3)] + [rn(1, Hkv, T, Dh, std=0.1), rn(1, Hkv, C, Dh, std=0.1)]
    valid = None
    if masked:
        valid = torch.rand((B, C), generator=g, device="cuda") < 0.8
        valid[:, 0] = True

    def grads(b):
        leaves = [x[b].clone().requires_grad_(True) for x in (q, k, v)]
        out = flashmvpa(leaves[0], *tabs[:3], leaves[1], *tabs[3:], leaves[2], True, Dh ** -0.5, window_size=window,
                        chan_valid=valid[b] if masked else None)
        return torch.autograd.grad(out, leaves, d[b])
    whole = grads(slice(0, B))
    for b in range(0, B, 5):
        for x, y in zip(whole, grads(slice(b, b + 1))):
            assert (x[b].double() - y[0].double()).norm() <= 2.0 ** -8 * y.double().norm()


@pytest.mark.parametrize("T,C,Dh,window,masked", [(267, 5, 128, 10, False), (268, 33, 128, 10, False), (269, 40, 128, 11, True),
                                                  (290, 70, 128, 2, False)])
def test_long_walks_against_the_fp32_kernels(T, C, Dh, window, masked):
    """Both sides of the line where the query pass becomes two launches, slabs that end inside and at the end of
    a walk, against the fp32 kernels on the same (bf16) inputs."""
    from attentions import flashmvpa
    g = torch.Generator(device="cuda").manual_seed(C * T)

    def rn(*s, std=1.0):
        return (torch.randn(s, generator=g, device="cuda") * std).bfloat16()
    args = [rn(1, 2, T * C, Dh)] + [rn(1, 1, 1, Dh, std=0.1) for _ in range(3)] + \
           [rn(1, 1, T * C, Dh, std=Dh ** -0.5), rn(1, 1, T, Dh, std=0.1), rn(1, 1, C, Dh, std=0.1), rn(1, 1, T * C, Dh)]
    d = rn(1, 2, T * C, Dh)
    valid = None
    if masked:
        valid = torch.ones((1, C), dtype=torch.bool, device="cuda")
        valid[0, 1::3] = False

    def grads(dtype):
        leaves = [x.to(dtype).requires_grad_(True) for x in args]
        out = flashmvpa(*leaves, True, Dh ** -0.5, window_size=window, chan_valid=valid)
        return torch.autograd.grad(out, leaves, d.to(dtype))
    for n, x, y in zip(NAMES, grads(torch.bfloat16), grads(torch.float32)):
        assert (x.double() - y.double()).norm() <= 2e-2 * y.double().norm(), n      # the bf16 bound of this file


@pytest.mark.parametrize("C,Dh,T,window", [
    *[(33, 64, T, 2) for T in range(4, 16)],      # 0 .. 6 units of far steps, whole and half; T even and odd
    (35, 64, 37, 31), (66, 64, 36, 3), (3, 64, 35, 2), (2, 64, 67, 30), (34, 64, 99, 1),      # rows and slabs of 1 .. 3
    (33, 128, 9, 2), (2, 128, 34, 1), (67, 128, 267, 3),
])
def test_query_pass_units_and_short_rows(C, Dh, T, window):
    """The query pass walks far steps in units of two and writes rows in fours: every remainder of both, against the
    fp32 kernels on the same (bf16) inputs."""
    inp = make_mvpa_inputs(seed=T + C, qkv_unit=True, B=1, C=C, T=T, H=2, Hkv=1, Dh=Dh).round_to(torch.bfloat16)
    d_out = torch.randn(inp.q.shape, generator=torch.Generator().manual_seed(T)).bfloat16().float()
    valid = None
    if T % 3 == 0 and C > 2:
        valid = torch.ones(1, C, dtype=torch.bool)
        valid[:, [0, C - 2]] = False
    _, ref = _gpu_grads(inp, d_out, window, torch.float32, chan_valid=valid)
    _, got = _gpu_grads(inp, d_out, window, torch.bfloat16, chan_valid=valid)
    for n in NAMES:
        a, b = got[n].double(), ref[n].double()
        assert torch.isfinite(a).all() and (a - b).norm() <= 2e-2 * b.norm(), n             # the bf16 bound of this file


@pytest.mark.parametrize("cfg,flags", [
    (dict(B=1, C=1, T=1, H=2, Hkv=1, Dh=64), {}),                   # one row
    (dict(B=1, C=64, T=64, H=3, Hkv=3, Dh=64), {}),                 # whole steps of 64 columns, whole tiles of 128 rows
    (dict(B=2, C=63, T=67, H=16, Hkv=4, Dh=64), {}),                # more row tiles than workgroups, ragged everything
    (dict(B=1, C=65, T=128, H=2, Hkv=2, Dh=64), {}),                # four steps, the last of one column
    (dict(B=1, C=65, T=129, H=2, Hkv=2, Dh=64), {}),                # five: the build of up to ten
    (dict(B=1, C=2, T=512, H=2, Hkv=1, Dh=64), {}),                 # nine
    (dict(B=1, C=1, T=640, H=1, Hkv=1, Dh=64), {}),                 # eleven: a pass by rows and one by columns
    (dict(B=2, C=32, T=70, H=4, Hkv=2, Dh=128), {}),                # three steps at Dh 128
    (dict(B=1, C=128, T=128, H=2, Hkv=1, Dh=128), {}),              # four
    (dict(B=1, C=5, T=257, H=2, Hkv=1, Dh=128), {}),                # six: the two passes
    (dict(B=33, C=3, T=90, H=16, Hkv=2, Dh=64), {}),                # a workgroup walks all of a head's three row tiles
    (dict(B=1, C=40, T=300, H=8, Hkv=4, Dh=64), {}),                # six steps, three of 94 row tiles a workgroup
    (dict(B=2, C=33, T=70, H=16, Hkv=8, Dh=128), {}),               # three of 19 at Dh 128
    (dict(B=1, C=40, T=37, H=2, Hkv=1, Dh=64), dict(time_bias=False)),
    (dict(B=1, C=40, T=37, H=2, Hkv=1, Dh=64), dict(chan_bias=False)),
    (dict(B=1, C=40, T=37, H=2, Hkv=1, Dh=128), dict(time_bias=False, chan_bias=False)),
], ids=lambda c: "-".join(f"{k}{int(v)}" for k, v in c.items()) or "both")
def test_backward_finish_against_table_products(cfg, flags):
    """mvpa_backward_full against mvpa_backward's fp32 results and the products of the table gradients in 64 bits.
    G is rounded to bf16 once (2^-8 of each term) and so is the result; the fp32 sums of up to 2^17 terms add less
    than 2^-10 of the sum of their magnitudes.  The sums over all rows, where that bound is far above the result, are held
    in the 2-norm as well: terms of random signs and their roundings (2^-9 of each) grow alike, which leaves 2^-9 of the
    result for the terms and as much for the result; 1e-2 allowed, and a row tile left out of n is n^-1/2."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=23, qkv_unit=True, **cfg).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, *tabs, return_lse=True, **flags)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).bfloat16()
    scale = cfg["Dh"] ** -0.5
    got = mvpa_hip.mvpa_backward_full(inp.q, inp.k, inp.v, out, d_o, lse, *tabs, sm_scale=scale, **flags)
    dq_c, dk, dv, dbt, dbc = (t.double() for t in mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, d_o, lse, *tabs,
                                                                         sm_scale=scale, **flags))
    B, H, N, Dh = inp.q.shape
    Hkv = cfg["Hkv"]

    def rows(t):
        return t.reshape(B, Hkv, -1, t.shape[-1])
    q, dq, size_q = rows(inp.q).double(), rows(dq_c), rows(dq_c).abs()
    want, size = {"u": dq.sum((0, 2))}, {"u": size_q.sum((0, 2))}
    for on, G, tab, bias, name, tname in ((flags.get("time_bias", True), dbt, inp.k_time, inp.vb, "vb", "k_time"),
                                          (flags.get("chan_bias", True), dbc, inp.k_chan, inp.z, "z", "k_chan")):
        G, tab, qb = rows(G) * int(on), tab.double(), q + bias.double()[None, :, None]
        dq, size_q = dq + G @ tab, size_q + G.abs() @ tab.abs()
        want[name], size[name] = (G @ tab).sum((0, 2)), (G.abs() @ tab.abs()).sum((0, 2))
        want[tname] = (G.transpose(2, 3).contiguous() @ qb).sum(0)
        size[tname] = (G.abs().transpose(2, 3).contiguous() @ (q.abs() + bias.double().abs()[None, :, None])).sum(0)
    want.update(q=dq.reshape(B, H, N, Dh), k=dk, v=dv)
    # dk, dv: the query heads of a kv head may come as parts that are added afterwards, another order of fp32 sums
    # whose terms are at least as large as a typical element
    size.update(q=size_q.reshape(B, H, N, Dh), k=dk.abs() + dk.pow(2).mean().sqrt(), v=dv.abs() + dv.pow(2).mean().sqrt())
    for n, g in zip(NAMES, got):
        bound = 1.02 * 2.0 ** -8 * (want[n].abs() + size[n]) + 2.0 ** -10 * size[n]
        assert ((g.double() - want[n]).abs() <= bound).all(), n
        if N > 1 and n not in ("q", "k", "v"):      # one row: a difference of equal numbers
            assert (g.double() - want[n]).norm() <= 1e-2 * want[n].norm(), n


@pytest.mark.parametrize("C,T,Dh,H,Hkv", [
    (5, 9, 64, 2, 2), (32, 20, 64, 2, 2), (33, 45, 64, 3, 3), (64, 130, 64, 16, 16), (65, 14, 64, 2, 2), (128, 33, 64, 2, 2),
    (20, 15, 128, 2, 2), (40, 13, 128, 2, 2), (100, 30, 128, 2, 2),
    (32, 160, 64, 32, 16),                        # two query heads walked by one workgroup
])
def test_key_gradients_rounded_where_they_are_summed(C, T, Dh, H, Hkv):
    """dk and dv of mvpa_backward_full are the fp32 results of mvpa_backward, rounded once: bit for bit."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=29, qkv_unit=True, B=1, C=C, T=T, H=H, Hkv=Hkv, Dh=Dh).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    if H > Hkv:
        assert C <= 32 and Hkv * ((T + 3) // 4) >= 512             # fewer: a workgroup per query head, sums of parts
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, *tabs, return_lse=True)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(3)).bfloat16()
    scale = Dh ** -0.5
    got = dict(zip(NAMES, mvpa_hip.mvpa_backward_full(inp.q, inp.k, inp.v, out, d_o, lse, *tabs, sm_scale=scale)))
    _, dk, dv, _, _ = mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, d_o, lse, *tabs, sm_scale=scale)
    assert torch.equal(got["k"], dk.bfloat16()) and torch.equal(got["v"], dv.bfloat16())


@pytest.mark.parametrize("over", [("k", "v"), ("v", "k"), ("d_o", "new"), ("new", "q"), ("o", "d_o")], ids="-".join)
@pytest.mark.parametrize("B,C,T,Dh", [(2, 100, 14, 64), (1, 70, 13, 128), (2, 20, 30, 64)])
def test_key_gradients_over_what_is_read(over, B, C, T, Dh):
    """dk and dv that lie over an input, which several launches read: what separate memory receives, bit for bit."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=37, qkv_unit=True, B=B, C=C, T=T, H=2, Hkv=2, Dh=Dh).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, *tabs, return_lse=True)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(7)).bfloat16()
    read = dict(q=inp.q, k=inp.k, v=inp.v, o=out, d_o=d_o)

    def grads(over):
        x = {n: t.contiguous().clone() for n, t in read.items()}
        to = [x[n] if n in x else torch.empty_like(inp.k) for n in over]
        return mvpa_hip.mvpa_backward_full(x["q"], x["k"], x["v"], x["o"], x["d_o"], lse, *tabs, sm_scale=Dh ** -0.5,
                                           out=(torch.empty_like(inp.q), *to))
    for n, want, got in zip(NAMES, grads(("new", "new")), grads(over)):
        assert torch.equal(got, want), n


@pytest.mark.parametrize("B,C,T,H,Hkv", [(2, 40, 256, 12, 4), (5, 64, 252, 4, 2), (10, 33, 508, 2, 1), (10, 33, 509, 2, 1), (3, 40, 63, 8, 4)])
def test_workgroups_per_query_head(B, C, T, H, Hkv):
    """Both sides of the lines where each query head gets its own workgroups in the key pass (and the far kernel with
    them): dk and dv against those of mvpa_backward, which never does.  Parts of fp32 sums in another order, one rounding."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=31, qkv_unit=True, B=B, C=C, T=T, H=H, Hkv=Hkv, Dh=64).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    out, lse = mvpa_hip.mvpa_forward(inp.q, inp.k, inp.v, *tabs, return_lse=True)
    d_o = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).bfloat16()
    got = dict(zip(NAMES, mvpa_hip.mvpa_backward_full(inp.q, inp.k, inp.v, out, d_o, lse, *tabs, sm_scale=0.125)))
    _, dk, dv, _, _ = mvpa_hip.mvpa_backward(inp.q, inp.k, inp.v, out, d_o, lse, *tabs, sm_scale=0.125)
    for n, want in (("k", dk.double()), ("v", dv.double())):
        # terms of the sums are at least as large as a typical element; 2^-10 of them for the order, as above
        bound = 1.01 * 2.0 ** -8 * want.abs() + 2.0 ** -10 * (want.abs() + want.pow(2).mean().sqrt())
        assert ((got[n].double() - want).abs() <= bound).all(), n


# (b, h) that do not divide over the XCDs, fewer than eight of them, just more, many; one tile, two, many; walks that take turns and ones that do not
@pytest.mark.parametrize("B,C,T,H,Hkv,Dh", [(3, 40, 33, 3, 1, 64), (3, 64, 1, 5, 5, 64), (5, 20, 3, 2, 1, 64), (3, 33, 90, 12, 4, 64), (2, 20, 70, 9, 9, 64),
                                            (3, 40, 20, 3, 3, 128), (6, 40, 26, 4, 4, 64), (5, 36, 140, 8, 8, 64),
                                            # parts of up to 32 channels in tiles of 32 and (the samples alone) of 64, without the far kernel and with it
                                            (6, 70, 24, 16, 16, 64), (8, 65, 60, 8, 8, 64), (2, 96, 52, 16, 8, 128), (2, 65, 20, 4, 2, 128)])
def test_every_workgroup_of_a_batch(B, C, T, H, Hkv, Dh):
    """A batch against its samples one by one, which other kernels may serve, their workgroups dealt in another order.  Either rounds its
    probabilities to 8 bits at a reference of its own, so a (b, h) is compared by its norm, as the kernels are with the oracle; a tile of rows that no
    workgroup wrote is at least sqrt(1 / 71) of it."""
    import mvpa_hip
    inp = make_mvpa_inputs(seed=37, qkv_unit=True, B=B, C=C, T=T, H=H, Hkv=Hkv, Dh=Dh).to("cuda", torch.bfloat16)
    tabs = (inp.u, inp.vb, inp.z, inp.k_time, inp.k_chan)
    d_o = torch.randn(inp.q.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(7)).bfloat16()

    def grads(s):
        q, k, v = inp.q[s], inp.k[s], inp.v[s]
        out, lse = mvpa_hip.mvpa_forward(q, k, v, *tabs, return_lse=True)
        g = dict(zip(NAMES, mvpa_hip.mvpa_backward_full(q, k, v, out, d_o[s], lse, *tabs, sm_scale=Dh ** -0.5)))
        return out, g["q"], g["k"], g["v"]
    for name, got, *want in zip(("o", "q", "k", "v"), grads(slice(None)), *(grads(slice(b, b + 1)) for b in range(B))):
        want = torch.cat(want).double()
        assert ((got.double() - want).flatten(2).norm(dim=-1) <= 2e-2 * want.flatten(2).norm(dim=-1)).all(), name
