"""Row operations of the training path (csrc/mvpa_train.hip) against the same formulas in 64 bits, and the
attention on packed projection rows against the operator on separate tensors."""
import pytest
import torch

import mvpa_hip
from attentions.attn import FlashMVPA, FlashMVPAPacked
from models.fftencoder import WaveEncoder
from models.mvpformer import MVPFormerConfig, MVPFormerModel
from mvpa_hip import autograd as AG

pytestmark = pytest.mark.gpu


def _close(got, ref, terms=1):
    """One rounding to the type of the result (half an ulp: 2^-8 of bf16 with its 8 significant bits, 2^-24 of fp32)
    terms whose roundings add up to at most 2^-24 sqrt(terms) of the result's scale, 8 sigma."""
    half = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -24
    ref = ref.double()
    scale = ref.pow(2).mean().sqrt()
    bound = half * 1.01 * ref.abs() + 8 * 2.0 ** -24 * (max(terms, 16) ** 0.5) * (ref.abs() + scale)
    assert ((got.double() - ref).abs() <= bound).all()


# columns: one chunk, rows that are no whole chunks, the edges of each build; rows: one, fewer than a
# workgroup's, a second round of rows for some workgroups only
@pytest.mark.parametrize("cols", [4, 7, 768, 772, 1024, 1030, 2048, 4092, 4096])
@pytest.mark.parametrize("rows,xt,wt,res", [(1, torch.bfloat16, torch.bfloat16, True), (5, torch.float32, torch.float32, False),
                                            (2051, torch.bfloat16, torch.float32, True),
                                            (2050, torch.float32, torch.bfloat16, True)])
def test_norm_backward(cols, rows, xt, wt, res):
    g = torch.Generator(device="cuda").manual_seed(cols * 31 + rows)

    def rn(*s):
        return torch.randn(s, generator=g, device="cuda")
    x, w, dy = rn(rows, cols).to(xt), (1 + 0.1 * rn(cols)).to(wt), rn(rows, cols).bfloat16()
    r = rn(rows, cols).to(xt) if res else None
    dx, dw = mvpa_hip.norm_backward(x, w, dy, r, 1e-5)
    xd, wd, gd = x.double(), w.double(), dy.double()
    inv = (xd.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
    parts = inv * gd * wd, xd * inv ** 3 * (xd * gd * wd).mean(-1, keepdim=True)
    ref = parts[0] - parts[1] + (r.double() if res else 0)
    half = 2.0 ** -8 if xt == torch.bfloat16 else 2.0 ** -24
    bound = half * 1.01 * ref.abs() + 2.0 ** -18 * (parts[0].abs() + parts[1].abs() + inv * wd.abs() + 1)
    assert ((dx.double() - ref).abs() <= bound).all()
    _close(dw, (gd * xd * inv).sum(0), rows * 4)
    only_x, none = mvpa_hip.norm_backward(x, w, dy, r, 1e-5, True, False)
    assert none is None and torch.equal(only_x, dx)
    none, only_w = mvpa_hip.norm_backward(x, w, dy, r, 1e-5, False, True)
    assert none is None and torch.equal(only_w, dw)


@pytest.mark.parametrize("cols,rows,res", [(1156, 34602, True), (1156, 34603, True), (2048, 21973, False), (1408, 31961, False),
                                           (1412, 31870, False)])
def test_norm_backward_of_many_rows(cols, rows, res):
    """Either side of the lines from which rows of more than 1024 columns are requested one ahead."""
    test_norm_backward(cols, rows, torch.bfloat16, torch.float32, res)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 2040), (4, 2048), (5, 2056), (33, 344), (130, 5632)])
def test_silu_gate(rows, n):
    g = torch.Generator(device="cuda").manual_seed(rows * n)
    gu = (torch.randn((rows, 2 * n), generator=g, device="cuda") * 4).bfloat16()
    gu[0, 0], gu[-1, n - 1] = -200.0, 200.0            # exp(-gate) overflows, underflows
    d = torch.randn((rows, n), generator=g, device="cuda").bfloat16()
    gate, up = gu.double().chunk(2, -1)
    s = torch.sigmoid(gate)
    _close(mvpa_hip.silu_gate(gu), gate * s * up)
    dgate, dup = mvpa_hip.silu_gate(gu, d).chunk(2, -1)
    _close(dgate, d.double() * up * s * (1 + gate * (1 - s)))
    _close(dup, d.double() * gate * s)


# one pair of steps, rows of less than a wave, of a chunk more, of several; one channel; a row of zeros, one shorter than eps
@pytest.mark.parametrize("B,T,C,E", [(1, 2, 1, 8), (2, 5, 7, 520), (3, 4, 5, 1032), (1, 25, 64, 768)])
def test_generative_score_gradients(B, T, C, E):
    g = torch.Generator(device="cuda").manual_seed(B * T * C + E)
    a, b = (torch.randn((B, T, C, E), generator=g, device="cuda").bfloat16().requires_grad_() for _ in range(2))
    with torch.no_grad():
        if T > 2:
            a[0, 1, 0], b[0, 2, -1] = 0, 1e-9 / E
    d = torch.randn((B, T - 1, C), generator=g, device="cuda")
    s = AG.cosine_steps(a, b)
    ad, bd = a.detach().double().requires_grad_(), b.detach().double().requires_grad_()
    ref = torch.cosine_similarity(ad[:, 1:], bd[:, :-1], dim=-1)
    _close(s, ref, E)
    want = torch.autograd.grad(ref, (ad, bd), d.double())
    for x, w in zip(torch.autograd.grad(s, (a, b), d, retain_graph=True), want):
        # a difference of two terms of about the result's size
        assert ((x.double() - w).abs() <= 2.0 ** -8 * 1.01 * w.abs() + 2.0 ** -18 * (w.abs() + w.norm(dim=-1, keepdim=True))).all()
        assert x.shape == a.shape and (w != 0).logical_or(x == 0).all()
    both = torch.autograd.grad(s, (a, b), torch.stack([d, 2 * d]), is_grads_batched=True, retain_graph=True)
    for x, y, w in zip(both, torch.autograd.grad(s, (a, b), d, create_graph=True), want):
        assert (x[0] - y).norm() <= 1e-2 * w.norm() and (y.double() - w).norm() <= 1e-2 * w.norm() and y.requires_grad
    only, = torch.autograd.grad(AG.cosine_steps(a.detach(), b), b, d)
    assert (only.double() - want[1]).norm() <= 1e-2 * want[1].norm()
    assert AG.cosine_steps(a[..., 4:], b[..., 4:]) is None and AG.cosine_steps(a[:, :1], b[:, :1]) is None


@pytest.mark.parametrize("E", [8, 1032])
def test_generative_score_gradients_of_rows_that_are_no_numbers(E):
    """A NaN or an infinity in either row of a pair makes every gradient of both NaN, with a zero gradient of the score too; finite
    elements whose squares are past the type give a score and gradients of zero; the other pairs are left alone."""
    g = torch.Generator(device="cuda").manual_seed(E)
    a, b = (torch.randn((2, 4, 3, E), generator=g, device="cuda").bfloat16() for _ in range(2))
    a[0, 1, 0, 5], b[0, 1, 1, E - 1], a[1, 3, 2, 0], b[1, 0, 0, 7] = float("nan"), float("nan"), float("inf"), -float("inf")
    a[1, 2, 0, 3], a[0, 2, 2] = float("nan"), 0
    # squares past fp32, with a.b past it and within: no similarity and no gradients, but numbers
    a[0, 3, 1, 4], b[0, 2, 1, 4], b[0, 2, 0, 6], a[1, 2, 1], b[1, 1, 1] = 3e38, 2, -2e19, 1e38, -1e30
    a, b, d = a.requires_grad_(), b.requires_grad_(), torch.randn((2, 3, 3), generator=g, device="cuda")
    d[1, 1, 0] = 0
    ref = torch.cosine_similarity(a[:, 1:].float(), b[:, :-1].float(), dim=-1)
    want = torch.autograd.grad(ref, (a, b), d)
    s = AG.cosine_steps(a, b)
    assert torch.equal(s.isnan(), ref.isnan()) and ref.isnan().sum() == 5
    assert ((s - ref).abs() <= 1e-5).logical_or(ref.isnan()).all()
    for graph in (False, True):
        for x, w in zip(torch.autograd.grad(s, (a, b), d, retain_graph=True, create_graph=graph), want):
            assert torch.equal(x.isnan(), w.isnan()) and w.isnan().sum() == 5 * E
            assert ((x - w).float().nan_to_num().norm(dim=-1) <= 1e-2 * w.float().nan_to_num().norm(dim=-1)).all()


@pytest.mark.parametrize("cols", [8, 768])
def test_add3_norm_gradients(cols):
    """Gradients through both results, through one of them, and of a gradient (the tensor expressions)."""
    def leaf(*s):
        return torch.randn(s, device="cuda").bfloat16().requires_grad_(True)
    torch.manual_seed(cols)
    a, b, c, w = leaf(70, cols), leaf(70, cols), leaf(70, cols), leaf(cols)
    ds, dn = torch.randn(70, cols, device="cuda").bfloat16(), torch.randn(70, cols, device="cuda").bfloat16()
    total, normed = AG.add3_rmsnorm(a, b, c, w, 1e-5)
    t64, w64 = total.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
    n64 = t64 * (t64.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt() * w64
    for outs, grads, ref_outs in (((total, normed), (ds, dn), (t64 + 0, n64)), ((normed,), (dn,), (n64,))):
        got = torch.autograd.grad(outs, (a, b, c, w), grads, retain_graph=True)
        ref = torch.autograd.grad(ref_outs, (t64, w64), [g.double() for g in grads], retain_graph=True)
        assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
        for x, y in ((got[0], ref[0]), (got[3], ref[1])):
            assert (x.double() - y).norm() <= 2.0 ** -8 * y.norm()
    first, = torch.autograd.grad(normed, (a,), dn, create_graph=True)
    second, = torch.autograd.grad(first.float().pow(2).sum(), (w,))
    assert torch.isfinite(second).all() and second.abs().sum() > 0


@pytest.mark.parametrize("B,C,T,H,Hkv,Dh,masked", [(1, 1, 1, 2, 1, 64, False), (2, 5, 13, 4, 2, 64, True),
                                                   (1, 33, 14, 6, 2, 64, False), (1, 70, 12, 2, 2, 128, True)])
def test_packed_attention(B, C, T, H, Hkv, Dh, masked):
    """Rows of one projection against separate tensors: the same kernels on other strides."""
    g = torch.Generator(device="cuda").manual_seed(C * T)

    def rn(*s, std=1.0):
        return (torch.randn(s, generator=g, device="cuda") * std).bfloat16().requires_grad_(True)
    N, row = T * C, (H + 2 * Hkv) * Dh
    qkv, tabs = rn(B, N, row), [rn(Hkv, Dh, std=0.1) for _ in range(3)] + [rn(Hkv, T, Dh, std=0.1), rn(Hkv, C, Dh, std=0.1)]
    valid = None
    if masked:
        valid = torch.ones(B, C, dtype=torch.bool, device="cuda")
        valid[:, C // 2] = False
    d = torch.randn((B, N, H, Dh), generator=g, device="cuda").bfloat16()
    scale = Dh ** -0.5
    out = FlashMVPAPacked.apply(qkv, *tabs, H, scale, 10, valid, True)
    got = torch.autograd.grad(out, [qkv, *tabs], d)
    q, k, v = FlashMVPAPacked._heads(qkv, H, Hkv, Dh)
    ref_out = FlashMVPA.apply(q, *tabs[:3], k, tabs[3], tabs[4], v, True, scale, 10, True, True, valid)
    ref = torch.autograd.grad(ref_out, [qkv, *tabs], d.transpose(1, 2))
    # bf16 rounding of the probabilities and of the result where the two take kernels of another split
    assert (out.transpose(1, 2).double() - ref_out.double()).norm() <= 2.0 ** -7 * ref_out.double().norm()
    for x, y in zip(got, ref):
        assert x.shape == y.shape
        assert (x.double() - y.double()).norm() <= 2.0 ** -6 * y.double().norm() + 1e-6


def test_operands_that_start_anywhere():
    """Rows, gradients and an fp32 norm weight at an offset of one element: the kernels that read 16 bytes at a
    time get copies or leave the work to the general path, and values and gradients are the aligned ones'."""
    g = torch.Generator(device="cuda").manual_seed(6)

    def at_one(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape).detach().requires_grad_(t.requires_grad)
    a, b, c = ((torch.randn(6, 64, generator=g, device="cuda")).bfloat16().requires_grad_(True) for _ in range(3))
    w = (1 + 0.1 * torch.randn(64, generator=g, device="cuda")).requires_grad_(True)
    # a random projection as the loss: the rows of a norm have the same length whatever goes in, so the gradient of
    # their squares is a difference of nearly equal terms, with errors above 1e-2 of what is left
    towards = torch.randn(6, 64, generator=g, device="cuda")
    results = []
    for where in (lambda t: t, at_one):
        x, weight = [where(t) for t in (a, b, c)], where(w)
        got = AG.add3_rmsnorm(*x, weight, 1e-5)
        if got is None:
            total = x[0] + x[1] + x[2]
            got = total, AG.rmsnorm(total, weight, 1e-5)
        results.append((*got, *torch.autograd.grad((got[1].float() * towards).sum(), [*x, weight])))
    for p, q in zip(*results):
        _near(q, p)
    gu, d = torch.randn(6, 64, generator=g, device="cuda").bfloat16(), torch.randn(6, 32, generator=g, device="cuda").bfloat16()
    assert torch.equal(mvpa_hip.silu_gate(at_one(gu)), mvpa_hip.silu_gate(gu))
    assert torch.equal(mvpa_hip.silu_gate(at_one(gu), at_one(d)), mvpa_hip.silu_gate(gu, d))
    # a training pass on embeddings that start anywhere
    torch.manual_seed(0)
    dims = dict(n_positions=8, n_channels=8, n_embd=128, n_layer=2, n_head=2, n_head_kv=1, n_inner=64, resid_pdrop=0.0,
                embd_pdrop=0.0, attn_pdrop=0.0)
    model = MVPFormerModel(MVPFormerConfig(**dims)).to("cuda", torch.bfloat16).train()
    x = torch.randn(1, 5, 6, 128, generator=g, device="cuda").bfloat16().requires_grad_(True)
    towards = torch.randn(1, 5, 6, 128, generator=g, device="cuda")
    grads = [torch.autograd.grad((model(inputs_embeds=t).float() * towards).sum(), t)[0] for t in (x, at_one(x))]
    _near(grads[1], grads[0])


def _near(got, ref):
    """The general path rounds the sum of three twice: half a unit of 2^-8, 0.11 % rms of a part of the sum, and
    the gradients, of the same size each, are rounded to bf16 on both sides: 0.4 % in all, of two blocks twice that."""
    assert ((got.double() - ref.double()).norm() / ref.double().norm()).item() <= 1e-2


# ranks around the eight that are summed together; columns around the 64 of a workgroup and the 1024 of a row's
# threads; rows around the 8 and the 32 shares; a slice without an adapter, a module without any
@pytest.mark.parametrize("r,cols,rows", [(1, 8, (1, 2)), (8, 768, (96, 64)), (9, 72, (33, 66)), (16, 1032, (8, 10)),
                                         (20, 2048, (64, 4)),
                                         (8, 16, (262148, 64))])      # more row groups than a grid takes along y
def test_stacked_weights_with_adapters(r, cols, rows):
    g = torch.Generator(device="cuda").manual_seed(r * cols)

    def rn(*s):
        return torch.randn(s, generator=g, device="cuda").bfloat16().requires_grad_(True)
    scale = 0.375
    mods = [((True,), rn(rows[0], cols), rn(r, cols), rn(rows[0], r)),
            ((False, True), rn(rows[1], cols), rn(r, cols), rn(rows[1] // 2, r)), ((), rn(3, cols), None, None),
            ((True, False, True), rn(6, cols), rn(2 * r, cols), rn(4, r))]
    d = torch.randn((sum(m[1].shape[0] for m in mods), cols), generator=g, device="cuda").bfloat16()
    leaves = [t for m in mods for t in m[1:] if t is not None]
    if rows[0] > 4 * 65535:                              # more than lora_stack hands to the kernel
        w = AG._LoRAStackFn.apply(scale, tuple(m[0] for m in mods), *(t for m in mods for t in m[1:]))
    else:
        w = AG.lora_stack(tuple(mods), scale)
    grads = torch.autograd.grad(w, leaves, d)
    ref = []
    for on, wm, a, b in mods:
        x = wm.detach().double().requires_grad_(True)
        y = x.clone()
        if a is not None:
            a, b, n = a.detach().double().requires_grad_(True), b.detach().double().requires_grad_(True), wm.shape[0] // len(on)
            at = [i for i, e in enumerate(on) if e]
            y = torch.cat([y[i * n:(i + 1) * n] + (scale * b[at.index(i) * n:][:n] @ a[at.index(i) * r:][:r] if i in at else 0)
                           for i in range(len(on))], 0)
        ref.append((y, [t for t in (x, a, b) if t is not None]))
    whole = torch.cat([y for y, _ in ref], 0)
    _close(w.detach(), whole.detach(), r)
    for got, want in zip(grads, torch.autograd.grad(whole, [t for _, ts in ref for t in ts], d.double())):
        _close(got, want, max(max(rows), cols))


def test_stacked_weights_that_the_kernel_refuses():
    from layers.mvpa import _LoRALinear, _stacked_weights
    mod = _LoRALinear(20, 6, 2, 4, enable=(False, True)).to("cuda", torch.bfloat16)     # rows of 20: no whole chunks
    with torch.no_grad():
        mod.lora_B.normal_()
    plain = torch.nn.Linear(20, 4, bias=False).to("cuda", torch.bfloat16)
    assert AG.lora_stack(((mod.enable, mod.weight, mod.lora_A, mod.lora_B),), 2.0) is None
    w = _stacked_weights((mod, plain))
    assert torch.equal(w, torch.cat([mod.effective_weight(), plain.weight], 0))
    w.sum().backward()
    assert mod.lora_B.grad.abs().sum() > 0


@pytest.mark.parametrize("r", [1, 8, 13])
def test_stacked_weights_with_infinite_adapters(r):
    """An infinity in the last row of a stays one: nothing past the rank is multiplied with it."""
    w, a, b = torch.zeros(6, 16), torch.zeros(r, 16), torch.ones(6, r)
    a[-1, 3], a[0, 5] = float("inf"), -float("inf")
    b[1] = -1
    got = AG.lora_stack((((True,), *(t.cuda().bfloat16() for t in (w, a, b))),), 0.5).float().cpu()
    want = torch.zeros(6, 16)
    for c, sign in ((3, 1), (5, -1)):
        want[:, c] = sign * b[:, 0] * float("inf")
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,kernel", [(1280, True), (1281, False)])
def test_stacked_weights_of_large_rank(rows, kernel):
    """Rank times rows of the largest part up to 160 * 1024 on the kernel."""
    from layers.mvpa import _LoRALinear, _stacked_weights
    mod = _LoRALinear(16, 2 * rows, 128, 4, enable=(False, True)).to("cuda", torch.bfloat16)
    with torch.no_grad():
        mod.lora_B.normal_()
    assert (AG.lora_stack(((mod.enable, mod.weight, mod.lora_A, mod.lora_B),), mod.scaling) is None) is not kernel
    _near(_stacked_weights((mod,)).detach(), mod.effective_weight().detach())


def test_stacked_weights_by_a_list_of_slices():
    """`enable` as any sequence of truth values, as effective_weight() takes it; the binding itself refuses what is no tuple."""
    from layers.mvpa import _LoRALinear, _stacked_weights
    mod = _LoRALinear(16, 6, 2, 4, enable=(False, True)).to("cuda", torch.bfloat16)
    with torch.no_grad():
        mod.lora_B.normal_()
    want = _stacked_weights((mod,))
    for enable in ([False, True], [0, 1], (0, 1)):
        mod.enable = enable
        assert torch.equal(_stacked_weights((mod,)), want)
    bad = (([False, True], mod.weight, mod.lora_A, mod.lora_B),)
    assert AG.lora_stack(bad, 2.0) is None and AG.lora_stack([bad[0]], 2.0) is None
    with pytest.raises(RuntimeError):
        mvpa_hip.lora_stack(bad, 2.0)


@pytest.mark.parametrize("unpack", [lambda t: t.t().contiguous().t(), lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape),
                                    lambda t: t.cpu()], ids=["columns", "offset", "host"])
def test_stacked_weights_with_hooks_on_what_is_saved(unpack):
    """A hook may hand the adapters back in another layout; on the host they are an error, not an address."""
    torch.manual_seed(4)
    w, a, b = (torch.randn(s, device="cuda").bfloat16().requires_grad_(True) for s in ((16, 32), (8, 32), (16, 8)))
    mods, d = (((True,), w, a, b),), torch.randn(16, 32, device="cuda").bfloat16()
    want = torch.autograd.grad(AG.lora_stack(mods, 0.5), (a, b), d)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = AG.lora_stack(mods, 0.5)
        if not unpack(a).is_cuda:
            with pytest.raises(RuntimeError):
                torch.autograd.grad(y, (a, b), d)
            return
        got = torch.autograd.grad(y, (a, b), d)
    assert all(torch.equal(x, z) and x.shape == z.shape for x, z in zip(got, want))


def test_stacked_weights_differentiate_twice():
    torch.manual_seed(3)
    w, a, b = (torch.randn(s, device="cuda").bfloat16().requires_grad_(True) for s in ((16, 32), (8, 32), (8, 8)))
    y = AG.lora_stack((((False, True), w, a, b),), 0.5)
    da, = torch.autograd.grad(y.float().pow(2).sum(), a, create_graph=True)
    grad, = torch.autograd.grad(da.float().sum(), b)
    wd, ad, bd = (t.detach().double().requires_grad_(True) for t in (w, a, b))
    yd = torch.cat([wd[:8], wd[8:] + 0.5 * bd @ ad], 0)
    dd, = torch.autograd.grad(yd.pow(2).sum(), ad, create_graph=True)
    ref, = torch.autograd.grad(dd.sum(), bd)
    assert ((grad.double() - ref).norm() / ref.norm()).item() <= 3e-2


# rows around the 32 of a block, the five blocks of the ring and the shares; outputs around tiles of 128, the smallest ones, operands with a row
# pitch; one share, several, one and two groups of waves
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (31, 8, 8), (63, 128, 128), (64, 136, 120), (65, 8, 264), (160, 8, 8), (161, 1664, 1664), (193, 136, 8), (129, 256, 1024), (700, 1280, 768),
                                   (6400, 768, 1728), (2561, 3456, 768), (1000, 2048, 2056), (20000, 8, 16)])
def test_weight_gradient(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n)
    dy, x = (torch.randn((m, c + 8), generator=g, device="cuda").bfloat16()[:, :c] for c in (n, k))
    dw = mvpa_hip.load_ext().linear_wgrad(dy, x)
    _close(dw, dy.double().t() @ x.double(), m)
    dw = mvpa_hip.load_ext().linear_wgrad(dy.contiguous(), x.contiguous())
    _close(dw, dy.double().t() @ x.double(), m)


# tiles of 256 x 128 and 128 x 256, one share and several; five blocks of rows a share, the last one whole, of one row, of all but one; ragged both ways
@pytest.mark.parametrize("m,n,k", [(289, 2512, 1552), (290, 3400, 1512), (640, 2056, 1928), (1260, 3000, 272), (2623, 1392, 1576), (3009, 3456, 768),
                                   (16001, 1280, 768)])
def test_weight_gradient_on_wide_tiles(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n)
    dy, x = (torch.randn((m, c + 8), generator=g, device="cuda").bfloat16()[:, :c] for c in (n, k))
    want = dy.double().t() @ x.double()
    for a, b in ((dy, x), (dy.contiguous(), x.contiguous())):
        _close(mvpa_hip.load_ext().linear_wgrad(a, b), want, m)


def test_weight_gradient_refuses_rows_off_16_bytes():
    x = torch.randn(64, 24, device="cuda").bfloat16()
    for dy in (x[:, 1:9], x[:, :12], x.t()):
        assert type(mvpa_hip.load_ext().linear_wgrad(dy, x[:dy.shape[0]])) is int
    w = torch.randn(24, 8, device="cuda").bfloat16().requires_grad_(True)
    x = torch.randn(3000, 8, device="cuda").bfloat16()                            # through the autograd function: any rows
    dy = torch.randn(3000 * 24 + 1, device="cuda").bfloat16()[1:].view(3000, 24)
    dw, = torch.autograd.grad(AG.linear(x, w), w, dy)
    _close(dw, dy.double().t() @ x.double(), 3000)


def test_weight_gradient_of_aligned_rows_is_the_kernels(monkeypatch):
    """Through the autograd function, from 2560 rows on: what it returns is what the kernel returned."""
    ext, seen = mvpa_hip.load_ext(), []
    kernel = ext.linear_wgrad

    def record(dy, x):
        seen.append(kernel(dy, x))
        return seen[-1]
    monkeypatch.setattr(ext, "linear_wgrad", record)
    for m in (2559, 2560):
        x, dy = torch.randn(m, 72, device="cuda").bfloat16(), torch.randn(m, 136, device="cuda").bfloat16()
        w = torch.randn(136, 72, device="cuda").bfloat16().requires_grad_(True)
        dw, = torch.autograd.grad(AG.linear(x, w), w, dy)
        _close(dw, dy.double().t() @ x.double(), m)
    assert len(seen) == 1 and isinstance(seen[0], torch.Tensor) and torch.equal(seen[0], dw)


def test_gradients_of_several_losses_at_once():
    """is_grads_batched through a projection of 2560 rows and more and through stacked weights with adapters."""
    torch.manual_seed(5)
    mods = tuple((on, *(torch.randn(s, device="cuda").bfloat16().requires_grad_(True) for s in ((rows, 64), (8, 64), (16, 8))))
                 for on, rows in (((True,), 16), ((False, True), 32)))
    leaves = [t for m in mods for t in m[1:]]
    y = AG.linear(torch.randn(2560, 64, device="cuda").bfloat16(), AG.lora_stack(mods, 0.5))
    d = torch.randn(3, *y.shape, device="cuda").bfloat16()
    got = torch.autograd.grad(y, leaves, d, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for whole, one in zip(got, torch.autograd.grad(y, leaves, d[i], retain_graph=True)):
            _near(whole[i], one)


def test_weight_gradient_of_rows_far_apart():
    """Row pitches past 32 bits of a block's bytes: 40 rows of a view into 5.4 GB, either operand."""
    pitch = (1 << 26) + 8
    far = torch.empty(40 * pitch, dtype=torch.bfloat16, device="cuda").view(40, pitch)[:, :136]
    near = torch.randn(40, 264, device="cuda").bfloat16()
    far.copy_(torch.randn(40, 136, device="cuda").bfloat16())
    for dy, x in ((far, near), (near, far)):
        got = mvpa_hip.load_ext().linear_wgrad(dy, x)
        _close(got, dy.double().T @ x.double(), 40)


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="two GPUs")
def test_operands_on_two_gpus_are_refused():
    """As tensor operations refuse them: no kernel reads another GPU's memory."""
    here, there = (torch.ones(16, 16, dtype=torch.bfloat16, device=f"cuda:{i}") for i in range(2))
    for mods in (((True,), here, there, here),), (((True,), here, here, here), ((), there, None, None)):
        assert AG.lora_stack(mods, 1.0) is None
        with pytest.raises(RuntimeError):
            mvpa_hip.lora_stack(mods, 1.0)
    with pytest.raises(RuntimeError):
        mvpa_hip.lora_stack((((True,), here, here, here),), 1.0, there)
    with pytest.raises(RuntimeError):
        mvpa_hip.load_ext().linear_wgrad(here, there)


# tiles of 128 columns and 128, 192 and 256 rows, of 192 and 256 columns, whole and ragged each way; two blocks of a contraction and many
@pytest.mark.parametrize("M,K,N,E", [(512, 128, 128, 128), (700, 192, 320, 192), (2600, 768, 1728, 768), (6400, 768, 1728, 768), (6001, 128, 832, 256),
                                     (6300, 256, 704, 128), (16000, 128, 1728, 128), (13000, 128, 192, 1024), (20001, 192, 576, 192)])
def test_gated_mlp(M, K, N, E):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)

    def rn(*s, std=1.0):
        return (std * torch.randn(s, generator=g, device="cuda")).bfloat16()
    x, wg, wu, wd = rn(M, K), rn(N, K, std=K ** -0.5), rn(N, K, std=K ** -0.5), rn(E, N, std=N ** -0.5)
    x[0] *= 60                                                        # exp(-gate) overflows, underflows
    dy, ext = rn(M, E), mvpa_hip.load_ext()
    # the launches against the products by themselves, the same sums and roundings, and the gates in 64 bits
    gu, mid = ext.gated_rows(x, wg, wu)
    w = torch.cat([wg, wu], 0)
    both = mvpa_hip.linear(x, w)
    assert torch.equal(gu, both)
    dgu = ext.gated_rows_backward(dy, wd, gu)
    gate, up = (t.double() for t in gu.chunk(2, -1))
    s, dm = torch.sigmoid(gate), ext.linear_nn(dy, wd).double()
    _close(mid, gate * s * up)
    _close(dgu, torch.cat([dm * up * s * (1 + gate * (1 - s)), dm * gate * s], -1))
    # and the same bits as the passes by themselves
    assert torch.equal(mid, mvpa_hip.silu_gate(gu)) and torch.equal(dgu, mvpa_hip.silu_gate(gu, dm.bfloat16()))
    assert torch.equal(ext.linear_nn2(dgu, wg, wu), ext.linear_nn(dgu, w))
    # and the whole with its gradients against 64 bits, rounded where the pass rounds
    leaves = [t.requires_grad_() for t in (x, wg, wu, wd)]
    y = AG.gated_mlp(x.view(1, M, K), wg, wu, wd)
    got = torch.autograd.grad(y, leaves, dy.view(1, M, E), retain_graph=True)
    xd, gd, ud, dd = (t.detach().double() for t in leaves)
    dm = dy.double() @ dd
    dgate, dup = dm * up * s * (1 + gate * (1 - s)), dm * gate * s
    want = dgate @ gd + dup @ ud, dgate.t() @ xd, dup.t() @ xd, dy.double().t() @ (gate * s * up)
    assert (y[0].double() - (gate * s * up) @ dd.t()).norm() <= 4e-3 * y.double().norm()
    for a, b in zip(got, want):
        assert (a.double() - b).norm() <= 6e-3 * b.norm()             # one rounding of the operands, one of the result
    if M < 3000:
        again = torch.autograd.grad(y, leaves, dy.view(1, M, E), create_graph=True)
        rows = torch.autograd.grad(y, leaves, torch.stack([dy, 2 * dy]).view(2, 1, M, E), is_grads_batched=True)
        for a, r, b in zip(again, rows, want):
            assert a.requires_grad and (a.double() - b).norm() <= 1e-2 * b.norm() and (r[1].double() - 2 * b).norm() <= 2e-2 * b.norm()
    frozen = AG.gated_mlp(x.detach(), wg.detach(), wu, wd.detach())
    assert torch.equal(torch.autograd.grad(frozen, wu, dy)[0], got[2])


def test_gated_mlp_refuses():
    def t(*s):
        return torch.zeros(s, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    assert AG.gated_mlp(t(511, 128), t(128, 128), t(128, 128), t(128, 128)) is None
    assert AG.gated_mlp(t(512, 96), t(128, 96), t(128, 96), t(128, 128)) is None
    assert AG.gated_mlp(t(512, 128), t(136, 128), t(136, 128), t(128, 136)) is None
    assert AG.gated_mlp(t(512, 128), t(128, 128), t(128, 128).float(), t(128, 128)) is None
    assert AG.gated_mlp(t(512, 128), t(128, 256)[:, :128], t(128, 128), t(128, 128)) is None


# one wave a row and a workgroup a row, odd sizes of every level, rows at odd boundaries of 16 bytes (odd L); rows: one, fewer
# than a wave's share, every group of rows and a remainder
@pytest.mark.parametrize("L,M,wt", [(97, 1, torch.float32), (512, 131, torch.bfloat16), (1001, 33, torch.float32),
                                    (2560, 2051, torch.bfloat16), (4095, 65, torch.bfloat16),
                                    (16032, 3, torch.float32)])                  # (the longest in one pass)
def test_encoder_norm(L, M, wt):
    """Analysis and norm of a training pass against the two kernels, the weight's gradient against 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(L + M)
    total = sum(mvpa_hip.dwt_sizes(L)[1])
    pitch = (total + 63) // 64 * 64
    x = torch.randn((M, L), generator=g, device="cuda")
    w = (1 + 0.1 * torch.randn(total, generator=g, device="cuda")).to(wt).requires_grad_()
    y = AG.encoder_norm(x, w, pitch, 1e-5)
    coeffs = mvpa_hip.wavedec_db4(x)
    ref = mvpa_hip.rmsnorm(coeffs, w.detach().float(), 1e-5, out=torch.empty(M, total, device="cuda"))
    assert (y[:, total:] == 0).all()
    assert ((y[:, :total].float() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-6).all()
    dy = torch.randn((M, pitch), generator=g, device="cuda").bfloat16()
    dw, = torch.autograd.grad(y, w, dy, retain_graph=True)
    c = coeffs.double()
    inv = (c.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
    assert dw.dtype == wt
    _close(dw, (dy[:, :total].double() * c * inv).sum(0), M * 4)
    again, = torch.autograd.grad(y, w, dy.clone().requires_grad_(), create_graph=True)      # the general expression
    assert ((again.double() - dw.double()).abs() <= 2.0 ** -7 * dw.double().abs() + 1e-3 * M ** 0.5).all()
    both, = torch.autograd.grad(y, w, torch.stack([dy, 2 * dy]), is_grads_batched=True)
    assert ((both[1].double() - 2 * again.double()).abs() <= 2.0 ** -7 * both[1].double().abs() + 1e-3 * M ** 0.5).all()


def test_weight_gradient_of_the_encoder_norm_takes_one_row_of_any_stride():
    total, pitch = 550, 576
    x, w = torch.randn(1, 512, device="cuda"), torch.ones(total, device="cuda", requires_grad=True)
    dy = torch.randn(pitch, 1, device="cuda").bfloat16()
    got, = torch.autograd.grad(AG.encoder_norm(x, w, pitch, 1e-5), w, dy.t())
    want, = torch.autograd.grad(AG.encoder_norm(x, w, pitch, 1e-5), w, dy.t().clone(memory_format=torch.contiguous_format).view(1, pitch))
    assert dy.t().stride(0) == 1 and torch.equal(got, want)


def test_a_frozen_encoder_norm_keeps_no_coefficients(monkeypatch):
    x, w = torch.randn(33, 512, device="cuda"), (1 + 0.1 * torch.randn(550, device="cuda")).requires_grad_()
    kept = AG.encoder_norm(x, w, 576, 1e-5)
    with torch.no_grad():
        assert torch.equal(AG.encoder_norm(x, w, 576, 1e-5), kept)
    monkeypatch.setattr(mvpa_hip, "wavedec_db4_rmsnorm_saved", None)
    got = AG.encoder_norm(x, w.detach(), 576, 1e-5)
    assert got.grad_fn is None and torch.equal(got, kept)


@pytest.mark.parametrize("how", ["subclass", "object", "class"])
def test_an_analysis_of_its_own_is_heard_in_training(monkeypatch, how):
    def block(self, x):
        return 2.0 + mvpa_hip.wavedec_db4(x.float())
    kind = type("Own", (WaveEncoder,), dict(block=block)) if how == "subclass" else WaveEncoder
    enc = kind(512, 64).to("cuda", torch.bfloat16).train()
    if how == "object":
        enc.block = lambda x: block(enc, x)
    elif how == "class":
        monkeypatch.setattr(WaveEncoder, "block", block)
    x = torch.randn(9, 512, device="cuda")
    normed = mvpa_hip.rmsnorm(2.0 + mvpa_hip.wavedec_db4(x), enc.ln.weight.detach(), 1e-5, out_dtype=torch.bfloat16)
    want = normed.double() @ enc.proj.weight.detach().double().T
    assert ((enc(x).double() - want).norm() / want.norm()).item() <= 1e-2          # one bf16 rounding of the product


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 3e38], ids=str)
@pytest.mark.parametrize("L", [97, 512, 2560])             # one wave a row, a workgroup a row
def test_columns_past_the_coefficients_are_zero_whatever_a_row_holds(L, bad):
    total = sum(mvpa_hip.dwt_sizes(L)[1])
    pitch = (total + 63) // 64 * 64 + 64
    x = torch.randn(9, L, device="cuda")
    good = mvpa_hip.wavedec_db4_rmsnorm(x, torch.ones(total, device="cuda"), pitch)
    x[4, L // 3] = bad
    w = torch.ones(total, device="cuda", requires_grad=True)
    for y in (mvpa_hip.wavedec_db4_rmsnorm(x, w.detach(), pitch), AG.encoder_norm(x, w, pitch, 1e-5)):
        assert (y[:, total:] == 0).all()
        rows = torch.arange(9, device="cuda") != 4
        assert torch.equal(y[rows], good[rows])


def test_encoder_norm_of_rows_beyond_the_one_pass():
    for L in (16033, 40000):
        assert AG.encoder_norm(torch.zeros(2, L, device="cuda"), torch.ones(sum(mvpa_hip.dwt_sizes(L)[1]), device="cuda"), 40960, 1e-5) is None
    assert AG.encoder_norm(torch.zeros(0, 512, device="cuda"), torch.ones(550, device="cuda"), 576, 1e-5) is None
