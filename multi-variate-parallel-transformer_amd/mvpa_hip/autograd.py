"""Differentiable wrappers of the library's dense ops, for gradients through the layer and stack
modules (the reference trains through layers/mvpa.py:280-337 and models/mvpformer.py:132-147).

Forward passes are the library's kernels.  Of the backward passes of the bf16 products dX = dY W and dW = dY^T X
run on kernels of the library where those are the faster ones (_input_gradient, _weight_gradient), elsewhere on the
vendor library through torch.matmul, which reads transposed operands in place too.  Norm,
gated activation and residual sums run on kernels of the library both ways (csrc/mvpa_train.hip).  The attention operator itself is
`attentions.attn.FlashMVPA` (mvpa_backward kernels).
"""
from __future__ import annotations

import torch

import mvpa_hip


def wants_grad(*tensors) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def _mapped(*tensors) -> bool:
    """Whether a vmap runs over one of them (autograd.grad with is_grads_batched, torch.func): such a tensor has no
    memory of its own that a kernel of the library could read."""
    f = torch._C._functorch
    return any(t is not None and (f.is_functorch_wrapped_tensor(t) or f.is_legacy_batchedtensor(t)) for t in tensors)


def _wgrad_on_kernel(m, n, k) -> bool:
    """Whether the kernel of csrc/mvpa_wgrad.hip is the faster one for dY^T X of [m, n] and [m, k], by the tiles of 128 x 128
    in its output.  us, both launches of it / the vendor library, eight sets of rows in turn:
        25 tiles  [640,640]    2560 rows 16 / 19, 6400 22 / 38, 25600 38 / 156
        36        [768,768]    2816 19 / 20, 3072 19 / 22, 6400 22 / 39, 25600 48 / 157
        60        [1280,768]   2560 23 / 19, 3072 23 / 22, 3584 23 / 25, 6400 26 / 42, 25600 70 / 172
        84        [768,1728]   2560 21 / 24, 6400 32 / 51, 25600 93 / 283
        162       [3456,768]   2560 26 / 29, 6400 52 / 72, 25600 171 / 280, 65536 410 / 541
        169       [1664,1664]  2560 27 / 29, 5120 46 / 55, 6400 53 / 72
        180       [2560,1152]  2560 27 / 29, 6400 65 / 72, 16384 144 / 174
        225       [1920,1920]  2560 29 / 31, 6400 64 / 74, 25600 232 / 259
        432       [2048,3456]  2560 49 / 49, 6400 116 / 108, 25600 484 / 437
    Fewer rows do not pay for the second launch, and with many tiles the vendor's larger ones fill the chip too; so they do
    where many tiles meet many rows, earlier where rows do not start at lines of 128 bytes (rows times tiles in millions: [3456,768]
    10.6 410 / 541, [1536,2048] 25 1008 / 1024; [640,4000] 5.2 241 / 312, 10.5 478 / 428).  Long thin outputs are padding for the most
    part (25600 rows of [8,16000] 144 / 139).  The limits of tiles and of rows from 162 tiles on were drawn with a kernel that took up to a
    fifth more (180 tiles 79 / 70, 225 80 / 73 over 6400 rows): they lie on the safe side, and farther since tiles of 256 x 128 took the larger
    problems ([3456,768] over 6400 rows 44, 25600 139; [768,1728] over 32768 111 -> 93)."""
    tiles = -(-n // 128) * -(-k // 128)
    if tiles > 170 or (min(n, k) < 64 and tiles > 96):
        return False
    least = 2560 if tiles <= 30 else 3072 if tiles <= 50 else 3584 if tiles <= 64 else 2560 if tiles <= 162 else 6400
    return m >= least and (tiles < 64 or m * tiles < (12 << 20 if n % 64 == 0 and k % 64 == 0 else 8 << 20))


def _weight_gradient(dy, x):
    """dy^T x of bf16 rows, on the library's kernel where that is the faster one."""
    if _mapped(dy, x):                                       # rows of several gradients: one product, no batched one
        return torch.matmul(dy.t().contiguous(), x)
    if _wgrad_on_kernel(*dy.shape, x.shape[-1]) and not torch.is_grad_enabled():
        dw = mvpa_hip.load_ext().linear_wgrad(dy, x)
        # rows that do not start at 16-byte boundaries or overlap are the vendor library's; any other status is an error
        if type(dw) is not int or dw not in (mvpa_hip.ERR_ALIGN, mvpa_hip.ERR_SHAPE, mvpa_hip.ERR_UNSUPPORTED):
            return mvpa_hip._taken(dw)
    return torch.matmul(dy.t(), x)


def _dx_on_kernel(m, n, k) -> bool:
    """Whether the library's product dY W of [m, k] and [k, n] is the faster one, by its tiles of 128 x 128.  us, it / the vendor
    library, four sets of operands in turn:
        k 192   [640,.]    600 rows (25 tiles) 4.6 / 4.9, 6400 5.4 / 7.9
        k 512   [512,.]    600 rows (20) 6.4 / 6.9, 6400 7.6 / 11.5
        k 768   [576,.]    1600 rows (65) 9.0 / 8.6, 2048 (80) 8.9 / 10.8
                [768,.]    1024 rows (48) 8.5 / 8.4, 1600 (78) 8.7 / 11.1, 6400 12.5 / 20.7, 20000 28.0 / 28.5
                [1728,.]   600 rows (70) 8.9 / 9.4, 6400 21.3 / 26.0, 20000 62 / 75
        k 1280  [768,.]    1024 rows (48) 11.5 / 11.2, 1600 (78) 11.7 / 12.3, 6400 18.8 / 27.2
        k 2048  [2048,.]   600 rows (80) 16.5 / 17.1, 2800 27 / 39, 5120 44.7 / 43.8, 20000 162 / 159
                [5632,.]   600 rows (220) 20.4 / 24.6, 1600 41.2 / 39.7, 6400 129 / 158
        k 3456  [768,.]    1024 rows (48) 23.7 / 19.9, 1600 (78) 23.8 / 23.6, 4096 29 / 41, 6400 39.9 / 40.7
        k 4096  [1024,.]   1024 rows (64) 27.4 / 23.3, 1600 (104) 27.7 / 32.0, 6400 57 / 61, 9000 83 / 80, 20000 166 / 156
        k 11264 [2048,.]   600 rows (80) 79 / 90, 1024 (128) 91 / 87, 6400 250 / 361
    Up to 191 columns are a tile or two across, half empty: few rows of them, and long contractions, are the vendor library's ([16,.] k 192 6920 rows
    5.2 / 4.5; [48,.] k 512 1330 6.9 / 5.7; [8,.] k 5632 13209 43 / 29, [152,.] k 3456 4517 23.9 / 19.7, 104 15888 37 / 32; taken: [160,.] k 384 10902
    6.8 / 11.1, [104,.] k 1728 25571 23 / 39).  Of 240 shapes of 192 columns or more that the rule takes, 0.79 of the vendor's time on average, 11 are
    slower, by 1 to 8 % and at no size in particular (k 2048 [512,.] 18785 rows 44.8 / 43.0, k 576 [320,.] 3010 7.6 / 7.0): the vendor library picks
    another tile there."""
    tiles = -(-m // 128) * -(-n // 128)
    return m >= 512 and (k <= 512 or tiles >= 72) and (n >= 192 or (tiles >= 72 and k <= 2048))


def _input_gradient(dy, w):
    """dy w of bf16 rows, on the library's kernel where that is the faster one."""
    if _dx_on_kernel(dy.shape[0], w.shape[1], w.shape[0]) and not torch.is_grad_enabled() and not _mapped(dy, w):
        dx = mvpa_hip.load_ext().linear_nn(dy, w)
        # contractions that are not whole blocks and rows that do not start at 16-byte boundaries are the vendor library's
        if type(dx) is not int or dx not in (mvpa_hip.ERR_ALIGN, mvpa_hip.ERR_SHAPE, mvpa_hip.ERR_UNSUPPORTED):
            return mvpa_hip._taken(dx)
    return torch.matmul(dy, w)


class _LinearFn(torch.autograd.Function):
    """y = x @ w^T, bf16, any leading shape of x: forward on the GPU library, backward dX and dW as above."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return mvpa_hip.linear(x, w)

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        k = x.shape[-1]
        dy2 = dy.reshape(-1, dy.shape[-1]).contiguous()
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = _input_gradient(dy2, w).view(x.shape)                            # [M,N] @ [N,K]
        if ctx.needs_input_grad[1]:
            dw = _weight_gradient(dy2, x.reshape(-1, k))                          # [N,M] @ [M,K]
        return dx, dw


class _LinearF32Fn(torch.autograd.Function):
    """The same in fp32 (the library's fp32 MFMA product, forward and both backward products)."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return mvpa_hip.linear_f32(x, w)

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.shape[-1]).contiguous()
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = mvpa_hip.linear_f32(dy2, w.t().contiguous()).view(x.shape)
        if ctx.needs_input_grad[1]:
            dw = mvpa_hip.linear_f32(dy2.t().contiguous(), x.reshape(-1, x.shape[-1]).t().contiguous())
        return dx, dw


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w^T on the GPU library, bf16 or fp32 (differentiably when a gradient is wanted);
    tensors that are not on the GPU take torch's own linear."""
    if x.is_cuda and x.dtype == torch.bfloat16:
        w = w.to(torch.bfloat16)
        if wants_grad(x, w):
            return _LinearFn.apply(x, w)
        return mvpa_hip.linear(x, w.detach())
    if x.is_cuda and x.dtype == torch.float32:
        w = w.to(torch.float32)
        if wants_grad(x, w):
            return _LinearF32Fn.apply(x, w)
        return mvpa_hip.linear_f32(x, w.detach())
    return torch.nn.functional.linear(x, w.to(x.dtype))


MAX_NORM_COLS = 4096          # the longest row of the library's RMSNorm backward


def _norm_backward(ctx, x, w, dy, res, need_x, need_w):
    """(dx, dw) of y = RMSNorm(x) w, dx with the gradient `res` of the rows themselves added where given."""
    if (x.is_cuda and dy.dtype == torch.bfloat16 and x.dtype in (torch.bfloat16, torch.float32) and x.numel()
            and w.dtype in (torch.bfloat16, torch.float32) and x.shape[-1] <= MAX_NORM_COLS
            and not torch.is_grad_enabled()):
        return mvpa_hip.norm_backward(x, w, dy, res, ctx.eps, need_x, need_w)
    # other types, and a backward that is differentiated itself (create_graph)
    xf, wf, g = x.float(), w.float(), dy.float()
    r = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + ctx.eps)
    gw = g * wf
    dx = dw = None
    if need_x:
        dx = r * gw - xf * r.pow(3) * (xf * gw).mean(-1, keepdim=True)
        dx = (dx if res is None else dx + res.float()).to(x.dtype)
    if need_w:
        dw = (g * xf * r).reshape(-1, x.shape[-1]).sum(0).to(w.dtype)
    return dx, dw


class _RMSNormFn(torch.autograd.Function):
    """y = x * rsqrt(mean(x^2) + eps) * w, forward and backward on the library's kernels."""

    @staticmethod
    def forward(ctx, x, w, eps, out_dtype):
        ctx.save_for_backward(x, w)
        ctx.eps = eps
        return mvpa_hip.rmsnorm(x, w, eps, out_dtype=out_dtype)

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        return (*_norm_backward(ctx, x, w, dy, None, *ctx.needs_input_grad[:2]), None, None)


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, out_dtype=None) -> torch.Tensor:
    if wants_grad(x, w):
        return _RMSNormFn.apply(x, w, eps, out_dtype)
    return mvpa_hip.rmsnorm(x, w, eps, out_dtype=out_dtype)


class _EncoderNormFn(torch.autograd.Function):
    """RMSNorm of the wavelet coefficients of signal rows, zeros past them up to whole blocks of the projection.  The transform has
    no parameters and carries no gradient (models/fftencoder.py:80: no_grad)."""

    @staticmethod
    def forward(ctx, x, w, pitch, eps):
        y, coeffs, inv = mvpa_hip.wavedec_db4_rmsnorm_saved(x, w, pitch, eps)
        ctx.save_for_backward(coeffs, inv, w)
        return y

    @staticmethod
    def backward(ctx, dy):
        coeffs, inv, w = ctx.saved_tensors
        if not ctx.needs_input_grad[1]:
            return None, None, None, None
        if not torch.is_grad_enabled() and not _mapped(dy) and dy.dtype == torch.bfloat16:
            return None, mvpa_hip.norm_dw(coeffs, inv, dy, w), None, None
        n = w.shape[0]                                       # a backward that is differentiated itself, or mapped over
        return None, (dy[:, :n].float() * coeffs[:, :n] * inv[:, None]).sum(0).to(w.dtype), None, None


def encoder_norm(x: torch.Tensor, w: torch.Tensor, pitch: int, eps: float):
    """[M, L] signal rows -> bf16 [M, pitch]: wavelet analysis, norm and zeros in one pass, or None where the rows are
    too long for it, are none, or the weight is of another type."""
    if not x.is_cuda or w.dtype not in (torch.float32, torch.bfloat16) or not mvpa_hip.wavedec_fits(x):
        return None
    if not wants_grad(w):                                    # a frozen norm: nothing is kept
        return mvpa_hip.wavedec_db4_rmsnorm(x, w, pitch, eps)
    return _EncoderNormFn.apply(x.detach().float(), w, pitch, eps)


class _Add3RMSNormFn(torch.autograd.Function):
    """(s, RMSNorm(s) w) with s = a + b + c: the residual update of a block and the norm behind it."""

    @staticmethod
    def forward(ctx, a, b, c, w, eps):
        ctx.set_materialize_grads(False)
        total, normed = mvpa_hip.add3_rmsnorm(a, b, c, w, eps)
        ctx.save_for_backward(total, w)
        ctx.eps = eps
        return total, normed

    @staticmethod
    def backward(ctx, d_total, d_normed):
        total, w = ctx.saved_tensors
        d, dw = d_total, None
        if d_normed is not None:
            d, dw = _norm_backward(ctx, total, w, d_normed, d_total, any(ctx.needs_input_grad[:3]),
                                   ctx.needs_input_grad[3])
        return d, d, d, dw, None


def add3_rmsnorm(a, b, c, w, eps):
    """(a + b + c, RMSNorm(a + b + c) * w) in one pass each way, or None where the operands are not bf16
    rows of whole 16-byte chunks on the GPU, or do not start at one."""
    if (not a.is_cuda or not a.dtype == b.dtype == c.dtype == torch.bfloat16 or not a.shape == b.shape == c.shape
            or a.shape[-1] % 8 or a.shape[-1] > MAX_NORM_COLS or not a.numel()
            or w.dtype not in (torch.bfloat16, torch.float32)
            or any(t.is_contiguous() and t.data_ptr() % 16 for t in (a, b, c))       # others are copied to a row of their own
            or w.dtype == torch.float32 and w.data_ptr() % 16):
        return None
    return _Add3RMSNormFn.apply(a, b, c, w, eps)


class _SiluGateFn(torch.autograd.Function):
    """silu(gate) * up of rows [gate | up], one pass each way."""

    @staticmethod
    def forward(ctx, gu):
        ctx.save_for_backward(gu)
        return mvpa_hip.silu_gate(gu)

    @staticmethod
    def backward(ctx, d):
        gu, = ctx.saved_tensors
        if not torch.is_grad_enabled():
            return mvpa_hip.silu_gate(gu, d)
        gate, up = gu.float().chunk(2, -1)                   # a backward that is differentiated itself
        s, df = torch.sigmoid(gate), d.float()
        return torch.cat([df * up * s * (1 + gate * (1 - s)), df * gate * s], -1).to(gu.dtype)


def gated_mid(x: torch.Tensor, w_gate_up: torch.Tensor) -> torch.Tensor:
    """silu(x @ gate^T) * (x @ up^T) for w_gate_up = [gate; up]: one product, one pass over its result."""
    return _SiluGateFn.apply(linear(x, w_gate_up))


class _GatedMLPFn(torch.autograd.Function):
    """(silu(x @ wg^T) * (x @ wu^T)) @ wd^T for bf16 rows x [M, K]: the gate and up rows and their product come out of one
    launch, and so do the gradients of gate and up with the product that the down projection's backward is."""

    @staticmethod
    def forward(ctx, x, wg, wu, wd):
        gu, mid = mvpa_hip._taken(mvpa_hip.load_ext().gated_rows(x, wg, wu))
        ctx.save_for_backward(x, wg, wu, wd, gu, mid)
        return mvpa_hip.linear(mid, wd)

    @staticmethod
    def backward(ctx, dy):
        x, wg, wu, wd, gu, mid = ctx.saved_tensors
        need_x, need_g, need_u, need_d = ctx.needs_input_grad
        if torch.is_grad_enabled() or _mapped(dy):           # a backward that is differentiated itself, or mapped over
            xf, g, u, d, df = x.float(), wg.float(), wu.float(), wd.float(), dy.float()
            gate, up, dm = xf @ g.t().contiguous(), xf @ u.t().contiguous(), df @ d
            s = torch.sigmoid(gate)
            dg, du = dm * up * s * (1 + gate * (1 - s)), dm * gate * s
            grads = (dg @ g + du @ u, dg.t().contiguous() @ xf, du.t().contiguous() @ xf, df.t().contiguous() @ (gate * s * up))
            return tuple(a.to(b.dtype) if n else None for a, b, n in zip(grads, (x, wg, wu, wd), ctx.needs_input_grad))
        ext, n = mvpa_hip.load_ext(), wg.shape[0]
        dy = dy.contiguous()
        dwd = _weight_gradient(dy, mid) if need_d else None
        dx = dwg = dwu = None
        if need_x or need_g or need_u:
            if dy.data_ptr() % 16:
                dy = dy.clone()
            dgu = mvpa_hip._taken(ext.gated_rows_backward(dy, wd, gu))
            if need_x:
                if _dx_on_kernel(x.shape[0], x.shape[1], 2 * n):
                    dx = mvpa_hip._taken(ext.linear_nn2(dgu, wg, wu))
                else:
                    dx = torch.matmul(dgu, torch.cat([wg, wu], 0))
            if need_g or need_u:
                dw = _weight_gradient(dgu, x)
                dwg, dwu = dw[:n] if need_g else None, dw[n:] if need_u else None
        return dx, dwg, dwu, dwd


def gated_mlp(x: torch.Tensor, wg: torch.Tensor, wu: torch.Tensor, wd: torch.Tensor):
    """wd applied to silu(x @ wg^T) * (x @ wu^T) with gradients, or None where the operands are not bf16 rows and weights in whole
    blocks on the GPU, at least 512 rows of them."""
    k, n, e = x.shape[-1], wg.shape[0], wd.shape[0]
    if (not all(t.is_cuda and t.dtype == torch.bfloat16 and t.device == x.device for t in (x, wg, wu, wd)) or _mapped(x, wg, wu, wd)
            or k % 64 or n % 64 or e % 64 or k < 128 or n < 128 or e < 128 or x.numel() < 512 * k
            or max(k, n, e) > 1 << 20 or wg.shape != (n, k) or wu.shape != (n, k) or wd.shape != (e, n)
            or not all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (wg, wu, wd))):
        return None
    rows = x.reshape(-1, k)
    if not rows.is_contiguous() or rows.data_ptr() % 16:
        rows = rows.clone(memory_format=torch.contiguous_format)
    return _GatedMLPFn.apply(rows, wg, wu, wd).view(*x.shape[:-1], e)


class _CosineStepsFn(torch.autograd.Function):
    """Cosine similarity of step t + 1 of nxt and step t of pred [B, T, C, E], one pass each way."""

    @staticmethod
    def forward(ctx, nxt, pred, eps):
        ctx.save_for_backward(nxt, pred)
        ctx.eps = eps
        return mvpa_hip.cosine_similarity_steps(nxt, pred, eps)

    @staticmethod
    def backward(ctx, d):
        nxt, pred = ctx.saved_tensors
        if not torch.is_grad_enabled() and not _mapped(d):
            return (*mvpa_hip.cosine_steps_backward(nxt, pred, d, ctx.eps, *ctx.needs_input_grad[:2]), None)
        # a backward that is differentiated itself, or mapped over
        a, b, d = nxt[:, 1:].float(), pred[:, :-1].float(), d[..., None]
        na, nb = a.norm(dim=-1, keepdim=True), b.norm(dim=-1, keepdim=True)
        ia, ib = 1 / na.clamp_min(ctx.eps), 1 / nb.clamp_min(ctx.eps)
        s, tiny = ((a * ia) * (b * ib)).sum(-1, keepdim=True), torch.finfo(torch.float32).tiny
        da = d * (b * ia * ib - a * s * ia / na.clamp_min(tiny))
        db = d * (a * ia * ib - b * s * ib / nb.clamp_min(tiny))
        pad = torch.nn.functional.pad
        return pad(da, (0, 0, 0, 0, 1, 0)).to(nxt.dtype), pad(db, (0, 0, 0, 0, 0, 1)).to(pred.dtype), None


def cosine_steps(nxt: torch.Tensor, pred: torch.Tensor, eps: float = 1e-8):
    """torch.cosine_similarity(nxt[:, 1:], pred[:, :-1], dim=-1) in fp32 with gradients, or None where the two are not bf16
    rows of whole 16-byte chunks on the GPU, or there is no pair of steps."""
    if (not nxt.is_cuda or not nxt.dtype == pred.dtype == torch.bfloat16 or nxt.shape != pred.shape or nxt.dim() != 4
            or nxt.shape[-1] % 8 or nxt.shape[1] < 2 or not nxt.numel() or nxt.device != pred.device or _mapped(nxt, pred)
            or any(t.is_contiguous() and t.data_ptr() % 16 for t in (nxt, pred))):     # others are copied to rows of their own
        return None
    return _CosineStepsFn.apply(nxt, pred, eps)


class _LoRAStackFn(torch.autograd.Function):
    """Weights of several modules, adapters added, stacked by rows; one launch each way.  tensors: w, a, b of
    each module in turn, a and b None where it has no adapter."""

    @staticmethod
    def forward(ctx, scale, enables, *tensors):
        ctx.conf = scale, enables, [w.shape[0] for w in tensors[::3]]
        ctx.save_for_backward(*(t for i, t in enumerate(tensors) if i % 3))       # w is not needed again
        return mvpa_hip.lora_stack(_lora_mods(enables, tensors[::3], tensors[1::3], tensors[2::3]), scale)

    @staticmethod
    def backward(ctx, d):
        scale, enables, rows = ctx.conf
        a, b = ctx.saved_tensors[::2], ctx.saved_tensors[1::2]
        dw = d.split(rows)
        needs = ctx.needs_input_grad[2:]
        adapters = [None] * (2 * len(rows))
        if torch.is_grad_enabled() or _mapped(d, *a, *b):     # a backward that is differentiated itself, or mapped over
            for m, (on, am, bm) in enumerate(zip(enables, a, b)):
                if am is None:
                    continue
                n, r = rows[m] // len(on), bm.shape[1]
                parts = [dw[m][i * n:(i + 1) * n] * scale for i, e in enumerate(on) if e]
                adapters[2 * m] = torch.cat([(x.t().contiguous() @ bm[j * n:(j + 1) * n]).t() for j, x in enumerate(parts)], 0)
                adapters[2 * m + 1] = torch.cat([x @ am[j * r:(j + 1) * r].t() for j, x in enumerate(parts)], 0)
        elif any(needs[1::3]) or any(needs[2::3]):
            adapters = mvpa_hip.lora_stack(_lora_mods(enables, dw, a, b), scale, d)
        grads = []
        for m in range(len(rows)):
            grads += [dw[m], adapters[2 * m], adapters[2 * m + 1]]
        return (None, None, *(g if n else None for g, n in zip(grads, needs)))


def _lora_mods(enables, w, a, b):
    return tuple(zip(enables, w, a, b))


def lora_stack(mods, scale: float):
    """cat([w + scale * b a over the enabled slices], 0) for mods = ((enable, w, a, b), ..), a and b None where a
    module has no adapter; None where they are not contiguous bf16 matrices on the GPU at 16-byte boundaries."""
    if not mvpa_hip.load_ext().lora_fits(mods):
        return None
    return _LoRAStackFn.apply(scale, tuple(m[0] for m in mods), *(t for m in mods for t in m[1:]))
