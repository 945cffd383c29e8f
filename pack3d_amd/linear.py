"""The layer's linear maps under autograd, with the weight gradients from the
HIP kernel ``p3d_weight_grad``.

For y = x W^T the weight gradient dW = dy^T x contracts over every token
(262,144 at 64^3) into a small matrix; the library GEMM runs it with a
handful of workgroups.  ``p3d_weight_grad`` splits the tokens over the whole
GPU and sums fp32 partials in a fixed order.  The three input projections
run as one kernel over the normalised tokens (``p3d_project_linear``), their
input gradient as one contraction (``p3d_input_grad``); the output
projection's products stay torch GEMMs.  These functions replace the to_q, to_kv,
gate (attention.py:64-67,85 of amilworks/Pack3D) and to_out + residual
(attention.py:89) steps of ``PACK3DAttention.forward`` when it runs in a
16-bit compute type with autograd active, and those of an fp32 model in
training (``fp32_training``; its products stay torch's, its LayerNorm and
gate torch modules); weight gradients are accumulated in fp32 (torch's
autocast path rounds them to the compute type first).
"""
from __future__ import annotations

import torch
from torch.autograd.function import once_differentiable

from . import _lib

# The kernel's workgroups own up to 256 output rows, up to 256 input columns
# and a range of rows of dy / x; splits are chosen for at most WORKGROUPS
# workgroups in all (one per compute unit: from 128 input columns on, one
# workgroup fills a compute unit's LDS, and a second round for a few
# workgroups would double the pass), with at least MIN_ROWS_PER_SPLIT rows
# each.  The fp32 partials ([splits, out, in]) stay below half of the bytes
# of dy and x at 64^3.
WG_ROWS = 256
WG_COLS = 256
WORKGROUPS = 256
MIN_ROWS_PER_SPLIT = 512


def splits_for(rows, out_features, in_features, dtype=torch.bfloat16):
    blocks = -(-out_features // WG_ROWS) * max(1, in_features // WG_COLS)
    # Small gradients may be split finer, as long as a split's partials (written
    # and read, 8 bytes an element) stay below the bytes of its rows of dy and
    # x: 4,096 rows of 64 x 64 run on 32 workgroups instead of 8 (21 -> 9 us).
    rows_per = max(128, min(MIN_ROWS_PER_SPLIT,
                            4 * out_features * in_features // (out_features + in_features)))
    # The fp32 products take 16 times as long and the partials no longer: 128
    # rows fill the GPU (18,711 rows of 192 x 192 on 147 workgroups instead of
    # 42, 105 -> 50 us; 968 x 192 on 236 instead of 132, 147 -> 91 us).
    if dtype == torch.float32:
        rows_per = 128
    splits = max(1, min(max(1, WORKGROUPS // blocks), rows // rows_per))
    # Several tiles to a split go to one XCD (eight of them, in turn): whole
    # rounds of eight splits load the XCDs alike.
    return splits // 8 * 8 if blocks > 1 and splits >= 8 else splits


def fp32_training(x, params):
    """Whether fp32 training takes InputProjections and OutputResidual (for their
    weight gradients; LayerNorm and the gate stay torch's): a CUDA fp32 x and
    fp32 parameters, without autocast."""
    return (x.is_cuda and x.dtype == torch.float32 and not torch.is_autocast_enabled("cuda")
            and all(type(p) in (torch.Tensor, torch.nn.Parameter) and p.dtype == torch.float32 for p in params))


def compute_dtype(x):
    """The 16-bit type the layer's linear maps run in: the autocast type when
    autocast is on for x's device, else x's own type (None when that is not
    fp16 / bf16)."""
    if x.is_cuda and torch.is_autocast_enabled("cuda"):
        dt = torch.get_autocast_dtype("cuda")
    else:
        dt = x.dtype
    return dt if dt in (torch.float16, torch.bfloat16) else None


def weight_grad_supported(out_features, in_features):
    cols_ok = (in_features % 32 == 0 and 32 <= in_features <= 256) or (
        in_features % 256 == 0 and 256 < in_features <= 2048)
    return out_features >= 8 and out_features % 8 == 0 and cols_ok


INPUT_GRAD_DIMS = (64, 96, 128, 192, 256, 384, 512)


def _rows_dense(t):
    """Whether t [rows, cols] lies as the kernels read it: unit column stride,
    16-byte aligned rows at a stride that covers them.  An expanded gradient
    (of y.sum(1), say) has a row stride of 0, a single row any."""
    return t.stride(1) == 1 and t.stride(0) >= t.shape[1] and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0


def input_grad(dys, ws):
    """dq Wq + dkv Wkv + dgl Wg for the three 16-bit gradients dys [rows, *]
    and the weights ws [*, dim] of the same type, as one contraction summed in
    fp32 (``p3d_input_grad``); None where the kernel does not take the shapes
    (the caller then runs the three products)."""
    if any(dy is None for dy in dys):
        return None
    dt, rows, dim = ws[0].dtype, dys[0].shape[0], ws[0].shape[1]
    outs = [w.shape[0] for w in ws]
    if (dt not in (torch.float16, torch.bfloat16) or dim not in INPUT_GRAD_DIMS or any(o % 8 for o in outs)
            or any(dy.dtype != dt or dy.shape != (rows, o) or not _rows_dense(dy) for dy, o in zip(dys, outs))):
        return None
    k = sum(outs)
    k_pad = -(-k // 64) * 64
    wt = torch.empty(dim, k_pad, dtype=dt, device=ws[0].device)
    ws = [w.contiguous() for w in ws]
    _lib.call("p3d_concat_transpose", ws[0].data_ptr(), outs[0], ws[1].data_ptr(), outs[1], ws[2].data_ptr(), outs[2],
              dim, wt.data_ptr(), k_pad, _lib.stream_of(wt.device))
    dx = torch.empty(rows, dim, dtype=dt, device=ws[0].device)
    _lib.call("p3d_input_grad", dys[0].data_ptr(), dys[0].stride(0), outs[0], dys[1].data_ptr(), dys[1].stride(0),
              outs[1], dys[2].data_ptr(), dys[2].stride(0), outs[2], wt.data_ptr(), k_pad, dx.data_ptr(), rows, dim,
              _lib.DTYPES[dt], _lib.stream_of(dx.device))
    return dx


PROJECT_DIMS = (64, 96, 128, 192, 256, 384, 512)


def project_linear(x16, ws, bg):
    """(x Wq^T, x Wkv^T, x Wg^T + bg) for x16 [rows, dim] and the weights ws
    [*, dim] of one 16-bit type, from one pass over x16 (``p3d_project_linear``:
    each output summed in fp32 and rounded once, as the torch products); None
    where the kernel does not take the shapes (the caller then runs the three
    products)."""
    dt, (rows, dim) = x16.dtype, x16.shape
    q_out, kv_out, g_out = (w.shape[0] for w in ws)
    if (dt not in (torch.float16, torch.bfloat16) or dim not in PROJECT_DIMS or q_out % 16 or kv_out % 16
            or g_out % 2 or not x16.is_contiguous() or x16.data_ptr() % 16
            or any(w.dtype != dt or w.shape[1] != dim or not w.is_contiguous() or w.data_ptr() % 16 for w in ws)
            or bg.numel() != g_out):
        return None
    bg = bg.to(dt).contiguous()  # the bias in dt, as torch.addmm(bg.to(dt), ...) adds it
    q = torch.empty(rows, q_out, dtype=dt, device=x16.device)
    kv = torch.empty(rows, kv_out, dtype=dt, device=x16.device)
    gl = torch.empty(rows, g_out, dtype=dt, device=x16.device)
    args = _lib.ProjectArgs(x=x16.data_ptr(), ln_weight=None, ln_bias=None, wq=ws[0].data_ptr(),
                            wkv=ws[1].data_ptr(), wg=ws[2].data_ptr(), gate_bias=bg.data_ptr(), q=q.data_ptr(),
                            kv=kv.data_ptr(), gate=gl.data_ptr(), rows=rows, dim=dim, q_out=q_out, kv_out=kv_out,
                            heads=g_out // 2, dtype=_lib.DTYPES[dt], ln_dtype=_lib.DTYPES[dt],
                            gate_bias_dtype=_lib.DTYPES[bg.dtype], eps=0.0)
    _lib.call("p3d_project_linear", args, _lib.stream_of(x16.device))
    return q, kv, gl


def _differentiated(*tensors):
    """fp32 backward passes under create_graph stay on torch ops, as they were."""
    return (torch.is_grad_enabled() and tensors[0].dtype == torch.float32
            and any(t.requires_grad for t in tensors))


def weight_grad(dy, x):
    """dW = dy^T x in fp32 for dy [rows, out], x [rows, in] of one type
    (``p3d_weight_grad``; torch's product in fp32 where the kernel does not
    take the shape, or where the gradient is itself to be differentiated)."""
    rows, out_f = dy.shape
    in_f = x.shape[1]
    if (not weight_grad_supported(out_f, in_f) or dy.dtype != x.dtype or dy.dtype not in _lib.DTYPES
            or _differentiated(dy, x)):
        return torch.mm(dy.t().float(), x.float())
    # A copy, not .contiguous(), which returns a single row as it lies.
    dy, x = (t if _rows_dense(t) else t.clone(memory_format=torch.contiguous_format) for t in (dy, x))
    splits = splits_for(rows, out_f, in_f, dy.dtype)
    dw = torch.empty(out_f, in_f, dtype=torch.float32, device=dy.device)
    work = torch.empty(splits, out_f, in_f, dtype=torch.float32, device=dy.device)
    _lib.call("p3d_weight_grad", dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), dw.data_ptr(),
              work.data_ptr(), rows, out_f, in_f, splits, _lib.DTYPES[dy.dtype], _lib.stream_of(dy.device))
    return dw


def weight_grads3(dys, x, out_dtype=torch.float32):
    """dW of three linear maps sharing the input x: [dy0^T x; dy1^T x;
    dy2^T x] summed in fp32 from one pass over x (``p3d_weight_grad3``) and
    returned as three tensors of out_dtype (fp32 or x's type); None where the
    kernel does not take the shapes (the caller then takes them one at a
    time)."""
    rows, in_f = x.shape
    outs = [dy.shape[1] for dy in dys]
    dt = x.dtype
    if (dt not in _lib.DTYPES or not all(weight_grad_supported(o, in_f) for o in outs) or _differentiated(x, *dys)
            or not _rows_dense(x) or any(dy.dtype != dt or dy.shape[0] != rows or not _rows_dense(dy) for dy in dys)):
        return None
    total = sum(outs)
    splits = splits_for(rows, total, in_f, dt)
    dw = torch.empty(total, in_f, dtype=out_dtype, device=x.device)
    work = torch.empty(splits, total, in_f, dtype=torch.float32, device=x.device)
    _lib.call("p3d_weight_grad3", dys[0].data_ptr(), dys[0].stride(0), outs[0], dys[1].data_ptr(), dys[1].stride(0),
              outs[1], dys[2].data_ptr(), dys[2].stride(0), outs[2], x.data_ptr(), x.stride(0), dw.data_ptr(),
              _lib.DTYPES[out_dtype], work.data_ptr(), rows, in_f, splits, _lib.DTYPES[dt], _lib.stream_of(x.device))
    return torch.split(dw, outs, 0)


def column_sums(x, dtype):
    """Sum over the rows of x [rows, cols] in fp32, rounded to dtype."""
    return x.float().sum(0).to(dtype)


def cast_all(tensors, dt):
    """The tensors in the 16-bit type dt, contiguous: those of another type cast
    in one launch (``p3d_cast``)."""
    out = [t.contiguous() if t.dtype == dt else None for t in tensors]
    todo = [i for i, t in enumerate(out) if t is None]
    if any(tensors[i].dtype not in _lib.DTYPES or tensors[i].numel() == 0 for i in todo) or len(todo) > 8:
        return [t.to(dt).contiguous() for t in tensors]
    if todo:
        jobs = (_lib.CastJob * len(todo))()
        keep = []
        for job, i in zip(jobs, todo):
            src = tensors[i].contiguous()
            keep.append(src)
            out[i] = torch.empty(src.shape, dtype=dt, device=src.device)
            job.src, job.dst, job.count = src.data_ptr(), out[i].data_ptr(), src.numel()
            job.src_dtype, job.dst_dtype = _lib.DTYPES[src.dtype], _lib.DTYPES[dt]
        _lib.call("p3d_cast", jobs, len(todo), _lib.stream_of(out[todo[0]].device))
    return out


class GateProbability(torch.autograd.Function):
    """The gate of attention.py:85 from its 16-bit logits gl [B, N, 2 H] (pairs
    per head): the second entry of each pair's softmax as [B, H, N] (a transposed
    view), in out_dtype.  Computed in fp32 from the logits in both directions,
    one kernel each (``p3d_gate_fwd`` / ``p3d_gate_bwd``).  bias: the bias that
    gl already holds, whose gradient is summed from the unrounded logit
    gradients in the same pass (the product that made gl takes the bias
    detached)."""

    @staticmethod
    def forward(ctx, gl, bias, heads, out_dtype):
        gl = gl.contiguous()
        b, n = gl.shape[0], gl.shape[1]
        gate = torch.empty(b, n, heads, dtype=out_dtype, device=gl.device)
        _lib.call("p3d_gate_fwd", gl.data_ptr(), _lib.DTYPES[gl.dtype], gate.data_ptr(), _lib.DTYPES[out_dtype],
                  gate.numel(), _lib.stream_of(gl.device))
        ctx.save_for_backward(gl)
        ctx.meta = (heads, bias.dtype)
        return gate.transpose(1, 2)

    @staticmethod
    @once_differentiable
    def backward(ctx, dgate):
        (gl,) = ctx.saved_tensors
        heads, bias_dtype = ctx.meta
        b, n = gl.shape[0], gl.shape[1]
        dgl = torch.empty_like(gl)
        part = torch.empty(-(-b * n // 256), 2 * heads, dtype=torch.float32, device=gl.device)
        _lib.call("p3d_gate_bwd", gl.data_ptr(), _lib.DTYPES[gl.dtype], _lib.view3(dgate), _lib.DTYPES[dgate.dtype],
                  dgl.data_ptr(), part.data_ptr(), b, heads, n, _lib.stream_of(gl.device))
        dbias = None
        if ctx.needs_input_grad[1]:
            dbias = torch.empty(2 * heads, dtype=bias_dtype if bias_dtype in _lib.DTYPES else torch.float32,
                                device=gl.device)
            _lib.sum_rows([(part, dbias)], gl.device)
            dbias = dbias.to(bias_dtype)
        return dgl, dbias, None, None


def _rows(t):
    return t.reshape(-1, t.shape[-1])


def layer_norm_train_supported(norm, x):
    """Whether LayerNormTrain takes this nn.LayerNorm and input."""
    dim = x.shape[-1]
    ep = 16 // x.element_size()
    return (x.dtype in _lib.DTYPES and norm.weight is not None and norm.bias is not None
            and norm.weight.dtype in _lib.DTYPES and norm.bias.dtype in _lib.DTYPES
            and norm.weight.dtype == norm.bias.dtype and tuple(norm.normalized_shape) == (dim,)
            and dim % ep == 0 and dim <= 512
            and not norm._forward_hooks and not norm._forward_pre_hooks)


class LayerNormTrain(torch.autograd.Function):
    """nn.LayerNorm of the layer input (attention.py:64) for 16-bit training,
    on ``p3d_layer_norm_train`` / ``p3d_layer_norm_bwd``: fp32 statistics, the
    output rounded straight to the compute type dt (the value the next
    linear maps would cast it to), and a backward that returns dx in x's
    dtype and the affine gradients summed in fp32.

    With residual=True the forward also returns x rounded to dt as a
    [rows, dim] tensor, written from the same read of x: the residual operand
    of the output product (OutputResidual with x_owned=True).  With
    residual="pass" it returns x itself as [rows, dim] (the unrounded residual
    of autocast over a wider x, for OutputResidualWide).  Either way the
    backward adds that output's gradient into dx inside the kernel, where
    autograd would otherwise sum the two gradients of x in a separate pass."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps, dt, residual=False):
        x2 = _rows(x).contiguous()
        rows, dim = x2.shape
        dev = x.device
        y = torch.empty(rows, dim, dtype=dt, device=dev)
        xc = torch.empty(rows, dim, dtype=dt, device=dev) if residual else None
        mean = torch.empty(rows, dtype=torch.float32, device=dev)
        rstd = torch.empty(rows, dtype=torch.float32, device=dev)
        _lib.call("p3d_layer_norm_train", x2.data_ptr(), weight.data_ptr(), bias.data_ptr(), _lib.DTYPES[weight.dtype],
                  y.data_ptr(), 0 if xc is None else xc.data_ptr(), mean.data_ptr(), rstd.data_ptr(), rows, dim,
                  _lib.DTYPES[x2.dtype], _lib.DTYPES[dt], float(eps), _lib.stream_of(dev))
        ctx.save_for_backward(x2, weight, mean, rstd)
        ctx.meta = (x.shape, bias.dtype)
        ctx.set_materialize_grads(False)
        if residual == "pass":
            return y.view(x.shape), x2
        if residual:
            return y.view(x.shape), xc
        return y.view(x.shape)

    @staticmethod
    def backward(ctx, dy, dres=None):
        x2, weight, mean, rstd = ctx.saved_tensors
        shape, b_dt = ctx.meta
        rows, dim = x2.shape
        if dy is None:
            dy = torch.zeros(rows, dim, dtype=torch.float32, device=x2.device)
        dy2 = _rows(dy).contiguous()
        if dy2.dtype not in _lib.DTYPES:
            dy2 = dy2.float()
        dx = torch.empty_like(x2)
        dr = None if dres is None else _rows(dres).to(dx.dtype).contiguous()
        # Row ranges of the affine partials, and with them workgroups: 256 rows
        # each left 64 workgroups at 16,384 rows (72 us at dim 512; 18 us).
        parts = max(1, min(1024, rows // 32))
        part = torch.empty(parts, 2, dim, dtype=torch.float32, device=x2.device)
        _lib.call("p3d_layer_norm_bwd", dy2.data_ptr(), 0 if dr is None else dr.data_ptr(), x2.data_ptr(),
                  weight.data_ptr(), _lib.DTYPES[weight.dtype], mean.data_ptr(), rstd.data_ptr(), dx.data_ptr(),
                  part.data_ptr(), rows, dim, _lib.DTYPES[dy2.dtype], _lib.DTYPES[x2.dtype], _lib.DTYPES[dx.dtype],
                  parts, _lib.stream_of(x2.device))
        dw, db = (torch.empty(dim, dtype=t, device=x2.device) for t in (weight.dtype, b_dt))
        _lib.sum_rows([(part[:, 0], dw), (part[:, 1], db)], x2.device)
        return dx.view(shape), dw, db, None, None, None


class InputProjections(torch.autograd.Function):
    """(x Wq^T, x Wkv^T, x Wg^T + bg) of the normalised tokens x in the type
    dt, 16-bit, or fp32 for an fp32 model (attention.py:64-67,85): x is rounded
    to dt once and shared by the three products; the backward returns dx in x's dtype (the three
    input gradients summed in fp32) and fp32 weight gradients cast to the
    parameters' dtypes."""

    @staticmethod
    def forward(ctx, x, wq, wkv, wg, bg, dt):
        x16 = _rows(x).to(dt).contiguous()
        *ws, bg16 = cast_all((wq, wkv, wg, bg), dt)
        made = project_linear(x16, ws, bg16)
        if made is not None:
            q, kv, gl = made
        else:
            q = torch.mm(x16, ws[0].t())
            kv = torch.mm(x16, ws[1].t())
            gl = torch.addmm(bg16, x16, ws[2].t())
        # x itself where it is what the products read, so that a differentiated
        # backward reaches it.
        ctx.save_for_backward(x if x.dtype == dt and x.is_contiguous() else x16, *ws)
        ctx.meta = (x.shape, x.dtype, wq.dtype, wkv.dtype, wg.dtype, bg.dtype)
        lead = x.shape[:-1]
        return q.view(*lead, -1), kv.view(*lead, -1), gl.view(*lead, -1)

    @staticmethod
    def backward(ctx, dq, dkv, dgl):
        x16, wq, wkv, wg = ctx.saved_tensors
        x16 = _rows(x16)
        shape, x_dt, wq_dt, wkv_dt, wg_dt, bg_dt = ctx.meta
        # dx = dq Wq + dkv Wkv + dgl Wg: for an fp32 x (autocast) the three
        # products are summed in fp32 as autograd would; for a 16-bit x the
        # GEMMs accumulate into one buffer of that type.
        wide = x_dt == torch.float32 and x16.dtype != x_dt
        dys = [None if dy is None else _rows(dy).to(x16.dtype) for dy in (dq, dkv, dgl)]
        # One kernel for the three products where it takes the shapes (16-bit x).
        need = ctx.needs_input_grad[0]
        dx = input_grad(dys, (wq, wkv, wg)) if need and not wide else None
        fused = dx is not None
        if need and wide:
            dx = torch.zeros(x16.shape, dtype=torch.float32, device=x16.device)
        # The three weight gradients from one pass over x16 where the kernel takes them.
        same = x16.dtype if wq_dt == wkv_dt == wg_dt == x16.dtype else torch.float32
        every = all(ctx.needs_input_grad[1:4]) and not any(dy is None for dy in dys)
        dws = weight_grads3(dys, x16, same) if every else None
        grads = []
        for i, (dy, w, w_dt) in enumerate(zip(dys, (wq, wkv, wg), (wq_dt, wkv_dt, wg_dt))):
            if dy is None:
                grads.append(None)
                continue
            if not need:
                pass
            elif wide:
                dx.add_(torch.mm(dy, w))
            elif dx is None:
                dx = torch.mm(dy, w)
            elif not fused:
                # in place: no copy of dx into a new result
                dx = torch.addmm(dx, dy, w) if _differentiated(dy, w) else dx.addmm_(dy, w)
            if not ctx.needs_input_grad[1 + i]:
                grads.append(None)
                continue
            grads.append((weight_grad(dy, x16) if dws is None else dws[i]).to(w_dt))
        if dx is None and need:
            dx = torch.zeros(x16.shape, dtype=x16.dtype, device=x16.device)
        dbg = column_sums(_rows(dgl), bg_dt) if dgl is not None and ctx.needs_input_grad[4] else None
        return dx.view(shape).to(x_dt) if need else None, grads[0], grads[1], grads[2], dbg, None


def wide_residual_supported(x, k, dim, dt):
    """Whether p3d_out_residual takes an fp32 residual x [.., dim] for the
    product of width k in the 16-bit type dt."""
    return (x.is_cuda and x.dtype == torch.float32 and dt in (torch.float16, torch.bfloat16)
            and k in (64, 96, 128, 192, 256, 384, 512) and dim % 32 == 0 and dim <= 512)


class OutputResidualWide(torch.autograd.Function):
    """x + y Wo^T under autocast over an fp32 input (attention.py:89): the
    product in the 16-bit type dt, rounded to dt, added to the unrounded fp32
    residual x [rows, dim], as the reference's ``residual + to_out(...)`` sums
    an fp32 tensor and a 16-bit one; y [rows, k].  One kernel
    (``p3d_out_residual`` with an fp32 residual) instead of the product, a
    16-bit intermediate and a torch add.  The backward gives dx = dout
    (fp32), dy = dout Wo and an fp32 weight gradient, as OutputResidual's."""

    @staticmethod
    def forward(ctx, x, y, wo, dt):
        y16 = y.to(dt).contiguous()
        wo16 = wo.to(dt).contiguous()
        x2 = x.contiguous()
        rows, dim = x2.shape
        out = torch.empty_like(x2)
        _lib.call("p3d_out_residual", y16.data_ptr(), wo16.data_ptr(), x2.data_ptr(), out.data_ptr(), rows,
                  y16.shape[1], dim, _lib.DTYPES[dt], _lib.DTYPES[torch.float32], _lib.stream_of(x2.device))
        ctx.save_for_backward(y16, wo16)
        ctx.meta = (y.dtype, wo.dtype)
        return out

    @staticmethod
    def backward(ctx, dout):
        y16, wo16 = ctx.saved_tensors
        y_dt, wo_dt = ctx.meta
        d16 = dout.to(y16.dtype)
        dy = torch.mm(d16, wo16).to(y_dt) if ctx.needs_input_grad[1] else None
        return dout, dy, weight_grad(d16, y16).to(wo_dt) if ctx.needs_input_grad[2] else None, None


class OutputResidual(torch.autograd.Function):
    """x + y Wo^T in the type dt (attention.py:89 with an x of that type):
    x [rows, dim], y [rows, k].  The product accumulates into the residual in
    place: into x itself when the caller owns it (x_owned: x is already a dt
    copy, such as the one LayerNormTrain returns; it is marked dirty and
    returned), else into a dt copy of x (addmm with a full matrix would copy
    it into a new result first).  With x None it returns the product y Wo^T
    alone, rounded to dt: the caller adds a residual of a wider type itself,
    as the reference's ``residual + to_out(...)`` does under autocast.  The
    backward gives dx = dout (in x's dtype), dy = dout Wo and an fp32 weight
    gradient."""

    @staticmethod
    def forward(ctx, x, y, wo, dt, x_owned=False):
        y16 = y.to(dt).contiguous()
        wo16 = wo.to(dt)
        if x is None:
            out = torch.mm(y16, wo16.t())
        elif x_owned and x.dtype == dt and x.dim() == 2 and x.is_contiguous():
            ctx.mark_dirty(x)
            out = x
            out.addmm_(y16, wo16.t())
        else:
            out = x.to(dt, copy=True)
            out.addmm_(y16, wo16.t())
        ctx.save_for_backward(y16, wo16)
        ctx.meta = (None if x is None else x.dtype, y.dtype, wo.dtype)
        return out

    @staticmethod
    def backward(ctx, dout):
        y16, wo16 = ctx.saved_tensors
        x_dt, y_dt, wo_dt = ctx.meta
        d16 = dout.to(y16.dtype)
        dy = torch.mm(d16, wo16).to(y_dt) if ctx.needs_input_grad[1] else None
        dx = None if x_dt is None else dout.to(x_dt)
        return dx, dy, weight_grad(d16, y16).to(wo_dt) if ctx.needs_input_grad[2] else None, None, None
