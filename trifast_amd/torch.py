"""PyTorch operator boundary of the MI355X triangle attention.

Mirrors the public surface of reference src/trifast/torch.py: two ``torch.library``
operators, ``trifast::triangle_attention`` (-> o, lse; reference :17-65) and
``trifast::triangle_attention_backward`` (-> dq, dk, dv, db, dmask; reference
:68-182), glued by ``register_autograd`` (reference :185-217), and the
``triangle_attention`` wrapper that drops lse (reference :220-228).  The device
work is done by hand-written HIP kernels behind the C ABI of
``libtrifast_hip.so``; PyTorch only owns the memory and the stream.
"""

from __future__ import annotations

import torch

from trifast_amd import _lib, tuner

_DTYPE_CODE = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}


def _dtype_code(t: torch.Tensor) -> int:
    try:
        return _DTYPE_CODE[t.dtype]
    except KeyError:
        raise TypeError(f"triangle_attention supports float32, bfloat16 and float16, got {t.dtype}") from None


def _check_inputs(q, k, v, b, mask) -> tuple[int, int, int, int]:
    if q.dim() != 5:
        raise ValueError(f"q must be [b, h, n, n, d], got shape {tuple(q.shape)}")
    bs, h, n, n2, d = q.shape
    if n != n2:
        raise ValueError(f"q must be square in its pair dims, got shape {tuple(q.shape)}")
    if k.shape != q.shape or v.shape != q.shape:
        raise ValueError("q, k, v must have the same shape")
    if tuple(b.shape) != (bs, h, n, n):
        raise ValueError(f"bias must be [b, h, n, n] = {(bs, h, n, n)}, got {tuple(b.shape)}")
    if tuple(mask.shape) != (bs, n, n):
        raise ValueError(f"mask must be [b, n, n] = {(bs, n, n)}, got {tuple(mask.shape)}")
    if mask.dtype != torch.bool:
        raise TypeError(f"mask must be bool, got {mask.dtype}")
    if not (k.dtype == q.dtype and v.dtype == q.dtype and b.dtype == q.dtype):
        raise TypeError("q, k, v and bias must share one dtype")
    for name, t in (("q", q), ("k", k), ("v", v), ("bias", b), ("mask", mask)):
        if not t.is_cuda:
            raise RuntimeError(f"{name} is on {t.device}: triangle_attention runs on the GPU only")
        if t.device != q.device:
            raise RuntimeError("all inputs must be on the same device")
    return bs, h, n, d


def _strides(t: torch.Tensor) -> list[int]:
    # the stride of a size-1 dim is never used for addressing; report 0
    return [0 if sz == 1 else st for sz, st in zip(t.shape, t.stride())]


def _vector_ready(t: torch.Tensor) -> torch.Tensor:
    """q-like tensors are read with 16-byte vector loads along d: the last stride
    must be 1, the base 16-byte aligned and the other strides multiples of the
    vector width.  Transposed (i<->j) views qualify and are read in place; anything
    else is copied, as the reference forward copies every non-contiguous input
    (src/trifast/torch.py:30-34)."""
    vec = 16 // t.element_size()
    st = _strides(t)
    if st[-1] == 1 and t.data_ptr() % 16 == 0 and all(s % vec == 0 for s in st[:-1]) and _j_stride_ok(t, st):
        return t
    return t.contiguous()


def _j_stride_ok(t: torch.Tensor, st: list[int]) -> bool:
    """The kernels address the rows of a tile through 32-bit offsets from a per-tile base:
    the stride between consecutive j, in bytes, must lie in [0, 2^24) (the library returns
    TRIFAST_EUNSUPPORTED otherwise)."""
    return t.dim() != 5 or 0 <= st[3] * t.element_size() < (1 << 24)


def _grad_like(t: torch.Tensor) -> torch.Tensor:
    """Empty gradient buffer for input ``t``: laid out like ``t`` when ``t`` is dense
    and the kernels can write that layout (d contiguous, 16-byte rows), so that a
    leaf that is a transposed view takes its gradient without a re-layout copy;
    contiguous otherwise."""
    vec = 16 // t.element_size()
    st = _strides(t)
    if t.dim() == 5 and st[-1] == 1 and all(s % vec == 0 for s in st[:-1]) and _j_stride_ok(t, st):
        out = torch.empty_like(t)  # preserves the strides of a dense tensor
        if out.stride() == t.stride():
            return out
    elif t.dim() == 4:
        out = torch.empty_like(t)
        if out.stride() == t.stride():
            return out
    return torch.empty(t.shape, dtype=t.dtype, device=t.device)


def _workspace(nbytes: int, device) -> torch.Tensor:
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)


def _ptr(t):
    return t.data_ptr()


def _tiles_to_keep(q: torch.Tensor, tiles: dict[int, int]) -> bool:
    """Whether the tiles just chosen (by kernel) may be remembered for the shape: they are what the
    tuner takes without timing from now on.  (A choice made under stream capture is the library's
    heuristic one, without the timing that eager mode does.)"""
    if torch.cuda.is_current_stream_capturing():
        return False
    _, h, n, _, d = q.shape
    return tuner.force_tune() or all(tuner.settled(kernel, n, h, d, q.dtype) == tile for kernel, tile in tiles.items())


def _choose_forward(q, k, v, b, mask) -> tuple[tuple[int, int, int], bool]:
    """Tile of the forward kernel for these tensors, timed on them where the tuner asks for it
    (the native host path calls this once per shape)."""
    bs, h, n, _, d = q.shape
    lib, code = _lib.load(), _dtype_code(q)
    args = []

    def launch(tile: int) -> None:
        if not args:
            o = torch.empty((bs, h, n, n, d), dtype=q.dtype, device=q.device)
            lse = torch.empty((bs, h, n, n), dtype=torch.float32, device=q.device)
            ws = _workspace(lib.trifast_fwd_workspace_bytes(bs, h, n, d, code), q.device)
            args.extend((o, lse, *(_vector_ready(t) for t in (q, k, v)), b, mask.view(torch.uint8), ws))
        o, lse, qr, kr, vr, br, mr, ws = args
        rc = lib.trifast_fwd(
            _ptr(o), _ptr(lse), _ptr(qr), _ptr(kr), _ptr(vr), _ptr(br), _ptr(mr), bs, h, n, d, code,
            *(_lib.i64_array(_strides(t)) for t in (qr, kr, vr, br, mr)),
            tile, _ptr(ws), ws.numel(), torch.cuda.current_stream(q.device).cuda_stream,
        )
        _lib.check(rc, "trifast_fwd")

    tile = tuner.pick(_lib.KERNEL_FWD, n, h, d, q.dtype, launch)
    return (tile, -1, -1), _tiles_to_keep(q, {_lib.KERNEL_FWD: tile})


def _choose_backward(do, q, k, v, b, o, l, mask) -> tuple[tuple[int, int, int], bool]:
    """Tiles of the three backward kernels, as :func:`_choose_forward`."""
    bs, h, n, _, d = q.shape
    lib, code = _lib.load(), _dtype_code(q)
    args = []

    def launch_one(kernel: int, tile: int) -> None:
        if not args:
            ins = [_vector_ready(t) for t in (do, q, k, v)] + [b, mask.view(torch.uint8)]
            outs = [_grad_like(t) for t in (q, k, v, b)]
            strides = [_lib.i64_array(_strides(t)) for t in ins + outs]
            args.extend((ins, outs, strides, _workspace(lib.trifast_bwd_workspace_bytes(bs, h, n, d, code), q.device)))
        ins, outs, strides, ws = args
        rc = lib.trifast_bwd_one(
            kernel, *map(_ptr, outs), *map(_ptr, ins), _ptr(o), _ptr(l), bs, h, n, d, code, *strides,
            tile, _ptr(ws), ws.numel(), torch.cuda.current_stream(q.device).cuda_stream,
        )
        _lib.check(rc, "trifast_bwd_one")

    # fixed launch order; _bwd_q also produces delta for the other two
    # (reference src/trifast/torch.py:110).  When a later kernel has to be timed
    # but _bwd_q's tile comes from the cache, _bwd_q runs once first so that the
    # timed kernels read a valid workspace.
    tiles = []
    primed = False
    kernels = (_lib.KERNEL_BWD_Q, _lib.KERNEL_BWD_KV, _lib.KERNEL_BWD_B)
    for kernel in kernels:
        def timed(t, kern=kernel):
            nonlocal primed
            if kern != _lib.KERNEL_BWD_Q and not primed:
                launch_one(_lib.KERNEL_BWD_Q, tiles[0])
            primed = True
            launch_one(kern, t)

        # a dk/dv tile that also produces dq saves the dq kernel's launch: the other
        # dk/dv tiles are charged with it
        extra = None
        if kernel == _lib.KERNEL_BWD_KV:
            dq_ms: list[float] = []

            def extra(t):
                if lib.trifast_bwd_kv_tile_writes_dq(t):
                    return 0.0
                if not dq_ms:
                    dq_ms.append(tuner._time_launch(lambda tile: launch_one(_lib.KERNEL_BWD_Q, tile), tiles[0]))
                return dq_ms[0]

        tiles.append(tuner.pick(kernel, n, h, d, q.dtype, timed, extra))
    return tuple(tiles), _tiles_to_keep(q, dict(zip(kernels, tiles)))


def _native():
    """The native host path (``csrc/host_torch.cpp``), with its tile choosers registered."""
    return _lib.host(_choose_forward, _choose_backward)


@torch.library.custom_op("trifast::triangle_attention", mutates_args=())
def _triangle_attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    b: torch.Tensor,
    mask: torch.Tensor,
) -> tuple[torch.Tensor, torch.Tensor]:
    native = _native()
    bs, h, n, d = _check_inputs(q, k, v, b, mask)
    _dtype_code(q)
    if q.numel() == 0 and d > 0:  # an empty batch (or no heads, or no tokens): nothing to launch
        return torch.empty_like(q, memory_format=torch.contiguous_format), torch.empty((bs, h, n, n), dtype=torch.float32, device=q.device)
    return native.forward(q, k, v, b, mask)


@_triangle_attention.register_fake
def _(q, k, v, b, mask):
    bs, h, n, _, d = q.shape
    o = q.new_empty((bs, h, n, n, d))
    lse = q.new_empty((bs, h, n, n), dtype=torch.float32)
    return o, lse


@torch.library.custom_op("trifast::triangle_attention_backward", mutates_args=())
def triangle_attention_bwd(
    do: torch.Tensor,
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    b: torch.Tensor,
    o: torch.Tensor,
    l: torch.Tensor,
    mask: torch.Tensor,
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    native = _native()
    bs, h, n, d = _check_inputs(q, k, v, b, mask)
    _dtype_code(q)
    if q.numel() == 0 and d > 0:  # an empty batch: empty gradients
        return _grad_like(q), _grad_like(k), _grad_like(v), _grad_like(b), torch.zeros_like(mask)
    dq, dk, dv, db = native.backward(do, q, k, v, b, o, l, mask)
    # the mask takes no gradient; autograd still wants a tensor in this slot
    # (reference src/trifast/torch.py:102)
    return dq, dk, dv, db, torch.zeros_like(mask)


@triangle_attention_bwd.register_fake
def _(do, q, k, v, b, o, l, mask):
    return (_grad_like(q), _grad_like(k), _grad_like(v), _grad_like(b), torch.zeros_like(mask))


def backwards(ctx, *grad):
    # reference src/trifast/torch.py:185-207
    do = grad[0]
    q, k, v, b, mask, o, l = ctx.saved_tensors
    if do is None:  # only lse was used downstream: nothing flows back through o
        do = torch.zeros_like(o)
    dq, dk, dv, db, _ = triangle_attention_bwd(do, q, k, v, b, o, l, mask)
    return dq, dk, dv, db, None


def setup_context(ctx, inputs, output) -> None:
    # reference src/trifast/torch.py:210-214
    q, k, v, b, mask, *_ = inputs
    o, l = output
    ctx.save_for_backward(q, k, v, b, mask, o, l)
    # lse takes no gradient: without this autograd fills a zero tensor of its size for every backward
    ctx.set_materialize_grads(False)


_triangle_attention.register_autograd(backwards, setup_context=setup_context)


def _no_forward_mode(*tensors: torch.Tensor) -> None:
    """Raises for tensors with a forward-mode tangent: a registered operator called without an input
    that requires grad would return a result without one."""
    for t in tensors:
        if torch.autograd.forward_ad.unpack_dual(t).tangent is not None:
            raise NotImplementedError("the triangle attention kernels have no forward-mode derivative (jvp)")


def _attend(q, k, v, b, mask, ending: bool) -> torch.Tensor:
    """The operator (``ending``: on the pair-transposed problem) on 5-D inputs.  Ordinary eager
    calls on plain GPU tensors run natively, with an autograd node of their own over the same
    launches, saved tensors and gradients: in Python the dispatcher passes, the marshalling and
    the backward's trips through the interpreter took 0.2 ms of a step, twice what its kernels
    take at n = 256.  The native path declines (None) anything else -- tracing, transforms,
    autocast, other devices, shapes that do not fit -- which goes through the registered
    operators; forward-mode differentiation raises."""
    if not torch.compiler.is_compiling():
        o = _native().attention(q, k, v, b, mask, ending)
        if o is not None:
            return o
        _no_forward_mode(q, k, v, b)
    if ending:
        t = lambda x: x.transpose(-3, -2)
        return t(_triangle_attention(t(q), t(k), t(v), b.transpose(-1, -2), mask.transpose(-1, -2))[0])
    return _triangle_attention(q, k, v, b, mask)[0]


def triangle_attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    b: torch.Tensor,
    mask: torch.Tensor,
) -> torch.Tensor:
    """Fused triangle self-attention (starting node).

    q, k, v: [b, h, n, n, d]; b (bias): [b, h, n, n]; mask: [b, n, n] bool with
    True = key masked out.  Returns o: [b, h, n, n, d].  Reference
    src/trifast/torch.py:220-228.

    Beyond the reference (its own TODO, src/trifast/torch.py:29,84): any number of
    leading batch dims, q [*batch, h, n, n, d] with bias [*batch, h, n, n] and mask
    [*batch, n, n], including none at all; they are folded into one batch dim (views
    where the layout allows it) and restored on the output.
    """
    if q.dim() == 5:
        return _attend(q, k, v, b, mask, False)
    if q.dim() < 4:
        raise ValueError(f"q must be [*batch, h, n, n, d], got shape {tuple(q.shape)}")
    lead = q.shape[:-4]
    if b.shape[:-3] != lead or mask.shape[:-2] != lead or k.shape != q.shape or v.shape != q.shape:
        raise ValueError(
            f"leading batch dims must agree: q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)}, "
            f"bias {tuple(b.shape)}, mask {tuple(mask.shape)}"
        )
    fold = lambda t, keep: t.reshape(-1, *t.shape[-keep:])
    o = _attend(fold(q, 4), fold(k, 4), fold(v, 4), fold(b, 3), fold(mask, 2), False)
    return o.reshape(*lead, *o.shape[1:])


def triangle_attention_ending_node(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    b: torch.Tensor,
    mask: torch.Tensor,
) -> torch.Tensor:
    """Triangle self-attention around the ending node, on tensors in the ordinary
    (untransposed) pair layout:

        a[i, j, k] = softmax_k(q[i, j] . k[k, j] / sqrt(d) + b[k, i] + mask[k, j] * finfo.min)
        o[i, j]    = sum_k a[i, j, k] v[k, j]

    with q, k, v: [*batch, h, n, n, d] indexed [.., i, j, :], b: [*batch, h, n, n],
    mask: [*batch, n, n] (True = masked out).  This is the starting-node operator on
    the pair-transposed problem; the transposes are views (q, k, v are read in place
    through their strides, bias and mask are re-tiled by the pre-passes anyway), so
    nothing is copied.  The result is a transposed view of a contiguous tensor.
    The reference has no such entry: its callers transpose and copy by hand.
    """
    if q.dim() == 5:
        return _attend(q, k, v, b, mask, True)
    t = lambda x: x.transpose(-3, -2)
    return t(triangle_attention(t(q), t(k), t(v), b.transpose(-1, -2), mask.transpose(-1, -2)))
