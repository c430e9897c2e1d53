"""The public functions as autograd sees them: what they keep for the backward and how, what they refuse, what a changed
mask or input does.  Results are compared with calls of the same functions that nothing interferes with."""
import gc

import pytest
import torch

from _util import cpu_mask, rel_fro
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu
BS, P = 64, 0.4


def _t(*shape, seed, scale=1.0, dtype=torch.float16):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=gen) * scale).to(dtype).cuda()


def _mask(rows, cols, seed=0):
    return cpu_mask(O.mask_shape(rows, cols, BS), P, torch.Generator().manual_seed(seed)).cuda()


def _linear():
    """(call, its tensors): call(mask) runs the function on them."""
    import flash_dropout.functional as F

    x, w = _t(192, 136, seed=1).requires_grad_(), _t(72, 136, seed=2, scale=0.1).requires_grad_()

    def call(mask="drawn"):
        if mask == "drawn":
            return F.hip_blockwise_dropout_matmul(x, w, BS, P, seed=5)
        return F.hip_blockwise_dropout_matmul_mask(x, mask, BS, P, w)

    return call, (x, w), _mask(192, 136)


def _mlp(act="gelu", rows=192):
    import flash_dropout.functional as F

    x = _t(rows, 136, seed=1).requires_grad_()
    ws = [_t(o, i, seed=3 + i, scale=i ** -0.5).requires_grad_() for i, o in ((136, 256), (256, 200), (200, 10))]

    def call(mask="drawn"):
        if mask == "drawn":
            return F.hip_blockwise_dropout_mlp(x, ws, BS, P, act, seed=5)
        return F.hip_blockwise_dropout_mlp(x, ws, BS, P, act, masks=[mask, _mask(rows, 256, 1), _mask(rows, 200, 2)])

    return call, (x, *ws), _mask(rows, 136)


# rows of 8 and 18 output positions: the routes without and with a patch matrix; a pointwise kernel on pixels in rows, whose
# patch matrix is the image itself
CONVS = {"implicit": (8, 3, 1, False), "explicit": (18, 3, 1, False), "pointwise": (12, 1, 0, True)}


def _conv(form):
    import flash_dropout.functional as F

    hw, r, pad, channels_last = CONVS[form]
    x, k = _t(4, 16, hw, hw, seed=1), _t(40, 16, r, r, seed=2, scale=0.1).requires_grad_()
    if channels_last:
        x = x.to(memory_format=torch.channels_last)
    x.requires_grad_()
    rows, cols = F.conv_patch_matrix_shape(x.shape, k.shape, (pad, pad))

    def call(mask="drawn"):
        if mask == "drawn":
            return F.blockwise_dropout_conv2d(x, k, BS, P, padding=pad, seed=5)
        return F.blockwise_dropout_conv2d_mask(x, mask, BS, P, k, padding=pad)

    return call, (x, k), _mask(rows, cols)


FUNCTIONS = {"linear": _linear, "mlp": _mlp, **{f"conv {f}": (lambda f=f: _conv(f)) for f in CONVS}}
every_function = pytest.mark.parametrize("name", FUNCTIONS)


def _grads(y, wrt, **kw):
    return torch.autograd.grad(y, wrt, _t(*y.shape, seed=9), **kw)


def _same(a, b):
    return all(torch.equal(s, t) for s, t in zip(a, b))


@every_function
def test_a_given_mask_changed_before_the_backward_is_refused(name):
    call, wrt, mask = FUNCTIONS[name]()
    want = _grads(call(mask.clone()), wrt)
    y = call(mask)
    assert _same(_grads(y, wrt, retain_graph=True), want)
    mask.logical_not_()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        _grads(y, wrt)


@every_function
def test_inputs_that_carry_a_forward_gradient_are_refused(name):
    import torch.autograd.forward_ad as fwd

    call, wrt, mask = FUNCTIONS[name]()
    import flash_dropout.functional as F

    with fwd.dual_level():
        for i in range(2):  # the input, a weight
            dual = [t.detach() for t in wrt]
            dual[i] = fwd.make_dual(dual[i], torch.ones_like(dual[i]))
            with pytest.raises(NotImplementedError, match="jvp"):
                if name == "linear":
                    F.hip_blockwise_dropout_matmul(*dual, BS, P, seed=5)
                elif name == "mlp":
                    F.hip_blockwise_dropout_mlp(dual[0], dual[1:], BS, P, "gelu", seed=5)
                else:
                    F.blockwise_dropout_conv2d(*dual, BS, P, seed=5)


@every_function
def test_function_transforms_are_refused(name):
    """The launches read raw pointers, which a transform's wrapped tensors do not have."""
    import flash_dropout.functional as F

    _, wrt, _ = FUNCTIONS[name]()
    plain = [t.detach() for t in wrt]

    def f(x):
        if name == "linear":
            return F.hip_blockwise_dropout_matmul(x, plain[1], BS, P, seed=5)
        if name == "mlp":
            return F.hip_blockwise_dropout_mlp(x, plain[1:], BS, P, "gelu", seed=5)
        return F.blockwise_dropout_conv2d(x, plain[1], BS, P, seed=5)

    for transformed in (lambda: torch.func.vmap(f)(torch.stack([plain[0]] * 2)),
                        lambda: torch.func.grad(lambda x: f(x).float().sum())(plain[0]),
                        lambda: torch.func.jvp(f, (plain[0],), (plain[0],))):
        with pytest.raises((RuntimeError, NotImplementedError, ValueError)):
            transformed()


@every_function
@pytest.mark.parametrize("given", [False, True])
def test_everything_kept_for_the_backward_goes_through_saved_tensor_hooks(name, given):
    """With hooks that take what is saved to host memory, the device holds the output and no more, and the gradients that
    come out of the copies are the same bits."""
    call, wrt, mask = FUNCTIONS[name]()
    args = (mask,) if given else ()
    want = _grads(call(*args), wrt)
    gc.collect()
    before = torch.cuda.memory_allocated()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        y = call(*args)
    gc.collect()
    # (the result of the convolution and of a layer is one buffer; the allocator hands out multiples of 512 bytes)
    assert torch.cuda.memory_allocated() - before <= -(-y.numel() * 2 // 512) * 512
    assert _same(_grads(y, wrt), want)


@every_function
def test_what_a_hook_hands_back_is_checked_and_may_have_other_strides(name):
    """The launches trust extents, types and devices; a hook may return any tensor."""
    call, wrt, mask = FUNCTIONS[name]()
    for unpack in (lambda t: t.cpu(), lambda t: t.double(), lambda t: t[:-1]):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            y = call(mask)
        with pytest.raises(ValueError, match="saved-tensor hook"):
            _grads(y, wrt)

    def strided(t):
        """The same values with a gap behind every element."""
        wide = torch.zeros(*t.shape, 2, dtype=t.dtype, device=t.device)
        wide[..., 0] = t
        return wide[..., 0]

    want = _grads(call(mask), wrt)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, strided):
        y = call(mask)
    # an image with gaps goes through a patch matrix: the same fp32 sums in another order, so an element may round to the
    # neighbouring fp16 value, 2^-10 of it at most
    assert all(rel_fro(g, r) <= 2 ** -10 for g, r in zip(_grads(y, wrt), want))


@every_function
def test_a_checkpoint_frees_what_the_function_keeps(name):
    from torch.utils.checkpoint import checkpoint

    call, wrt, _ = FUNCTIONS[name]()
    want = _grads(call(), wrt)
    gc.collect()
    before = torch.cuda.memory_allocated()
    y = checkpoint(call, use_reentrant=False)
    gc.collect()
    assert torch.cuda.memory_allocated() - before <= -(-y.numel() * 2 // 512) * 512
    assert _same(_grads(y, wrt), want)


@every_function
def test_a_second_backward(name):
    call, wrt, _ = FUNCTIONS[name]()
    y = call()
    want = _grads(y, wrt, retain_graph=True)
    assert _same(_grads(y, wrt), want)
    with pytest.raises(RuntimeError, match="second time"):
        _grads(y, wrt)


@every_function
@pytest.mark.parametrize("which", [0, 1])
def test_an_operand_changed_before_the_backward_is_refused_where_it_is_read(name, which):
    """(the image behind a patch matrix is not: the matrix is what was kept)"""
    call, wrt, _ = FUNCTIONS[name]()
    want = _grads(call(), wrt)
    y = call()
    with torch.no_grad():
        wrt[which].mul_(2)
    if name == "conv explicit" and which == 0:
        assert _same(_grads(y, wrt), want)
    else:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            _grads(y, wrt)


def test_the_convolution_keeps_the_image_or_its_patch_matrix():
    call, wrt, _ = _conv("explicit")
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
        call()
    assert (4 * 18 * 18, 16 * 9) in kept and tuple(wrt[0].shape) not in kept
    for form in ("implicit", "pointwise"):
        call, wrt, _ = _conv(form)
        kept.clear()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
            call()
        big = [s for s in kept if len(s) == 4 or s[0] >= 256]
        assert big == [tuple(wrt[0].shape)], form


@every_function
@pytest.mark.parametrize("along", [0, 1])
def test_an_expanded_mask_is_the_mask_it_shows(name, along):
    call, wrt, mask = FUNCTIONS[name]()
    expanded = mask.narrow(along, 0, 1).expand(mask.shape)
    y, want = call(expanded), call(expanded.contiguous())
    assert torch.equal(y, want) and _same(_grads(y, wrt), _grads(want, wrt))


def test_masks_may_be_given_for_some_layers_only():
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    _, (x, *ws), m0 = _mlp()
    drawn = GEMM().random_lists(O.mask_shape(192, 256, BS), P, seed=7 + 1)[0]  # layer i draws from seed + i
    m2 = _mask(192, 200, 2)
    y = F.hip_blockwise_dropout_mlp(x, ws, BS, P, "relu", masks=[m0, None, m2], seed=7)
    ref = F.hip_blockwise_dropout_mlp(x, ws, BS, P, "relu", masks=[m0, drawn, m2])
    assert torch.equal(y, ref) and _same(_grads(y, (x, *ws)), _grads(ref, (x, *ws)))


@every_function
def test_a_gradient_that_is_not_there_counts_as_zeros(name):
    class Blocks(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    call, wrt, _ = FUNCTIONS[name]()
    Blocks.apply(call()).float().sum().backward()
    for t in wrt:
        assert t.grad is not None and not t.grad.any()


@every_function
def test_a_trace_records_the_function(name):
    """The traced program computes on what it is given, gradients included."""
    import flash_dropout.functional as F

    _, wrt, _ = FUNCTIONS[name]()

    def f(x, *ws):
        if name == "linear":
            y = F.hip_blockwise_dropout_matmul(x, ws[0], BS, P, seed=5)
        elif name == "mlp":
            y = F.hip_blockwise_dropout_mlp(x, list(ws), BS, P, "gelu", seed=5)
        else:
            y = F.blockwise_dropout_conv2d(x, ws[0], BS, P, seed=5)
        return y * 2

    traced = torch.jit.trace(f, wrt, check_trace=False)
    other = [(t.detach() * 0.5).requires_grad_() for t in wrt]
    y, want = traced(*other), f(*other)
    assert torch.equal(y, want)
    assert _same(_grads(y, other), _grads(want, other))
    with torch.no_grad():
        assert torch.equal(torch.jit.trace(f, wrt, check_trace=False)(*other), want)


def test_a_trace_under_autocast_keeps_its_casts():
    import flash_dropout.functional as F

    x, w = _t(192, 136, seed=1, dtype=torch.float32), _t(72, 136, seed=2, dtype=torch.float32)
    f = lambda a, b: F.hip_blockwise_dropout_matmul(a, b, BS, P, seed=5)  # noqa: E731
    with torch.autocast("cuda", torch.bfloat16):
        traced, want = torch.jit.trace(f, (x, w), check_trace=False), f(x, w)
    assert torch.equal(traced(x, w), want) and want.dtype == torch.bfloat16


def test_draws_do_not_depend_on_the_gradient_mode():
    """A stack whose first layer keeps everything and whose input asks for a gradient takes the same draws of the
    generator when nothing is recorded."""
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    _, (x, *ws), _ = _mlp()
    ps = (0.0, P, P)
    GEMM().manual_seed(11)
    want = F.hip_blockwise_dropout_mlp(x, ws, BS, ps, "relu")
    after = GEMM().rng_state().clone()
    GEMM().manual_seed(11)
    with torch.no_grad():
        got = F.hip_blockwise_dropout_mlp(x, ws, BS, ps, "relu")
    assert torch.equal(GEMM().rng_state(), after) and torch.equal(got, want)


@every_function
def test_an_output_changed_in_place_counts_in_the_gradients(name):
    """No backward reads the result, so it may be overwritten; what the change does to the gradient is not lost."""
    call, wrt, _ = FUNCTIONS[name]()
    want = _grads(call().relu(), wrt)
    assert _same(_grads(call().relu_(), wrt), want)
