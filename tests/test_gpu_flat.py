"""The flat concat route (rows padded to a 16-byte pitch, tiles of 256
positions) between the fused generator and the fuse convolution, and the flat
copies of the stand-alone fuse convolution, against the fp64 oracle."""

import pytest
import torch

from dynamicconvolutionoperator_amd import DDPM, _lib, ops
from oracle import unfold_ref
from oracle.unfold_ref import UnfoldDDPM
from tests.gpu_helpers import DEV, DIL, TOL, assert_close, default_generator_params, randn, say

pytestmark = pytest.mark.gpu

# (n, c, h, w): one position over and under a tile of 256, rows shorter than
# the halo, a single row, a padded pitch of exactly one tile, several images,
# channel counts below and between the 16-, 32- and 64-channel blocks (24 and
# 40 channels in fp32 are not whole blocks of the pair planes: there the module
# runs the plain concat and the stand-alone fuse convolution)
SHAPES = [
    (1, 16, 1, 5), (2, 16, 15, 17), (1, 32, 3, 251), (1, 48, 9, 249), (3, 64, 20, 30),
    (1, 64, 31, 257), (2, 96, 11, 35), (1, 128, 24, 40), (1, 24, 30, 50), (2, 40, 17, 8),
    (1, 64, 70, 300),
]


def _modules(c, k, dtype):
    torch.manual_seed(7)
    ref = UnfoldDDPM(c, k)
    mod = DDPM(c, k, fused_generator_training=True)
    mod.load_state_dict(ref.state_dict())
    mod = mod.to(DEV, dtype)
    with torch.no_grad():
        for p, q in zip(ref.parameters(), mod.parameters()):
            p.copy_(q.float().cpu())
    return ref.double(), mod


def _nan_memory():
    """Leaves NaN in the memory that the allocator hands out next, in its
    large and its small blocks."""
    junk = [torch.full((1 << 24,), float("nan"), device=DEV)]
    junk += [torch.full((1 << 17,), float("nan"), device=DEV) for _ in range(64)]
    del junk


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", SHAPES)
def test_flat_training_matches_oracle(shape, dtype):
    _check_training(shape, dtype, 5)


# wide modules whose weight gradients take fewer splits than their steps allow
# (two rounds of workgroups instead of a third partly filled one): flat, and
# plain rows
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,guard", [((2, 96, 60, 66), 5), ((1, 96, 34, 256), 0), ((1, 128, 25, 256), 0)])
def test_wide_training_matches_oracle(shape, guard, dtype):
    _check_training(shape, dtype, guard)


def _check_training(shape, dtype, guard):
    n, c, h, w = shape
    say(f"training {shape} {dtype}")
    ref, mod = _modules(c, 3, dtype)
    x, y, g = (randn(shape, s, dtype=dtype) for s in (1, 2, 3))
    xg, yg = (t.to(DEV).requires_grad_() for t in (x, y))
    xr, yr = (t.double().requires_grad_() for t in (x, y))
    _nan_memory()
    out = mod(xg, yg)
    # the layout that the forward took, as its autograd node keeps it
    one_pair = dtype != torch.float32 or c % 16 == 0
    assert getattr(out.grad_fn, "guard", None) == (guard if one_pair else None), out.grad_fn
    out_ref = ref(xr, yr)
    grads = torch.autograd.grad(out, (xg, yg, *mod.parameters()), g.to(DEV))
    grads_ref = torch.autograd.grad(out_ref, (xr, yr, *ref.parameters()), g.double())
    assert_close(out, out_ref, *TOL["module_fwd"][dtype], "out")
    with torch.no_grad():  # (its layout has one guard row, the training one five)
        assert_close(mod(xg, yg), out_ref, *TOL["module_fwd"][dtype], "inference")
    atol, rtol = TOL["module_bwd"][dtype]
    for name, a, e in zip(("dx", "dy", "dgw", "dgb", "dfw", "dfb"), grads, grads_ref):
        assert_close(a, e, atol * max(e.abs().max().item(), 1e-6), rtol, name)


# one tap, and other dilations than 1, 3, 5 (the largest halo, the smallest, a
# first branch wider than the others), through the channel blocks of the
# kernels: 16, 48 (three blocks), 64, and halves of 64
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,k,dil", [
    ((1, 64, 21, 43), 1, DIL), ((2, 96, 13, 35), 1, DIL), ((1, 16, 20, 30), 3, (1, 1, 1)),
    ((2, 48, 19, 29), 3, (2, 7, 8)), ((1, 80, 18, 37), 3, (8, 1, 4)), ((1, 128, 20, 50), 3, (3, 3, 2)),
])
def test_flat_kernel_sizes_and_dilations(shape, k, dil, dtype):
    say(f"flat {shape} K={k} dilations={dil} {dtype}")
    n, c, h, w = shape
    gw, gb = default_generator_params(c, k, 5, dtype)
    torch.manual_seed(6)
    conv = torch.nn.Conv2d(4 * c, c, 3, 1, 1)
    fw, fb = conv.weight.detach().to(dtype), conv.bias.detach().to(dtype)
    tensors = (randn(shape, 1, dtype), randn(shape, 2, dtype), gw, gb, fw, fb)
    g = randn(shape, 3, dtype)
    dev = [t.to(DEV).requires_grad_() for t in tensors]
    x, y, gw, gb, fw, fb = ref = [t.double().requires_grad_() for t in tensors]
    _nan_memory()
    out = ops._fused_ddpm_checked(*dev, k, dil, flat=True)
    assert out.grad_fn.guard == max(1, k // 2 * max(dil))
    cat = unfold_ref.generator_dynamic_cat(x, y, gw, gb, k, dil)
    out_ref = torch.nn.functional.conv2d(cat, fw, fb, padding=1)
    got, want = torch.autograd.grad(out, dev, g.to(DEV)), torch.autograd.grad(out_ref, ref, g.double())
    assert_close(out, out_ref, *TOL["module_fwd"][dtype], "out")
    with torch.no_grad():
        assert_close(ops._fused_ddpm_checked(*dev, k, dil, flat=True), out_ref, *TOL["module_fwd"][dtype], "inference")
    atol, rtol = TOL["module_bwd"][dtype]
    for name, a, e in zip(("dx", "dy", "dgw", "dgb", "dfw", "dfb"), got, want):
        assert_close(a, e, atol * max(e.abs().max().item(), 1e-6), rtol, name)


def test_flat_plain_fp32_concat(monkeypatch):
    """The flat entry points take a plain fp32 concat (dtype 0) too; the module's
    fp32 concat is pair planes."""
    _, mod = _modules(48, 3, torch.float32)
    x, y, g = (randn((2, 48, 13, 21), s).to(DEV).requires_grad_() for s in (1, 2, 3))
    leaves = (x, y, *mod.parameters())

    def run():
        out = mod(x, y)
        return out, *torch.autograd.grad(out, leaves, g)

    want = run()
    monkeypatch.setattr(ops, "_cat_code", lambda dtype: ops._DTYPES[dtype])
    for a, e in zip(run(), want):
        # the concat's bf16 halves formed at another place, the sums' order as before
        assert_close(a, e.double().cpu(), 2e-5 * e.abs().max().item(), 2e-5, "")


def test_flat_partial_gradients_match_all():
    """Each subset of the gradients is bit for bit the full backward's."""
    shape, dtype = (2, 32, 13, 21), torch.bfloat16
    _, mod = _modules(32, 3, dtype)
    x, y, g = (randn(shape, s, dtype=dtype).to(DEV) for s in (1, 2, 3))
    tensors = (x, y, *(p.detach() for p in mod.parameters()))

    def grads(needs):
        t = [v.clone().requires_grad_(f) for v, f in zip(tensors, needs)]
        out = ops._fused_ddpm_checked(*t, 3, DIL, flat=True)
        it = iter(torch.autograd.grad(out, [v for v, f in zip(t, needs) if f], g))
        return [next(it) if f else None for f in needs]

    full = grads((True,) * 6)
    for needs in [(1, 0, 0, 0, 0, 0), (0, 1, 0, 0, 0, 0), (0, 0, 1, 1, 0, 0), (0, 0, 0, 0, 1, 1),
                  (1, 1, 0, 0, 0, 0), (1, 0, 0, 1, 0, 0), (0, 1, 1, 0, 1, 0)]:
        for a, e in zip(grads([bool(f) for f in needs]), full):
            assert a is None or torch.equal(a, e), needs


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 24, 15, 17), (1, 20, 9, 33), (1, 64, 7, 255), (2, 100, 13, 31), (1, 136, 9, 33)])
def test_stand_alone_fuse_conv_copies_flat(shape, dtype):
    """Odd widths: the public NCHW fuse convolution lays its operands out flat
    (C % 8 != 0: the weight gradient does not; above 128 channels it is the
    library's)."""
    n, c, h, w = shape
    cat, g = randn((n, 4 * c, h, w), 1, dtype=dtype), randn(shape, 2, dtype=dtype)
    wt, b = randn((c, 4 * c, 3, 3), 3, dtype=dtype, scale=0.05), randn((c,), 4, dtype=dtype)
    dev = [t.to(DEV).requires_grad_() for t in (cat, wt, b)]
    ref = [t.double().requires_grad_() for t in (cat, wt, b)]
    out = ops.fuse_conv3x3(*dev)
    out_ref = torch.nn.functional.conv2d(ref[0], ref[1], ref[2], padding=1)
    own = 3 if c <= 128 else 1
    got = torch.autograd.grad(out, dev[:own], g.to(DEV))
    want = torch.autograd.grad(out_ref, ref[:own], g.double())
    assert_close(out, out_ref, *TOL["module_fwd"][dtype], "out")
    atol, rtol = TOL["module_bwd"][dtype]
    for name, a, e in zip(("dcat", "dw", "db"), got, want):
        assert_close(a, e, atol * e.abs().max().item(), rtol, name)


# more than 64 channels: (c, h, w) whose grids take each tile width of the
# paired forward (16, 32 and 64 columns beside three chunks' weights, 16 and
# 32 beside four's) with a ragged last chunk, tile row and tile column, and a
# channel count the paired forward does not take
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [
    (72, 33, 40), (72, 45, 397), (72, 99, 397), (104, 20, 37), (120, 30, 395), (72, 97, 384), (76, 20, 37),
])
def test_wide_modules_match_oracle(shape, dtype):
    c, h, w = shape
    say(f"wide inference {shape} {dtype}")
    ref, mod = _modules(c, 3, dtype)
    x, y = (randn((1, c, h, w), s, dtype=dtype) for s in (1, 2))
    with torch.no_grad():
        out_ref = ref(x.double(), y.double())
        assert_close(mod(x.to(DEV), y.to(DEV)), out_ref, *TOL["module_fwd"][dtype], "module")
        cat = ops.fused_generator_dynamic_cat(x.to(DEV), y.to(DEV), mod.generator.weight,
                                              mod.generator.bias, 3, DIL)
        out = torch.nn.functional.conv2d(cat.double().cpu(), ref.fuse.weight, ref.fuse.bias, padding=1)
        assert_close(out, out_ref, *TOL["module_fwd"][dtype], "plain concat")


# 104 to 128 channels at a halo of one pixel, where a 64-column tile fits the
# LDS and takes the fewest rounds of workgroups, but no kernel has that tile
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,w", [(104, 256), (128, 256), (120, 250)])
def test_wide_forward_at_unit_dilations(c, w, dtype):
    shape, dil = (1, c, 128, w), (1, 1, 1)
    say(f"unit dilations {shape} {dtype}")
    x, y = randn(shape, 1, dtype), randn(shape, 2, dtype)
    wt, b = default_generator_params(c, 3, 3, dtype)
    _nan_memory()
    out = ops.fused_generator_dynamic_cat(x.to(DEV), y.to(DEV), wt.to(DEV), b.to(DEV), 3, dil)
    kernels = unfold_ref.generated_kernels(y.double(), wt.double(), b.double(), 3).to(dtype).double()
    atol, rtol = TOL["gen_fwd"][dtype]
    assert_close(out, unfold_ref.dynamic_cat(x.double(), kernels, 3, dil), atol, rtol, "concat")


@pytest.mark.parametrize("dtype,c", [(torch.float32, 16), (torch.float32, 48), (torch.bfloat16, 24), (torch.float16, 64)])
def test_flat_gradient_is_written_whole(dtype, c):
    """The concat's flat gradient passes through autograd: every element of it
    is a number, whatever its memory held (3C a multiple of 16 and not), so
    that NaN detection accepts a step."""
    say(f"anomaly detection C={c} {dtype}")
    _, mod = _modules(c, 3, dtype)
    x, y, g = (randn((2, c, 45, 51), s, dtype=dtype).to(DEV).requires_grad_() for s in (1, 2, 3))
    seen = []
    out = mod(x, y)
    out.grad_fn.register_hook(lambda grads_in, grads_out: seen.append(grads_in[0]))
    _nan_memory()
    out.backward(g)
    assert seen[0].ndim == 1 and bool(torch.isfinite(seen[0]).all())
    with torch.autograd.detect_anomaly():
        out = mod(x, y)
        _nan_memory()
        out.backward(g)


# an infinite x reaches the weight gradients of the taps that meet it inside
# the image and no others (dilated taps from the first and last columns and
# rows lie outside): finite where the oracle is, and equal there
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,k", [(32, 3), (96, 3), (64, 1)])
def test_flat_infinities_stay_in_their_taps(c, k, dtype):
    say(f"infinities C={c} K={k} {dtype}")
    shape = (2, c, 20, 30)
    oracle, mod = _modules(c, k, dtype)
    x, y, g = (randn(shape, s, dtype=dtype) for s in (1, 2, 3))
    x[0, 1, 7, 0] = x[1, 5, 19, 12] = x[1, 9, 3, 29] = float("inf")
    x[0, 20, 0, 0] = -float("inf")
    xg, yg = (t.to(DEV).requires_grad_() for t in (x, y))
    xr, yr = (t.double().requires_grad_() for t in (x, y))
    got = torch.autograd.grad(mod(xg, yg), (xg, yg, *mod.parameters()), g.to(DEV))
    want = torch.autograd.grad(oracle(xr, yr), (xr, yr, *oracle.parameters()), g.double())
    atol, rtol = TOL["module_bwd"][dtype]
    for name, a, e in zip(("dx", "dy", "dgw", "dgb", "dfw", "dfb"), got, want):
        a, finite = a.detach().double().cpu(), torch.isfinite(e)
        assert torch.equal(torch.isfinite(a), finite), name
        assert_close(a[finite], e[finite], atol * e[finite].abs().max().item(), rtol, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_stand_alone_fuse_conv_infinities_stay_in_their_taps(dtype):
    n, c, h, w = 2, 32, 61, 125
    cat, g = randn((n, 4 * c, h, w), 1, dtype=dtype), randn((n, c, h, w), 2, dtype=dtype)
    cat[0, 3, 7, 0] = cat[1, 50, h - 1, 12] = cat[1, 9, 3, w - 1] = float("inf")
    wt = randn((c, 4 * c, 3, 3), 3, dtype=dtype, scale=0.05)
    wd, wr = wt.to(DEV).requires_grad_(), wt.double().requires_grad_()
    (got,) = torch.autograd.grad(ops.fuse_conv3x3(cat.to(DEV), wd, None), wd, g.to(DEV))
    (want,) = torch.autograd.grad(torch.nn.functional.conv2d(cat.double(), wr, padding=1), wr, g.double())
    assert torch.equal(torch.isfinite(got.cpu()), torch.isfinite(want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c", [64, 72, 128])
def test_paired_forward_of_infinite_kernels(c, dtype):
    """An infinite y makes the generated kernels infinite, and the branches
    with them, not NaN: the last tap of a branch has no partner to pair with."""
    shape = (1, c, 20, 40)
    x, y = randn(shape, 1, dtype).abs() + 0.5, randn(shape, 2, dtype)
    wt, b = default_generator_params(c, 3, 3, dtype)
    wt = wt.abs() + 2.0**-6  # (no zero weight, no cancelling signs)
    y[0, 5, 9, 11] = float("inf")
    out = ops.fused_generator_dynamic_cat(x.to(DEV), y.to(DEV), wt.to(DEV), b.to(DEV), 3, DIL).cpu()
    want = unfold_ref.generator_dynamic_cat(x.double(), y.double(), wt.double(), b.double(), 3)
    assert torch.equal(torch.isinf(out), torch.isinf(want)) and not bool(torch.isnan(out).any())


@pytest.mark.parametrize("code,dtype", [(0, torch.float32), (1, torch.bfloat16)])
def test_stand_alone_fuse_conv_workspaces(code, dtype):
    """At an odd width the fuse convolution copies its operands flat; a
    workspace without room for the copies (the packed weight and the partial
    sums alone), one off a 16-byte boundary for the weight gradient, and none
    where a single split needs none, give the same gradients without them."""
    lib = _lib.load()
    n, c, h, w = 1, 64, 135, 181
    stream = torch.cuda.current_stream().cuda_stream
    cat, g = randn((n, 4 * c, h, w), 1).to(dtype).to(DEV), randn((n, c, h, w), 2).to(dtype).to(DEV)
    wt, b = randn((c, 4 * c, 3, 3), 3, scale=0.05).to(dtype).to(DEV), randn((c,), 4).to(dtype).to(DEV)

    def buffers():
        shapes = (g.shape, cat.shape, wt.shape, b.shape)
        return [torch.full(s, float("nan"), dtype=dtype, device=DEV) for s in shapes]

    def memory(nbytes, off=0):
        return torch.empty(nbytes + 16, dtype=torch.uint8, device=DEV)[off:]

    query = lib.ddpm_fuse_conv_workspace_bytes(n, c, h, w, code)
    query_w = lib.ddpm_fuse_conv_bwd_weight_workspace_bytes(n, c, h, w, code)
    # forward: 8 chunks of 32 planes x 9 taps x 4 blocks x 1 KB (fp32: hi and lo),
    # two plane splits; weight gradient: 16 splits of 36 C^2 + C
    plain = 8 * 9 * 4 * 1024 * (2 if code == 0 else 1) + 2 * n * c * h * w * 4
    plain_w = 16 * (36 * c * c + c) * 4
    assert plain < query and plain_w < query_w
    results = []
    for size, size_w, off in ((query, query_w, 0), (plain, plain_w, 0), (query, plain_w, 0),
                              (plain, query_w, 0), (query, query_w, 4)):
        out, gc, gw, gb = buffers()
        ws, wsw = memory(size), memory(size_w, off)
        rc = lib.ddpm_fuse_conv_fwd(cat.data_ptr(), wt.data_ptr(), b.data_ptr(), out.data_ptr(), ws.data_ptr(),
                                    size, n, c, h, w, code, stream)
        assert rc == 0, rc
        rc = lib.ddpm_fuse_conv_bwd(cat.data_ptr(), wt.data_ptr(), g.data_ptr(), gc.data_ptr(), gw.data_ptr(),
                                    gb.data_ptr(), ws.data_ptr(), size, wsw.data_ptr(), size_w, n, c, h, w,
                                    code, stream)
        assert rc == 0, rc
        results.append((out, gc, gw, gb))
        _, _, gw, gb = buffers()
        rc = lib.ddpm_fuse_conv_bwd_weight(cat.data_ptr(), g.data_ptr(), gw.data_ptr(), gb.data_ptr(),
                                           wsw.data_ptr(), size_w, n, c, h, w, code, stream)
        assert rc == 0, rc
        assert torch.equal(gw, results[-1][2]) and torch.equal(gb, results[-1][3])
    for got in results[1:]:
        for name, a, e in zip(("out", "dcat", "dw", "db"), got, results[0]):
            # the same products in another order: fp32 sums, then one rounding
            tol = 2e-5 if dtype == torch.float32 else 1e-2
            assert_close(a, e.double().cpu(), tol * e.abs().max().item(), tol, name)
    _, _, gw, gb = buffers()
    few = cat[:, :, :1, :17].contiguous(), g[:, :, :1, :17].contiguous()
    rc = lib.ddpm_fuse_conv_bwd_weight(few[0].data_ptr(), few[1].data_ptr(), gw.data_ptr(), gb.data_ptr(), None,
                                       0, n, c, 1, 17, code, stream)
    torch.cuda.synchronize()
    assert rc == 0 and not bool(torch.isnan(gw).any()), rc


def test_flat_backward_of_tensors_off_16_bytes():
    """Saved-tensor and gradient hooks may hand back tensors that start anywhere."""
    _, mod = _modules(32, 3, torch.bfloat16)
    x, y, g = (randn((1, 32, 45, 51), s, dtype=torch.bfloat16).to(DEV).requires_grad_() for s in (1, 2, 3))
    leaves = (x, y, *mod.parameters())

    def unaligned(t):
        if t is None or t.dtype != torch.bfloat16:
            return t
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        return buf[1:].view(t.shape).copy_(t)

    want = torch.autograd.grad(mod(x, y), leaves, g)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unaligned):
        out = mod(x, y)
        out.grad_fn.register_hook(lambda grads_in, grads_out: tuple(unaligned(t) for t in grads_in))
        got = torch.autograd.grad(out, leaves, g)
    for a, e in zip(got, want):
        assert torch.equal(a, e)
