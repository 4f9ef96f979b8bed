"""Products on the bf16 matrix instruction with operands split in three (csrc/conv_split.hip): edges of their tiles,
ragged channel counts, reduction splits, operands that are not finite; against the oracle."""
import numpy as np
import pytest

from util import F, rel_max

pytestmark = pytest.mark.gpu

# Both sides add R products in fp32 in some order: each within R 2^-24 of sum |x w| of the exact sum, in practice sqrt(R)
# of it, and max |y| is a few times the typical sum: 1e-5 covers R up to 3000 with a factor of three.
TOL = 1e-5

CASES = [  # x (H, W, C, N), f (FH, FW, FC, K), stride, pad, dilate
    ((16, 16, 16, 1), (1, 1, 16, 5), 1, 0, 1),          # one chunk, one group of taps: padding to a slab; five channels out
    ((12, 11, 6, 1), (3, 3, 6, 33), 1, 1, 1),           # fewest channels in, a second channel block of one
    ((13, 10, 17, 2), (3, 3, 17, 31), 1, 1, 1),         # a chunk of one channel; one pixel tile and a bit
    ((9, 14, 20, 3), (5, 3, 20, 65), (2, 1), (2, 1, 0, 1), 1),   # strided, asymmetric padding, a third block of one channel
    ((16, 16, 32, 1), (2, 2, 32, 64), 1, (1, 0, 1, 0), 1),       # 256 pixels exactly; groups 8
    ((17, 16, 48, 2), (3, 3, 48, 96), 1, 2, 2),         # odd number of groups (27), dilation, three channel blocks
    ((8, 17, 16, 1), (3, 3, 16, 128), 1, 1, 1),         # nine groups, a tile of 8 pixels at the end
    ((23, 29, 64, 2), (3, 3, 64, 200), 1, 1, 1),        # 128-channel tiles, 72 channels in the last
]


@pytest.fixture
def any_size(capi):
    """Split operands at every size: the edges of tiles are tested on small layers."""
    capi.set_tunable("conv_any_size", 1)
    yield
    capi.set_tunable("conv_any_size", 0)


@pytest.mark.parametrize("wa", [0, 1, 2, 4])
@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("xs,fs,stride,pad,dilate", CASES)
def test_forward_and_backward_data(capi, ob, xs, fs, stride, pad, dilate, splits, wa):
    r = np.random.default_rng(sum(xs) + sum(fs))
    x, f = F(r.standard_normal(xs)), F(r.standard_normal(fs) / np.sqrt(np.prod(fs[:3])))
    b = r.standard_normal(fs[3]).astype(np.float32)
    g, og = capi.conv_geom(xs, fs, stride, pad, dilate), ob.conv_geom(xs, fs, stride, pad, dilate)
    want = ob.conv_forward(x, f, b, og)
    dy, y0, dx0 = F(r.standard_normal(want.shape)), F(r.standard_normal(want.shape)), F(r.standard_normal(xs))
    wdx = ob.conv_backward(x, f, dy, og, want=(True, False, False))[0]
    xd, fd, bd, dyd = (capi.to_device(v) for v in (x, f, b, dy))
    capi.set_tunable("conv_split_wa", wa)
    capi.set_tunable("conv_split_splits", splits)
    capi.set_tunable("conv_short", -1)
    try:
        capi.profile_begin("conv_split_mfma")
        y = capi.to_host(capi.conv_forward(xd, fd, bd, g))
        launches, _ = capi.profile_end()
        y2 = capi.to_host(capi.conv_forward(xd, fd, bd, g, y=capi.to_device(y0), out_mult=0.5, in_mult=2.0))
        dx = capi.to_host(capi.conv_backward_data_acc(capi.empty(xs), 0.0, fd, dyd, g))
        dx2 = capi.to_host(capi.conv_backward_data_acc(capi.to_device(dx0), 1.0, fd, dyd, g))
    finally:
        capi.set_tunable("conv_split_wa", 0)
        capi.set_tunable("conv_split_splits", 0)
        capi.set_tunable("conv_short", 0)
    assert launches == 1
    b4 = b.reshape(1, 1, -1, 1)
    assert rel_max(y, want) <= TOL and rel_max(y2, 0.5 * y0 + 2.0 * (want - b4) + b4) <= TOL
    assert rel_max(dx, wdx) <= TOL and rel_max(dx2, dx0 + wdx) <= TOL


@pytest.fixture(params=[0, -1], ids=["few pixels apart", "tiles of 128 pixels"])
def either(capi, request):
    """Products over few pixels by the kernel that takes them, and by the one for all."""
    capi.set_tunable("conv_short", request.param)
    yield
    capi.set_tunable("conv_short", 0)


def test_no_less_accurate_than_the_fp32_instruction(capi, either):
    """The same product through this kernel and through the fp32 matrix instruction, both against double: the error here
    is not the larger one (it is about 0.85 of the other: fewer roundings of the accumulator)."""
    import torch
    g = capi.conv_geom((14, 14, 256, 8), (3, 3, 256, 128), 1, 1, 1)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    x = torch.randn(8, 256, 14, 14, device="cuda", generator=gen)
    f = torch.randn(128, 256, 3, 3, device="cuda", generator=gen) / 48
    want = torch.nn.functional.conv2d(x.cpu().double(), f.cpu().double(), padding=1)
    got = {}
    for fp32 in (0, 1):
        capi.set_tunable("conv_no_ws", fp32)
        try:
            got[fp32] = float((capi.conv_forward(x, f, None, g).cpu().double() - want).norm() / want.norm())
        finally:
            capi.set_tunable("conv_no_ws", 0)
    assert got[0] <= 1.02 * got[1], got


@pytest.mark.parametrize("xs,fs", [((12, 12, 32, 2), (3, 3, 32, 40)), ((11, 9, 20, 2), (1, 1, 20, 72))])
def test_operands_that_are_not_finite_or_round_to_infinity(capi, ob, either, xs, fs):
    """Infinities, NaNs and magnitudes above bf16's largest give what fp32 arithmetic gives, and only where they reach."""
    r = np.random.default_rng(9)
    x, f = F(r.uniform(0.5, 1.0, xs)), F(r.uniform(0.5, 1.0, fs) / np.prod(fs[:3]))
    x[3, 4, 5, 0], x[7, 2, 1, 1], x[0, 0, 0, 0], x[5, 5, xs[2] - 1, 1] = np.inf, np.nan, -np.inf, 3.4e38
    f[0, 0, 2, 3] = np.inf
    pad = fs[0] // 2
    g, og = capi.conv_geom(xs, fs, 1, pad, 1), ob.conv_geom(xs, fs, 1, pad, 1)
    want = ob.conv_forward(x, f, None, og)
    got = capi.to_host(capi.conv_forward(capi.to_device(x), capi.to_device(f), None, g))
    assert np.isnan(want).any() and np.isinf(want).any() and (np.abs(want[np.isfinite(want)]) > 1e30).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    rest = ~np.isnan(want)
    assert np.array_equal(np.isinf(got[rest]), np.isinf(want[rest]))
    fin = np.isfinite(want)
    assert np.max(np.abs(got[fin] - want[fin]) / np.abs(want[fin])) <= TOL  # (all terms positive: no cancellation)


@pytest.mark.usefixtures("any_size")
@pytest.mark.parametrize("xs,k", [((6, 6, 256, 6), 911), ((7, 5, 61, 37), 1003), ((1, 1, 2048, 128), 200), ((1, 1, 64, 128), 6200), ((3, 3, 250, 128), 177),
                                  ((6, 6, 256, 5), 1100)])
def test_fully_connected(capi, xs, k):
    """Layers of one output pixel: products over rows of the bank and of x, in the derivatives dzdy in the bank's place
    (fewest images it takes, pixels and channels beside whole tiles; five images: the filters with the general kernel)."""
    import torch
    h, w, c, n = xs
    gen = torch.Generator(device="cuda")
    gen.manual_seed(k)
    x = torch.randn(n, c, w, h, device="cuda", generator=gen)
    f = torch.randn(k, c, w, h, device="cuda", generator=gen) / np.sqrt(h * w * c)
    dy = torch.randn(n, k, 1, 1, device="cuda", generator=gen)
    g = capi.conv_geom((h, w, c, n), (h, w, c, k), 1, 0, 1)
    rows = lambda t: t.double().reshape(t.shape[0], -1)
    wdx, wdf, wdb = rows(dy) @ rows(f), rows(dy).t() @ rows(x), rows(dy).sum(0)
    b = torch.randn(k, device="cuda", generator=gen)
    wy = rows(x) @ rows(f).t() + b.double()
    capi.profile_begin("conv_wgrad_mfma_split")
    y = capi.conv_forward(x, f, b, g)
    launches, _ = capi.profile_end()
    y2 = capi.conv_forward(x, f, b, g, y=y.clone(), out_mult=0.5, in_mult=2.0)
    assert launches == (1 if n >= 16 else 0)
    close = lambda a, b: float((a.double() - b).abs().max() / b.abs().max())
    assert close(rows(y), wy) <= TOL and close(rows(y2), 2.5 * wy - b.double()) <= TOL
    launches = 0
    for kernel in ("conv_split_mfma", "conv_split_short"):  # (few values to an image: few pixels here)
        capi.profile_begin(kernel)
        dx = capi.conv_backward_data_acc(torch.empty_like(x), 0.0, f, dy, g)
        _, df, db = capi.conv_backward(x, f, dy, g, want=(False, True, True))
        launches += capi.profile_end()[0]
    dx2 = capi.conv_backward_data_acc(x.clone(), 1.0, f, dy, g)
    assert launches == (1 if n < 6 else 2)
    assert close(rows(dx), wdx) <= TOL and close(rows(dx2), wdx + rows(x)) <= TOL
    assert close(rows(df), wdf) <= TOL and close(db.reshape(-1), wdb) <= 1e-6  # (sums in double, rounded once)


FILTER_CASES = [  # x (H, W, C, N), f (FH, FW, FC, K), stride, pad, dilate
    ((8, 8, 16, 1), (1, 1, 16, 16), 1, 0, 1),           # one half-block each way, two steps
    ((5, 6, 17, 1), (1, 1, 17, 19), 1, 0, 1),           # one pixel short of a step; all but one row computed twice
    ((9, 7, 48, 3), (3, 3, 48, 40), 1, 1, 1),           # half-blocks of different taps in a block; tile of 64 filters
    ((9, 14, 44, 3), (5, 3, 44, 130), (2, 1), (2, 1, 0, 1), 1),  # strided, asymmetric padding, a second filter tile of two
    ((17, 16, 64, 2), (3, 3, 64, 64), 1, 2, 2),         # 192-row tiles, dilation
    ((13, 13, 32, 4), (5, 5, 16, 48), 1, 2, 1),         # two groups, 24 filters each: 32-filter tiles
    ((14, 14, 256, 3), (1, 1, 64, 512), 2, 0, 1),       # four groups, 64-row tiles of 128 filters
    ((12, 12, 64, 9), (3, 3, 64, 128), 1, 1, 1),        # 128 x 128
    ((30, 30, 130, 2), (1, 1, 130, 66), 1, 0, 1),       # a third block of two filters, 130 rows
]


@pytest.mark.usefixtures("any_size")
@pytest.mark.parametrize("xs,fs,stride,pad,dilate", FILTER_CASES)
def test_filter_gradient(capi, ob, xs, fs, stride, pad, dilate):
    r = np.random.default_rng(sum(xs) + sum(fs))
    x, f = F(r.standard_normal(xs)), F(r.standard_normal(fs))
    g, og = capi.conv_geom(xs, fs, stride, pad, dilate), ob.conv_geom(xs, fs, stride, pad, dilate)
    dy = F(r.standard_normal(capi.conv_out_shape(g)))
    want = ob.conv_backward(x, f, dy, og, want=(False, True, False))[1]
    xd, fd, dyd = (capi.to_device(v) for v in (x, f, dy))
    capi.profile_begin("conv_wgrad_mfma_split")
    df = capi.to_host(capi.conv_backward(xd, fd, dyd, g, want=(False, True, False))[1])
    launches, _ = capi.profile_end()
    assert launches == xs[2] // fs[2]
    assert rel_max(df, want) <= TOL


@pytest.mark.usefixtures("any_size")
@pytest.mark.parametrize("tile", [48, 44, 82, 42, 28, 24, 26, 22, 14])
@pytest.mark.parametrize("xs,fs,stride,pad,dilate", FILTER_CASES[1:4] + FILTER_CASES[6:7] + [
    ((9, 11, 144, 3), (1, 1, 144, 272), 1, 0, 1),   # second tiles of nearly nothing in every shape; a last step of nine pixels
    ((11, 7, 35, 11), (3, 3, 35, 37), 1, 1, 1),     # split over the pixels, ragged both ways
])
def test_filter_gradient_in_every_tile(capi, ob, tile, xs, fs, stride, pad, dilate):
    r = np.random.default_rng(sum(xs) + sum(fs))
    x, f = F(r.standard_normal(xs)), F(r.standard_normal(fs))
    g, og = capi.conv_geom(xs, fs, stride, pad, dilate), ob.conv_geom(xs, fs, stride, pad, dilate)
    dy = F(r.standard_normal(capi.conv_out_shape(g)))
    want = ob.conv_backward(x, f, dy, og, want=(False, True, False))[1]
    x2 = x.copy(order="F")
    x2[xs[0] // 4 * 2, xs[1] // 4 * 2, xs[2] - 1, xs[3] - 1] = np.inf  # (a tile that is done again on the fp32 instruction)
    want2 = ob.conv_backward(x2, f, dy, og, want=(False, True, False))[1]
    capi.set_tunable("conv_wsplit_tile", tile)
    try:
        df, df2 = (capi.to_host(capi.conv_backward(*(capi.to_device(v) for v in (a, f, dy)), g, want=(False, True, False))[1]) for a in (x, x2))
    finally:
        capi.set_tunable("conv_wsplit_tile", 0)
    assert rel_max(df, want) <= TOL
    fin = np.isfinite(want2)
    assert not fin.all() and np.array_equal(df2[~fin], want2[~fin], equal_nan=True)
    assert rel_max(df2[fin], want2[fin]) <= TOL


def test_filter_gradient_no_less_accurate_than_the_fp32_instruction(capi):
    import torch
    g = capi.conv_geom((14, 14, 96, 32), (3, 3, 96, 128), 1, 1, 1)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    x = torch.randn(32, 96, 14, 14, device="cuda", generator=gen)
    dy = torch.randn(32, 128, 14, 14, device="cuda", generator=gen)
    f = torch.zeros(128, 96, 3, 3, device="cuda")
    want = torch.nn.grad.conv2d_weight(x.cpu().double(), (128, 96, 3, 3), dy.cpu().double(), padding=1)
    got = {}
    for fp32 in (0, 1):
        capi.set_tunable("conv_wgrad_no_split", fp32)
        try:
            got[fp32] = float((capi.conv_backward(x, f, dy, g, want=(False, True, False))[1].cpu().double() - want).norm() / want.norm())
        finally:
            capi.set_tunable("conv_wgrad_no_split", 0)
    assert got[0] <= 1.02 * got[1], got


def test_filter_gradient_of_operands_that_are_not_finite(capi, ob):
    r = np.random.default_rng(10)
    xs, fs = (10, 9, 40, 3), (3, 3, 40, 72)
    x, f = F(r.uniform(0.5, 1.0, xs)), F(np.zeros(fs))
    g, og = capi.conv_geom(xs, fs, 1, 1, 1), ob.conv_geom(xs, fs, 1, 1, 1)
    dy = F(r.uniform(0.5e-3, 1e-3, capi.conv_out_shape(g)))
    x[3, 4, 5, 0], x[7, 2, 38, 1], x[5, 5, 20, 2] = np.inf, np.nan, 3.4e38
    dy[2, 2, 3, 1] = -np.inf
    want = ob.conv_backward(x, f, dy, og, want=(False, True, False))[1]
    got = capi.to_host(capi.conv_backward(*(capi.to_device(v) for v in (x, f, dy)), g, want=(False, True, False))[1])
    assert np.isnan(want).any() and np.isinf(want).any() and (np.abs(want[np.isfinite(want)]) > 1e30).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    rest = ~np.isnan(want)
    assert np.array_equal(np.isinf(got[rest]), np.isinf(want[rest]))
    fin = np.isfinite(want)
    assert np.max(np.abs(got[fin] - want[fin]) / np.abs(want[fin])) <= TOL


@pytest.mark.parametrize("xs,fs,stride,pad,splits", [
    ((7, 7, 64, 3), (3, 3, 64, 96), 1, 1, 3),       # planes of 49: no 16-byte accesses; split reduction
    ((7, 7, 64, 3), (3, 3, 64, 96), 1, 1, 0),       # the same by the kernel for few pixels
    ((14, 14, 512, 2), (1, 1, 512, 64), 1, 0, 4),   # split, 16-byte accesses
    ((13, 11, 48, 2), (3, 3, 48, 32), 2, 1, 1),     # one launch, a last tile of pixels
    ((28, 28, 32, 90), (1, 1, 32, 160), 1, 0, 0),   # whole rounds; 32 channels in the last tile of 128
    ((48, 48, 256, 48), (3, 3, 256, 128), 1, 1, 0), # a round left over: its tiles split, added up and normalised apart
])
@pytest.mark.parametrize("relu,add", [(True, False), (True, True), (False, False)])
def test_normalised_output_has_the_bits_of_separate_calls(capi, xs, fs, stride, pad, splits, relu, add):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(xs))
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f = normal(*xs[::-1]), normal(*fs[::-1]) / np.sqrt(np.prod(fs[:3]))
    g = capi.conv_geom(xs, fs, stride, pad, 1)
    K = fs[3]
    moments = torch.stack([normal(K), 0.5 + torch.rand(K, device="cuda", generator=gen)])
    mult, bias = normal(K), normal(K)
    res = normal(*capi.conv_out_shape(g)[::-1]) if add else None
    capi.set_tunable("conv_split_splits", splits)
    try:
        a = capi.conv_forward(x, f, None, g)
        capi.profile_begin("conv_pix_reduce_bn")
        got = capi.conv_forward_bnorm(x, f, g, moments, mult, bias, res, relu)
        launches, _ = capi.profile_end()
    finally:
        capi.set_tunable("conv_split_splits", 0)
    assert launches == (1 if splits > 1 else 0)
    want = capi.bnorm_forward_fused(a, mult, bias, residual=res, relu=relu, moments=moments)[0]
    assert got is not None and torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_normalised_output_is_refused_where_there_is_no_such_form(capi):
    for xs, fs in [((8, 8, 20, 2), (3, 3, 20, 32)), ((8, 8, 32, 2), (3, 3, 32, 33)), ((8, 8, 32, 2), (3, 3, 16, 32)), ((6, 6, 32, 2), (6, 6, 32, 64))]:
        g = capi.conv_geom(xs, fs, 1, 0, 1)
        assert capi.lib().mcn_conv_forward_bnorm_supported(g) == 0
        x, f = capi.empty(xs, 1.0), capi.empty(fs, 1.0)
        ones = capi.empty((fs[3], 2), 1.0)
        rc = capi.lib().mcn_conv_forward_bnorm(capi.stream(), g, capi.ptr(capi.empty(capi.conv_out_shape(g))), capi.ptr(x), capi.ptr(f), None, 0,
                                               capi.ptr(ones), capi.ptr(ones), capi.ptr(ones), None, 0, None, 0)
        assert rc != 0


@pytest.mark.parametrize("product", ["forward", "input", "filters"])
@pytest.mark.parametrize("xs,fs", [((28, 28, 64, 8), (3, 3, 64, 64)), ((28, 28, 64, 8), (1, 1, 64, 256)), ((14, 14, 256, 8), (3, 3, 256, 128))])
def test_errors_behind_a_relu_are_no_larger_and_centred(capi, either, xs, fs, product):
    """Where half of an operand is zeros the fp32 instruction rounds half as often: its error is the smaller one of the two
    operand kinds, and what this kernel's is held to.  And its errors are centred: the mean over the n pixels of a channel
    (batch normalisation and bias gradients add them up) lies within a few sigma / sqrt(n); the rms over the channels of
    the mean in those units is 1 for independent errors, 3 leaves room for neighbouring pixels' common operands."""
    import torch
    h, w, c, n = xs
    k = fs[3]
    pad = fs[0] // 2
    g = capi.conv_geom(xs, fs, 1, pad, 1)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f, dy = normal(n, c, w, h).clamp_min(0), normal(k, c, *fs[:2]) / np.sqrt(np.prod(fs[:3])), normal(n, k, w, h).clamp_min(0)
    xc, fc, dc = (t.cpu().double() for t in (x, f, dy))
    want, call = {"forward": (lambda: torch.nn.functional.conv2d(xc, fc, padding=pad), lambda: capi.conv_forward(x, f, None, g)),
                  "input": (lambda: torch.nn.grad.conv2d_input(xc.shape, fc, dc, padding=pad),
                            lambda: capi.conv_backward_data_acc(torch.empty_like(x), 0.0, f, dy, g)),
                  "filters": (lambda: torch.nn.grad.conv2d_weight(xc, fc.shape, dc, padding=pad),
                              lambda: capi.conv_backward(x, f, dy, g, want=(False, True, False))[1])}[product]
    want = want()
    switch = "conv_wgrad_no_split" if product == "filters" else "conv_no_ws"
    error = {}
    for fp32 in (1, 0):
        capi.set_tunable(switch, fp32)
        try:
            e = call().cpu().double() - want
        finally:
            capi.set_tunable(switch, 0)
        error[fp32] = float(e.norm() / want.norm())
    assert error[0] <= 1.02 * error[1], error
    e = (e.transpose(0, 1) if product != "filters" else e).reshape(e.shape[0 if product == "filters" else 1], -1)
    z = e.mean(1) / (e.std(1) / np.sqrt(e.shape[1]))
    assert float(z.pow(2).mean().sqrt()) <= 3.0


@pytest.mark.parametrize("ex,ef", [(-116, 40), (-124, 60), (-140, 100), (60, -110), (104, -60), (124, -120), (-100, 126)])
def test_operands_of_every_magnitude_keep_their_bits(capi, either, ex, ef):
    """x around 2^ex (down to subnormal numbers), the other operand around 2^ef: 576 and 784 products each, which fp32
    arithmetic sums to 4.2e-7 of the 2-norm (measured on the fp32 instruction); 5e-7 leaves none of them a bit of an
    operand less."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(ex + 1000)
    def around(e, *s):
        return (torch.randn(*s, device="cuda", generator=gen, dtype=torch.float64).clamp(-3.9, 3.9) * 2.0 ** e).float()
    x, f, dy = around(ex, 4, 64, 14, 14), around(ef, 128, 64, 3, 3), around(ef, 4, 128, 14, 14)
    g = capi.conv_geom((14, 14, 64, 4), (3, 3, 64, 128), 1, 1, 1)
    xc, fc, dc = (t.double().cpu() for t in (x, f, dy))
    error = lambda got, want: float((got.cpu().double() - want).norm() / want.norm())
    assert error(capi.conv_forward(x, f, None, g), torch.nn.functional.conv2d(xc, fc, padding=1)) <= 5e-7
    assert error(capi.conv_backward(x, f, dy, g, want=(False, True, False))[1], torch.nn.grad.conv2d_weight(xc, fc.shape, dc, padding=1)) <= 5e-7
    # and with the magnitudes the other way round
    y, w = around(ex, 4, 128, 14, 14), around(ef, 128, 64, 3, 3)
    got = capi.conv_backward_data_acc(torch.empty_like(x), 0.0, w, y, g)
    assert error(got, torch.nn.grad.conv2d_input(xc.shape, w.double().cpu(), y.double().cpu(), padding=1)) <= 5e-7
    y, w = around(ef, 4, 64, 14, 14), around(ex, 128, 64, 3, 3)
    assert error(capi.conv_forward(y, w, None, g), torch.nn.functional.conv2d(y.double().cpu(), w.double().cpu(), padding=1)) <= 5e-7


def test_ragged_channels_of_a_tensor_just_under_two_gigabytes(capi):
    """17 channels of 126 MB: the second chunk holds one channel, its other rows lie behind the tensor.  Compared with
    double precision around the corners, where taps leave the image as well, and along the last columns."""
    import torch
    free, _ = torch.cuda.mem_get_info()
    if free < 12 << 30:
        pytest.skip("needs 12 GB of device memory")
    n, c, k = 5611, 17, 6
    assert (1 << 31) - (16 << 20) < 4 * n * n * c < 1 << 31
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    x = torch.randn(1, c, n, n, device="cuda", generator=gen)
    f = torch.randn(k, c, 3, 3, device="cuda", generator=gen) / np.sqrt(9 * c)
    g = capi.conv_geom((n, n, c, 1), (3, 3, c, k), 1, 1, 1)
    capi.profile_begin("conv_split_mfma")
    y = capi.conv_forward(x, f, None, g)
    launches, _ = capi.profile_end()
    assert launches >= 1
    for ws, hs in [(slice(0, 40), slice(0, 40)), (slice(n - 40, n), slice(n - 40, n)), (slice(0, 40), slice(n - 40, n)), (slice(n - 4, n), slice(0, n))]:
        wide = [slice(max(0, s.start - 1), min(n, s.stop + 1)) for s in (ws, hs)]
        crop = x[:, :, wide[0], wide[1]].double().cpu()
        pads = [(int(s.start == 0), int(s.stop == n)) for s in (hs, ws)]
        want = torch.nn.functional.conv2d(torch.nn.functional.pad(crop, pads[0] + pads[1]), f.double().cpu())
        got = y[:, :, ws, hs].double().cpu()
        assert float((got - want).abs().max() / want.abs().max()) <= TOL


@pytest.mark.parametrize("c,k,last", [(129, 32, "channel"), (32, 129, "filter"), (129, 129, "filter")])
def test_every_row_of_a_filter_gradient_is_stored_by_one_workgroup(capi, c, k, last):
    """The last half-block of 16 rows starts before the end and shares rows with the one before, in another workgroup here.
    An infinity in the last row, the only one its workgroup stores, makes that workgroup repeat its tile on the fp32
    instruction: the rows they share have the bits they have without the infinity."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(c)
    x, dy = torch.randn(3, c, 12, 12, device="cuda", generator=gen), torch.randn(3, k, 12, 12, device="cuda", generator=gen)
    f = torch.zeros(k, c, 1, 1, device="cuda")
    g = capi.conv_geom((12, 12, c, 3), (1, 1, c, k), 1, 0, 1)
    clean = capi.conv_backward(x, f, dy, g, want=(False, True, False))[1].reshape(k, c)
    (x if last == "channel" else dy)[1, -1, 5, 5] = float("inf")
    got = capi.conv_backward(x, f, dy, g, want=(False, True, False))[1].reshape(k, c)
    if last == "channel":
        assert not torch.isfinite(got[:, -1]).any() and torch.equal(got[:, :-1], clean[:, :-1])
    else:
        assert not torch.isfinite(got[-1]).any() and torch.equal(got[:-1], clean[:-1])


@pytest.mark.parametrize("xs,fs,pad", [((56, 56, 256, 64), (1, 1, 256, 128), 0), ((69, 53, 32, 109), (4, 4, 32, 64), 2)])
def test_channel_sums_where_a_round_is_left_over(capi, xs, fs, pad):
    """The tiles of the last round are split and added up apart: their partial sums come from there (whole tiles; a last tile
    of 116 pixels).  Same output bits as the plain call; sums against double (128 values added in double per partial)."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(xs[0])
    x = torch.randn(*xs[::-1], device="cuda", generator=gen) + 0.3
    f = torch.randn(*fs[::-1], device="cuda", generator=gen) / np.sqrt(np.prod(fs[:3]))
    g = capi.conv_geom(xs, fs, 1, pad, 1)
    assert capi.conv_forward_sums_groups(g) > 0
    want = capi.conv_forward(x, f, None, g)
    capi.profile_begin("conv_split_tail_reduce")
    y, sums = capi.conv_forward_sums(x, f, g)
    launches, _ = capi.profile_end()
    assert launches == 1 and torch.equal(y, want)
    yd = y.double()
    for i, s in enumerate((yd.sum(dim=(0, 2, 3)), (yd * yd).sum(dim=(0, 2, 3)))):
        assert float((sums.sum(dim=1)[:, i] - s).abs().max() / s.abs().max()) < 1e-12


@pytest.fixture(params=[0, -1], ids=["staged", "per_tap"])
def tail_kernel(request, capi):
    """The kernel that splits pixels once for all taps, and the one that does it per tap: the name their tails run under."""
    capi.set_tunable("conv_staged", request.param)
    yield "conv_split_mfma_staged_tail" if request.param == 0 else "conv_split_mfma_tail"
    capi.set_tunable("conv_staged", 0)


@pytest.mark.parametrize("xs,fs,pad", [((56, 56, 64, 128), (3, 3, 64, 64), 1), ((40, 28, 256, 104), (3, 3, 256, 64), 1)])
def test_masked_second_term_where_a_round_is_left_over(capi, tail_kernel, xs, fs, pad):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(xs[0])
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    f, g = normal(*fs[::-1]) / np.sqrt(9 * fs[3]), capi.conv_geom(xs, fs, 1, pad, 1)
    assert capi.lib().mcn_conv_backward_data_masked_add_supported(g) == 1
    dy, addend, y = normal(*capi.conv_out_shape(g)[::-1]), normal(*xs[::-1]), normal(*xs[::-1])
    words = ((y.reshape(-1) > 0).to(torch.int64).reshape(-1, 32) * (1 << torch.arange(32, device="cuda", dtype=torch.int64))).sum(dim=1)
    bits = torch.where(words >= (1 << 31), words - (1 << 32), words).to(torch.int32)
    want = capi.conv_backward_data_acc(capi.relu_backward(y, addend), 1.0, f, dy, g)
    capi.profile_begin("conv_split_tail_reduce")
    got = capi.conv_backward_data_masked_add(f, dy, g, addend, bits)
    launches, _ = capi.profile_end()
    assert launches == 1 and torch.equal(got.view(torch.int32), want.view(torch.int32))
    capi.profile_begin(tail_kernel)
    capi.conv_backward_data_masked_add(f, dy, g, addend, bits)
    assert capi.profile_end()[0] == 1


@pytest.mark.parametrize("xs,k", [((6, 6, 64, 16), 1500), ((1, 1, 2048, 32), 1000), ((3, 3, 250, 128), 177)])
def test_fully_connected_packed_ahead_and_deferred_give_the_same_bits(capi, xs, k):
    """Layers of 1e8 operations and more: nothing is packed ahead, a call with a packed buffer in hand is the plain call, and
    the filter gradient of the deferred form is the plain one's."""
    import ctypes as C
    import torch
    h, w, c, n = xs
    gen = torch.Generator(device="cuda")
    gen.manual_seed(k)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f, dy, b = normal(n, c, w, h), normal(k, c, w, h) / np.sqrt(h * w * c), normal(n, k, 1, 1), normal(k)
    g = capi.conv_geom((h, w, c, n), (h, w, c, k), 1, 0, 1)
    assert capi.conv_packed_bytes(g, capi.CONV_FORWARD) == 0 and capi.conv_packed_bytes(g, capi.CONV_BACKWARD_DATA) == 0
    some = torch.empty(16, device="cuda", dtype=torch.uint8)  # (a buffer that holds nothing)
    same = lambda a, b: torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert same(capi.conv_forward_packed(x, f, some, b, g), capi.conv_forward(x, f, b, g))
    want = capi.conv_backward_data_acc(x.clone(), 1.0, f, dy, g)
    assert same(capi.conv_backward_data_packed(x.clone(), 1.0, f, some, dy, g), want)
    assert capi.lib().mcn_conv_backward_filter_partial_bytes(C.byref(g)) > 0
    got = capi.conv_backward_filter_deferred([(x, dy, g)])[0]
    assert same(got, capi.conv_backward(x, f, dy, g, want=(False, True, False))[1])


@pytest.mark.parametrize("xs,fs,pad,product,kernel,launches", [
    ((8, 8, 90, 1), (3, 3, 90, 62), 1, "filters", "conv_wgrad_mfma_split", 0),      # two steps of pixels: one launch of the fp32 kernel
    ((14, 14, 90, 2), (3, 3, 90, 62), 1, "filters", "conv_wgrad_mfma_split", 1),
    ((8, 8, 64, 1), (3, 3, 64, 65), 1, "filters", "conv_wgrad_mfma_split", 1),      # channels by 32: two launches there too
    ((28, 28, 64, 1), (3, 3, 64, 64), 1, "filters", "conv_wgrad_mfma_split", 0),    # but tiles of 64 filters
    ((28, 28, 64, 9), (3, 3, 64, 64), 1, "filters", "conv_wgrad_mfma_split", 1),    # 5.2e8 operations
    ((4, 4, 111, 16), (4, 4, 111, 2500), 0, "filters", "conv_split_mfma", 0),       # 1.4e8 operations, values no multiple of 32
    ((4, 4, 111, 68), (4, 4, 111, 600), 0, "filters", "conv_split_mfma", 1),
    ((28, 28, 8, 4), (1, 1, 8, 259), 0, "forward", "conv_split_mfma", 0),           # half a chunk of channels
    ((28, 28, 16, 4), (1, 1, 16, 259), 0, "forward", "conv_split_mfma", 1),
    ((28, 28, 40, 4), (3, 3, 40, 7), 1, "input", "conv_split_mfma", 0),
    ((28, 28, 40, 4), (3, 3, 40, 8), 1, "input", "conv_split_mfma", 1),
])
def test_small_products_stay_with_the_kernel_that_is_faster(capi, ob, xs, fs, pad, product, kernel, launches):
    r = np.random.default_rng(sum(xs) + sum(fs))
    x, f = F(r.standard_normal(xs)), F(r.standard_normal(fs) / np.sqrt(np.prod(fs[:3])))
    g, og = capi.conv_geom(xs, fs, 1, pad, 1), ob.conv_geom(xs, fs, 1, pad, 1)
    dy = F(r.standard_normal(capi.conv_out_shape(g)))
    xd, fd, dyd = (capi.to_device(v) for v in (x, f, dy))
    n = 0
    for name in [kernel] + ["conv_split_short"] * (kernel == "conv_split_mfma"):  # (few pixels: the same operands, another kernel)
        capi.profile_begin(name)
        if product == "forward":
            got, want = capi.conv_forward(xd, fd, None, g), ob.conv_forward(x, f, None, og)
        else:
            which = (product == "input", product == "filters", False)
            at = which.index(True)
            got, want = capi.conv_backward(xd, fd, dyd, g, want=which)[at], ob.conv_backward(x, f, dy, og, want=which)[at]
        n += capi.profile_end()[0]
    assert n == launches
    assert rel_max(capi.to_host(got), want) <= TOL


@pytest.fixture(params=[108, 116, 204])
def short(capi, request):
    """The kernel for few pixels wherever it can."""
    capi.set_tunable("conv_short", request.param)
    yield
    capi.set_tunable("conv_short", 0)


@pytest.mark.parametrize("xs,fs,stride,pad,dilate", [
    ((5, 6, 16, 3), (1, 1, 16, 17), 1, 0, 1),           # one group: a pair half of padding, wavefronts without work; a channel alone
    ((9, 10, 288, 2), (1, 1, 288, 96), (2, 1), 0, 1),   # strided 1x1, second pairs for all wavefronts, a tile of 26 pixels
    ((7, 7, 48, 1), (3, 3, 48, 33), 1, 1, 1),           # odd number of groups, pixels before and behind the one image
    ((4, 11, 80, 3), (3, 5, 80, 64), 1, (1, 1, 2, 2), 1),   # tiles across images
    ((13, 9, 32, 2), (3, 3, 32, 48), 1, 2, 2),          # dilation
])
def test_few_pixels(capi, ob, short, xs, fs, stride, pad, dilate):
    r = np.random.default_rng(sum(xs) + sum(fs))
    x, f = F(r.standard_normal(xs)), F(r.standard_normal(fs) / np.sqrt(np.prod(fs[:3])))
    b = r.standard_normal(fs[3]).astype(np.float32)
    g, og = capi.conv_geom(xs, fs, stride, pad, dilate), ob.conv_geom(xs, fs, stride, pad, dilate)
    y0 = F(r.standard_normal(capi.conv_out_shape(g)))
    dy = F(r.standard_normal(y0.shape))
    inf = x.copy(order="F")
    inf[2, 3, 5, 0], inf[3, 0, 15, xs[3] - 1], inf[0, 4, 11, 0] = np.inf, np.nan, 3e38
    for v in (x, inf):
        want = ob.conv_forward(v, f, b, og)
        fin = np.isfinite(want)
        capi.profile_begin("conv_split_short")
        y = capi.to_host(capi.conv_forward(*(capi.to_device(t) for t in (v, f, b)), g))
        launches, _ = capi.profile_end()
        assert launches == 1
        assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(y[~fin], want[~fin], equal_nan=True)
        scale = np.maximum(np.abs(want[fin]), 1.0)  # (outputs are of order one; one that holds 3e38 holds one such term)
        assert np.max(np.abs(y[fin] - want[fin]) / scale) <= TOL
    want = ob.conv_forward(x, f, b, og)
    y = capi.to_host(capi.conv_forward(*(capi.to_device(t) for t in (x, f, b)), g, y=capi.to_device(y0), out_mult=0.5, in_mult=2.0))
    assert rel_max(y, 0.5 * y0 + 2 * (want - b.reshape(1, 1, -1, 1)) + b.reshape(1, 1, -1, 1)) <= TOL
    want = ob.conv_backward(x, f, dy, og, want=(True, False, False))[0]
    dx = capi.to_host(capi.conv_backward(*(capi.to_device(t) for t in (x, f, dy)), g, want=(True, False, False))[0])
    assert rel_max(dx, want) <= TOL


@pytest.mark.parametrize("size,n", [(1, 130), (3, 3)])  # (1x1 input gradients under 1e8 operations run on the fp32 instruction)
def test_few_pixels_sums_masked_add_and_normalisation(capi, short, size, n):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(size)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f = normal(n, 64, 8, 8), normal(96, 64, size, size) / (8.0 * size)
    g = capi.conv_geom((8, 8, 64, n), (size, size, 64, 96), 1, size // 2, 1)
    y = capi.conv_forward(x, f, None, g)
    y1, sums = capi.conv_forward_sums(x, f, g)
    assert torch.equal(y, y1)
    d = y.double()
    want = torch.stack([d.sum((0, 2, 3)), (d * d).sum((0, 2, 3))], 1)
    assert float(((sums.sum(1) - want).abs() / (d * d).sum((0, 2, 3))[:, None]).max()) <= 1e-12  # (double sums of up to 8320 terms)
    dy, addend = normal(n, 96, 8, 8), normal(n, 64, 8, 8)
    bits = torch.randint(-2 ** 31, 2 ** 31 - 1, (addend.numel() // 32,), device="cuda", generator=gen, dtype=torch.int32)
    mask = (bits[:, None] >> torch.arange(32, device="cuda", dtype=torch.int32)[None] & 1).reshape(addend.shape).bool()
    dx = capi.conv_backward(x, f, dy, g, want=(True, False, False))[0]
    assert torch.equal(capi.conv_backward_data_masked_add(f, dy, g, addend, bits), dx + torch.where(mask, addend, addend * 0))
    moments, mult, bias, res = torch.stack([normal(96), 0.5 + torch.rand(96, device="cuda", generator=gen)]), normal(96), normal(96), normal(n, 96, 8, 8)
    got = capi.conv_forward_bnorm(x, f, g, moments, mult, bias, res, True)
    assert torch.equal(got, capi.bnorm_forward_fused(y, mult, bias, residual=res, relu=True, moments=moments)[0])


@pytest.mark.parametrize("wa,K", [(2, 64), (2, 128), (4, 128), (4, 256)])
@pytest.mark.parametrize("size,staged", [(1, 0), (3, 0), (3, -1)])  # (3x3: pixels split once for all taps, and per tap)
@pytest.mark.parametrize("left", [1, 30, "most"])  # tiles beyond whole rounds, the last of them half full
def test_left_over_tiles_in_narrower_ones(capi, wa, K, size, staged, left):
    """Every form of the product with them and without: the same products in the same order, the same bits.  Of a filter that is
    not finite the wider tile does its neighbours again on the fp32 instruction too, the narrower one fewer of them: rounding apart."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tilesC = K // (32 * wa)
    left = cus // wa if left == "most" else left
    mTiles = -(-(cus + left) // tilesC)  # (two channel tiles: 1 is rounded up to 2)
    N = 2 * mTiles - 1  # (images of 64 pixels)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f, b = normal(N, 32, 8, 8), normal(K, 32, size, size) / (32 * size * size) ** 0.5, normal(K, 1)
    x[N - 1, 5, 6, 7] = float("inf")
    bad = f.clone()
    bad[K - 7, 3, size // 2, 0] = float("inf")
    g = capi.conv_geom((8, 8, 32, N), (size, size, 32, K), 1, size // 2, 1)
    # backward-data of a layer of K channels and 32 filters: the same product
    back, gb = normal(32, K, size, size) / (32 * size * size) ** 0.5, capi.conv_geom((8, 8, K, N), (size, size, K, 32), 1, size // 2, 1)
    addend = normal(N, K, 8, 8)
    bits = torch.randint(-2 ** 31, 2 ** 31 - 1, (addend.numel() // 32,), device="cuda", generator=gen, dtype=torch.int32)
    moments, mult, res = torch.stack([normal(K), 0.5 + torch.rand(K, device="cuda", generator=gen)]), normal(K), normal(N, K, 8, 8)
    calls = [lambda: capi.conv_forward(x, f, b, g), lambda: capi.conv_forward_sums(x, f, g),
             lambda: capi.conv_forward_bnorm(x, f, g, moments, mult, b.reshape(-1), res, True),
             lambda: capi.conv_backward_data_masked_add(back, x, gb, addend, bits), lambda: capi.conv_forward(x, bad, b, g)]
    got = []
    capi.set_tunable("conv_split_wa", wa)
    capi.set_tunable("conv_sb_tail", 0)
    capi.set_tunable("conv_staged", staged)
    try:
        for name in ("conv_split_mfma_staged", "conv_split_mfma_ends_staged"):
            capi.profile_begin(name)
            calls[0]()
            assert capi.profile_end()[0] == (1 if name == "conv_split_mfma_ends_staged" and size == 3 and staged == 0 else 0)
        for ends in (1, 0):
            capi.set_tunable("conv_split_ends", ends)
            outs = []
            for call in calls:
                capi.profile_begin("conv_split_mfma_ends")
                out = call()
                assert capi.profile_end()[0] == ends
                outs += out if isinstance(out, tuple) else [out]
            got.append(outs)
    finally:
        capi.set_tunable("conv_split_wa", 0)
        capi.set_tunable("conv_sb_tail", 1)
        capi.set_tunable("conv_split_ends", 1)
        capi.set_tunable("conv_staged", 0)
    for a, c in zip(got[0][:-1], got[1][:-1]):
        assert torch.equal(a.view(torch.int32), c.view(torch.int32))
    for weights, ys in ((f, got[0][:1]), (bad, [got[0][-1], got[1][-1]])):
        want = torch.nn.functional.conv2d(x.double().cpu(), weights.double().cpu(), padding=size // 2) + b.double().cpu().reshape(1, -1, 1, 1)
        fin = torch.isfinite(want)
        for y in ys:
            y = y.double().cpu()
            assert torch.equal(torch.isfinite(y), fin)
            assert float((y[fin] - want[fin]).abs().max() / want[fin].abs().max()) <= TOL


@pytest.mark.parametrize("n", [1, 2, 3, 4])
@pytest.mark.parametrize("h,c,k", [(1, 1, 1), (1, 64, 10), (1, 1027, 33), (1, 1028, 5), (3, 115, 7), (6, 256, 130)])  # ragged volumes, one step and many
def test_fully_connected_few_images(capi, n, h, c, k):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(h + c + k + n)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    FV = h * h * c
    x, f, b, y0 = normal(n, c, h, h), normal(k, c, h, h) / FV ** 0.5, normal(k, 1), normal(n, k, 1, 1)
    g = capi.conv_geom((h, h, c, n), (h, h, c, k), 1, 0, 1)
    want = x.double().reshape(n, FV) @ f.double().reshape(k, FV).t().contiguous()
    bd = b.double().reshape(1, k)
    if c > 6 or h > 1:
        capi.profile_begin("conv_dot")
    y = capi.conv_forward(x, f, b, g)
    if c > 6 or h > 1:
        assert capi.profile_end()[0] == 1
    y2 = capi.conv_forward(x, f, b, g, y=y0.clone(), out_mult=0.5, in_mult=2.0)
    big = max(1.0, float(want.abs().max()))
    assert float((y.double().reshape(n, k) - want - bd).abs().max()) <= TOL * big
    assert float((y2.double().reshape(n, k) - 0.5 * y0.double().reshape(n, k) - 2 * want - bd).abs().max()) <= 2 * TOL * big
    x[n - 1, c - 1, h - 1, h - 1], x[0, 0, 0, 0] = float("inf"), float("nan")
    y = capi.conv_forward(x, f, None, g).reshape(n, k)
    assert bool(torch.isnan(y[0]).all()) and (n == 1 or bool(torch.isinf(y[n - 1]).all()))


@pytest.mark.parametrize("h,c,k,n", [(6, 256, 4096, 3), (6, 256, 4096, 4), (7, 512, 4096, 2), (6, 256, 1001, 4),   # two filters to a workgroup, a last one alone
                                     (6, 256, 1001, 1), (1, 2048, 1000, 4), (1, 1027, 33, 2), (1, 30, 3, 4)])
def test_fully_connected_few_images_run_by_geometry_alone(capi, h, c, k, n):
    """No bank is packed ahead; with a packed buffer in hand (of any content) and without, with the workspace a call must have and
    with more, it is the same kernel and the same bits.  What a call must bring is what it was for the tiles."""
    import ctypes as C
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(h + c + k + n)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f, b = normal(n, c, h, h), normal(k, c, h, h) / (h * h * c) ** 0.5, normal(k, 1)
    g = capi.conv_geom((h, h, c, n), (h, h, c, k), 1, 0, 1)
    L, ptr = capi.lib(), capi.ptr
    assert capi.conv_packed_bytes(g, capi.CONV_FORWARD) == 0 and capi.conv_pack_filters(f, g, capi.CONV_FORWARD) is None
    capi.profile_begin("conv_dot")
    want = capi.conv_forward(x, f, b, g)
    assert capi.profile_end()[0] == 1
    some = torch.zeros(64, device="cuda", dtype=torch.uint8)
    most = L.mcn_conv_workspace_bytes(C.byref(g), capi.CONV_FORWARD)
    bank = 4 * -(-h * h * c // 16) * 16 * k  # (no call gets by with less than the bank, padded or not)
    ws = torch.empty(most + 16, device="cuda", dtype=torch.uint8)

    def call(packed, offset, size):
        y = torch.full((n, k, 1, 1), float("nan"), device="cuda")
        rc = L.mcn_conv_forward_packed(capi.stream(), C.byref(g), ptr(y), 0.0, ptr(x), 1.0, ptr(f), ptr(packed) if packed is not None else None,
                                       64 if packed is not None else 0, ptr(b), ptr(ws[offset:]) if size else None, size)
        if rc == 0:
            assert torch.equal(y.view(torch.int32), want.view(torch.int32))
        return rc

    assert call(some, 0, most) == 0 and call(None, 0, most) == 0
    refused = [size for size in (0, bank // 2, most // 2, most - 16) if call(None, 0, size)]
    assert refused[:2] == [0, bank // 2] and call(None, 1, most) != 0  # too small; not aligned
    for size in (0, bank // 2, most // 2, most - 16):
        call(some, 0, size)  # (the same bits wherever it is accepted)
    rows = lambda t: t.double().reshape(t.shape[0], -1)
    exact = rows(x) @ rows(f).t().contiguous() + b.double().reshape(1, k)
    assert float((rows(want) - exact).abs().max()) <= TOL * max(1.0, float(exact.abs().max()))


@pytest.mark.usefixtures("any_size")
@pytest.mark.parametrize("tile,room", [(48, 0), (44, 0), (82, 0), (42, 1), (28, 0), (24, 1), (26, 1), (22, 1), (14, 1)])
def test_filter_gradient_beside_another_stream_in_every_tile(capi, tile, room):
    """On a marked stream every tile asks for local memory that leaves a CU no room for a second workgroup (those under 84 KB for
    more than they use), with the same bits."""
    import ctypes as C
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tile)
    x, dy = torch.randn(3, 80, 17, 15, device="cuda", generator=gen), torch.randn(3, 272, 17, 15, device="cuda", generator=gen)
    f = torch.zeros(272, 80, 3, 3, device="cuda")
    g = capi.conv_geom((15, 17, 80, 3), (3, 3, 80, 272), 1, 1, 1)
    side, L = torch.cuda.Stream(), capi.lib()
    capi.set_tunable("conv_wsplit_tile", tile)
    try:
        want = capi.conv_backward(x, f, dy, g, want=(False, True, False))[1]
        torch.cuda.synchronize()
        capi.check(L.mcn_stream_beside(C.c_void_p(side.cuda_stream), 1))
        with torch.cuda.stream(side):
            capi.profile_begin("_beside")
            got = capi.conv_backward(x, f, dy, g, want=(False, True, False))[1]
            launches, _ = capi.profile_end()
        side.synchronize()
    finally:
        capi.set_tunable("conv_wsplit_tile", 0)
        capi.check(L.mcn_stream_beside(C.c_void_p(side.cuda_stream), 0))
    assert launches == room and torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("product", ["forward", "input", "input of a strided layer"])
def test_taps_outside_planes_of_two_to_the_25_pixels(capi, product):
    """Nine reduction channels over planes of 2^27 bytes: the upper half-wave's channel lies eight planes, 2^30 bytes, further on,
    also for a lane whose tap lies outside the image, which must still load nothing.  Compared with double precision around the
    corners and along the last columns."""
    import torch
    free, _ = torch.cuda.mem_get_info()
    if free < 12 << 30:
        pytest.skip("needs 12 GB of device memory")
    H, W, C, K = 8192, 4096, 9, 6
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    x = torch.randn(1, C, W, H, device="cuda", generator=gen)
    step = 2 if product == "input of a strided layer" else 1  # (down the columns)
    if product == "forward":
        f = torch.randn(K, C, 3, 3, device="cuda", generator=gen) / np.sqrt(9 * C)
        call = lambda: capi.conv_forward(x, f, None, capi.conv_geom((H, W, C, 1), (3, 3, C, K), 1, 1, 1))
    else:
        f = torch.randn(C, K, 3, 3, device="cuda", generator=gen) / np.sqrt(9 * C)
        g = capi.conv_geom((step * H, W, K, 1), (3, 3, K, C), (step, 1), 1, 1)
        call = lambda: capi.conv_backward_data_acc(torch.zeros(1, K, W, step * H, device="cuda"), 0.0, f, x, g)
    capi.profile_begin("conv_split_mfma")
    y = call()
    launches, _ = capi.profile_end()
    assert launches >= 1
    n, m = W, step * H
    for ws, hs in [((0, 40), (0, 40)), ((n - 40, n), (m - 40, m)), ((0, 40), (m - 40, m)), ((n - 4, n), (0, m))]:
        # what is read for this part of the result: [first, last) of either dimension, and where it lies in the product over them
        if product == "forward":
            read = [(max(0, a - 1), min(size, b + 1)) for (a, b), size in ((ws, W), (hs, H))]
            crop = x[:, :, read[0][0]:read[0][1], read[1][0]:read[1][1]].double().cpu()
            want = torch.nn.functional.conv2d(crop, f.double().cpu(), padding=2)
            at = [a + 1 - r[0] for (a, _), r in zip((ws, hs), read)]
        else:
            read = [(max(0, (a - 1) // s), min(size, b // s + 1)) for (a, b), s, size in ((ws, 1, W), (hs, step, H))]
            crop = x[:, :, read[0][0]:read[0][1], read[1][0]:read[1][1]].double().cpu()
            want = torch.nn.functional.conv_transpose2d(crop, f.double().cpu(), stride=(1, step))
            at = [a + 1 - r[0] * s for (a, _), r, s in zip((ws, hs), read, (1, step))]
        want = want[:, :, at[0]:at[0] + ws[1] - ws[0], at[1]:at[1] + hs[1] - hs[0]]
        got = y[:, :, ws[0]:ws[1], hs[0]:hs[1]].double().cpu()
        assert got.shape == want.shape
        assert float((got - want).abs().max() / want.abs().max()) <= TOL
