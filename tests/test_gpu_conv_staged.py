"""Filters with taps over pixels that are split once into LDS (csrc/conv_staged.hpp): the same products in the same order as
csrc/conv_split.hip, so the same bits, where the tiles, the pixels staged and the taps have their edges; against double too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # x (H, W, C, N), f (FH, FW, FC, K), pad, dilate, wa, splits
    ((14, 14, 16, 3), (3, 3, 16, 64), 1, 1, 2, 1),       # one chunk; 192 pixels in LDS, six units for four wavefronts
    ((7, 7, 48, 5), (3, 3, 48, 128), 1, 1, 4, 1),        # tiles over three images
    ((62, 9, 32, 2), (3, 3, 32, 96), 1, 1, 2, 1),        # 254 pixels, 256 with the zeros' place; a third of a tile's channels missing
    ((63, 9, 32, 2), (3, 3, 32, 128), 1, 1, 4, 1),       # 256 pixels and the zeros: too many under nine taps, the other kernel
    ((13, 10, 64, 2), (3, 3, 64, 200), 2, 2, 4, 1),      # dilation; 72 channels in the last tile
    ((15, 11, 32, 2), (1, 9, 32, 64), (0, 0, 4, 4), 1, 2, 1),   # nine taps in a row, in a column
    ((20, 11, 32, 2), (9, 1, 32, 128), (4, 4, 0, 0), 1, 4, 1),
    ((27, 27, 48, 1), (5, 5, 48, 128), 2, 1, 4, 1),      # 25 taps
    ((40, 9, 32, 2), (5, 5, 32, 128), 2, 1, 4, 1),       # 25 taps, three units to a wavefront
    ((30, 9, 32, 2), (5, 5, 32, 64), 2, 1, 2, 1),        # 252 pixels: the most for tiles of 64 channels
    ((31, 9, 32, 2), (5, 5, 32, 64), 2, 1, 2, 1),        # 256: the other kernel
    ((62, 9, 32, 2), (5, 5, 32, 128), 2, 1, 4, 1),       # 380 pixels: the most
    ((63, 9, 32, 2), (5, 5, 32, 128), 2, 1, 4, 1),       # too many: the other kernel
    ((14, 14, 80, 2), (3, 3, 80, 128), 1, 1, 4, 3),      # five chunks in three splits: two, two, one
    ((14, 14, 64, 2), (3, 3, 32, 128), 1, 1, 2, 1),      # two groups: a slice of a wider tensor
]


@pytest.mark.parametrize("xs,fs,pad,dilate,wa,splits", CASES)
def test_same_bits(capi, xs, fs, pad, dilate, wa, splits):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(xs) + sum(fs))
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    H, W, C, N = xs
    K = fs[3]
    g = capi.conv_geom(xs, fs, 1, pad, dilate)
    x, f, b = normal(N, C, W, H), normal(*fs[::-1]) / np.prod(fs[:3]) ** 0.5, normal(K, 1)
    dy, y0 = normal(N, K, W, H), normal(N, K, W, H)
    inf = x.clone()
    inf[N - 1, C - 1, W // 2, H - 1] = float("inf")  # (that pixel's tiles again on the fp32 instruction)
    nan = f.clone()
    nan[K - 1, 0, 0, 0] = float("nan")
    whole = C == fs[2] and K % 32 == 0 and fs[0] * fs[1] == 9 and splits == 1  # (what the fused forms ask for)
    calls = [lambda: capi.conv_forward(x, f, b, g), lambda: capi.conv_forward(x, f, b, g, y=y0.clone(), out_mult=0.5, in_mult=2.0),
             lambda: capi.conv_backward_data_acc(torch.zeros_like(x), 0.0, f, dy, g), lambda: capi.conv_forward(inf, f, b, g),
             lambda: capi.conv_forward(x, nan, b, g)]
    if whole:
        moments = torch.stack([normal(K), 0.5 + torch.rand(K, device="cuda", generator=gen)])
        calls += [lambda: capi.conv_forward_sums(x, f, g), lambda: capi.conv_forward_bnorm(x, f, g, moments, b.reshape(-1), b.reshape(-1), y0, True)]
    got = []
    capi.set_tunable("conv_short", -1)
    capi.set_tunable("conv_split_wa", wa)
    capi.set_tunable("conv_split_splits", splits)
    try:
        for staged in (1, -1):
            capi.set_tunable("conv_staged", staged)
            outs = []
            for i, call in enumerate(calls):
                capi.profile_begin("conv_split_mfma_staged")
                out = call()
                launches, _ = capi.profile_end()
                if i == 0:
                    assert launches == ((C // fs[2]) if staged > 0 and H not in (31, 63) else 0)
                outs += [(i, o) for o in (out if isinstance(out, tuple) else (out,))]
            got.append(outs)
    finally:
        for name in ("conv_staged", "conv_split_splits", "conv_split_wa", "conv_short"):
            capi.set_tunable(name, 0)
    for (i, a), (_, c) in zip(*got):
        if i in (3, 4):  # (what is finite beside it is done again or not, as the wavefronts have their channels: rounding apart)
            assert torch.equal(torch.isfinite(a), torch.isfinite(c)) and torch.equal(torch.isnan(a), torch.isnan(c))
            fin = torch.isfinite(a)
            assert float((a[fin] - c[fin]).abs().max()) <= 1e-5 * float(c[fin].abs().max())
        elif splits == 1:
            assert torch.equal(a.contiguous().view(torch.int32), c.contiguous().view(torch.int32)), i
        else:  # (cut elsewhere: the same products in other partial sums)
            assert float((a - c).abs().max()) <= 1e-5 * float(c.abs().max()), i
    # R products in fp32, each sum within R 2^-24 of sum |x w|, in practice its root: as for the kernel beside it
    pads = pad if isinstance(pad, tuple) else (pad,) * 4
    form = dict(padding=(pads[2], pads[0]), dilation=dilate, groups=C // fs[2])
    host = lambda t: t.double().cpu()
    product = torch.nn.functional.conv2d(host(x), host(f), **form)
    bias = host(b).reshape(1, -1, 1, 1)
    dx = torch.nn.grad.conv2d_input(x.shape, host(f), host(dy), **form)
    for (_, a), want in zip(got[0], (product + bias, 0.5 * host(y0) + 2 * product + bias, dx)):
        assert float((host(a) - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("C,size,K,H,wa,over,staged", [
    (32, 3, 64, 8, 2, 0, 0),      # one workgroup to a CU
    (32, 3, 64, 8, 2, 1, 1),      # and one more
    (32, 3, 128, 8, 4, 0, 0),
    (32, 3, 128, 8, 4, 1, 1),
    (16, 3, 64, 8, 2, 1, 0),      # one chunk
    (24, 3, 64, 8, 2, 1, 0),      # a chunk and a half
    (32, 3, 32, 8, 1, 1, 0),      # tiles of 32 channels
    (32, 1, 64, 8, 2, 1, 0),      # one tap
    (32, 7, 64, 8, 2, 1, 0),      # 49
    (32, 5, 64, 8, 2, 1, 1),
    (32, 3, 64, 62, 2, 1, 1),     # 254 pixels under a tile
    (32, 3, 64, 63, 2, 1, 0),     # 256
    (32, 5, 64, 31, 2, 1, 0),     # 256 under a tile of 64 channels
    (32, 5, 128, 31, 4, 1, 1),
    (32, 5, 128, 62, 4, 1, 1),    # 380
    (32, 5, 128, 63, 4, 1, 0),    # 384
])
def test_which_products_are_staged(capi, C, size, K, H, wa, over, staged):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    W = 128 // H if H == 8 else -(-128 * (cus + over) // H)  # (planes of one tile, or one image of so many)
    N = cus + over if H == 8 else 1
    if H != 8:
        W -= W * H > 128 * (cus + over)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(C + K + H)
    x, f = torch.randn(N, C, W, H, device="cuda", generator=gen), torch.randn(K, C, size, size, device="cuda", generator=gen) / (size * size * C) ** 0.5
    for name, value in (("conv_short", -1), ("conv_split_wa", wa), ("conv_split_splits", 1)):
        capi.set_tunable(name, value)
    try:
        capi.profile_begin("staged")
        y = capi.conv_forward(x, f, None, capi.conv_geom((H, W, C, N), (size, size, C, K), 1, size // 2, 1))
        assert (capi.profile_end()[0] > 0) == bool(staged)
    finally:
        for name in ("conv_split_splits", "conv_split_wa", "conv_short"):
            capi.set_tunable(name, 0)
    want = torch.nn.functional.conv2d(x[-1:].double().cpu(), f.double().cpu(), padding=size // 2)
    assert float((y[-1:].double().cpu() - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("xs,k,K,staged", [
    ((56, 56, 96, 4), 5, 128, 0),    # planned five splits of 30 groups; whole chunks are three of 50
    ((27, 27, 192, 8), 5, 64, 0),    # eleven of 28; six of 50, in tiles of 64 channels
    ((24, 24, 192, 4), 3, 192, 1),   # nine of 12; six of 18
    ((24, 24, 512, 1), 5, 192, 1),   # 31 of 26; 16 of 50, half the partial results
    ((14, 14, 384, 32), 5, 384, 1),  # five of 120; five of 125
])
def test_split_reductions_are_staged_where_whole_chunks_fit_the_plan(capi, xs, k, K, staged):
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("planned for 256 compute units")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(xs))
    H, W, C, N = xs
    x, f = torch.randn(N, C, W, H, device="cuda", generator=gen), torch.randn(K, C, k, k, device="cuda", generator=gen) / (k * k * C) ** 0.5
    capi.profile_begin("conv_split_mfma_staged")
    y = capi.conv_forward(x, f, None, capi.conv_geom(xs, (k, k, C, K), 1, k // 2, 1))
    assert capi.profile_end()[0] == staged
    want = torch.nn.functional.conv2d(x[-1:].double().cpu(), f.double().cpu(), padding=k // 2)
    assert float((y[-1:].double().cpu() - want).abs().max()) <= 1e-5 * float(want.abs().max())
