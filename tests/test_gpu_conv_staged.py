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
    # R products in fp32, each sum within R 2^-24 of sum |x w|, in practice its root: as for the kernel beside it
    pads = pad if isinstance(pad, tuple) else (pad,) * 4
    want = torch.nn.functional.conv2d(x.double().cpu(), f.double().cpu(), b.double().cpu().reshape(-1), padding=(pads[2], pads[0]), dilation=dilate,
                                      groups=C // fs[2]).numpy()
    y = got[0][0][1].double().cpu().numpy()
    assert np.abs(y - want).max() <= 1e-5 * np.abs(want).max()


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
