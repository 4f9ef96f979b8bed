"""First layers with a normalisation with given moments in their epilogue (csrc/conv_first.hip): the bits of the convolution
followed by the normalisation, where the tiles have their edges; and the network's stem, whose own output is handed out all
the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xs,fs,stride,pad", [
    ((64, 64, 3, 2), (7, 7, 3, 64), 2, 3),      # the stem
    ((37, 23, 3, 3), (7, 7, 3, 64), 2, 3),      # rows no multiple of four, a part of a tile at every end
    ((32, 32, 3, 5), (5, 5, 3, 32), 1, 2),      # 32 filters: four wavefronts side by side
    ((9, 70, 4, 1), (5, 3, 4, 32), 1, 1),       # an even number of rows of the volume
    ((224, 224, 3, 1), (7, 7, 3, 64), 2, 3),
])
@pytest.mark.parametrize("residual,relu", [(False, True), (True, False)])
def test_normalised_first_layers(capi, xs, fs, stride, pad, residual, relu):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(xs) + sum(fs))
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    K = fs[3]
    g = capi.conv_geom(xs, fs, stride, pad, 1)
    assert capi.lib().mcn_conv_forward_bnorm_supported(g) == 1
    x, f = normal(*xs[::-1]), normal(*fs[::-1]) / np.prod(fs[:3]) ** 0.5
    x[0, 0, 1, 2] = float("inf")
    moments, mult, bias = torch.stack([normal(K), 0.5 + torch.rand(K, device="cuda", generator=gen)]), normal(K), normal(K)
    capi.profile_begin("conv_first_fwd")
    a = capi.conv_forward(x, f, None, g)
    res = normal(*a.shape) if residual else None
    got = capi.conv_forward_bnorm(x, f, g, moments, mult, bias, res, relu)
    assert capi.profile_end()[0] == 2
    want = capi.bnorm_forward_fused(a, mult, bias, residual=res, relu=relu, moments=moments)[0]
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got).view(torch.int32), torch.nan_to_num(want).view(torch.int32))


def test_the_stem_hands_out_its_convolutions_output(capi):
    import torch
    from matconvnet_amd import vlapi as vl
    r, outs = np.random.default_rng(5), []
    net = vl.ResNet50(N=2, image_size=64, classes=10, fused=True, seed=7)
    try:
        net.set("input", r.standard_normal(net.get("input").shape))
        net.forward()
        net.set("running.stem.m", net.get("stem.m"))
        net.set_test_mode(True)
        x = torch.from_numpy(net.get("input")).cuda().reshape(2, 3, 64, 64)
        f = torch.from_numpy(net.get("stem.f")).cuda().reshape(64, 3, 7, 7)
        for turn in range(2):  # (the first pass does not write it, the second does)
            x.mul_(-0.5)
            net.set("input", x.cpu().numpy().reshape(-1))
            net.forward()
            if turn == 0:
                outs.append(net.get("stem.r"))
            want = capi.conv_forward(x, f, None, capi.conv_geom((64, 64, 3, 2), (7, 7, 3, 64), 2, 3, 1))
            assert np.array_equal(net.get("stem.a").view(np.int32).reshape(-1), want.cpu().numpy().view(np.int32).reshape(-1)), turn
        net.set("input", (x * -2).cpu().numpy().reshape(-1))  # (the first turn's input; the normalisation in its own pass now)
        net.forward()
        assert np.array_equal(net.get("stem.r").view(np.int32), outs[0].view(np.int32))
    finally:
        net.close()


def test_replays_hand_out_the_stems_output_of_their_own_input(capi):
    import torch
    from matconvnet_amd import vlapi as vl
    r = np.random.default_rng(6)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        net = vl.ResNet50(N=2, image_size=64, classes=10, fused=True, seed=8)
        try:
            net.set("input", r.standard_normal(net.get("input").shape))
            net.forward()
            net.set("running.stem.m", net.get("stem.m"))
            net.set_test_mode(True)
            net.forward()
            net.capture(False)
            f = torch.from_numpy(net.get("stem.f")).cuda().reshape(64, 3, 7, 7)
            for turn in range(4):  # (before the third an eager pass, which writes it)
                if turn == 2:
                    net.forward()
                    torch.cuda.synchronize()
                x = torch.from_numpy(r.standard_normal((2, 3, 64, 64)).astype(np.float32)).cuda()
                net.set("input", x.cpu().numpy().reshape(-1))
                net.replay()
                want = capi.conv_forward(x, f, None, capi.conv_geom((64, 64, 3, 2), (7, 7, 3, 64), 2, 3, 1))
                assert np.array_equal(net.get("stem.a").view(np.int32).reshape(-1), want.cpu().numpy().view(np.int32).reshape(-1)), turn
        finally:
            net.close()


@pytest.mark.parametrize("xs,fs,stride,pad", [
    ((37, 23, 3, 3), (7, 7, 3, 64), 2, 3),
    ((32, 32, 3, 5), (5, 5, 3, 32), 1, 2),
    ((9, 70, 4, 1), (5, 3, 4, 32), 1, 1),
])
@pytest.mark.parametrize("residual,relu", [(False, True), (True, False)])
def test_the_convolutions_output_beside_the_normalised_one(capi, xs, fs, stride, pad, residual, relu):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(xs) + sum(fs))
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    K = fs[3]
    g = capi.conv_geom(xs, fs, stride, pad, 1)
    x, f = normal(*xs[::-1]), normal(*fs[::-1]) / np.prod(fs[:3]) ** 0.5
    x[0, 0, 1, 2] = float("inf")
    moments, mult, bias = torch.stack([normal(K), 0.5 + torch.rand(K, device="cuda", generator=gen)]), normal(K), normal(K)
    want = capi.conv_forward(x, f, None, g)
    res = normal(*want.shape) if residual else None
    both = capi.conv_forward_bnorm_keep(x, f, g, moments, mult, bias, res, relu)
    for a, b in zip(both, (capi.conv_forward_bnorm(x, f, g, moments, mult, bias, res, relu), want)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a).view(torch.int32), torch.nan_to_num(b).view(torch.int32))


def test_the_stems_output_is_there_whenever_it_is_looked_at(capi):
    """In test mode: through an address taken before a pass or a replay, and taken after the next input has been uploaded."""
    import ctypes
    import torch
    from matconvnet_amd import vlapi as vl
    r = np.random.default_rng(8)
    stream = torch.cuda.Stream()

    class At:
        def __init__(self, address, count):
            self.__cuda_array_interface__ = dict(shape=(count,), typestr="<f4", data=(address, False), version=2, strides=None)

    with torch.cuda.stream(stream):
        net = vl.ResNet50(N=2, image_size=64, classes=10, fused=True, seed=9)
        try:
            upload = lambda: net.set("input", r.standard_normal(net.get("input").shape)) or torch.from_numpy(net.get("input")).cuda().reshape(2, 3, 64, 64)
            upload()
            net.forward()
            net.set("running.stem.m", net.get("stem.m"))
            net.set_test_mode(True)
            net.forward()
            net.capture(False)
            f = torch.from_numpy(net.get("stem.f")).cuda().reshape(64, 3, 7, 7)
            conv = lambda x: capi.conv_forward(x, f, None, capi.conv_geom((64, 64, 3, 2), (7, 7, 3, 64), 2, 3, 1)).reshape(-1)
            held = None
            for go in (net.forward, net.replay, net.replay):
                want = conv(upload())
                go()
                torch.cuda.synchronize()
                if held is None:
                    upload()
                    n = ctypes.c_size_t(0)
                    held = torch.as_tensor(At(net.L.vlh_resnet50_buffer(net.h, b"stem.a", ctypes.byref(n)), want.numel()), device="cuda")
                    assert n.value == want.numel()
                assert torch.equal(held.view(torch.int32), want.view(torch.int32))
        finally:
            net.close()
