"""GPU tests of the learned denoiser: forward activations and gradients of
the hand-written bf16 MFMA kernels against the CPU fp32 reference network
(oracle/unet_ref.py), the denoise entry point, and a short training run on
pairs rendered by the tracer that must beat its 1-spp input."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import unet_ref
from voxelpathtracer_amd.unet import UNet, bf16_bits, bf16_to_f32, make_dataset, tonemap_psnr, train

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


def _inputs(rng, n, h, w):
    x = np.zeros((n, h, w, 32), np.float32)
    x[..., :10] = rng.normal(0.3, 0.6, size=(n, h, w, 10))
    xb = bf16_bits(x)
    return xb, bf16_to_f32(xb).reshape(n, h, w, 32)


def _rel(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture(scope="module")
def net(ctx):
    u = UNet(ctx, 8, 64, 64)
    yield u
    u.close()


@pytest.mark.parametrize("n,h,w", [(2, 32, 32), (1, 36, 20)])
def test_forward_matches_cpu(net, n, h, w):
    torch = _torch()
    rng = np.random.default_rng(5)
    xb, xf = _inputs(rng, n, h, w)
    net.init(11)
    params = net.get_params()
    out = torch.empty((n, h, w, 3), dtype=torch.float32, device="cuda")
    print(f"unet forward {n}x{h}x{w}", flush=True)
    net.forward(torch.from_numpy(xb.view(np.int16)).cuda(), n, h, w, out)
    torch.cuda.synchronize()
    with torch.no_grad():
        ref_out, acts = unet_ref.forward(unet_ref.unpack(params), torch.from_numpy(xf))
    # every stored activation: bf16 values of an fp32-accumulated product;
    # summation order differs, so a value may round to a neighbouring bf16
    for i, name in enumerate(["x", "e0a", "e0b", "p0", "e1a", "e1b", "p1", "b0", "b1", "d1a", "d1b", "d0a", "d0b"]):
        got = bf16_to_f32(net.activation(i, n, h, w))
        ref = acts[name].numpy()
        assert got.shape == ref.shape, name
        err = _rel(got, ref)
        assert err < 1e-2, (name, err)
        assert np.abs(got - ref).max() <= 0.02 * np.abs(ref).max() + 1e-6, name
    assert _rel(out.cpu().numpy(), ref_out.numpy()) < 1e-2


@pytest.mark.timeout(300)
def test_forward_matches_cpu_1080p(ctx):
    """The workload's resolution, 1920x1080: the persistent convolution
    kernels loop over many 16x32 tiles per workgroup and the pooled levels
    run at 960x540 and 480x270; every activation and the output equal the
    CPU fp32 reference to the same tolerance as the small cases."""
    torch = _torch()
    n, h, w = 1, 1080, 1920
    u = UNet(ctx, n, h, w)
    rng = np.random.default_rng(17)
    xb, xf = _inputs(rng, n, h, w)
    u.init(13)
    params = u.get_params()
    out = torch.empty((n, h, w, 3), dtype=torch.float32, device="cuda")
    print("unet forward 1x1080x1920", flush=True)
    u.forward(torch.from_numpy(xb.view(np.int16)).cuda(), n, h, w, out)
    torch.cuda.synchronize()
    with torch.no_grad():
        ref_out, acts = unet_ref.forward(unet_ref.unpack(params), torch.from_numpy(xf))
    for i, name in enumerate(["x", "e0a", "e0b", "p0", "e1a", "e1b", "p1", "b0", "b1", "d1a", "d1b", "d0a", "d0b"]):
        got = bf16_to_f32(u.activation(i, n, h, w))
        ref = acts[name].numpy()
        assert got.shape == ref.shape, name
        err = _rel(got, ref)
        assert err < 1e-2, (name, err)
        assert np.abs(got - ref).max() <= 0.02 * np.abs(ref).max() + 1e-6, name
    assert _rel(out.cpu().numpy(), ref_out.numpy()) < 1e-2
    u.close()


def test_gradients_match_cpu(net):
    torch = _torch()
    rng = np.random.default_rng(9)
    n, h, w = 2, 32, 48
    xb, xf = _inputs(rng, n, h, w)
    target = rng.normal(0.2, 0.5, size=(n, h, w, 3)).astype(np.float32)
    net.init(21)
    params = net.get_params()
    print("unet backward 2x32x48", flush=True)
    loss = net.backward(torch.from_numpy(xb.view(np.int16)).cuda(), torch.from_numpy(target).cuda(), n, h, w)
    g = net.get_grads()
    ref_loss, ref_g = unet_ref.loss_and_grads(params, xf, target)
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
    from voxelpathtracer_amd.unet import param_layout
    layout, total = param_layout()
    assert total == g.size == ref_g.size
    for name, off, shape in layout:
        size = int(np.prod(shape))
        a, b = g[off:off + size], ref_g[off:off + size]
        cos = float(np.dot(a, b) / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
        # bf16 storage of activation gradients on the GPU: a few percent
        assert _rel(a, b) < 0.06 and cos > 0.998, (name, _rel(a, b), cos)


@pytest.mark.parametrize("n,h,w", [(1, 4, 4), (2, 12, 36), (3, 20, 100), (1, 60, 68), (5, 64, 64)])
def test_gradients_at_tile_edges(net, n, h, w):
    """Weight gradients where the 4 x 32 pixel tiles, their groups over the
    four waves and the slices have remainders.  The target lies above every
    prediction, so that no sign of the L1 loss hangs on a rounding; bf16
    gradients as in test_gradients_match_cpu, same tolerance."""
    torch = _torch()
    rng = np.random.default_rng(31)
    xb, xf = _inputs(rng, n, h, w)
    target = rng.normal(40.0, 0.5, size=(n, h, w, 3)).astype(np.float32)
    net.init(22)
    params = net.get_params()
    print(f"unet backward {n}x{h}x{w}", flush=True)
    loss = net.backward(torch.from_numpy(xb.view(np.int16)).cuda(), torch.from_numpy(target).cuda(), n, h, w)
    g = net.get_grads()
    ref_loss, ref_g = unet_ref.loss_and_grads(params, xf, target)
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
    from voxelpathtracer_amd.unet import param_layout
    for name, off, shape in param_layout()[0]:
        size = int(np.prod(shape))
        assert _rel(g[off:off + size], ref_g[off:off + size]) < 0.06, name
    again = net.backward(torch.from_numpy(xb.view(np.int16)).cuda(), torch.from_numpy(target).cuda(), n, h, w)
    assert again == loss
    np.testing.assert_array_equal(net.get_grads(), g)   # a fixed order of sums


def _bf16_tensor(a):
    torch = _torch()
    return torch.from_numpy(bf16_to_f32(a.cpu().numpy().view(np.uint16))).cuda()


def test_denoise_entry_point(ctx, net):
    """vpt_unet_denoise (assemble + forward + exp) equals the separate calls."""
    torch = _torch()
    from voxelpathtracer_amd.unet import PairMaker
    net.init(4)
    pm = PairMaker(ctx, worlds=1, size=64, spp=2, seed=9)
    x1 = torch.empty((64, 64, 32), dtype=torch.int16, device="cuda")
    t1 = torch.empty((64, 64, 3), dtype=torch.float32, device="cuda")
    pm.pair(net, x1, t1)
    rgb = torch.empty((64, 64, 3), dtype=torch.float32, device="cuda")
    out = torch.empty((64, 64, 3), dtype=torch.float32, device="cuda")
    net.denoise(pm.gb, pm.tex, rgb)
    net.forward(x1, 1, 64, 64, out, mode=1)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(rgb.cpu().numpy(), out.cpu().numpy())
    pm.close()


@pytest.mark.parametrize("h,w", [(4, 4), (8, 16), (20, 12), (16, 36), (64, 60), (132, 100), (360, 640), (1080, 1920)])
def test_denoise_activations(ctx, h, w):
    """vpt_unet_denoise (16-channel input, head in the last convolution) and
    vpt_unet_forward on the assembled input give the same activations and
    output bit for bit, with odd tile remainders and with both tile sizes;
    the last activation is the one of the weights that the pass ran with."""
    torch = _torch()
    from voxelpathtracer_amd import World, generate_terrain, gi_params, make_camera
    from voxelpathtracer_amd.world import DeviceGBuffer
    world = World(ctx, 64, 64, 64)
    world.m_WorldData[...] = generate_terrain(64, 64, 64, h_min=10, h_max=45)
    world.Buffer()
    world.GenerateDistanceField()
    cam, _, _ = make_camera((32.5, 52.5, 32.5), 40.0, -20.0, w, h)
    gb = DeviceGBuffer(w, h)
    tex = torch.empty((h, w, 8), dtype=torch.int16, device="cuda")
    rgb = torch.empty((h, w, 3), dtype=torch.float32, device="cuda")
    world.trace_primary(cam, gb, 350)
    world.trace_gi(cam, gb, gi_params(50.0, 3), rgb, tex)
    u = UNet(ctx, 1, h, w)
    u.init(5)
    x = torch.empty((h, w, 32), dtype=torch.int16, device="cuda")
    a = torch.empty((h, w, 3), dtype=torch.float32, device="cuda")
    b = torch.empty((h, w, 3), dtype=torch.float32, device="cuda")
    u.assemble(gb, tex, x)
    u.forward(x, 1, h, w, a, mode=1)
    fwd = [u.activation(i, 1, h, w) for i in range(13)]
    params = u.get_params()
    u.denoise(gb, tex, b)
    u.set_params(params * 1.5)   # the activations read below are the denoise pass's
    den = [u.activation(i, 1, h, w) for i in range(13)]
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
    for i in range(13):
        np.testing.assert_array_equal(fwd[i], den[i], err_msg=str(i))
    xf = bf16_to_f32(fwd[0])
    with torch.no_grad():
        ref_out, acts = unet_ref.forward(unet_ref.unpack(params), torch.from_numpy(xf))
    # bf16 values of fp32 sums in another order, as in test_forward_matches_cpu
    for i, name in ((9, "d1a"), (12, "d0b")):
        assert _rel(bf16_to_f32(fwd[i]), acts[name].numpy()) < 1e-2, name
    assert _rel(a.cpu().numpy(), np.maximum(np.expm1(ref_out.numpy()[0]), 0.0)) < 2e-2
    u.close()
    world.close()


def test_last_activation(ctx):
    """The last activation, which an inference pass does not store, read in
    parts and again, after the weights changed, and after replays of a
    captured pass of another size: always the values that a pass which stores
    it (the backward pass) has with the same weights, bit for bit."""
    torch = _torch()
    rng = np.random.default_rng(71)
    n, h, w = 3, 16, 20
    x = {k: torch.from_numpy(_inputs(rng, *k)[0].view(np.int16)).cuda() for k in ((n, h, w), (2, 12, 36))}
    tgt = {k: torch.zeros(k + (3,), device="cuda") for k in x}
    out = {k: torch.empty(k + (3,), device="cuda") for k in x}
    small = (2, 12, 36)
    u = UNet(ctx, n, h, 64)
    u.init(3)
    want = {}
    for k in x:
        u.backward(x[k], tgt[k], *k)
        want[k] = u.activation(12, *k)
    other = torch.from_numpy(_inputs(rng, n, h, w)[0].view(np.int16)).cuda()

    def soil():   # another pass's values in every buffer
        u.backward(other, tgt[n, h, w], n, h, w)

    soil()
    u.forward(x[n, h, w], n, h, w, out[n, h, w])
    one = u.activation(12, 1, h, w)
    np.testing.assert_array_equal(one, want[n, h, w][:1])
    np.testing.assert_array_equal(u.activation(12, n, h, w), want[n, h, w])
    tall = u.activation(12, 1, n * h, w)            # the same values under another shape
    np.testing.assert_array_equal(tall.ravel(), want[n, h, w].ravel())
    np.testing.assert_array_equal(u.activation(12, n, h, w), want[n, h, w])

    soil()
    u.forward(x[n, h, w], n, h, w, out[n, h, w])
    params = u.get_params()
    u.adam_step(0.05)
    np.testing.assert_array_equal(u.activation(12, n, h, w), want[n, h, w])
    u.set_params(params)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        u.forward(x[small], *small, out[small])
    u.forward(x[n, h, w], n, h, w, out[n, h, w])
    np.testing.assert_array_equal(u.activation(12, n, h, w), want[n, h, w])   # recorded, not run
    for _ in range(3):
        soil()
        graph.replay()
        np.testing.assert_array_equal(u.activation(12, *small), want[small])
        u.forward(x[n, h, w], n, h, w, out[n, h, w])
        np.testing.assert_array_equal(u.activation(12, n, h, w), want[n, h, w])
        u.forward(x[n, h, w], n, h, w, out[n, h, w])
        graph.replay()
        u.adam_step(0.05)
        np.testing.assert_array_equal(u.activation(12, *small), want[small])
        u.set_params(params)
    del graph
    u.close()


def test_training_beats_input(ctx, net):
    """Tracer-rendered pairs (1 spp -> 64 spp at 64x64), 150 Adam steps: the
    loss falls and the network beats its own 1-spp input on held-out pairs."""
    torch = _torch()
    net.init(3)
    print("unet dataset", flush=True)
    x, t = make_dataset(ctx, net, 40, size=64, spp=64, seed=5, worlds=2)
    xtr, ttr, xte, tte = x[:32], t[:32], x[32:], t[32:]
    print("unet training", flush=True)
    losses = train(net, xtr, ttr, steps=150, batch=8, lr=2e-3)
    assert np.mean(losses[-10:]) < 0.7 * np.mean(losses[:5])
    out = torch.empty((8, 64, 64, 3), dtype=torch.float32, device="cuda")
    net.forward(xte, 8, 64, 64, out, mode=1)
    torch.cuda.synchronize()
    ref = torch.expm1(tte).cpu().numpy()
    noisy = torch.expm1(_bf16_tensor(xte)[..., :3]).cpu().numpy()
    p_net, p_noisy = tonemap_psnr(out.cpu().numpy(), ref), tonemap_psnr(noisy, ref)
    print(f"held-out PSNR: network {p_net:.2f} dB, 1-spp input {p_noisy:.2f} dB", flush=True)
    assert p_net > p_noisy + 3.0
