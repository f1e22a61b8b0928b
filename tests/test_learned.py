"""Learned absorbing boundary: the CPU conv oracle is pinned (adjoints, finite differences,
dense brute force; Adam against torch.optim.Adam and its first-step closed form; bf16
rounding against torch's cast, on values where truncation differs); the BF16-MFMA training
kernels match it; the fused per-step inference
kernel writes the layer the oracle predicts; a trained network beats the same grid without
it."""
import ctypes as ct

import numpy as np
import pytest

from oracle import conv
from pyfds_amd import _native as nat
from pyfds_amd.learned import LAYER, BAND, lbc_cell


# ------------------------------------------------------------------ CPU: oracle pins
def test_conv_oracle_adjoints_and_brute_force():
    rng = np.random.default_rng(0)
    B, P, Ci, Co, K, S = 3, 19, 16, 32, 5, 2
    x = rng.standard_normal((B, P, Ci))
    w = rng.standard_normal((S, Co, K, Ci))
    side = np.array([0, 1, 1])
    dy = rng.standard_normal((B, P, Co))
    y = conv.conv_fwd(x, w, side)
    # dense brute force of one output
    b, p, co = 1, 0, 7
    want = sum(w[side[b], co, k, ci] * x[b, p + k - 2, ci]
               for k in range(K) for ci in range(Ci) if 0 <= p + k - 2 < P)
    assert np.isclose(y[b, p, co], want)
    ip = np.sum(y * dy)
    assert np.isclose(ip, np.sum(x * conv.conv_bwd_data(dy, w, side)))
    assert np.isclose(ip, np.sum(w * conv.conv_bwd_weight(dy, x, side, S, K)))


def test_mse_gradient_finite_differences():
    rng = np.random.default_rng(1)
    y, t = rng.standard_normal((2, 9, 4)), rng.standard_normal((2, 9, 4))
    wch = rng.random(4)
    lo, hi = [0, 2], [9, 7]
    loss, grad = conv.mse(y, t, lo, hi, wch, 0.1)
    eps = 1e-6
    for idx in [(0, 3, 1), (1, 1, 2), (1, 5, 0)]:
        yp = y.copy()
        yp[idx] += eps
        fd = (conv.mse(yp, t, lo, hi, wch, 0.1)[0] - loss) / eps
        assert np.isclose(fd, grad[idx], rtol=1e-4, atol=1e-8)


def _torch_bf16_bits(a):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(torch.bfloat16)
    return t.view(torch.int16).numpy().view(np.uint16)


# values where round-to-nearest-even, round-half-up and truncation disagree
BF16_EDGES = np.array([65504.0, 1 + 2 ** -8 + 2 ** -16, 1 + 2 ** -8, 1 + 3 * 2 ** -8,
                       -(1 + 2 ** -8 + 2 ** -16), 3.14159, 1e-3, -2.5, 1.0, 2 ** -130,
                       3.0e38], np.float32)


def _bf16_cases():
    rng = np.random.default_rng(3)
    return np.concatenate([BF16_EDGES, rng.standard_normal(20000).astype(np.float32) * 1e3,
                           rng.standard_normal(20000).astype(np.float32) * 1e-20])


def test_bf16_rounding_matches_torch():
    a = _bf16_cases()
    np.testing.assert_array_equal(conv.to_bf16_bits(a), _torch_bf16_bits(a))
    r = conv.from_bf16_bits(conv.to_bf16_bits(BF16_EDGES[:4]))
    np.testing.assert_array_equal(r, np.array([65536.0, 1 + 2 ** -7, 1.0, 1 + 2 ** -6],
                                              np.float32))


def test_bf16_planted_truncation_is_caught():
    a = _bf16_cases()
    truncated = (np.ascontiguousarray(a).view(np.uint32) >> 16).astype(np.uint16)
    assert np.count_nonzero(truncated != _torch_bf16_bits(a)) > 0


def _torch_adam(w, grads, lr, b1, b2, eps):
    import torch
    p = torch.nn.Parameter(torch.from_numpy(w.copy()))
    opt = torch.optim.Adam([p], lr=lr, betas=(b1, b2), eps=eps)
    out = []
    for g in grads:
        p.grad = torch.from_numpy(g.copy())
        opt.step()
        out.append(p.detach().numpy().copy())
    return out


def _oracle_adam(w, grads, lr, b1, b2, eps, step_fn=None):
    step_fn = step_fn or conv.adam_step
    m1, m2, out = np.zeros_like(w), np.zeros_like(w), []
    for i, g in enumerate(grads):
        w, m1, m2 = step_fn(w, m1, m2, g, lr, b1, b2, eps, i + 1)
        out.append(w.copy())
    return out


ADAM = dict(lr=3e-3, b1=0.9, b2=0.999, eps=1e-8)


def _adam_case():
    rng = np.random.default_rng(4)
    w = rng.standard_normal(500)
    return w, [rng.standard_normal(500) * s for s in (1.0, 0.3, 2.0)]


def test_adam_oracle_matches_torch_and_first_step_closed_form():
    w, grads = _adam_case()
    ours, ref = _oracle_adam(w, grads, **ADAM), _torch_adam(w, grads, **ADAM)
    for a, b in zip(ours, ref):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-14)
    # step 1: bias-corrected moments are g and g**2, so w1 = w - lr g / (|g| + eps)
    g = grads[0]
    np.testing.assert_allclose(ours[0], w - ADAM['lr'] * g / (np.abs(g) + ADAM['eps']),
                               rtol=0, atol=1e-15)


def test_adam_planted_mistake_is_caught():
    # the second moment without its bias correction: the same comparison must fail
    def planted(w, m1, m2, g, lr, b1, b2, eps, step):
        m1 = b1 * m1 + (1 - b1) * g
        m2 = b2 * m2 + (1 - b2) * g * g
        return w - lr * (m1 / (1 - b1 ** step)) / (np.sqrt(m2) + eps), m1, m2
    w, grads = _adam_case()
    ours, ref = _oracle_adam(w, grads, step_fn=planted, **ADAM), _torch_adam(w, grads, **ADAM)
    assert max(np.abs(a - b).max() for a, b in zip(ours, ref)) > 1e-6


def test_layer_cells_are_written_once():
    """Top/bottom own the full width, left/right the rows between: every layer cell of the
    G x G frame is written by exactly one side and no interior cell is written."""
    g = 56
    count = np.zeros(g * g, int)
    a = np.arange(g)
    for s in range(4):
        span = a if s < 2 else a[LAYER:g - LAYER]
        for d in range(LAYER):
            np.add.at(count, lbc_cell(s, d, span, g), 1)
    frame = np.ones((g, g), bool)
    frame[LAYER:g - LAYER, LAYER:g - LAYER] = False
    assert np.all(count.reshape(g, g)[frame] == 1)
    assert np.all(count.reshape(g, g)[~frame] == 0)


# ------------------------------------------------------------------ GPU
def _torch():
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    return torch


def _bf16_tensor(torch, a):
    return torch.from_numpy(conv.to_bf16_bits(a).view(np.int16)).cuda()


@pytest.mark.gpu
def test_mfma_training_kernels_match_oracle():
    torch = _torch()
    lib = nat.load()
    rng = np.random.default_rng(2)
    B, P, Ci, Co, K, S = 5, 70, 48, 32, 5, 4
    x = conv.round_bf16(rng.standard_normal((B, P, Ci)))
    w = conv.round_bf16(rng.standard_normal((S, Co, K, Ci)) * 0.1)
    dy = conv.round_bf16(rng.standard_normal((B, P, Co)))
    side = np.array([0, 3, 1, 3, 2], np.int32)
    xd, wd, dyd = _bf16_tensor(torch, x), _bf16_tensor(torch, w), _bf16_tensor(torch, dy)
    wt = _bf16_tensor(torch, np.ascontiguousarray(w.transpose(0, 3, 2, 1)))
    sd = torch.from_numpy(side).cuda()
    p = lambda t: ct.c_void_p(t.data_ptr())
    s = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    y = torch.empty((B, P, Co), dtype=torch.float32, device='cuda')
    nat.check(lib.fds_lbc_conv_fwd(p(xd), p(wd), p(sd), p(y), None, B, P, Ci, Co, K, s))
    dx = torch.empty((B, P, Ci), dtype=torch.float32, device='cuda')
    nat.check(lib.fds_lbc_conv_bwd_data(p(dyd), p(wt), p(sd), p(dx), None, B, P, Ci, Co, K, s))
    part = torch.empty((B, Co, K, Ci), dtype=torch.float32, device='cuda')
    dw = torch.empty((S, Co, K, Ci), dtype=torch.float32, device='cuda')
    nat.check(lib.fds_lbc_conv_bwd_weight(p(dyd), p(xd), p(part), B, P, Ci, Co, K, s))
    nat.check(lib.fds_lbc_reduce_weight(p(part), p(sd), p(dw), B, S, Co * K * Ci, s))
    torch.cuda.synchronize()
    for got, want, name in ((y, conv.conv_fwd(x, w, side), 'fwd'),
                            (dx, conv.conv_bwd_data(dy, w, side), 'bwd_data'),
                            (dw, conv.conv_bwd_weight(dy, x, side, S, K), 'bwd_weight')):
        g = got.cpu().numpy().astype(np.float64)
        err = np.linalg.norm(g - want) / np.linalg.norm(want)
        print(name, 'rel err', err)
        assert err < 2e-6, (name, err)

    # loss + gradient, Adam
    t_ = rng.standard_normal((B, P, Co)).astype(np.float32)
    yv = y.cpu().numpy()
    lo = np.array([0, 3, 0, 16, 0], np.int32)
    hi = np.array([P, P - 3, P, P - 16, 50], np.int32)
    wch = rng.random(Co).astype(np.float32)
    norm = 1.0 / (B * P)
    loss_ref, grad_ref = conv.mse(yv.astype(np.float64), t_, lo, hi, wch, norm)
    dyb = torch.empty((B, P, Co), dtype=torch.int16, device='cuda')
    lp = torch.zeros(64, dtype=torch.float32, device='cuda')
    tt, lod, hid, wd_ = (torch.from_numpy(a).cuda() for a in (t_, lo, hi, wch))
    nat.check(lib.fds_lbc_mse(p(y), p(tt), p(lod), p(hid), p(wd_), p(dyb), p(lp), 64, B, P, Co,
                              norm, s))
    torch.cuda.synchronize()
    assert np.isclose(lp.sum().item(), loss_ref, rtol=1e-4)
    g_dev = conv.from_bf16_bits(dyb.cpu().numpy().view(np.uint16))
    assert np.allclose(g_dev, grad_ref, rtol=2 ** -7, atol=1e-12)
    wv = rng.standard_normal(1000).astype(np.float32)
    gv = rng.standard_normal(1000).astype(np.float32)
    m1 = np.zeros(1000, np.float32)
    m2 = np.zeros(1000, np.float32)
    wd2, gd, m1d, m2d = (torch.from_numpy(a.copy()).cuda() for a in (wv, gv, m1, m2))
    for step in (1, 2):
        nat.check(lib.fds_lbc_adam(p(wd2), p(m1d), p(m2d), p(gd), 1000, 1e-2, 0.9, 0.999, 1e-8,
                                   step, s))
        wv, m1, m2 = conv.adam_step(wv.astype(np.float64), m1, m2, gv, 1e-2, 0.9, 0.999, 1e-8,
                                    step)
    torch.cuda.synchronize()
    assert np.allclose(wd2.cpu().numpy(), wv, rtol=1e-5, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize('g, B, iters', [(33, 1, 1), (64, 3, 2), (65, 70, 2), (129, 5, 3),
                                         (190, 32, 2)])
def test_training_iterations_equal_the_single_kernels(g, B, iters):
    """fds_lbc_train against the kernels of one operation each, which the oracle checks above:
    the same sums in the same order, so the same bits; the loss is summed in another order
    (a few hundred float32 terms: 1e-5).  Strips shorter than a segment, of whole segments and
    with remainders; sides without a sample; more samples than lanes."""
    torch = _torch()
    lib = nat.load()
    rng = np.random.default_rng(g)
    T, D, L, K, Ci, Ch, Co = 6, 24, 16, 5, 48, 32, 48
    frames = torch.from_numpy(rng.standard_normal((2 * T, 3, 4, D, g)).astype(np.float32)).cuda()
    pick = [rng.integers(lo, hi, (iters, B)).astype(np.int32)
            for lo, hi in ((0, 2), (1, T), (0, 4 if B > 3 else 2))]
    scale = rng.uniform(0.5, 2.0, (iters, B)).astype(np.float32)
    run, step, side, scale = (torch.from_numpy(a).cuda() for a in pick + [scale])
    wch = torch.from_numpy(rng.random(Co).astype(np.float32)).cuda()
    cs = np.array([1.0, 2.0, 0.5], np.float32)
    s = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda t: ct.c_void_p(t.data_ptr())

    def layers():
        gen = torch.Generator().manual_seed(g)
        out = []
        for co, ci in ((Ch, Ci), (Co, Ch)):
            w = (torch.randn(4, co, K, ci, generator=gen) * 0.1).cuda()
            wb = torch.empty(w.shape, dtype=torch.int16, device='cuda')
            wt = torch.empty((4, ci, K, co), dtype=torch.int16, device='cuda')
            nat.check(lib.fds_lbc_pack(p(w), p(wb), p(wt), 4, co, K, ci, s))
            out.append([w, torch.zeros_like(w), torch.zeros_like(w), wb, wt])
        return out

    got = layers()
    size = ct.c_int64()
    nat.check(lib.fds_lbc_train_workspace(B, g, ct.byref(size)))
    work = torch.full((size.value,), 0xff, dtype=torch.uint8, device='cuda')
    loss = torch.empty(B * -(-g // 64), dtype=torch.float32, device='cuda')
    arg = (nat.LbcLayer * 2)(*[nat.LbcLayer(*[t.data_ptr() for t in row]) for row in got])
    nat.check(lib.fds_lbc_train(p(frames), p(run), p(step), p(side), p(scale), p(wch), arg,
                                p(work), p(loss), iters, B, T, D, g, L,
                                cs.ctypes.data_as(ct.c_void_p), 1e-2, 0.9, 0.999, 1e-8, 3, s))
    want = layers()
    new = lambda dt, *shape: torch.empty(shape, dtype=dt, device='cuda')
    f4, i2 = torch.float32, torch.int16
    x, tgt = new(i2, B, g, Ci), new(f4, B, g, Co)
    h, hb, y, dyb = new(f4, B, g, Ch), new(i2, B, g, Ch), new(f4, B, g, Co), new(i2, B, g, Co)
    dh, dhb = new(f4, B, g, Ch), new(i2, B, g, Ch)
    lp = new(f4, 64)
    (w1, m1, v1, w1b, w1t), (w2, m2, v2, w2b, w2t) = want
    part1, part2 = new(f4, B, Ch, K, Ci), new(f4, B, Co, K, Ch)
    g1, g2 = torch.empty_like(w1), torch.empty_like(w2)
    for i in range(iters):
        sd = side[i]
        edge = torch.where(sd < 2, 0, L).int()
        lo, hi = edge, (g - edge).int()
        nat.check(lib.fds_lbc_gather(p(frames), p(run[i]), p(step[i]), p(sd), p(scale[i]), p(x),
                                     p(tgt), B, T, D, g, L, cs.ctypes.data_as(ct.c_void_p), s))
        nat.check(lib.fds_lbc_conv_fwd(p(x), p(w1b), p(sd), p(h), p(hb), B, g, Ci, Ch, K, s))
        nat.check(lib.fds_lbc_conv_fwd(p(hb), p(w2b), p(sd), p(y), None, B, g, Ch, Co, K, s))
        nat.check(lib.fds_lbc_mse(p(y), p(tgt), p(lo), p(hi), p(wch), p(dyb), p(lp), 64, B, g, Co,
                                  1.0 / (B * g * 4.0), s))
        nat.check(lib.fds_lbc_conv_bwd_weight(p(dyb), p(hb), p(part2), B, g, Ch, Co, K, s))
        nat.check(lib.fds_lbc_reduce_weight(p(part2), p(sd), p(g2), B, 4, Co * K * Ch, s))
        nat.check(lib.fds_lbc_conv_bwd_data(p(dyb), p(w2t), p(sd), p(dh), p(dhb), B, g, Ch, Co, K,
                                            s))
        nat.check(lib.fds_lbc_conv_bwd_weight(p(dhb), p(x), p(part1), B, g, Ci, Ch, K, s))
        nat.check(lib.fds_lbc_reduce_weight(p(part1), p(sd), p(g1), B, 4, Ch * K * Ci, s))
        for (w, m, v, wb, wt), gr, co, ci in ((want[0], g1, Ch, Ci), (want[1], g2, Co, Ch)):
            nat.check(lib.fds_lbc_adam(p(w), p(m), p(v), p(gr), w.numel(), 1e-2, 0.9, 0.999, 1e-8,
                                       3 + i, s))
            nat.check(lib.fds_lbc_pack(p(w), p(wb), p(wt), 4, co, K, ci, s))
    torch.cuda.synchronize()
    for a, b, layer in zip(got, want, (1, 2)):
        for u, v, name in zip(a, b, ('w', 'm', 'v', 'wb', 'wt')):
            assert torch.equal(u, v), (layer, name, (u != v).sum().item())
    assert np.isclose(loss.sum().item(), lp.sum().item(), rtol=1e-5)


@pytest.mark.gpu
def test_fused_inference_writes_oracle_layer():
    """One step of a 64 x 64 FP32 grid with the learned layer: the layer cells equal the
    network evaluated by the oracle on the band rows (bf16 inputs and hidden activations
    rounded as on the device)."""
    torch = _torch()
    import pyfds_amd as fds
    from pyfds_amd.learned import LearnedBoundary, CIN, HIDDEN, COUT, TAPS
    g = 64
    rng = np.random.default_rng(3)
    lb = LearnedBoundary.__new__(LearnedBoundary)
    lb.torch, lb.lib, lb.dev = torch, nat.load(), torch.device('cuda', 0)
    lb.cs = np.array([1.0, 1.5e6, 1.5e6], np.float32)
    w1 = conv.round_bf16(rng.standard_normal((4, HIDDEN, TAPS, CIN)) * 0.05)
    w2 = conv.round_bf16(rng.standard_normal((4, COUT, TAPS, HIDDEN)) * 0.05)
    lb.w1b, lb.w2b = _bf16_tensor(torch, w1), _bf16_tensor(torch, w2)
    fld = fds.Acoustic2D(x_samples=g, x_delta=1e-4, y_samples=g, y_delta=1e-4, t_samples=2,
                         t_delta=1e-8, material=fds.AcousticMaterial(1500.0, 1000.0))
    fld.form = 'fp32'
    p0 = rng.standard_normal(g * g).astype(np.float32).astype(np.float64)
    vx0 = (rng.standard_normal(g * g) * 1e-6).astype(np.float32).astype(np.float64)
    vy0 = (rng.standard_normal(g * g) * 1e-6).astype(np.float32).astype(np.float64)
    fld.pressure.values, fld.velocity_x.values, fld.velocity_y.values = p0, vx0, vy0
    p0_in, vx0_in, vy0_in = p0.copy(), vx0.copy(), vy0.copy()
    lb.attach(fld)
    fld.simulate(1)
    cur = [np.asarray(c.values, np.float64) for c in (fld.pressure, fld.velocity_x,
                                                      fld.velocity_y)]
    # copies: the run updates the held arrays in place (as the reference's values -= ...)
    prev = [p0_in, vx0_in, vy0_in]
    for s in range(4):
        x = np.zeros((1, g, CIN))
        for a in range(LAYER, g - LAYER):
            for h, src in ((0, cur), (1, prev)):
                for c in range(3):
                    for j in range(BAND):
                        v = np.float32(src[c][lbc_cell(s, LAYER + j, a, g)]) * lb.cs[c]
                        x[0, a, h * 24 + c * 8 + j] = v
        x = conv.round_bf16(x)
        hdn = conv.round_bf16(conv.conv_fwd(x, w1, np.array([s])))
        y = conv.conv_fwd(hdn, w2, np.array([s]))[0]
        span = range(g) if s < 2 else range(LAYER, g - LAYER)
        for c in range(3):
            for d in (0, LAYER // 2, LAYER - 1):
                got = np.array([cur[c][lbc_cell(s, d, a, g)] for a in span]) * lb.cs[c]
                want = np.array([y[a, c * LAYER + d] for a in span])
                scale = np.abs(want).max() + 1e-30
                # bf16 rounding of the hidden layer may flip by one ulp between the fp32
                # device sum and the float64 oracle sum
                assert np.abs(got - want).max() <= 2e-2 * scale, (s, c, d)
    fld._runner().close()


def _ring_field(torch, g, case, tile, steps):
    import pyfds_amd as fds
    from pyfds_amd.learned import LearnedBoundary, CIN, HIDDEN, COUT, TAPS
    rng = np.random.default_rng(g)
    lb = LearnedBoundary.__new__(LearnedBoundary)
    lb.torch, lb.lib, lb.dev = torch, nat.load(), torch.device('cuda', 0)
    lb.cs = np.array([1.0, 1.5e6, 1.5e6], np.float32)
    lb.w1b = _bf16_tensor(torch, rng.standard_normal((4, HIDDEN, TAPS, CIN)) * 0.05)
    lb.w2b = _bf16_tensor(torch, rng.standard_normal((4, COUT, TAPS, HIDDEN)) * 0.05)
    dt = 1e-8
    fld = fds.Acoustic2D(x_samples=g, x_delta=1e-4, y_samples=g,
                         y_delta=1.25e-4 if case == 'anisotropic' else 1e-4, t_samples=steps,
                         t_delta=dt, material=fds.AcousticMaterial(1500.0, 1000.0))
    fld.form = 'fp32_kahan' if case == 'kahan' else 'fp32'
    fld.tile = tile
    cells = [x + g * y for x in range(3, g // 2) for y in range(g // 3, g // 2)]
    fld.add_material_region(fds.regions.Region(cells), fds.AcousticMaterial(2500.0, 1800.0))
    n = g * g
    for comp, scale in ((fld.pressure, 1.0), (fld.velocity_x, 1e-6), (fld.velocity_y, 1e-6)):
        comp.values = (rng.standard_normal(n) * scale).astype(np.float32).astype(np.float64)
    src = 20 if case == 'source' else g // 2
    fld.pressure.add_boundary(fds.regions.Region([src + g * (g // 2)]),
                              value=np.sin(np.arange(steps + 1)), additive=True)
    last = g - 1
    at = {'layer': [(5, 40)], 'many': [(x, 18) for x in range(20, g - 20)] +
          [(20, y) for y in range(20, g - 20)]}.get(case, [])
    at = at + [(16, 16), (23, 16), (16, last - 16), (last - 17, last - 20), (last - 16, 33),
               (33, 20), (g // 2, 16), (24, 24), (g // 2, g // 2), (g // 2, g // 2)]
    for comp in (fld.pressure, fld.velocity_x, fld.velocity_y):
        comp.add_output(fds.regions.Region([x + g * y for x, y in at]))
    lb.attach(fld)
    return fld, lb


@pytest.mark.gpu
@pytest.mark.parametrize('g, case, stages', [
    (66, '', 4), (67, '', 4), (127, '', 4), (129, '', 4), (256, '', 4), (511, '', 4),
    (512, '', 6), (573, '', 6), (65, '', 1), (130, 'source', 1), (130, 'layer', 1),
    (130, 'many', 1), (130, 'kahan', 1), (130, 'anisotropic', 1)])
def test_steps_per_launch_with_the_layer_equal_single_steps(g, case, stages):
    """The learned layer with several steps per launch against the LDS-tile engine with the
    network after every step: the same bits.  Smallest grids, segments of every length, corners,
    remainders of a run; and the fields that keep single steps."""
    torch = _torch()
    plan = (13, 1, 6)
    got = []
    for tile in (None, 0):
        fld, lb = _ring_field(torch, g, case, tile, sum(plan))
        assert lb.lib.fds_steps_per_launch(fld._runner().ctx) == (1 if tile == 0 else stages)
        for n in plan:
            fld.simulate(n)
        comps = (fld.pressure, fld.velocity_x, fld.velocity_y)
        got.append([np.array(c.values) for c in comps] +
                   [np.array(c.outputs[0].signals) for c in comps])
        fld._runner().close()
    assert np.isfinite(got[0][0]).all() and np.abs(got[0][0]).max() > 0
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.fixture(scope='module')
def trained_small():
    """A network trained at reduced size (interior 256, enlarged 768) on three recorded runs."""
    _torch()
    from pyfds_amd.learned import LearnedBoundary
    lb = LearnedBoundary(n_int=256, big=768, seed=0)
    lb.generate(n_runs=3, seed=100, after=500)
    hist = lb.train(iters=600, batch=32, lr=2e-3, log_every=100)
    print('loss history', hist)
    return lb


@pytest.mark.gpu
def test_trained_network_beats_plain_small_grid(trained_small):
    """After training, the learned layer reflects under 1 % of the interior energy (against
    the enlarged run), far less than the same small grid without it, and stays finite."""
    from pyfds_amd.learned import Scene
    res = trained_small.evaluate(Scene.random(np.random.default_rng(7), 256), after=500)
    print('evaluation', res)
    assert res['finite']
    assert res['learned'] <= 0.01
    assert res['learned'] < 0.05 * res['plain_small']


@pytest.mark.gpu
@pytest.mark.parametrize('seed', [11, 12, 13])
def test_held_out_scenes_stay_under_one_percent(trained_small, seed):
    """Scenes the training never saw (other sources, inclusions and incidence angles)."""
    from pyfds_amd.learned import Scene
    scene = Scene.random(np.random.default_rng(seed), 256)
    res = trained_small.evaluate(scene, after=500, timing=False)
    print('held-out scene', seed, scene.source, res)
    assert res['finite'] and res['learned'] <= 0.01
    assert res['learned'] < 0.05 * res['plain_small']


@pytest.mark.gpu
def test_run_falls_back_to_the_enlarged_domain(trained_small):
    """LearnedBoundary.run uses the net only when its validated reflected energy is within
    the tolerance; otherwise it runs the plain enlarged domain, whose interior is exactly what
    a direct enlarged run computes."""
    from pyfds_amd.learned import Scene
    lb = trained_small
    scene = Scene.random(np.random.default_rng(21), 256)
    steps = 300
    saved = lb.validated, getattr(lb, 'tolerance', 0.01)
    try:
        lb.validated = None                       # never validated: fallback
        inner, how = lb.run(scene, steps)
        assert how == 'enlarged'
        f = lb.field(scene, lb.big, lb.off, steps)
        f.simulate(steps)
        p = np.asarray(f.pressure.values).reshape(lb.big, lb.big)
        o = lb.off + LAYER
        np.testing.assert_array_equal(inner, p[o:o + lb.n_int, o:o + lb.n_int])
        f._runner().close()
        lb.validated, lb.tolerance = 0.5, 0.01    # validated but above the tolerance
        assert lb.run(scene, steps)[1] == 'enlarged'
        lb.validated = 0.001                      # within it: the learned grid
        inner_l, how = lb.run(scene, steps)
        assert how == 'learned' and inner_l.shape == inner.shape
        assert np.all(np.isfinite(inner_l))
    finally:
        lb.validated, lb.tolerance = saved


@pytest.mark.gpu
def test_full_size_learned_run_is_faster_than_the_enlarged_run():
    """At the bench's size (interior 1024, enlarged 3072) the learned grid costs less
    wall-clock than the enlarged plain run for the same steps, at under 1 % reflected energy.
    (At reduced sizes the enlarged grid's steps cost less than the net's, so the method pays
    only where the enlarged domain is large.)"""
    _torch()
    from pyfds_amd.learned import LearnedBoundary, Scene
    lb = LearnedBoundary(n_int=1024, big=3072, seed=0)
    lb.generate(n_runs=3, seed=100, after=1200)
    lb.train(iters=600, batch=32, lr=2e-3)
    res = lb.evaluate(Scene.random(np.random.default_rng(7), 1024), after=1200)
    print('full size', res)
    assert res['finite'] and res['learned'] <= 0.01
    assert res['speedup'] > 1.0
