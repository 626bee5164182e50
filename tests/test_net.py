"""Learned preconditioner network (stratiflow_amd.Net, sf_net_*).

CPU: the numpy restatement (oracle/convnet.py) against FP64 finite differences
and against closed forms (identity taps, linearity in the last layer).
GPU: the MFMA forward pass and parameter gradients against the restatement
with the same BF16 roundings; training lowers the loss; the preconditioner is
the identity until trained.
"""
import numpy as np
import pytest

CH = [32, 64, 64, 64, 32]


def _rand_params(rng, channels, creal_in, creal_out, scale=1.0, last_zero=False):
    from oracle import convnet
    layers = []
    for l in range(len(channels) - 1):
        ci, co = channels[l], channels[l + 1]
        rin = creal_in if l == 0 else ci
        rout = creal_out if l == len(channels) - 2 else co
        W = np.zeros((5, co, ci))
        W[:, :rout, :rin] = rng.standard_normal((5, rout, rin)) * scale * np.sqrt(2.0 / (5 * rin))
        if last_zero and l == len(channels) - 2:
            W[:] = 0
        b = np.zeros(co)
        b[:rout] = 0.1 * rng.standard_normal(rout)
        layers.append((W, b))
    return convnet.pack(layers)


@pytest.mark.parametrize("dil", [None, [1, 2, 3]])
def test_restatement_gradient_matches_finite_differences(dil):
    from oracle import convnet
    rng = np.random.default_rng(0)
    ch = [4, 6, 5, 3]
    p = _rand_params(rng, ch, 4, 3)
    x = rng.standard_normal((2, 11, 4))
    tgt = rng.standard_normal((2, 11, 3))
    loss, g = convnet.loss_and_grad(p, ch, x, tgt, 3, bf16=False, dil=dil)
    eps = 1e-6
    for k in rng.choice(p.size, 40, replace=False):
        pp, pm = p.copy(), p.copy()
        pp[k] += eps
        pm[k] -= eps
        fd = (convnet.loss_and_grad(pp, ch, x, tgt, 3, bf16=False, dil=dil)[0]
              - convnet.loss_and_grad(pm, ch, x, tgt, 3, bf16=False, dil=dil)[0]) / (2 * eps)
        assert abs(fd - g[k]) <= 1e-6 * max(1.0, abs(fd)), (k, fd, g[k])


def test_restatement_closed_forms():
    """A centre-tap identity layer copies its input; profile ends see zero padding."""
    from oracle import convnet
    x = np.arange(12, dtype=float).reshape(1, 6, 2)
    W = np.zeros((5, 2, 2))
    W[2] = np.eye(2)
    assert np.allclose(convnet.conv(x, W, None), x)
    W = np.zeros((5, 2, 2))
    W[4] = np.eye(2)  # out[p] = in[p + 2]
    out = convnet.conv(x, W, None)
    assert np.allclose(out[0, :4], x[0, 2:]) and np.allclose(out[0, 4:], 0)
    out = convnet.conv(x, W, None, 2)  # dilation 2: out[p] = in[p + 4]
    assert np.allclose(out[0, :2], x[0, 4:]) and np.allclose(out[0, 2:], 0)
    W = np.zeros((5, 2, 2))
    W[0] = np.eye(2)  # out[p] = in[p - 2 d]
    out = convnet.conv(x, W, None, 2)
    assert np.allclose(out[0, 4:], x[0, :2]) and np.allclose(out[0, :4], 0)
    assert convnet.to_bf16(np.float32(1.0 + 2 ** -9)) == np.float32(1.0)
    assert convnet.to_bf16(np.float32(1.0 + 3 * 2 ** -9)) == np.float32(1.0 + 2 ** -7)


def _net(N1=48, N3=64, prec=4, seed=3):
    import stratiflow_amd as sf
    s = sf.IMEXRK(N1, 1, N3, sf.TWO_D, 2 * np.pi / 0.44, 1.0, 10.0, 1000.0, 0.1, 1.0, precision=prec)
    return s, sf.Net(s, hidden=64, layers=4, seed=seed)


@pytest.mark.gpu
@pytest.mark.parametrize("dil", [None, [1, 2, 4, 8]])
def test_forward_and_gradient_match_restatement(dil):
    from oracle import convnet
    s, net = _net()
    assert net.channels == CH
    if dil:
        net.set_dilations(dil)
    rng = np.random.default_rng(1)
    p = _rand_params(rng, CH, 8, 6).astype(np.float32)
    net.set_params(p)
    x = np.zeros((5, net.Z, 32), np.float32)
    x[..., :8] = rng.standard_normal((5, net.Z, 8))
    out = net.forward_raw(x)
    ref, _, _ = convnet.forward(p, CH, x, bf16=True, dil=dil)
    err = np.abs(out - ref).max() / np.abs(ref).max()
    print("forward rel err", err)
    assert err < 2e-3
    tgt = np.zeros_like(out)
    tgt[..., :6] = rng.standard_normal((5, net.Z, 6))
    loss, g = net.grad_raw(x, tgt)
    lref, gref = convnet.loss_and_grad(p, CH, x, tgt, 6, bf16=True, dil=dil)
    print("loss gpu %.6e ref %.6e" % (loss, lref))
    assert abs(loss - lref) / lref < 1e-3
    eg = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print("gradient rel err", eg)
    assert eg < 2e-2


@pytest.mark.gpu
def test_training_lowers_loss_and_identity_until_trained():
    import stratiflow_amd as sf
    from stratiflow_amd import ic
    s, net = _net()
    z, zf = s.vertical_points()
    pert = ic.perturbation(48, 1, 64, sf.TWO_D, z, zf, 5, amplitude=1e-2)
    for n, a in pert.items():
        s.set(n, a)
    fin = [s.state(n) for n in ("u1", "u2", "u3", "b")]
    outs = [s.field(sf.MODAL, sf.DIRICHLET if n == "u3" else sf.NEUMANN) for n in ("u1", "u2", "u3", "b")]
    net.apply(fin, outs)
    for f, o in zip(fin, outs):
        assert np.array_equal(f.download(), o.download())
    # pairs of a fixed per-field scaling q = (0.5 u1, 2 u3, b): the direction
    # target q/RMS(q) - w/RMS(w) is a per-channel scaling of the input
    scale = {"u1": 0.5, "u2": 1.0, "u3": 2.0, "b": 1.0}
    for k in range(6):
        w = [s.field(sf.MODAL, sf.DIRICHLET if n == "u3" else sf.NEUMANN) for n in ("u1", "u2", "u3", "b")]
        q = [s.field(sf.MODAL, sf.DIRICHLET if n == "u3" else sf.NEUMANN) for n in ("u1", "u2", "u3", "b")]
        pk = ic.perturbation(48, 1, 64, sf.TWO_D, z, zf, 100 + k, amplitude=1.0)
        for i, n in enumerate(("u1", "u2", "u3", "b")):
            if n in pk:
                w[i].upload(pk[n])
                q[i].upload(scale[n] * pk[n])
        net.add_pair(w, q)
    assert net.samples() == 6 * 16
    l0, l1 = net.train(epochs=60, batch=32, lr=2e-3)
    print("loss first epoch %.4e last %.4e" % (l0, l1))
    assert l1 < 0.1 * l0


@pytest.mark.gpu
@pytest.mark.parametrize("shape,prec,hidden,layers", [((6, 1, 8, 1), 8, 64, 2), ((12, 1, 20, 1), 4, 32, 3),
                                                      ((48, 1, 64, 1), 8, 64, 4), ((24, 1, 100, 1), 4, 64, 8),
                                                      ((24, 1, 256, 1), 8, 64, 4), ((24, 1, 260, 1), 8, 32, 5),
                                                      ((12, 1, 512, 1), 4, 64, 4), ((24, 12, 36, 0), 8, 64, 4)])
def test_fused_application_matches_layers(shape, prec, hidden, layers):
    """apply() keeps a profile in LDS through all layers; the layer-by-layer
    forward pass of the packed input gives the same correction: fewer positions
    than a wave's tile, ragged tiles, one and two tiles per wave, both widths,
    the fewest and most layers, the largest dilation, 2D and 3D."""
    import stratiflow_amd as sf
    N1, N2, N3, dim = shape
    s = sf.IMEXRK(N1, N2, N3, dim, 2 * np.pi / 0.44, np.pi / 0.44, 10.0, 1000.0, 0.1, 1.0, precision=prec)
    net = sf.Net(s, hidden=hidden, layers=layers, seed=3)
    net.set_dilations([1, 2, 4, 8, 1, 3, 8, 1][:layers])
    rng = np.random.default_rng(2)
    names = ("u1", "u2", "u3", "b") if dim == 0 else ("u1", "u3", "b")
    nf = len(names)
    net.set_params(_rand_params(rng, net.channels, 2 * nf + 2, 2 * nf).astype(np.float32))
    fin, fout, a = {}, {}, {}
    for n in names:
        bc = sf.DIRICHLET if n == "u3" else sf.NEUMANN
        fin[n], fout[n] = s.field(sf.MODAL, bc), s.field(sf.MODAL, bc)
        fin[n].upload(rng.standard_normal(fin[n].shape) + 1j * rng.standard_normal(fin[n].shape))
        a[n] = fin[n].download()
    order = ("u1", "u2", "u3", "b")
    net.apply([fin.get(n) for n in order], [fout.get(n) for n in order])
    A1, h = N1 // 3, N2 // 3
    rows = list(range(h)) + list(range(N2 - h + 1, N2)) if dim == 0 else [0]
    act = {n: a[n][rows][:, :A1].reshape(len(rows) * A1, N3) for n in names}
    rms = np.sqrt(sum((np.abs(v) ** 2).sum() for v in act.values()) / (nf * act["b"].size))
    x = np.zeros((len(rows) * A1, N3, 32), np.float32)
    for i, n in enumerate(names):
        x[..., 2 * i], x[..., 2 * i + 1] = act[n].real * (1 / rms), act[n].imag * (1 / rms)
    x[..., 2 * nf] = np.tile(np.arange(A1) / (A1 - 1), len(rows))[:, None]
    if dim == 0:
        ky = np.array([j if j <= N2 // 2 else j - N2 for j in rows]) / (h - 1)
        x[..., 2 * nf + 1] = np.repeat(ky, A1)[:, None]
    y = net.forward_raw(x).astype(np.float64)
    eps = np.finfo(np.float32 if prec == 4 else np.float64).eps
    print(shape, prec, hidden, layers, flush=True)
    for i, n in enumerate(names):
        want = act[n] + rms * (y[..., 2 * i] + 1j * y[..., 2 * i + 1])
        got = fout[n].download()[rows][:, :A1].reshape(want.shape)
        # the sums differ by roundings of the RMS and of the result; an input within
        # those of a BF16 rounding boundary may fall to its other side
        off = np.abs(got - want) > 16 * eps * (np.abs(act[n]) + np.abs(want)).max()
        assert off.mean() < 1e-3 and np.abs(got - want).max() <= 2.0 ** -7 * np.abs(want).max(), n
    s.close()


@pytest.mark.gpu
def test_parameters_take_their_turn():
    """set_params and get_params after calls that are still queued: an apply uses
    the parameters that it was called with, and those read back are the last set."""
    import stratiflow_amd as sf
    s = sf.IMEXRK(64, 1, 64, sf.TWO_D, 2 * np.pi / 0.44, np.pi / 0.44, 10.0, 1000.0, 0.1, 1.0, precision=8)
    net = sf.Net(s, hidden=32, layers=3, seed=5)
    rng = np.random.default_rng(6)
    first, second = (_rand_params(rng, net.channels, 8, 6).astype(np.float32) for _ in range(2))
    fin, quiet, queued = ([s.field(sf.MODAL, sf.DIRICHLET if i == 2 else sf.NEUMANN) if i != 1 else None for i in range(4)]
                          for _ in range(3))
    for f in fin:
        if f is not None:
            f.upload(rng.standard_normal(f.shape) + 1j * rng.standard_normal(f.shape))
    net.set_params(first)
    net.apply(fin, quiet)
    s.synchronize()
    for _ in range(3):
        net.set_params(first)
        s.TimeStep(200)  # milliseconds of work in front of the call
        net.apply(fin, queued)
        net.set_params(second)
        for a, b in zip(quiet, queued):
            assert a is None or np.array_equal(a.download(), b.download())
    assert np.array_equal(net.get_params(), second)
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,prec,hidden,layers", [((192, 1, 360, 1), 8, 64, 2), ((192, 1, 364, 1), 4, 32, 2),
                                                      ((48, 24, 100, 0), 8, 32, 3)])
def test_rms_on_both_sides_of_the_second_launch(shape, prec, hidden, layers):
    """Up to 90 blocks the last one adds the sums of the RMS, of more (90, 91 and
    94 blocks here) a second launch does."""
    test_fused_application_matches_layers(shape, prec, hidden, layers)
