"""Whole-field kernels (sf_fields.hip) against numpy at the sizes where their
work split changes: fields smaller than one block, remainders of the four
elements a thread takes, several blocks, and more than one round of blocks."""
import numpy as np
import pytest

import stratiflow_amd as sf

pytestmark = pytest.mark.gpu

LX = 2 * np.pi / 0.44


def solver(shape, prec):
    N1, N2, N3, dim = shape
    s = sf.IMEXRK(N1, N2, N3, dim, LX, LX / 2, 10.0, 1000.0, 0.1, 1.0, precision=prec)
    s.SetBackground(np.tanh(s.vertical_points()[1]))
    return s


def random_field(s, bc, seed):
    rng = np.random.default_rng(seed)
    f = s.field(sf.MODAL, bc)
    f.upload(rng.standard_normal(f.shape) + 1j * rng.standard_normal(f.shape))
    return f, f.download()


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("shape", [(6, 1, 8, 1), (12, 1, 64, 1), (24, 1, 132, 1), (256, 1, 256, 1), (12, 6, 36, 0),
                                   (96, 48, 100, 0), (192, 96, 256, 0)])
def test_inner_products(shape, prec):
    s = solver(shape, prec)
    z, zf = s.vertical_points()
    N3 = s.N3
    for bc in (sf.NEUMANN, sf.DIRICHLET):
        w = np.zeros(N3)
        if bc == sf.NEUMANN:
            w[1:-1] = z[2:] - z[1:-1]
        else:
            w[2:-1] = zf[2:-1] - zf[1:-2]
        w = w.astype(np.float32 if prec == 4 else np.float64).astype(np.float64)
        f, a = random_field(s, bc, 1)
        g, b = random_field(s, bc, 2)
        terms = 2 * w * (a * b.conj()).real
        terms[0, 0] *= 0.5
        print(shape, prec, bc, flush=True)
        # FP64 sums in another order: a few roundings per term at most
        assert abs(s.InnerProd(f, g) - terms.sum()) <= 1e-14 * np.abs(terms).sum()
        assert s.InnerProd(f, g) == s.InnerProd(f, g)
    s.close()


def test_energies_follow_the_queue():
    """KE and PE are read while steps are still queued and equal the inner
    products of the state."""
    s = solver((64, 1, 64, 1), 8)
    for n in ("u1", "u3", "b"):
        s.state(n).assign(random_field(s, sf.DIRICHLET if n == "u3" else sf.NEUMANN, 3)[0])
        s.state(n).__imul__(1e-4)
    s.deltaT = 1e-3
    for _ in range(3):
        s.TimeStep(200)
        ke, pe = s.energies()
        u1, u3, b = (s.InnerProd(s.state(n), s.state(n)) for n in ("u1", "u3", "b"))
        assert ke == 0.5 * (u1 + u3) and pe == 0.1 * 0.5 * b
    s.close()


@pytest.mark.parametrize("shape,prec", [((6, 1, 8, 1), 8), ((24, 1, 64, 1), 4), ((24, 1, 132, 1), 8),
                                        ((24, 1, 256, 1), 8), ((24, 1, 260, 1), 4), ((24, 1, 384, 1), 4),
                                        ((24, 1, 448, 1), 4), ((24, 1, 512, 1), 4), ((96, 48, 100, 0), 8),
                                        ((128, 48, 36, 0), 8), ((128, 48, 64, 0), 4), ((128, 48, 256, 0), 8)])
@pytest.mark.parametrize("bc", [sf.NEUMANN, sf.DIRICHLET])
def test_advected_preconditioner(shape, prec, bc):
    """The wavefront solver for every number of rows per lane, one and eight
    modes per block, whole and ragged columns and blocks, against dense solves
    of some modes; within the rounding that the systems' condition allows."""
    s = solver(shape, prec)
    N1, N2, N3, dim = shape
    z, zf = s.vertical_points()
    dy, dyf = np.ones(N3), np.ones(N3)
    dy[1:], dyf[:-1] = np.diff(zf), np.diff(z)
    f, a = random_field(s, bc, 4)
    out = s.field(sf.MODAL, bc)
    tnu, delta, tadv, kmax = 0.02, 0.3, 2.0, 9.0
    print(shape, prec, bc, flush=True)
    f.diffusion_precondition(out, tnu, delta, kmax, tadv)
    o = out.download()
    dirichlet = bc == sf.DIRICHLET
    U = np.tanh(zf)
    rng = np.random.default_rng(5)
    A1 = N1 // 3
    rows = list(range(N2 // 3)) + list(range(N2 - N2 // 3 + 1, N2)) if dim == 0 else [0]
    modes = [(j2, j1) for j2 in rows for j1 in range(A1)]
    picked = {modes[0], modes[-1]} | {modes[i] for i in rng.integers(0, len(modes), 10)}
    for j2, j1 in picked:
        kx = 0.44 * j1
        ky = 2 * np.pi / (LX / 2) * (j2 if j2 <= N2 // 2 else j2 - N2) if dim == 0 else 0.0
        if kx * kx + ky * ky > kmax * kmax:
            assert np.array_equal(o[j2, j1], -a[j2, j1])
            continue
        A = np.eye(N3, dtype=np.complex128)
        rhs = -a[j2, j1] / delta
        ends = [0, 1, N3 - 2, N3 - 1] + ([2] if dirichlet else [])
        rhs[ends] = 0
        for j in range(1, N3 - 1):
            if j in ends:
                continue
            if dirichlet:
                lo, up = 1 / dyf[j - 1] / dy[j], 1 / dyf[j] / dy[j]
            else:
                lo, up = 1 / dy[j] / dyf[j], 1 / dy[j + 1] / dyf[j]
            c = tnu / delta
            A[j, j - 1], A[j, j + 1] = -c * lo, -c * up
            A[j, j] = 1 - c * (-lo - up - kx * kx - ky * ky) + 1j * tadv * kx * U[j] / delta
        if not dirichlet:
            A[1, 2] = -1
            A[N3 - 2, N3 - 3], A[N3 - 2, N3 - 2] = 1, -1
        x = np.linalg.solve(A, rhs)
        eps = np.finfo(np.float32 if prec == 4 else np.float64).eps
        tol = 32 * eps * np.linalg.cond(A, np.inf) * np.abs(x).max() + 4 * eps * np.abs(a[j2, j1]).max()
        assert np.abs(o[j2, j1] - (x - 0.5 * a[j2, j1])).max() <= tol, (j2, j1)
    s.close()


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("shape", [(6, 1, 8, 1), (16, 1, 12, 1), (64, 1, 64, 1), (12, 6, 36, 0), (16, 12, 100, 0),
                                   (192, 96, 64, 0)])
def test_states_to_and_from_the_solver(shape, prec):
    """CopyToSolver and CopyFromSolver in one launch: odd and even rows (two
    FP32 values share a 16-byte access), each end condition, absent fields,
    several rounds of blocks; the solver's fields as arguments keep the order
    of the copies."""
    s = solver(shape, prec)
    names = ["u1", "u2", "u3", "b", "p"] if s.N2 > 1 else ["u1", "u3", "b", "p"]
    bc = {n: sf.DIRICHLET if n == "u3" else sf.NEUMANN for n in names}
    f, a = {}, {}
    for i, n in enumerate(names):
        f[n], a[n] = random_field(s, bc[n], 10 + i)
    s.CopyToSolver(f["u1"], f.get("u2"), f["u3"], f["b"], f["p"])
    out = {n: s.field(sf.MODAL, bc[n]) for n in names}
    s.CopyFromSolver(out["u1"], out.get("u2"), out["u3"], out["b"], out["p"])
    print(shape, prec, flush=True)
    for n in names:
        assert np.array_equal(s.get(n), a[n]), n
        w = a[n].copy()
        if n == "u3":
            w[..., [0, 1, 2, -2, -1]] = 0
        elif n != "p":
            w[..., 0], w[..., -1] = w[..., 1], w[..., -2]
        assert np.array_equal(out[n].download(), w), n
    # p absent: zero; b bound to the solver's u1, which the first copy has replaced
    s.CopyToSolver(f["b"], f.get("u2"), f["u3"], s.state("u1"))
    assert np.array_equal(s.get("b"), a["b"]) and not s.get("p").any()
    # two results in one field: the last one stays
    s.CopyToSolver(f["u1"], f.get("u2"), f["u3"], f["b"], f["p"])
    s.CopyFromSolver(out["u1"], None, out["u3"], out["u1"])
    w = a["b"].copy()
    w[..., 0], w[..., -1] = w[..., 1], w[..., -2]
    assert np.array_equal(out["u1"].download(), w)
    # the linearisation state
    s.SetLinearBackground(f["u1"], None, f["u3"], f["b"])
    assert np.array_equal(s.get("b_tot"), a["b"]) and not s.get("u2_tot").any()
    s.SetLinearBackground(s.state("b_tot"), f["p"], f["u3"], s.state("u2_tot"))
    assert np.array_equal(s.get("u1_tot"), a["b"]) and np.array_equal(s.get("b_tot"), a["p"])
    s.close()


@pytest.mark.parametrize("shape,prec", [((6, 1, 8, 1), 4), ((8, 1, 12, 1), 8), ((12, 1, 36, 1), 4), ((16, 1, 100, 1), 8),
                                        ((64, 1, 20, 1), 4), ((96, 1, 36, 1), 8), ((192, 1, 24, 1), 8),
                                        ((256, 1, 28, 1), 8), ((384, 1, 20, 1), 8), ((384, 1, 52, 1), 4),
                                        ((512, 1, 20, 1), 4), ((24, 12, 36, 0), 4), ((48, 24, 16, 0), 8)])
def test_whole_field_transforms(shape, prec):
    """ToNodal and ToModal against numpy for every length class (one register
    DFT and two passes of N1/2 points), 16 and 8 levels per block, and levels
    that do not fill a block; a level's result does not depend on its
    neighbours, bit for bit."""
    s = solver(shape, prec)
    N1, N2, N3, dim = shape
    f, a = random_field(s, sf.NEUMANN, 6)
    a[0, 0] = a[0, 0].real
    for j2 in range(1, (N2 + 1) // 2):  # a real field's j1 = 0 column
        a[N2 - j2, 0] = a[j2, 0].conj()
    a[..., 1] = a[..., 0]  # equal levels
    f.upload(a)
    a = f.download()
    n, back = s.field(sf.NODAL, sf.NEUMANN), s.field(sf.MODAL, sf.NEUMANN)
    f.ToNodal(n)
    want = np.fft.irfft2(a, s=(N2, N1), axes=(0, 1)) * (N1 * N2)
    got = n.download()
    tol = 8 * np.finfo(np.float32 if prec == 4 else np.float64).eps * np.log2(N1 * N2)
    e = np.linalg.norm(got - want) / np.linalg.norm(want)
    n.ToModal(back)
    b = np.linalg.norm(back.download() - a) / np.linalg.norm(a)
    print(shape, prec, "%.2e %.2e" % (e / tol, b / tol), flush=True)
    assert e < tol and b < 2 * tol
    assert np.array_equal(got[..., 0], got[..., 1])
    s.close()


@pytest.mark.parametrize("shape", [(24, 1, 64, 1), (192, 96, 192, 0)])
def test_many_inner_products(shape):
    """The number that the results of a call carry starts 256 calls before its
    overflow: the results on both sides of it are those of the first calls (on
    the blocks' own sums and on the total of a second launch)."""
    s = solver(shape, 8)
    for n in ("u1", "u3", "b"):
        s.state(n).assign(random_field(s, sf.DIRICHLET if n == "u3" else sf.NEUMANN, 4)[0])
    u, b = s.state("u1"), s.state("b")
    first = s.energies() + (s.InnerProd(u, b),)
    assert all(np.isfinite(first)) and first[0] > 0 and first[1] > 0
    for i in range(300):
        assert s.energies() + (s.InnerProd(u, b),) == first, i
    s.close()


@pytest.mark.parametrize("shape,prec", [((48, 1, 36, 1), 4), ((64, 1, 68, 1), 8), ((48, 12, 20, 0), 8), ((64, 6, 16, 0), 8),
                                        ((32, 16, 48, 0), 8), ((64, 12, 64, 0), 4)])
def test_transforms_of_short_lines(shape, prec):
    """Lines of 24 and 32 points (N1 = 48, 64) in two passes, with blocks that fill
    or do not fill their levels, and FP64 blocks of whole lines in their own
    order: a random nodal field against numpy, there and back."""
    s = solver(shape, prec)
    N1, N2, N3, dim = shape
    n, m, back = s.field(sf.NODAL, sf.NEUMANN), s.field(sf.MODAL, sf.NEUMANN), s.field(sf.NODAL, sf.NEUMANN)
    n.upload(np.random.default_rng(8).standard_normal(n.shape))
    v = n.download()
    n.ToModal(m)
    m.ToNodal(back)
    want = np.fft.rfft2(v, axes=(0, 1)) / (N1 * N2)
    want[:, N1 // 3:] = 0
    if dim == 0:
        want[N2 // 3:N2 - N2 // 3 + 1] = 0
    tol = 8 * np.finfo(np.float32 if prec == 4 else np.float64).eps * np.log2(N1 * N2)
    e = np.linalg.norm(m.download() - want) / np.linalg.norm(want)
    back_want = np.fft.irfft2(want, s=(N2, N1), axes=(0, 1)) * (N1 * N2)
    b = np.linalg.norm(back.download() - back_want) / np.linalg.norm(back_want)
    print(shape, prec, "%.2e %.2e" % (e / tol, b / tol), flush=True)
    assert e < tol and b < 2 * tol
    s.close()
