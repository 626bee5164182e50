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
