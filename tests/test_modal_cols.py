"""The stage kernel of grids with few modes (one block per mode, one wavefront
per field) against the FP64 oracle: every number of rows per lane, whole and
ragged columns, 2D and 3D, and both sides of the rule that picks it."""
import numpy as np
import pytest

from helpers import fields, make_pair, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(6, 1, 8, 1), (24, 1, 64, 1), (24, 1, 68, 1), (24, 1, 192, 1), (24, 1, 256, 1),
                                   (12, 1, 300, 1), (12, 1, 384, 1), (12, 1, 448, 1), (12, 1, 512, 1), (6, 6, 12, 0),
                                   (24, 12, 64, 0), (24, 12, 132, 0), (24, 12, 320, 0), (64, 32, 100, 0),
                                   (96, 48, 48, 0), (96, 48, 100, 0)])
def test_stages_and_projection(shape):
    s, o = make_pair(*shape, gpu_prec=8, amplitude=0.05, seed=8)
    s.TimeStep(2)
    o.step(2)
    s.RemoveDivergence(0.5)
    o.remove_divergence(0.5)
    for f in fields(shape[3]):  # a step's last stage keeps no explicit terms
        e = rel_l2(s.get(f), o.get_modal(f))
        print(shape, f, "%.2e" % e, flush=True)
        # two steps of FP64 rounding; p is rescaled by 1/h (1/0.00133)
        assert e < (1e-9 if f == "p" else 1e-11), f
    s.close()


@pytest.mark.parametrize("shape", [(64, 1, 64, 1), (256, 1, 256, 1), (24, 12, 100, 0)])
def test_fp32(shape):
    """FP32 within three times the FP32 oracle's own error (the (0,0) mode's
    Poisson problem in FP64, as in the tiled kernel)."""
    s, o64 = make_pair(*shape, gpu_prec=4, amplitude=0.05, seed=9)
    _, o32 = make_pair(*shape, gpu_prec=4, oracle_prec=4, amplitude=0.05, seed=9)
    s.TimeStep(2)
    o64.step(2)
    o32.step(2)
    for f in fields(shape[3]):
        eg, er = rel_l2(s.get(f), o64.get_modal(f)), rel_l2(o32.get_modal(f), o64.get_modal(f))
        print(shape, f, "%.2e %.2e" % (eg, er), flush=True)
        assert eg <= max(3 * er, 1e-6), f
    s.close()
