"""TimeStepLinear (IMEXRK.cpp:26-41, BuildRHSLinear :195-258) on the GPU vs the oracle."""
import numpy as np
import pytest

import stratiflow_amd as sf
from stratiflow_amd import ic
from helpers import fields, make_pair, rel_l2

pytestmark = pytest.mark.gpu


def _with_base(shape, prec, oracle_prec=8):
    N1, N2, N3, dim = shape
    s, o = make_pair(N1, N2, N3, dim, gpu_prec=prec, oracle_prec=oracle_prec, amplitude=0.01, project=False)
    z, zf = s.vertical_points()
    base = ic.perturbation(N1, N2, N3, dim, z, zf, 99, amplitude=0.2)
    names = {"u1": "u1t", "u2": "u2t", "u3": "u3t", "b": "bt"}
    gpu_fields = {}
    for n, a in base.items():
        f = s.field(sf.MODAL, sf.DIRICHLET if n == "u3" else sf.NEUMANN)
        f.upload(a)
        gpu_fields[n] = f
        o.set_modal(names[n], a)
    s.SetLinearBackground(gpu_fields["u1"], gpu_fields.get("u2"), gpu_fields["u3"], gpu_fields["b"])
    o.set_linear_background()
    # LinearEvolve's start-up (StateVector.cpp:109-115)
    s.FilterAll()
    s.PopulateNodalVariables()
    s.RemoveDivergence(0.0)
    o.filter_all()
    o.populate_nodal()
    o.remove_divergence(0.0)
    return s, o, gpu_fields


@pytest.mark.parametrize("shape", [(48, 1, 64, 1), (24, 12, 32, 0)])
def test_linear_steps_fp64(shape):
    s, o, keep = _with_base(shape, 8)
    s.TimeStepLinear(5)
    o.step_linear(5)
    for f in fields(shape[3]):
        e = rel_l2(s.get(f), o.get_modal(f))
        print("linear fp64", f, e)
        assert e < 1e-9, f


@pytest.mark.parametrize("shape", [(48, 1, 64, 1), (24, 12, 32, 0)])
def test_linear_steps_fp32(shape):
    s, o, keep = _with_base(shape, 4)
    s.TimeStepLinear(10)
    o.step_linear(10)
    for f in fields(shape[3]):
        if f == "p":
            continue
        e = rel_l2(s.get(f), o.get_modal(f))
        print("linear fp32", f, e)
        assert e < 1e-4, f


@pytest.mark.parametrize("shape,prec", [((6, 1, 8, 1), 8), ((256, 1, 36, 1), 8), ((384, 1, 24, 1), 8),
                                        ((384, 1, 20, 1), 4), ((512, 1, 20, 1), 4), ((96, 12, 36, 0), 8),
                                        ((384, 6, 12, 0), 8), ((384, 6, 20, 0), 4)])
def test_linear_base_of_every_point_split(shape, prec):
    """The base state held per x point: one and two points per thread, levels
    that do not fill a block of the base transform, and a base that changes
    between calls (steps, then single stages) is the one the next call uses."""
    s, o, keep = _with_base(shape, prec)
    s.TimeStepLinear(1)
    o.step_linear(1)
    for f in ("u1", "b"):  # another base, through the solver's own field
        keep[f] *= 0.5
        s.state(f + "_tot").assign(keep[f])
        o.set_modal(f + "t", keep[f].download())
    o.set_linear_background()
    s.TimeStepLinear(1)
    o.step_linear(1)
    s.Stage(0, linear=True)
    o.stage(0, linear=True)
    for f in fields(shape[3]):
        if prec == 4 and f == "p":
            continue
        e = rel_l2(s.get(f), o.get_modal(f))
        print(shape, prec, f, "%.2e" % e, flush=True)
        assert e < (1e-9 if prec == 8 else 1e-4), f
    s.close()


@pytest.mark.parametrize("linear", [False, True])
@pytest.mark.parametrize("shape", [(6, 6, 8, 0), (64, 6, 20, 0), (96, 48, 36, 0), (128, 64, 92, 0), (192, 6, 20, 0)])
def test_products_of_every_block_size(shape, linear):
    """x-pass blocks of 64, 128 and 256 threads, with one and two points of a
    line per thread and columns that end inside a block's levels."""
    s, o, keep = _with_base(shape, 8)
    for _ in range(2):
        s.TimeStepLinear(1) if linear else s.TimeStep(1)
        o.step_linear(1) if linear else o.step(1)
    for f in fields(shape[3]):
        e = rel_l2(s.get(f), o.get_modal(f))
        print(shape, linear, f, "%.2e" % e, flush=True)
        assert e < 1e-9, f  # as the steps above
    s.close()
