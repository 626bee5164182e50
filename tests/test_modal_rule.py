"""The rule that picks the stage kernel (sf_modal_cols.hip): one block per mode
or tiles of eight modes.  On the CPU against measured times of both, on the GPU
against the FP64 oracle on both sides of its lines."""
import ctypes
import os

import pytest

# us per launch, tiles and one block per mode, on an MI355X: (N1, N2, N3,
# precision) of every class of the rule next to its line
STAGE = {
    (48, 48, 512, 4): (45.1, 34.1), (24, 96, 512, 4): (41.7, 30.1), (48, 48, 384, 8): (47.0, 40.3),
    (48, 48, 512, 8): (77.2, 82.3), (96, 32, 256, 4): (30.3, 23.3), (192, 16, 384, 4): (34.0, 36.9),
    (96, 32, 192, 8): (35.9, 29.9), (96, 32, 384, 8): (45.0, 54.5), (96, 48, 128, 4): (22.5, 17.4),
    (96, 48, 192, 4): (25.9, 27.3), (384, 12, 192, 4): (23.7, 26.5), (96, 48, 128, 8): (30.5, 28.7),
    (96, 48, 256, 8): (35.0, 47.0), (64, 32, 256, 4): (31.9, 23.8), (64, 32, 384, 4): (36.9, 39.0),
    (64, 32, 192, 8): (37.8, 32.8), (64, 32, 256, 8): (36.0, 38.7), (64, 48, 128, 4): (23.0, 20.8),
    (64, 48, 192, 4): (26.4, 32.1), (64, 48, 100, 8): (30.7, 28.2), (64, 48, 192, 8): (38.4, 48.7),
    (64, 64, 100, 4): (23.4, 22.0), (64, 64, 128, 4): (23.6, 26.7), (64, 64, 64, 8): (25.7, 22.0),
    (64, 64, 100, 8): (31.6, 37.9), (128, 48, 64, 4): (19.9, 21.4), (128, 48, 64, 8): (26.7, 30.1),
}
PROJECTION = {
    (48, 48, 256, 4): (10.5, 8.9), (48, 48, 384, 4): (12.7, 14.4), (96, 32, 100, 4): (6.8, 6.1),
    (96, 32, 192, 4): (8.5, 10.2), (96, 48, 48, 4): (5.7, 5.2), (96, 48, 192, 4): (9.8, 14.5),
    (64, 32, 256, 4): (12.5, 13.6), (64, 48, 100, 4): (8.4, 10.2),
    (48, 48, 192, 8): (9.9, 8.5), (48, 48, 384, 8): (15.5, 17.3), (96, 32, 128, 8): (8.6, 7.5),
    (96, 32, 192, 8): (10.0, 11.9), (96, 48, 64, 8): (7.2, 6.5), (96, 48, 100, 8): (8.7, 10.2),
    (64, 32, 192, 8): (13.3, 14.0), (64, 48, 100, 8): (11.2, 13.0), (24, 96, 192, 8): (9.9, 8.5),
}


def test_rule_takes_the_faster_kernel():
    import stratiflow_amd as sf
    if not os.path.exists(sf.LIB_PATH):
        pytest.skip("libsfhip.so not built")
    fit = ctypes.CDLL(sf.LIB_PATH)._ZN2sf14modal_cols_fitEiiiib
    fit.restype = ctypes.c_bool
    fit.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool]
    for step, times in ((True, STAGE), (False, PROJECTION)):
        for (N1, N2, N3, prec), (tiles, columns) in times.items():
            assert fit(N1 // 3, 2 * (N2 // 3) - 1, N3, 2 * prec, step) == (columns < tiles), (step, N1, N2, N3, prec)
        # 2D grids have up to 170 modes: always columns
        for N1, N3, prec in ((6, 8, 4), (256, 512, 8), (512, 512, 4)):
            assert fit(N1 // 3, 1, N3, 2 * prec, step)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(48, 48, 132, 0), (48, 48, 388, 0), (96, 32, 196, 0), (96, 48, 132, 0),
                                   (64, 32, 196, 0), (64, 48, 104, 0), (64, 64, 64, 0), (64, 64, 68, 0), (6, 512, 16, 0)])
def test_both_sides_of_the_lines(shape):
    """Two steps and a projection, in FP64 (the tolerances of the other tests of
    these kernels: FP64 rounding of two steps, p rescaled by 1/h)."""
    from helpers import fields, make_pair, rel_l2
    s, o = make_pair(*shape, gpu_prec=8, amplitude=0.05, seed=11)
    s.TimeStep(2)
    o.step(2)
    s.RemoveDivergence(0.5)
    o.remove_divergence(0.5)
    for f in fields(shape[3]):
        e = rel_l2(s.get(f), o.get_modal(f))
        print(shape, f, "%.2e" % e, flush=True)
        assert e < (1e-9 if f == "p" else 1e-11), f
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("N3", [260, 320, 324, 384])
def test_projection_of_long_columns_fp32(N3):
    """Tiles of five and six rows per lane, whole and ragged, read their
    coefficients by level in the projection and by lane in a stage: FP32 within
    three times the FP32 oracle's own error."""
    from helpers import fields, make_pair, rel_l2
    shape = (96, 64, N3, 0)
    s, o64 = make_pair(*shape, gpu_prec=4, amplitude=0.05, seed=12, project=False)
    _, o32 = make_pair(*shape, gpu_prec=4, oracle_prec=4, amplitude=0.05, seed=12, project=False)
    s.RemoveDivergence(0.5)
    o64.remove_divergence(0.5)
    o32.remove_divergence(0.5)
    for f in fields(shape[3]):
        eg, er = rel_l2(s.get(f), o64.get_modal(f)), rel_l2(o32.get_modal(f), o64.get_modal(f))
        print(shape, f, "%.2e %.2e" % (eg, er), flush=True)
        assert eg <= max(3 * er, 1e-6), f
    s.close()
