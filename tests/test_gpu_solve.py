"""The triangular solves by panels of 256 rows, at the sizes where panels end (one panel, an edge, a
remainder, several): a launch per panel (few items) against the oracle, and against one workgroup per item
(many items), which does the same arithmetic and so has to give the same bits; FP64, and FP32 with its
refinement."""
import numpy as np
import pytest

from oracle import oracle as O
from qlens_amd import qlx
from qlens_amd import workloads as W

TOL = 1e-9          # FP64: the oracle's sums in another order
TOL_MIXED = 1e-4    # mixed: refined to an FP64 residual of 1e-10 of the right side, on systems of condition below 1e6,
                    # formed from entries rounded to 11 bits (2^-11, averaged over the rows that a cell is seen in)


@pytest.mark.gpu
@pytest.mark.parametrize("src_n", [(5, 4), (14, 9), (16, 16), (17, 15), (20, 18), (26, 24), (30, 29)])
@pytest.mark.parametrize("precision", [qlx.QLX_PREC_FP64, qlx.QLX_PREC_MIXED])
def test_panel_solves(qlx_ctx, src_n, precision):
    case = W.c1()
    case["src_n"] = src_n
    data = O.mock_image(case)
    _, arr = O.invert(case, data)
    qlx_ctx.load_workload(case, data, precision=precision)
    models = [case["lenses"]] + W.proposals(case, 99, 3)
    one = qlx_ctx.invert_image_surface_brightness_map(models[0])[0]
    src1 = qlx_ctx.get_source()["src"]
    tol = TOL_MIXED if precision == qlx.QLX_PREC_MIXED else TOL
    assert one["status"] == 0
    assert np.linalg.norm(src1 - arr["src"]) <= tol * np.linalg.norm(arr["src"])
    many = qlx_ctx.invert_image_surface_brightness_map(models)
    for k in ("minus2lnE", "chisq0", "Es"):
        assert one[k] == many[0][k], k
    assert np.array_equal(qlx_ctx.get_source(0)["src"], src1)


@pytest.mark.gpu
@pytest.mark.parametrize("lam,steps", [(1e3, 1), (0.1, 2)])
def test_refinement_of_large_systems(qlx_ctx, lam, steps):
    """Above 8192 columns every refinement step goes by panels, and none is launched once the items are done:
    forty more allowed steps take no time (two launches of at least a microsecond per panel and step would
    take over 2.5 ms) and change nothing.  The evidence stays within the mixed path's contract of FP64, and an
    item's bits do not depend on its neighbours."""
    case = W.c1()
    case.update(xvals=W.corners(-2.5, 2.5, 240), yvals=W.corners(-2.5, 2.5, 240), src_n=(92, 90), regparam=lam)
    data = O.mock_image(case)
    qlx_ctx.load_workload(case, data)
    ref = qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]
    assert ref["n_src_active"] > 8192
    qlx_ctx.load_workload(case, data, precision=qlx.QLX_PREC_MIXED)
    got, ms = [], []
    for iters in (6, 46):
        qlx_ctx.set_settings(case["nsplit"], case["srcgrid"], case["src_n"], lam, case["integral_tol"],
                             precision=qlx.QLX_PREC_MIXED, refine_iters=iters)
        t = []
        for _ in range(4):
            r = qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]
            t.append(qlx_ctx.kernel_time("solve")[0])
        got.append(r)
        ms.append(min(t))
    assert got[0] == got[1] and got[0]["status"] == 0
    assert got[0]["refine_steps"] >= steps and got[0]["refine_resid"] <= 1e-10
    assert abs(got[0]["minus2lnE"] - ref["minus2lnE"]) / 2 < 0.1
    assert ms[1] - ms[0] < 1.0, ms
    many = qlx_ctx.invert_image_surface_brightness_map([case["lenses"]] + W.proposals(case, 2, 5))
    assert many[0] == got[0]
