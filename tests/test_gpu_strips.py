"""The blurred-L pool's strips and the SYRK over them, at the sizes where strips, column blocks, chunks
and the tap table end: chunks that span two ends of an image row (thin masks and images), PSFs of one pixel
to wider than the padded tap table takes, partly reached source grids of various sizes, and more chunks than
one list holds (test_strips_match_oracle); whole source grids whose data column opens a strip or a column
block of its own or closes one (test_data_column_at_every_edge); against the oracle, FP64 and mixed."""
import numpy as np
import pytest

from oracle import oracle as O
from qlens_amd import qlx
from qlens_amd import workloads as W

TOL = 1e-9         # FP64: the oracle's sums in another order
TOL_MIXED = 0.1    # |delta ln E| of the mixed path's contract
TOL_SRC = 2e-3     # mixed path's source: both factors of F and D hold entries rounded to 11 bits (2^-11 each),
                   # and twice that for a regularized solve, which damps more than it amplifies


def _psf(n, m):
    x, y = np.arange(n) - n // 2, np.arange(m) - m // 2
    p = np.exp(-0.5 * ((x[:, None] / (0.25 * n)) ** 2 + (y[None, :] / (0.25 * m)) ** 2))
    return p / p.sum()


def _thin(nx, ny):
    m = np.zeros((nx, ny), np.uint8)
    m[::3] = 1       # every third column of pixels: chunks of many image tiles
    m[:, :5] = 1
    m[:, -4:] = 1
    return m


CASES = [
    # nx, ny, nsplit, source grid, psf, mask
    (40, 44, 2, (15, 1 + 16), (1, 1), None),
    (40, 44, 2, (8, 16), (3, 5), "thin"),
    (61, 37, 1, (12, 10), (9, 3), "thin"),
    (50, 50, 2, (23, 23), (61, 61), None),   # no padded tap table in FP64
    (60, 50, 2, (16, 16), (65, 65), None),   # none in either precision
    (36, 220, 0, (31, 9), (5, 5), None),
    (200, 190, 0, (17, 13), (3, 3), None),   # over 512 chunks: more than one list
]


def _case(nx, ny, nsplit, src_n, psf, mask):
    xv, yv = W.corners(-2.2, 2.2, nx), W.corners(-2.0, 2.0, ny)
    base = W.c1()
    return dict(name="strips", xvals=xv, yvals=yv, nsplit=nsplit, lenses=base["lenses"], sources=base["sources"],
                psf=_psf(*psf), sigma=0.02, seed=3, srcgrid=(-2.4, 2.4, -2.3, 2.3), src_n=src_n, regparam=50.0, integral_tol=1e-6,
                mask=_thin(nx, ny) if mask else None)


@pytest.mark.gpu
@pytest.mark.parametrize("args", CASES)
@pytest.mark.parametrize("precision", [qlx.QLX_PREC_FP64, qlx.QLX_PREC_MIXED])
def test_strips_match_oracle(qlx_ctx, args, precision):
    case = _case(*args)
    data = O.mock_image(case)
    ref, arr = O.invert(case, data)
    qlx_ctx.load_workload(case, data, precision=precision)
    r = qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]
    assert r["status"] == 0 and (r["n_src_active"], r["n_img_active"]) == (ref["n_src"], ref["n_img"])
    if precision == qlx.QLX_PREC_MIXED:
        assert abs(r["minus2lnE"] - ref["minus2lnE"]) / 2 < TOL_MIXED
        return
    for k in ("minus2lnE", "chisq0", "logdetF", "logdetR"):
        assert abs(r[k] - ref[k]) <= TOL * max(1.0, abs(ref[k])), k
    src = qlx_ctx.get_source()["src"]
    assert np.linalg.norm(src - arr["src"]) <= TOL * np.linalg.norm(arr["src"])


@pytest.mark.gpu
@pytest.mark.parametrize("src_n,thin", [((4, 4), False), ((8, 8), False), ((16, 8), False), ((17, 15), False), ((16, 16), False),
                                        ((24, 16), False), ((20, 20), True)])
@pytest.mark.parametrize("precision", [qlx.QLX_PREC_FP64, qlx.QLX_PREC_MIXED])
def test_data_column_at_every_edge(qlx_ctx, src_n, thin, precision):
    """n_src a multiple of 16, 64, 128 and 256 and one less: a strip, a column block and a padded system that
    hold the data column alone, or that it fills; up to four column blocks of the mixed path."""
    case = W.c1()
    case["src_n"] = src_n
    case["mask"] = _thin(100, 100) if thin else None
    data = O.mock_image(case)
    ref, arr = O.invert(case, data)
    qlx_ctx.load_workload(case, data, precision=precision)
    r = qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]
    assert r["status"] == 0 and r["n_src_active"] == ref["n_src"] == src_n[0] * src_n[1]
    err = np.linalg.norm(qlx_ctx.get_source()["src"] - arr["src"]) / np.linalg.norm(arr["src"])
    if precision == qlx.QLX_PREC_MIXED:
        assert abs(r["minus2lnE"] - ref["minus2lnE"]) / 2 < TOL_MIXED and err <= TOL_SRC
        return
    for k in ("minus2lnE", "chisq0", "logdetF", "logdetR"):
        assert abs(r[k] - ref[k]) <= TOL * max(1.0, abs(ref[k])), k
    assert err <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("thin,psf,precision", [(False, 121, qlx.QLX_PREC_MIXED), (True, 121, qlx.QLX_PREC_MIXED), (True, 89, qlx.QLX_PREC_FP64)])
def test_chunk_support_costs_less_than_the_pool(qlx_ctx, thin, psf, precision):
    """Finding the columns that a chunk reaches looks at each pixel of its reach once; the pool's build
    multiplies each of that pixel's entries for 64 rows.  So the stage ahead of the build (L's rows and
    columns, the supports) takes less time than the build also where large PSFs meet chunks of many image
    tiles."""
    case = _case(200, 200, 2, (60, 60), (psf, psf), "thin" if thin else None)
    case["srcgrid"] = (-0.7, 0.7, -0.7, 0.7)
    qlx_ctx.load_workload(case, np.ones((200, 200)), precision=precision)
    ahead, build = [], []
    for _ in range(6):
        assert qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]["n_src_active"] > 3000  # of 3600
        build.append(qlx_ctx.kernel_time("lbkernel")[0])
        ahead.append(qlx_ctx.kernel_time("lbuild")[0] - build[-1])
    assert min(ahead) < min(build), (min(ahead), min(build))


@pytest.mark.gpu
@pytest.mark.parametrize("src_n", [(5, 3), (9, 9), (20, 14)])
def test_executed_flops_are_those_of_the_products(qlx_ctx, src_n):
    """A PSF wider than the image: every chunk holds every strip (the last one with the data column), so the
    products are known: FP64 multiplies the lower pairs, the mixed kernel each strip against four column
    strips from the strip's own block of 64 columns down."""
    case = _case(40, 44, 2, src_n, (89, 89), None)
    case["srcgrid"] = (-0.7, 0.7, -0.7, 0.7)
    n = src_n[0] * src_n[1]
    strips = n // 16 + 1
    pairs = {qlx.QLX_PREC_FP64: strips * (strips + 1) // 2,
             qlx.QLX_PREC_MIXED: 4 * sum(strips - h for h in range(0, strips, 4))}
    for precision, want in pairs.items():
        qlx_ctx.load_workload(case, np.ones((40, 44)), precision=precision)
        r = qlx_ctx.invert_image_surface_brightness_map(case["lenses"])[0]
        st = qlx.get_stats(qlx_ctx)
        assert r["n_src_active"] == n
        assert st["syrk_exec_flops"] == want * st["rows_pad"] // 64 * 2 * 64 * 16 * 16
