"""Potentials of few points split the sources into chunks of less than a tile; many points do not."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 320 triangles: 1,920 sources, 8 tiles of 256. 32,768 points fill the chip with whole tiles; 1, 255 and 2,049
# points take chunks of 32, 8,193 points of 64, 16,385 points of 128 sources. 20 triangles: 120 sources, less than a tile
@pytest.mark.parametrize("family,name,k", [("laplace", "double_layer", 0.0), ("helmholtz", "single_layer", 2.0),
                                           ("helmholtz", "double_layer", 2.0 + 0.5j),
                                           ("maxwell", "electric_field", 1.5 + 0.2j),
                                           ("maxwell", "magnetic_field", 1.5)])
@pytest.mark.parametrize("level", [0, 2])
def test_few_points_equal_many(family, name, k, level, hip_available):
    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere

    space = bempp.function_space(icosphere(level), *(("RWG", 0) if family == "maxwell" else ("DP", 0)))
    rng = np.random.default_rng(level)
    coefficients = rng.standard_normal(space.global_dof_count) + 1j * rng.standard_normal(space.global_dof_count)
    fun = bempp.GridFunction(space, coefficients=coefficients)
    points = rng.standard_normal((3, 262144 if level == 0 else 32768))
    points *= rng.uniform(1.5, 3.0, points.shape[1]) / np.linalg.norm(points, axis=0)
    make = getattr(getattr(bempp.operators.potential, family), name)

    def evaluate(x):
        options = () if family == "laplace" else (k,)
        return make(space, np.ascontiguousarray(x), *options, precision="double").evaluate(fun)

    many = evaluate(points)
    for count in (1, 255, 2049, 8193, 16385):
        few = evaluate(points[:, :count])
        # the same terms summed in another grouping: about sqrt(1,920) roundings of terms that partly cancel
        assert np.linalg.norm(few - many[:, :count]) < 1e-13 * np.linalg.norm(many[:, :count])


# 1,920 sources: 2,049 points take chunks of 64, 8,193 of 128 sources (electric field); scalar potentials of up
# to 13,107 points (25,165,440 pairs) are evaluated in FP64, 13,108 in FP32
@pytest.mark.parametrize("family,name,k", [("laplace", "double_layer", 0.0), ("helmholtz", "single_layer", 2.0),
                                           ("maxwell", "electric_field", 1.5),
                                           ("maxwell", "magnetic_field", 1.5 + 0.2j)])
@pytest.mark.parametrize("count", [1, 2049, 8193, 13107, 13108])
def test_mixed_against_fp64(family, name, k, count, hip_available):
    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere

    space = bempp.function_space(icosphere(2), *(("RWG", 0) if family == "maxwell" else ("DP", 0)))
    rng = np.random.default_rng(count)
    fun = bempp.GridFunction(space, coefficients=1.0 + rng.random(space.global_dof_count))
    points = rng.standard_normal((3, count))
    points *= rng.uniform(1.5, 3.0, count) / np.linalg.norm(points, axis=0)
    options = () if family == "laplace" else (k,)
    make = getattr(getattr(bempp.operators.potential, family), name)
    single, double = (make(space, points, *options, precision=p).evaluate(fun) for p in ("single", "double"))
    # the mode's stated accuracy; a scalar call in FP64 rounds its output only
    exact = family != "maxwell" and count * 1920 <= 3 << 23
    assert np.linalg.norm(single - double) < (1e-7 if exact else 2e-6) * np.linalg.norm(double)


@pytest.mark.parametrize("precision", ["double", "single"])
def test_workspace_of_the_largest_batch_serves_smaller_ones(precision, hip_available):
    """320 triangles: 24,000 points take more chunks than 32,768, and fit the workspace sized for these."""
    import ctypes

    import torch

    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.api.integration.triangle_gauss import rule as triangle_rule
    from bempp_amd.core import hip_backend as hb

    L = hb.lib()
    space = hb.device_space(bempp.function_space(icosphere(2), "DP", 0))
    rule = hb.quad_rule(*triangle_rule(4))
    mode = hb.PRECISION_FP64 if precision == "double" else hb.PRECISION_MIXED
    size = L.bem_potential_workspace_size(3, ctypes.byref(space.struct), ctypes.byref(rule), 32768, mode)
    work = torch.empty(size, dtype=torch.uint8, device=hb.device())
    c = torch.ones(320, dtype=torch.complex128, device=hb.device())
    points = torch.randn((32768, 3), dtype=torch.float64, device=hb.device())
    points *= 2.0 / torch.linalg.vector_norm(points, dim=1, keepdim=True)
    for count in (32768, 24000, 5000, 1):
        out = torch.empty((1, count), dtype=torch.complex128, device=hb.device())
        hb.check(L.bem_potential_evaluate(3, ctypes.byref(space.struct), hb.ptr(c), count, hb.ptr(points), ctypes.byref(rule),
                                          2.0, 0.0, mode, hb.ptr(out), hb.DTYPES["complex128"], hb.ptr(work), size,
                                          hb.stream_handle()))
        assert torch.isfinite(torch.view_as_real(out)).all()


FP64_PAIRS = 3 << 23  # scalar potentials of up to this many (point, source) pairs are evaluated in FP64 in either mode


def _mixed_error(space, family, name, k, points, seed):
    """Error of the single precision potential of a random density against the double precision one."""
    import bempp_amd.api as bempp

    rng = np.random.default_rng(seed)
    c = rng.standard_normal(space.global_dof_count)
    if family == "helmholtz":
        c = c + 1j * rng.standard_normal(space.global_dof_count)
    fun = bempp.GridFunction(space, coefficients=c)
    make = getattr(getattr(bempp.operators.potential, family), name)
    single, double = (make(space, points, *(() if family == "laplace" else (k,)), precision=p).evaluate(fun)
                      for p in ("single", "double"))
    return np.linalg.norm(single - double) / np.linalg.norm(double)


def _shell(count, low, high, seed=5):
    rng = np.random.default_rng(seed)
    points = rng.standard_normal((3, count))
    return points * rng.uniform(low, high, count) / np.linalg.norm(points, axis=0)


# 320 and 1,280 triangles: every target is close to its tiles of 43 triangles, away from most groups of 5 or 6
@pytest.mark.parametrize("family,name,k", [("laplace", "single_layer", 0.0), ("laplace", "double_layer", 0.0),
                                           ("helmholtz", "single_layer", 1.2), ("helmholtz", "double_layer", 1.2),
                                           ("helmholtz", "single_layer", 1.2 + 0.12j),
                                           ("helmholtz", "double_layer", 1.2 + 0.12j)])
@pytest.mark.parametrize("level,count,low,high", [(2, 13200, 1.5, 3.0), (3, 3300, 1.02, 1.3)])
@pytest.mark.parametrize("kind", ["P", "DP"])
def test_mixed_rounds_the_result_only_close_to_the_mesh(kind, level, count, low, high, family, name, k, hip_available):
    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere

    space = bempp.function_space(icosphere(level), kind, int(kind == "P"))
    sources = 6 * space.grid.number_of_elements
    assert sources * count > FP64_PAIRS
    # the result's rounding to FP32, 2.5e-8 (2^-24 / sqrt 6), and a remainder of some tenths of the sum in FP32
    assert _mixed_error(space, family, name, k, _shell(count, low, high), level) < 4e-8


# 7,680 sources, 30 tiles. k h = 0.07 to 3.5 of a group's radius and beyond: all series of e^{ik delta} - 1, the
# hardware sine, both forms of the damping
@pytest.mark.parametrize("family,k", [("laplace", 0.0)] + [("helmholtz", k) for k in (0.5, 2.0, 5.0, 8.0, 12.0, 30.0, 2.0 + 0.5j,
                                                                                      30.0 + 2.0j, 3.0 + 5.0j, 2.0 - 0.3j)])
@pytest.mark.parametrize("name", ["single_layer", "double_layer"])
@pytest.mark.parametrize("kind", ["P", "DP"])
def test_mixed_scalar_at_every_distance(kind, name, family, k, hip_available):
    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere

    space = bempp.function_space(icosphere(3), kind, int(kind == "P"))
    for low, high in ((0.9, 1.1), (1.02, 1.05), (1.2, 2.5), (6.0, 12.0)):
        points = _shell(3300, low, high)
        assert 7680 * points.shape[1] > FP64_PAIRS
        assert _mixed_error(space, family, name, k, points, 7) < 1e-6  # the mode's stated accuracy


@pytest.mark.parametrize("family,name,k", [("laplace", "double_layer", 0.0), ("helmholtz", "single_layer", 6.0),
                                           ("helmholtz", "double_layer", 4.0 + 0.4j)])
def test_parts_of_a_tile_take_the_paths_of_the_tile(family, name, k, hip_available):
    """30,720 sources: 1,024 points take parts of 128 sources, 9,216 points whole tiles of 256; the sums differ in
    the order of FP64 additions only, so their roundings to FP32 by at most a unit."""
    import bempp_amd.api as bempp
    from bempp_amd.api.grid.shapes import icosphere

    space = bempp.function_space(icosphere(4), "DP", 0)
    rng = np.random.default_rng(3)
    fun = bempp.GridFunction(space, coefficients=rng.standard_normal(space.global_dof_count))
    points = _shell(9216, 1.02, 3.0)
    assert 30720 * 1024 > FP64_PAIRS
    make = getattr(getattr(bempp.operators.potential, family), name)
    many, few = (make(space, np.ascontiguousarray(points[:, :n]), *(() if family == "laplace" else (k,)),
                      precision="single").evaluate(fun) for n in (9216, 1024))
    many = many[:, :1024]
    for a, b in ((few.real, many.real), (few.imag, many.imag)):
        np.testing.assert_array_max_ulp(a.astype(np.float32), b.astype(np.float32), maxulp=1)
