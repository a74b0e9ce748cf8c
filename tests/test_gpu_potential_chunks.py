"""Potentials of few points split the sources into chunks of less than a tile; many points do not."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 320 triangles: 1,920 sources, 8 tiles of 256. 32,768 points fill the chip with whole tiles; 1 and 255 points
# take chunks of 32, 2,049 points of 64, 16,385 points of 128 sources. 20 triangles: 120 sources, less than a tile
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
    for count in (1, 255, 2049, 16385):
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
