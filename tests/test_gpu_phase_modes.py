"""FP64 phase and damping modes of the regular pass, on both sides of |k| (diam_e + diam_f) = 1."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op,space", [("helmholtz_single_layer", "P1"), ("helmholtz_double_layer", "P1"),
                                      ("helmholtz_adjoint_double_layer", "DP0"), ("helmholtz_hypersingular", "P1"),
                                      ("maxwell_electric_field", "RWG")])
@pytest.mark.parametrize("k", [1.0, 1.0 + 0.5j, 0.3 + 1.2j, 6.0, 6.0 + 0.5j, 0.5 + 6.0j])
def test_complex_wavenumbers_vs_oracle(op, space, k, default_parameters, hip_available):
    """Real and damped wavenumbers whose Re k or Im k puts the mesh's pairs in the series mode (the
    factored e^{ik R0}) or beyond it, against the FP64 oracle: the operators' 1e-12 parity bound."""
    import bempp_amd.api.operators.boundary as B
    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from oracle import oracle as O

    grid = icosphere(2)
    dom = function_space(grid, *{"P1": ("P", 1), "DP0": ("DP", 0), "RWG": ("RWG", 0)}[space])
    dual = function_space(grid, "SNC", 0) if space == "RWG" else dom
    limit = 1.0 / (2.0 * grid.diameters.max())
    assert (max(abs(np.real(k)), abs(np.imag(k))) < limit) == (abs(k) < 2)  # one side of the bound or the other
    family, _, name = op.partition("_")
    a = getattr(getattr(B, family), name)(dom, dom, dual, k, parameters=default_parameters,
                                          precision="double").weak_form().A
    ref = O.assemble(op, grid.vertices, grid.elements, dom, dual, k)
    assert np.linalg.norm(a - ref) < 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("op,space", [("helmholtz_single_layer", "P1"), ("helmholtz_adjoint_double_layer", "DP0"),
                                      ("helmholtz_hypersingular", "P1"), ("maxwell_electric_field", "RWG")])
@pytest.mark.parametrize("k", [1.0 - 0.5j, 0.3 - 1.2j, 6.0 - 0.5j, 0.5 - 6.0j])
def test_growing_wavenumbers_vs_oracle(op, space, k, default_parameters, hip_available):
    """Im k < 0: the exponential grows with the distance, in the series mode (the factored e^{ik R0}) and beyond."""
    import bempp_amd.api.operators.boundary as B
    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from oracle import oracle as O

    grid = icosphere(2)
    dom = function_space(grid, *{"P1": ("P", 1), "DP0": ("DP", 0), "RWG": ("RWG", 0)}[space])
    dual = function_space(grid, "SNC", 0) if space == "RWG" else dom
    family, _, name = op.partition("_")
    a = getattr(getattr(B, family), name)(dom, dom, dual, k, parameters=default_parameters,
                                          precision="double").weak_form().A
    ref = O.assemble(op, grid.vertices, grid.elements, dom, dual, k)
    assert np.linalg.norm(a - ref) < 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("space", ["P1", "DP0"])
@pytest.mark.parametrize("k", [1.0, 1.0 + 0.5j, 0.3 + 1.2j, 0.3 - 1.2j, 6.0 + 0.5j, 0.5 + 6.0j])
def test_fused_pass_vs_oracle(space, k, default_parameters, hip_available):
    """Single and double layer assembled together in FP64, on both sides of the series mode's bound."""
    import bempp_amd.api.operators.boundary as B
    from bempp_amd.api import function_space
    from bempp_amd.api.assembly.boundary_operator import assemble_weak_forms
    from bempp_amd.api.grid.shapes import icosphere
    from oracle import oracle as O

    grid = icosphere(2)
    dom = function_space(grid, *{"P1": ("P", 1), "DP0": ("DP", 0)}[space])
    names = ("single_layer", "double_layer")
    forms = assemble_weak_forms([getattr(B.helmholtz, n)(dom, dom, dom, k, parameters=default_parameters,
                                                         precision="double") for n in names])
    for name, form in zip(names, forms):
        ref = O.assemble("helmholtz_" + name, grid.vertices, grid.elements, dom, dom, k)
        assert np.linalg.norm(form.A - ref) < 1e-12 * np.linalg.norm(ref)
