"""API behaviour that needs no GPU: descriptors, argument checks and error classes
(test/unit/operators/test_boundary_operators.py:117-147)."""

import numpy as np
import pytest


def test_descriptor_fields(sphere_grid):
    from bempp_amd.api import function_space
    from bempp_amd.api.operators.boundary import helmholtz

    sp = function_space(sphere_grid, "P", 1)
    op = helmholtz.single_layer(sp, sp, sp, 2.5 + 1j)
    d = op.descriptor
    assert d.options == [2.5, 1.0] and d.kernel_type == "helmholtz_single_layer"
    assert d.assembly_type == "default_scalar" and d.is_complex and d.precision == "double"


def test_efie_space_checks(sphere_grid):
    from bempp_amd.api import function_space
    from bempp_amd.api.operators.boundary.maxwell import electric_field

    rwg = function_space(sphere_grid, "RWG", 0)
    snc = function_space(sphere_grid, "SNC", 0)
    p1 = function_space(sphere_grid, "P", 1)
    with pytest.raises(ValueError):
        electric_field(p1, rwg, snc, 1.0)
    with pytest.raises(ValueError):
        electric_field(rwg, rwg, rwg, 1.0)


def test_unknown_interface_and_assembler(sphere_grid):
    from bempp_amd.api import function_space
    from bempp_amd.api.operators.boundary import laplace

    sp = function_space(sphere_grid, "DP", 0)
    with pytest.raises(ValueError):
        laplace.single_layer(sp, sp, sp, device_interface="numba").weak_form()
    with pytest.raises(ValueError):
        laplace.single_layer(sp, sp, sp, assembler="fmm")
    with pytest.raises(ValueError):
        laplace.single_layer(sp, sp, sp, precision="half")


def test_modified_helmholtz_rejected(sphere_grid):
    from bempp_amd.api import function_space
    from bempp_amd.api.operators.boundary import helmholtz

    sp = function_space(sphere_grid, "DP", 0)
    with pytest.raises(ValueError):
        helmholtz.single_layer(sp, sp, sp, 1j)


def test_unknown_space(sphere_grid):
    from bempp_amd.api import function_space

    with pytest.raises(ValueError):
        function_space(sphere_grid, "DUAL", 0)


def test_singular_pair_arrays(sphere_grid):
    """Pair offsets point at the remapped rule blocks (singular_assembler.py:322-448)."""
    from bempp_amd.api import function_space
    from bempp_amd.core.singular_assembler import singular_rule

    sp = function_space(sphere_grid, "DP", 0)
    r = singular_rule(sphere_grid, 4, sp.support, sp.support, on_device=False)
    n = 6 * 4**4, 5 * 4**4, 2 * 4**4
    assert r.counts == {"coincident": 230, "edge_adjacent": 690, "vertex_adjacent": r.counts["vertex_adjacent"]}
    p = r.pairs
    assert np.all(p[:230, 5] == n[0]) and np.all(p[230:920, 5] == n[1]) and np.all(p[920:, 5] == n[2])
    assert np.all(p[:, 2] + p[:, 5] <= r.test_points.shape[1])
    assert np.all(p[:, 4] + p[:, 5] <= len(r.weights))
    # the remapped test points of an edge pair lie on the shared edge when the Duffy parameter hits it
    el = sphere_grid.elements
    ea = sphere_grid.edge_adjacency[:, 0]
    assert el[ea[2], ea[0]] == el[ea[4], ea[1]]


def test_benchmark_line_is_short():
    """The benchmark's line: the contract's keys, under 2,000 characters whatever the record holds."""
    import importlib.util
    import json
    import os

    spec = importlib.util.spec_from_file_location("bench", os.path.join(os.path.dirname(__file__), "..", "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    roofline = {"kernel": "k" * 80, "bound": "valu", "achieved": 75.4900442540644, "peak": 157.3, "unit": "TFLOP/s",
                "frac": 0.479911279428254, "traffic": 7275989813.3333, "traffic_record": {"measured_at_commit": "0" * 40}}
    cpu = {"value": 3881374.3029187405, "unit": "matrix entries/s", "cores": 16, "kind": "port", "how": "h" * 200}
    errors = {"helmholtz_single_layer": 1.0572978997602936e-07, "helmholtz_double_layer": 1.2901930099823879e-07}
    part = {"workload": "w" * 200, "entries_per_s": 16838712594.886068, "evals_per_s": 11812088.588358318,
            "ms": 1.0 / 3.0, "rel_err_vs_fp64": 2.0 / 3e7, "rel_err_vs_oracle": 2.0 / 3e15, "max_rel_err_vs_fp64": 2.0 / 3e7,
            "forward_s": 0.08611553999999444, "backward_s": 0.15687844300000364, "backward_over_forward": 1.8217204815764236,
            "grad_vertices_rel_err_vs_fp64": 6.507629797871003e-08, "roofline": roofline, "roofline_backward": roofline,
            "cpu_baseline": cpu}
    result = {"metric": "BEM matrix entries/s at ≤1e-6 rel err vs FP64 (mixed vs FP64 GPU); fwd+bwd s",
              "value": 11841807764.189985, "unit": "matrix entries/s", "n_gpus": 1, "steps": 5, "warmup": 1,
              "ms_per_step": 17.716646999998886, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
              "dtype": "f32+f64", "data": "synthetic", "speedup_vs_fp64": 2.8609456970050497,
              "fp64_entries_per_s": 4139123569.0304976, "rel_err_vs_fp64": errors, "roofline": roofline,
              "cpu_baseline": cpu, "c1": part, "potential": part, "frequency_sweep": part,
              "efie": dict(part, potential=part), "adjoint": part,
              "config": {"workload": "w" * 180, "triangles": 20480, "dofs": 10242, "wavenumber": 4.0, "quadrature": "q" * 60}}
    result["configs"] = bench.config_summary(result)
    line = json.dumps(bench.result_line(result))
    assert len(line) < 2000
    back = json.loads(line)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data"):
        assert back[key] == result[key]
    assert back["config"]["workload"] == result["config"]["workload"]
    assert set(back["configs"]) == {"C1", "C2_potential", "C3", "C4", "C4_potential", "C5"}
    assert back["roofline"]["bound"] == "valu" and back["roofline"]["frac"] == 0.4799
