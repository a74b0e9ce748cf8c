"""The singular kernel's grouping of pairs: workgroups take consecutive pairs of the table, a wave's pairs
may follow several rules, and the split of a pair's points depends on the number of pairs."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 3, 63 and 3,071 pairs: the smallest launches and their last workgroup (4 pairs, remainder 3); 3,072 to
# 4,607 and 4,608 to 10,239 (Laplace 16,383): 8 pairs per workgroup, whole parts and chunks of points; 10,241:
# 16 pairs, remainder 1; 49,153 (electric field) and 131,073: one lane per pair (64 pairs, remainder 1). Order 2:
# up to 96 points a pair, less than one chunk; order 5: 3,750, several chunks of 64, 128 and 384 points
@pytest.mark.parametrize("op,space,k", [("laplace_single_layer", "P1", 0.0), ("helmholtz_double_layer", "DP0", 2.0),
                                        ("helmholtz_hypersingular", "P1", 2.0 + 0.3j),
                                        ("maxwell_electric_field", "RWG", 3.0)])
@pytest.mark.parametrize("count,order", [(c, 2) for c in (3, 63, 3071, 3072, 4095, 4096, 4607, 4608, 10239, 10241, 15777, 16383,
                                                          16385, 49153, 131073)] +
                         [(c, 5) for c in (65, 3073, 4609, 10241, 16385, 49153, 131073)])
def test_singular_pairs_in_any_order(op, space, k, count, order, hip_available):
    """A table of `count` pairs gives the same sum whether the pairs of one rule stand together (every
    wave reads one set of points) or the table is shuffled (every wave runs many rules)."""
    import torch

    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.core import hip_backend as hb
    from bempp_amd.core.singular_assembler import singular_rule

    grid = icosphere(3 if count <= 15777 else 5)
    sp = function_space(grid, *{"P1": ("P", 1), "DP0": ("DP", 0), "RWG": ("RWG", 0)}[space])
    rule = singular_rule(grid, order, sp.support, sp.support)
    rng = np.random.default_rng(count)
    chosen = np.sort(rng.permutation(len(rule.host.pairs))[:count])
    complex_op = not op.startswith("laplace")
    results = []
    for order in (chosen, rng.permutation(chosen)):
        pairs = torch.from_numpy(np.ascontiguousarray(rule.host.pairs[order])).to(hb.device())
        out = torch.zeros((sp.global_dof_count,) * 2, dtype=torch.complex128 if complex_op else torch.float64,
                          device=hb.device())
        hb.singular_assemble(op, hb.device_space(sp), hb.device_space(sp), pairs, rule.test_points, rule.trial_points,
                             rule.weights, k, out)
        results.append(out)
    assert torch.linalg.norm(results[0]) > 0
    # the same FP64 terms in another order of the atomics: a few roundings per entry
    assert torch.linalg.norm(results[0] - results[1]) < 1e-14 * torch.linalg.norm(results[0])


@pytest.mark.parametrize("op,space,count", [("laplace_single_layer", "DP0", 500), ("helmholtz_double_layer", "P1", 3500),
                                            ("maxwell_electric_field", "RWG", 12000)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_point_tables_of_any_double_alignment(op, space, count, shuffled, hip_available):
    """The points of the rules may start at any double, not only at a multiple of 16 bytes."""
    import torch

    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.core import hip_backend as hb
    from bempp_amd.core.singular_assembler import singular_rule

    sp = function_space(icosphere(3), *{"P1": ("P", 1), "DP0": ("DP", 0), "RWG": ("RWG", 0)}[space])
    rule = singular_rule(sp.grid, 4, sp.support, sp.support)
    pairs = rule.pairs[torch.randperm(count, generator=torch.Generator().manual_seed(1)) if shuffled else slice(count)]
    pairs = pairs.contiguous()

    def shifted(table):
        out = torch.empty(table.numel() + 1, dtype=torch.float64, device=table.device)[1:]
        return out.copy_(table.reshape(-1))

    results = []
    for points in ((rule.test_points, rule.trial_points), (shifted(rule.test_points), shifted(rule.trial_points))):
        out = torch.zeros((sp.global_dof_count,) * 2, dtype=torch.complex128 if "laplace" not in op else torch.float64,
                          device=hb.device())
        ds = hb.device_space(sp)
        hb.singular_assemble(op, ds, ds, pairs, *points, rule.weights, 2.0, out)
        results.append(out)
    assert points[0].data_ptr() % 16 == 8
    # the same terms, only the order of the atomics may differ
    assert torch.linalg.norm(results[0] - results[1]) < 1e-14 * torch.linalg.norm(results[0])
