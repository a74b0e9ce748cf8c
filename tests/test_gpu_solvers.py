"""Solves on operators assembled by the HIP path.

* The reference's mixed Dirichlet / Neumann Laplace problem on cube_grid.msh
  (test/validation/computations/test_mixed_neumann_dirichlet_.py): a 2 x 2 blocked system of
  single, double, adjoint double layer and hypersingular operators with the L2 identity,
  right-hand sides projected from callables, GMRES, then the solution on the element centres
  against the reference's golden values (mixed_dirichlet_neumann_sol.npz) at the reference's
  tolerances (rtol 1e-10 double, 6e-4 single).
* Device GMRES / CG / LU against scipy / numpy on the same assembled matrices (host copies).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["double", "single"])
def test_laplace_mixed_neumann_dirichlet(precision, helpers, default_parameters, hip_available):
    import bempp_amd.api as bempp
    from bempp_amd.api.operators.boundary import laplace, sparse

    grid = helpers.load_grid("cube_grid")
    dirichlet_segments = [1, 3]
    neumann_segments = [2, 4, 5, 6]
    fs = bempp.function_space
    global_neumann_space = fs(grid, "DP", 0)
    global_dirichlet_space = fs(grid, "P", 1)
    neumann_space_dirichlet_segment = fs(grid, "DP", 0, segments=dirichlet_segments)
    neumann_space_neumann_segment = fs(grid, "DP", 0, segments=neumann_segments)
    dirichlet_space_dirichlet_segment = fs(grid, "P", 1, segments=dirichlet_segments, include_boundary_dofs=True,
                                           truncate_at_segment_edge=False)
    dirichlet_space_neumann_segment = fs(grid, "P", 1, segments=neumann_segments)
    dual_dirichlet_space = fs(grid, "P", 1, segments=dirichlet_segments, include_boundary_dofs=True)
    kw = dict(parameters=default_parameters, precision=precision)
    slp_DD = laplace.single_layer(neumann_space_dirichlet_segment, dirichlet_space_dirichlet_segment,
                                  neumann_space_dirichlet_segment, **kw)
    dlp_DN = laplace.double_layer(dirichlet_space_neumann_segment, dirichlet_space_dirichlet_segment,
                                  neumann_space_dirichlet_segment, **kw)
    adlp_ND = laplace.adjoint_double_layer(neumann_space_dirichlet_segment, neumann_space_neumann_segment,
                                           dirichlet_space_neumann_segment, **kw)
    hyp_NN = laplace.hypersingular(dirichlet_space_neumann_segment, neumann_space_neumann_segment,
                                   dirichlet_space_neumann_segment, **kw)
    slp_DN = laplace.single_layer(neumann_space_neumann_segment, dirichlet_space_dirichlet_segment,
                                  neumann_space_dirichlet_segment, **kw)
    dlp_DD = laplace.double_layer(dirichlet_space_dirichlet_segment, dirichlet_space_dirichlet_segment,
                                  neumann_space_dirichlet_segment, **kw)
    id_DD = sparse.identity(dirichlet_space_dirichlet_segment, dirichlet_space_dirichlet_segment,
                            neumann_space_dirichlet_segment)
    adlp_NN = laplace.adjoint_double_layer(neumann_space_neumann_segment, neumann_space_neumann_segment,
                                           dirichlet_space_neumann_segment, **kw)
    id_NN = sparse.identity(neumann_space_neumann_segment, neumann_space_neumann_segment,
                            dirichlet_space_neumann_segment)
    hyp_ND = laplace.hypersingular(dirichlet_space_dirichlet_segment, neumann_space_neumann_segment,
                                   dirichlet_space_neumann_segment, **kw)

    blocked = bempp.BlockedOperator(2, 2)
    blocked[0, 0] = slp_DD
    blocked[0, 1] = -dlp_DN
    blocked[1, 0] = adlp_ND
    blocked[1, 1] = hyp_NN

    @bempp.real_callable
    def dirichlet_data(x, n, domain_index, res):
        res[0] = 1

    @bempp.real_callable
    def neumann_data(x, n, domain_index, res):
        res[0] = 1

    dirichlet_grid_fun = bempp.GridFunction(dirichlet_space_dirichlet_segment, fun=dirichlet_data,
                                            dual_space=dual_dirichlet_space)
    neumann_grid_fun = bempp.GridFunction(neumann_space_neumann_segment, fun=neumann_data,
                                          dual_space=dirichlet_space_neumann_segment)
    rhs_fun1 = (0.5 * id_DD + dlp_DD) * dirichlet_grid_fun - slp_DN * neumann_grid_fun
    rhs_fun2 = -hyp_ND * dirichlet_grid_fun + (0.5 * id_NN - adlp_NN) * neumann_grid_fun

    (neumann_solution, dirichlet_solution), info, its = bempp.linalg.gmres(
        blocked, [rhs_fun1, rhs_fun2], return_iteration_count=True)
    assert info == 0

    embed = sparse.identity
    dirichlet = (embed(dirichlet_space_dirichlet_segment, global_dirichlet_space, global_dirichlet_space)
                 * dirichlet_grid_fun
                 + embed(dirichlet_space_neumann_segment, global_dirichlet_space, global_dirichlet_space)
                 * dirichlet_solution)
    neumann = (embed(neumann_space_neumann_segment, global_neumann_space, global_neumann_space) * neumann_grid_fun
               + embed(neumann_space_dirichlet_segment, global_neumann_space, global_neumann_space) * neumann_solution)
    data = helpers.load_npz_data("mixed_dirichlet_neumann_sol")
    actual_dirichlet = dirichlet.evaluate_on_element_centers()
    actual_neumann = neumann.evaluate_on_element_centers()
    tol = helpers.default_tolerance(precision)
    print(f"{precision}: {its} GMRES iterations; max rel err dirichlet "
          f"{np.max(np.abs(actual_dirichlet - data['dirichlet_vals']) / np.abs(data['dirichlet_vals'])):.2e}, "
          f"neumann {np.max(np.abs(actual_neumann - data['neumann_vals']) / np.abs(data['neumann_vals'])):.2e}",
          flush=True)
    np.testing.assert_allclose(actual_dirichlet, data["dirichlet_vals"], rtol=tol)
    np.testing.assert_allclose(actual_neumann, data["neumann_vals"], rtol=tol)


@pytest.fixture(scope="module")
def helmholtz_system():
    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.api.operators.boundary import helmholtz

    grid = icosphere(3)
    p1 = function_space(grid, "P", 1)
    return grid, p1, helmholtz


@pytest.mark.parametrize("precision,restart", [("double", None), ("single", 10)])
def test_gmres_vs_scipy_on_assembled_matrix(precision, restart, helmholtz_system, default_parameters,
                                            hip_available):
    import scipy.sparse.linalg as sla

    import bempp_amd.api as bempp

    grid, p1, helmholtz = helmholtz_system
    op = helmholtz.single_layer(p1, p1, p1, 3.0, parameters=default_parameters, precision=precision)

    @bempp.complex_callable
    def wave(x, n, domain_index, res):
        res[0] = np.exp(3.0j * x[0])

    rhs = bempp.GridFunction(p1, fun=wave)
    sol, info, res, its = bempp.linalg.gmres(op, rhs, tol=1e-8, restart=restart, return_residuals=True,
                                             return_iteration_count=True)
    A = op.weak_form().to_dense()
    b = rhs.projections()
    ref_res = []
    x_ref, info_ref = sla.gmres(A, b, rtol=1e-8, restart=restart, callback=ref_res.append, callback_type="legacy")
    print(f"{precision}: {its} iterations (scipy {len(ref_res)})", flush=True)
    assert info == info_ref == 0
    assert its == len(ref_res) == len(res)
    np.testing.assert_allclose(res, ref_res, rtol=1e-5, atol=1e-12)
    x = sol.coefficients
    # the same Krylov iterate: differences come from the products' rounding (FP64 accumulation
    # on the device, the matrix's dtype in numpy)
    assert np.linalg.norm(x - x_ref) / np.linalg.norm(x_ref) < (1e-9 if precision == "double" else 1e-5)
    assert np.linalg.norm(A.astype(np.complex128) @ x - b) <= 1e-8 * np.linalg.norm(b) * 1.01


def test_cg_and_lu_on_laplace_single_layer(default_parameters, hip_available):
    import scipy.sparse.linalg as sla

    import bempp_amd.api as bempp
    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.api.operators.boundary import laplace

    grid = icosphere(3)
    dp0 = function_space(grid, "DP", 0)
    op = laplace.single_layer(dp0, dp0, dp0, parameters=default_parameters)

    @bempp.real_callable
    def data(x, n, domain_index, res):
        res[0] = x[2] + 0.5 * x[0] * x[1]

    rhs = bempp.GridFunction(dp0, fun=data)
    sol, info, its = bempp.linalg.cg(op, rhs, tol=1e-10, return_iteration_count=True)
    A = op.weak_form().to_dense()
    b = rhs.projections()
    xs = []
    x_ref, info_ref = sla.cg(A, b, rtol=1e-10, callback=xs.append)
    assert info == info_ref == 0 and its == len(xs)
    assert sol.coefficients.dtype == np.float64
    np.testing.assert_allclose(sol.coefficients, x_ref, rtol=1e-8, atol=1e-10 * np.abs(x_ref).max())
    lu_sol = bempp.linalg.lu(op, rhs)
    x_np = np.linalg.solve(A, b)
    np.testing.assert_allclose(lu_sol.coefficients, x_np, rtol=1e-9, atol=1e-12 * np.abs(x_np).max())
    factors = bempp.linalg.compute_lu_factors(op)
    np.testing.assert_allclose(bempp.linalg.lu(op, rhs, lu_factor=factors).coefficients, x_np, rtol=1e-9,
                               atol=1e-12 * np.abs(x_np).max())


@pytest.mark.parametrize("dtype", ["float64", "complex64"])
def test_discrete_operator_products(dtype, default_parameters, hip_available):
    from bempp_amd.api import function_space
    from bempp_amd.api.grid.shapes import icosphere
    from bempp_amd.api.operators.boundary import helmholtz, laplace, sparse

    grid = icosphere(2)
    p1 = function_space(grid, "P", 1)
    if dtype == "float64":
        op = laplace.double_layer(p1, p1, p1, parameters=default_parameters)
    else:
        op = helmholtz.double_layer(p1, p1, p1, 2.0, parameters=default_parameters, precision="single")
    W = op.weak_form()
    A = W.to_dense()
    rng = np.random.default_rng(1)
    x = rng.standard_normal(A.shape[1]) + 1j * rng.standard_normal(A.shape[1])
    np.testing.assert_allclose(W @ x, A.astype(np.complex128) @ x, rtol=1e-12, atol=1e-14)
    xr = rng.standard_normal(A.shape[1])
    y = W @ xr
    assert y.dtype == np.result_type(A.dtype, xr.dtype)
    S = (0.5 * sparse.identity(p1, p1, p1) + op).weak_form()
    M = sparse.identity(p1, p1, p1).weak_form().to_dense()
    np.testing.assert_allclose(S.to_dense(), (0.5 * M + A).astype(S.dtype), rtol=1e-6, atol=1e-12)


@pytest.mark.parametrize("k,n", [(1, 37), (5, 1000), (21, 10242), (40, 200000), (300, 2000)])
def test_gmres_cgs2_entry_point(k, n, hip_available):
    """bem_gmres_cgs2 against the same CGS2 arithmetic in numpy (FP64): the coefficients, both
    norms, the updated vector and the next basis vector (row k of V: w2 / |w2|, or w2 itself when
    the breakdown test |w2| <= eps |w| holds); n past one block, past the 512-block grid cap
    (grid-stride), k past the restart length used elsewhere and past the 256 dot products staged
    per barrier."""
    import torch

    from bempp_amd.core import hip_backend as hb

    rng = np.random.default_rng(k + n)
    V = rng.standard_normal((k + 2, n)) + 1j * rng.standard_normal((k + 2, n))
    V[:k] = np.linalg.qr(V[:k].T)[0].T  # orthonormal rows, as in GMRES
    w = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    c1 = V[:k].conj() @ w
    w1 = w - V[:k].T @ c1
    c2 = V[:k].conj() @ w1
    w2 = w1 - V[:k].T @ c2
    dev = hb.device()
    Vt = torch.as_tensor(V, device=dev)
    wt = torch.as_tensor(w, device=dev)
    out = torch.full((2 * k + 2,), 7.0 + 7.0j, dtype=torch.complex128, device=dev)  # overwritten
    hb.gmres_cgs2(Vt, k, wt, out, Vt[k], 1e-14)
    g = out.cpu().numpy()
    scale = np.linalg.norm(w)
    np.testing.assert_allclose(g[:k], c1, rtol=0, atol=1e-12 * scale)
    np.testing.assert_allclose(g[k + 1 : 2 * k + 1], c2, rtol=0, atol=1e-12 * scale)
    assert abs(g[k].real - np.vdot(w, w).real) <= 1e-12 * scale**2 and g[k].imag == 0.0
    assert abs(g[2 * k + 1].real - np.vdot(w2, w2).real) <= 1e-12 * scale**2
    np.testing.assert_allclose(wt.cpu().numpy(), w2, rtol=0, atol=1e-12 * scale)
    Vh = Vt.cpu().numpy()
    np.testing.assert_allclose(Vh[k], w2 / np.linalg.norm(w2), rtol=0, atol=1e-12)
    # the other rows are untouched
    np.testing.assert_array_equal(Vh[:k], V[:k])
    np.testing.assert_array_equal(Vh[k + 1], V[k + 1])
    # breakdown test (eps so large that it holds): row k + 1 receives w_out unscaled
    w3 = wt.clone()
    hb.gmres_cgs2(Vt, k, w3, out, Vt[k + 1], 1e300)
    np.testing.assert_array_equal(Vt[k + 1].cpu().numpy(), w3.cpu().numpy())



@pytest.mark.parametrize("n", [1, 2, 65, 2047, 2048, 2049])
@pytest.mark.parametrize("dtype", ["float32", "float64", "complex64", "complex128"])
def test_gmres_step_equals_its_parts(n, dtype, hip_available):
    """One call per Arnoldi step (product, CGS2, next basis vector, coefficients on the host) against the same
    step in torch, on both sides of the vector length at which one workgroup does the orthogonalisation."""
    import torch

    from bempp_amd.core import hip_backend as hb

    dev = hb.device()
    torch.manual_seed(n)
    A = torch.randn((n, n), dtype=getattr(torch, dtype), device=dev)
    m = min(n, 4)
    Q = torch.linalg.qr(torch.randn((n, m), dtype=torch.complex128, device=dev))[0].T.contiguous()
    V = torch.zeros((m + 1, n), dtype=torch.complex128, device=dev)
    V[:m] = Q
    buf = 2 * (m + 1)
    out = [torch.empty(buf, dtype=torch.complex128, device=dev) for _ in range(2)]
    host = [torch.empty(buf, dtype=torch.complex128, pin_memory=True) for _ in range(2)]
    step = hb.gmres_stepper(A, V, torch.empty(n, dtype=torch.complex128, device=dev), out, host, 0.0)
    step(m, 1)
    torch.cuda.synchronize()
    w = A.to(torch.complex128) @ Q[m - 1]
    norm = torch.linalg.vector_norm(w)
    c1 = Q.conj() @ w
    w1 = w - Q.T @ c1
    w2 = w1 - Q.T @ (Q.conj() @ w1)
    got = host[1].to(dev)
    # sums of n FP64 products: n eps sqrt-wise; 1e-13 covers n = 2,049
    assert torch.linalg.vector_norm(got[:m] - c1) < 1e-13 * norm
    assert abs(got[m].real.sqrt() - norm) < 1e-13 * norm
    assert abs(got[2 * m + 1].real.sqrt() - torch.linalg.vector_norm(w2)) < 1e-13 * norm
    if n > m:  # else nothing is left of w but rounding
        assert torch.linalg.vector_norm(V[m] - w2 / torch.linalg.vector_norm(w2)) < 1e-12
    assert torch.equal(V[:m], Q)


@pytest.mark.parametrize("rows,cols,ld", [(1, 1, 2), (3, 1001, 1002), (2048, 33, 34), (2049, 70, 72), (5000, 1030, 1032)])
@pytest.mark.parametrize("dtype", ["float32", "float64", "complex64", "complex128"])
def test_product_by_whole_rows(rows, cols, ld, dtype, hip_available):
    """Products whose 32-row tiles would not fill the chip: one or two rows per wavefront, remainders of rows
    and of 16-byte loads (float32 takes rows of a multiple of 4, the others of 2 values)."""
    import torch

    from bempp_amd.core import hip_backend as hb

    torch.manual_seed(rows)
    ld = (ld + 3) // 4 * 4
    A = torch.randn((rows, ld), dtype=getattr(torch, dtype), device=hb.device())[:, :cols]
    x = torch.randn(cols, dtype=torch.complex128, device=hb.device())
    y = hb.dense_matvec(A, x)
    ref = A.to(torch.complex128) @ x
    assert torch.linalg.vector_norm(y - ref) < 1e-14 * cols**0.5 * torch.linalg.vector_norm(ref)


def _delayed_stepper(monkeypatch, cycles):
    """Each library step of GMRES behind `cycles` of device time."""
    import torch

    from bempp_amd.core import hip_backend as hb

    make = hb.gmres_stepper

    def delayed(*args):
        step = make(*args)

        def slow(*args):
            torch.cuda._sleep(cycles)
            step(*args)

        return slow

    monkeypatch.setattr(hb, "gmres_stepper", delayed)


@pytest.mark.parametrize("stop_at", [1, 3])
def test_gmres_left_by_an_exception_waits_for_its_copies(stop_at, monkeypatch, hip_available):
    """A callback that raises leaves while the next step is in flight: its copy into page-locked memory is
    finished before the exception reaches the caller, who frees that memory."""
    import torch

    from bempp_amd.api.linalg.iterative_solvers import device_gmres
    from bempp_amd.core import hip_backend as hb

    _delayed_stepper(monkeypatch, 20_000_000)  # about 10 ms each
    rng = np.random.default_rng(0)
    n, count = 60, 0
    A = torch.from_numpy(np.eye(n) + 0.05 * rng.standard_normal((n, n))).to(hb.device())

    class Stop(Exception):
        pass

    def callback(residual):
        nonlocal count
        count += 1
        if count == stop_at:
            raise Stop

    with pytest.raises(Stop):
        device_gmres(A, rng.standard_normal(n), rtol=1e-12, callback=callback)
    assert torch.cuda.current_stream().query()


def _product_error(A, x):
    """|A x - ref| / |ref| against the FP64 product, the reference by chunks of columns."""
    import torch

    from bempp_amd.core import hip_backend as hb

    ref = sum(A[:, c : c + 50000].to(torch.complex128) @ x[c : c + 50000] for c in range(0, A.shape[1], 50000))
    return (torch.linalg.vector_norm(hb.dense_matvec(A, x) - ref) / torch.linalg.vector_norm(ref)).item()


# tiles of 32 x 1,024: more than 1,023 of them (remainders of rows, columns and 16-byte loads); wide matrices of
# fewer; the last shapes that take whole rows (1,022 tiles; 2 x rows + 256 columns; 32 tiles) and their
# neighbours that do not
@pytest.mark.parametrize("rows,cols", [(6001, 6003), (33, 600001), (64, 20480), (5, 70001), (4672, 7168), (4673, 7168),
                                       (640, 1536), (640, 1537), (256, 4096), (257, 4096), (1024, 1030), (1025, 1030)])
@pytest.mark.parametrize("dtype", ["float32", "float64", "complex64", "complex128"])
def test_product_by_tiles_and_by_rows(rows, cols, dtype, hip_available):
    import torch

    from bempp_amd.core import hip_backend as hb

    torch.manual_seed(rows)
    A = torch.randn((rows, (cols + 7) // 4 * 4), dtype=getattr(torch, dtype), device=hb.device())[:, :cols]
    x = torch.randn(cols, dtype=torch.complex128, device=hb.device())
    # sums of cols FP64 products: rounding grows with the root of their number
    assert _product_error(A, x) < 1e-15 * cols**0.5


def test_product_of_a_wide_matrix_fills_the_chip(hip_available):
    """32 rows x 1,000,000 columns: about twice the time of a copy of the matrix when the columns are shared among
    workgroups, 30 times when every row is one wavefront's."""
    import torch

    from bempp_amd.core import hip_backend as hb

    A = torch.randn((32, 1000000), dtype=torch.complex64, device=hb.device())
    x = torch.randn(1000000, dtype=torch.complex128, device=hb.device())
    B, y = torch.empty_like(A), torch.empty(32, dtype=torch.complex128, device=hb.device())

    def best(f):
        times = []
        for _ in range(6):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            f()
            stop.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(stop))
        return min(times)

    assert best(lambda: hb.dense_matvec(A, x, out=y)) < 8 * best(lambda: B.copy_(A))
    assert _product_error(A, x) < 1e-15 * 1000000**0.5


def test_gmres_callback_may_change_the_stream(monkeypatch, hip_available):
    """A callback that finishes the work of one stream and makes another current: later steps run on the new
    stream, and the host reads their coefficients only after they have arrived."""
    import torch

    from bempp_amd.api.linalg.iterative_solvers import device_gmres
    from bempp_amd.core import hip_backend as hb

    rng = np.random.default_rng(1)
    n = 60
    A = torch.from_numpy(np.eye(n) + 0.05 * rng.standard_normal((n, n))).to(hb.device())
    b = rng.standard_normal(n)
    expected, _ = device_gmres(A, b, rtol=1e-10)
    _delayed_stepper(monkeypatch, 2_000_000)
    first, other, calls = torch.cuda.current_stream(), torch.cuda.Stream(), 0

    def callback(residual):
        nonlocal calls
        calls += 1
        if calls == 2:
            torch.cuda.synchronize()
            torch.cuda.set_stream(other)

    try:
        x, info = device_gmres(A, b, rtol=1e-10, callback=callback)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_stream(first)
    assert info == 0 and calls > 4
    # the same arithmetic: atomics of the product may reorder a row's sums, times the condition (below 100)
    assert torch.linalg.vector_norm(x - expected) < 1e-12 * torch.linalg.vector_norm(expected)
