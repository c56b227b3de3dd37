"""Kernels at the sizes where their launch shape or staging can go wrong:
patches below and above the rounds a workgroup holds in registers, sources of
every word alignment, empty owned sets, meshes of one to a few patches. Each
against a plain FP64 restatement."""
import numpy as np
import pytest

from rxmesh_amd import meshgen as mg

pytestmark = pytest.mark.gpu


def _mesh(V, F, patch_size):
    import rxmesh_amd as rx
    import torch
    m = rx.Mesh(F, patch_size=patch_size)
    x = torch.from_numpy(np.ascontiguousarray(V[m.array("v_l2g")].T.astype(np.float32))).cuda()
    return m, x


def _cg64(rp, col, val, b, x, diag, iters):
    """`iters` (preconditioned) CG iterations on the CSR system, FP64."""
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))

    def prod(v):
        y = np.zeros_like(v)
        np.add.at(y, rows, val[:, None] * v[col])
        return y
    x = x.copy()
    r = b - prod(x)
    z = r / diag
    p, delta = z.copy(), (r * z).sum()
    for _ in range(iters):
        s = prod(p)
        a = delta / (p * s).sum()
        x += a * p
        r -= a * s
        z = r / diag
        new = (r * z).sum()
        p, delta = z + (new / delta) * p, new
    return x


@pytest.mark.parametrize("patch_size", [16, 64, 512, 2048])
@pytest.mark.parametrize("mis", [0, 1, 2, 3])
def test_cg_patch_sizes_and_alignment(patch_size, mis):
    """Both implicit solves, six iterations, against the FP64 CG on the same
    fp32 system; the value array starts at every word of a 16-byte line.
    Tolerance 1e-5 of the largest coordinate, the forward error the solves
    keep at dt = 1e-2."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(4, seed=3, sigma=0.01), seed=3)
    m, x = _mesh(V, F, patch_size)
    dt, iters = 1e-2, 6
    nnz = m.cot_nnz()
    val = torch.empty(nnz + 4, dtype=torch.float32, device="cuda")[mis:mis + nnz]
    A = m.cot_assemble(x, dt, out=(torch.empty(m.nV + 1, dtype=torch.int32, device="cuda"),
                                   torch.empty(nnz, dtype=torch.int32, device="cuda"), val,
                                   torch.empty(m.nV, dtype=torch.float32, device="cuda")))
    rp, col, v64, mass = (t.cpu().numpy() for t in A)
    v64, x64 = v64.astype(np.float64), x.cpu().numpy().T.astype(np.float64)
    b = mass.astype(np.float64)[:, None] * x64
    X, it, _, _ = m.mcf_implicit_cg(A, x, max_iter=iters, abs_tol=0.0)
    ref = _cg64(rp, col, v64, b, x64, np.ones((m.nV, 1)), iters)
    assert it == iters
    assert np.abs(X.cpu().numpy().T - ref).max() <= 1e-5 * np.abs(ref).max()
    Y, it, _, _ = m.mcf_matfree_cg(x, x, dt, precond=True, max_iter=iters, abs_tol=0.0)
    ref = _cg64(rp, col, v64, b, x64, v64[rp[:-1]][:, None], iters)
    assert it == iters
    assert np.abs(Y.cpu().numpy().T - ref).max() <= 1e-5 * np.abs(ref).max()


def test_cg_stops_inside_and_after_the_loop():
    """A relative tolerance met by the last iteration allowed, by an earlier
    one, and by the start itself: the solution and the counts are those of the
    same number of unconditional iterations."""
    import torch
    V, F = mg.icosphere(4, seed=1, sigma=0.01)
    m, x = _mesh(V, F, 128)
    A = m.cot_assemble(x, 1e-2)
    full = [m.mcf_implicit_cg(A, x, max_iter=k, abs_tol=0.0) for k in range(1, 7)]
    start = full[0][2]
    for k in range(1, 6):
        tol = 1.001 * full[k - 1][3] / start  # met by the k-th update
        assert all(f[3] / start >= tol for f in full[:k - 1])
        for limit in (k, k + 3):
            X, it, r0, r1 = m.mcf_implicit_cg(A, x, max_iter=limit, abs_tol=0.0, rel_tol=tol)
            assert it == k - 1 and r0 == start and r1 == full[k - 1][3]
            assert torch.equal(X, full[k - 1][0])
    X, it, r0, r1 = m.mcf_implicit_cg(A, x, max_iter=3, abs_tol=2.0 * start)
    assert it == 0 and r1 == start and torch.equal(X, x)


def _dirichlet_grad64(x, fv, rest):
    """Gradient of sum A |J|^2 (1 + 1 / det(J^T J)) by FP64 autograd; x (V, 3), rest (4, F) m00 m10 m01 m11."""
    import torch
    x = torch.from_numpy(x).requires_grad_(True)
    f = torch.from_numpy(fv.astype(np.int64))
    m00, m10, m01, m11 = torch.from_numpy(rest)
    det = m00 * m11 - m01 * m10
    e1, e2 = x[f[:, 1]] - x[f[:, 0]], x[f[:, 2]] - x[f[:, 0]]
    j0 = e1 * (m11 / det)[:, None] - e2 * (m10 / det)[:, None]
    j1 = -e1 * (m01 / det)[:, None] + e2 * (m00 / det)[:, None]
    a, b, c = (j0 * j0).sum(1), (j1 * j1).sum(1), (j0 * j1).sum(1)
    (0.5 * det * (a + b) * (1 + 1 / (a * b - c * c))).sum().backward()
    return x.grad.numpy()


@pytest.mark.parametrize("patch_size", [16, 256, 512, 1024, 4096])
def test_symdir3_patch_sizes(patch_size):
    """The gradient and the step over patches from a few faces to more than a
    workgroup's registers and (4096) LDS hold, every workgroup size: the same
    bits, and within 1e-5 of the largest entry of the FP64 gradient (the bound
    the gradient keeps elsewhere)."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(5, seed=4, sigma=0.01), seed=4)
    m, x = _mesh(V, F, patch_size)
    Mr = m.symdir_rest(x)
    y = (x * 1.1 + 0.01 * torch.sin(5.0 * x.flip(0))).contiguous()
    g = m.symdir3_grad(Mr, y)
    step = m.symdir3_grad_step(Mr, y, 1e-3)
    for threads in (128, 256, 512):
        m.set_launch_threads(1, threads)
        for queue in (0, 1):
            m.set_launch_threads(2, queue)
            assert torch.equal(step, m.symdir3_grad_step(Mr, y, 1e-3))
    l2g, f_l2g = m.array("v_l2g"), m.array("f_l2g")
    yg = np.empty((m.nV, 3))
    yg[l2g] = y.cpu().numpy().T
    rest = np.empty((4, m.nF))
    rest[:, f_l2g] = Mr.cpu().numpy()
    ref = _dirichlet_grad64(yg, F, rest)[l2g].T
    assert np.abs(g.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    assert torch.allclose(step, y - 1e-3 * g, rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("shape", ["sphere", "grid", "tiny"])
@pytest.mark.parametrize("patch_size", [16, 256, 512, 1024, 4096])
def test_multi_step_smoothing_equals_single_steps(shape, patch_size):
    """Smoothing over the device-built ring plan (every number of steps per
    launch, and the automatic choice after build_vv_plan) gives the bits of
    single steps, whose values other tests check against FP64; patches of 4096
    faces are beyond the plan kernel's tables and take the host walk."""
    import torch
    V, F = {"sphere": lambda: mg.permute_mesh(*mg.icosphere(5, seed=6, sigma=0.01), seed=6),
            "grid": lambda: mg.grid(67, seed=6), "tiny": lambda: mg.icosphere(1, seed=6, sigma=0.01)}[shape]()
    m, x = _mesh(V, F, patch_size)
    m.set_launch_threads(8, 0)
    ref = {k: m.smooth(x, 0.5, k) for k in range(1, 8)}
    n, xn = _mesh(V, F, patch_size)
    assert torch.equal(x, xn)
    n.build_vv_plan()
    for k in ref:
        assert torch.equal(n.smooth(x, 0.5, k), ref[k])
    for steps in range(1, 7):
        for threads in (64, 128, 256, 512):
            m.set_launch_threads(0, threads)
            m.set_launch_threads(8, steps)
            assert torch.equal(m.smooth(x, 0.5, 7), ref[7])


def _arap64(V, F, P, X, w):
    """Covariances, best proper rotations (SVD), energy and gradient; w per (i, j) pair with i the larger id."""
    e = np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]).astype(np.int64), 1), axis=0)
    i, j = e[:, 1], e[:, 0]
    dp, dx = P[i] - P[j], X[i] - X[j]
    wt = np.array([w[(a, b)] for a, b in zip(i, j)])
    S = np.zeros((len(V), 3, 3))
    t = wt[:, None, None] * dp[:, :, None] * dx[:, None, :]
    np.add.at(S, i, t)
    np.add.at(S, j, t)
    u, s, vt = np.linalg.svd(S)
    sign = np.sign(np.linalg.det(np.swapaxes(vt, 1, 2) @ np.swapaxes(u, 1, 2)))
    gap = s[:, 1] + sign * s[:, 2]
    u[:, :, 2] *= sign[:, None]
    R = np.swapaxes(vt, 1, 2) @ np.swapaxes(u, 1, 2)
    return R, gap > 1e-2 * s[:, 0], (i, j, wt, dp, dx)


@pytest.mark.parametrize("patch_size", [16, 512, 2048])
@pytest.mark.parametrize("mirror", [False, True])
def test_arap_patch_sizes(patch_size, mirror):
    """Rotations, energy and gradient against FP64 over patches from a few
    faces to more than the register rounds; mirrored poses have negative
    determinants everywhere. Tolerances of the other ARAP tests: 1e-4 per
    entry where the covariance fixes R, 1e-5 of the energy, 1e-4 of the
    largest gradient entry."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(4, seed=7, sigma=0.02), seed=7)
    m, x = _mesh(V, F, patch_size)
    pose = (x + 0.3 * torch.sin(2.0 * x.flip(0))).contiguous()
    if mirror:
        pose[0] = -pose[0]
    w = m.arap_weights(x)
    R = m.arap_rotations(x, pose, w)
    E, g = m.arap_energy_grad(x, pose, w, R)
    l2g, e_l2g = m.array("v_l2g"), m.array("e_l2g")
    P, X = np.empty((m.nV, 3)), np.empty((m.nV, 3))
    P[l2g], X[l2g] = x.cpu().numpy().T, pose.cpu().numpy().T
    ev = m.array("ev").reshape(-1, 2).astype(np.int64)[e_l2g]
    wd = {(max(a, b), min(a, b)): v for (a, b), v in zip(ev.tolist(), w.cpu().numpy().astype(np.float64))}
    R64, fixed, (i, j, wt, dp, dx) = _arap64(V, F, P, X, wd)
    Rg = np.empty((m.nV, 9))
    Rg[l2g] = R.cpu().numpy()
    assert np.abs(Rg.reshape(-1, 3, 3) - R64)[fixed].max() <= 1e-4
    assert np.abs(Rg.reshape(-1, 3, 3) @ np.swapaxes(Rg.reshape(-1, 3, 3), 1, 2) - np.eye(3)).max() <= 1e-5
    d = dx - np.einsum("nij,nj->ni", Rg.reshape(-1, 3, 3)[i], dp)
    grad = np.zeros((m.nV, 3))
    np.add.at(grad, i, 2 * wt[:, None] * d)
    np.add.at(grad, j, -2 * wt[:, None] * d)
    e64 = (wt * (d * d).sum(1)).sum()
    assert abs(float(E[0]) - e64) <= 1e-5 * e64
    assert np.abs(g.cpu().numpy().T - grad[l2g]).max() <= 1e-4 * np.abs(grad).max()


def test_arap_rotations_of_undetermined_covariances():
    """No weight at all gives the identity; an unmoved pose the identity; a
    pose squeezed to a line or a point, where the covariance does not fix R, a
    proper rotation."""
    import torch
    V, F = mg.icosphere(3, seed=8, sigma=0.02)
    m, x = _mesh(V, F, 64)
    eye = torch.eye(3, device="cuda").reshape(1, 9)
    w = m.arap_weights(x)
    assert torch.equal(m.arap_rotations(x, x.flip(0).contiguous(), torch.zeros_like(w)), eye.expand(m.nV, 9))
    assert (m.arap_rotations(x, x, w) - eye).abs().max() <= 1e-5
    for keep in (1, 0):
        pose = x.clone()
        pose[keep:] = 0.0
        R = m.arap_rotations(x, pose, w).reshape(-1, 3, 3).double()
        assert (R @ R.transpose(1, 2).contiguous() - torch.eye(3, device="cuda")).abs().max() <= 1e-5
        assert (torch.linalg.det(R.cpu()) - 1.0).abs().max() <= 1e-5


@pytest.mark.parametrize("patch_size", [16, 512, 2048])
def test_evd_rows_at_any_alignment(patch_size):
    """The EVDiamond columns leave as 16-byte stores where the array allows:
    the same rows from an array that starts at every word of a line."""
    import torch
    V, F = mg.grid(37, seed=9)
    m, _ = _mesh(V, F, patch_size)
    n = m.query_nnz("EVD")
    rp, col = m.query("EVD")
    for mis in (1, 2, 3):
        c = torch.full((n + 8,), -7, dtype=torch.int32, device="cuda")
        r2, _ = m.query("EVD", col=c[mis:mis + n])
        assert torch.equal(r2, rp) and torch.equal(c[mis:mis + n], col[:n])
        assert (c[:mis] == -7).all() and (c[mis + n:] == -7).all()


def test_calls_go_to_the_current_stream():
    """A call without a stream argument is queued on torch's current stream,
    also inside a stream context and in another thread."""
    import threading
    import rxmesh_amd as rx
    import torch
    side = torch.cuda.Stream()
    assert rx._stream(None) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert rx._stream(None) == side.cuda_stream == rx._stream(side)
        got = []
        th = threading.Thread(target=lambda: got.append((rx._stream(None), torch.cuda.current_stream().cuda_stream)))
        th.start()
        th.join()
    assert got[0][0] == got[0][1]
    assert rx._stream(None) == torch.cuda.current_stream().cuda_stream


def _fan(k, closed):
    """One vertex with k neighbours in a closed or open fan."""
    ring = np.arange(1, k + 1)
    nxt = np.roll(ring, -1)
    f = np.stack([np.zeros(k, np.int64), ring, nxt], 1)
    return (f if closed else f[:-1]).astype(np.uint32)


def _query_mesh(name):
    if name == "sphere":
        return mg.permute_mesh(*mg.icosphere(4, seed=2, sigma=0.01), seed=2)[1]
    if name == "grid":
        return mg.grid(45, seed=2)[1]
    if name == "torus":  # valence 4 and 8
        return mg.permute_mesh(*mg.torus(40, 30), seed=2)[1]
    if name == "triangle":
        return np.array([[0, 1, 2]], np.uint32)
    if name == "fan7":
        return _fan(7, False)
    if name == "fan8":
        return _fan(8, True)
    if name == "fan9":  # one row beyond the fixed slots
        return np.concatenate([mg.grid(20, seed=2)[1], _fan(9, True) + 400])
    if name == "fan40":
        return _fan(40, True)
    if name == "bowtie":  # two fans, and three, sharing one vertex
        a, b = _fan(6, True), _fan(4, False)
        b[b > 0] += 10
        c = _fan(5, False)
        c[c > 0] += 20
        f = np.concatenate([a, b, c])
        return np.unique(f, return_inverse=True)[1].reshape(-1, 3).astype(np.uint32)
    if name == "flipped":
        f = mg.grid(20, seed=2)[1].copy()
        f[37] = f[37][::-1]
        return f
    f = mg.grid(12, seed=2)[1]  # "fin": an edge with three faces
    return np.concatenate([f, np.array([[f[50][0], f[50][1], 144]], np.uint32)])


@pytest.mark.parametrize("name", ["sphere", "grid", "torus", "triangle", "fan7", "fan8", "fan9", "fan40", "bowtie",
                                  "flipped", "fin"])
@pytest.mark.parametrize("patch_size", [16, 256, 512, 1024, 4096])
def test_query_kernels_over_forms(name, patch_size):
    """Every relation of the default kernels against the oracle: meshes inside
    and outside what the fixed-slot and direct-slot kernels take (long rows,
    flipped faces, edges with three faces), patches on either side of their
    register rounds, vertices of several fans for the oriented rows, and the
    general kernels (knob 10 = 0) on the same mesh."""
    import rxmesh_amd as rx
    import torch
    from oracle.oracle import OracleMesh
    F = _query_mesh(name)
    m = rx.Mesh(F, patch_size=patch_size)
    o = OracleMesh(F).set_patches(m.array("face_patch"), m.array("patches_val"), m.array("patches_offset"))
    for knob in (2, 0):
        m.set_launch_threads(10, knob)
        for op in ("VV", "VE", "VF", "EF", "FF", "EV", "FV", "FE", "EVD"):
            rp, col = m.query(op)
            orp, ocol = o.query(op)
            assert np.array_equal(rp.cpu().numpy(), orp), (op, knob)
            assert np.array_equal(col.cpu().numpy()[:len(ocol)], ocol), (op, knob)
        (vr, vc), (fr, fc) = m.query_vv_vf()
        for (rp, col), op in (((vr, vc), "VV"), ((fr, fc), "VF")):
            orp, ocol = o.query(op)
            assert np.array_equal(rp.cpu().numpy(), orp) and np.array_equal(col.cpu().numpy()[:len(ocol)], ocol)
    if name in ("flipped", "fin"):
        return
    for threads in (256, 512):
        m.set_launch_threads(6, threads)
        for op in ("VV", "VE"):
            rp, col = m.query(op, oriented=True)
            orp, ocol = o.query(op, oriented=True)
            assert np.array_equal(rp.cpu().numpy(), orp) and np.array_equal(col.cpu().numpy()[:len(ocol)], ocol), op


@pytest.mark.parametrize("level,patch_size", [(7, 512), (7, 1024), (7, 128), (6, 256), (8, 700)])
def test_query_kernels_of_many_patches(level, patch_size):
    """The workgroup sizes chosen for hundreds and thousands of patches: the
    rows of the general kernels, bit for bit."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(level, seed=5), seed=5)
    m, _ = _mesh(V, F, patch_size)
    for op in ("VV", "VE", "VF", "EF", "FF"):
        m.set_launch_threads(10, 2)
        rp, col = m.query(op)
        m.set_launch_threads(10, 0)
        r2, c2 = m.query(op)
        assert torch.equal(rp, r2) and torch.equal(col, c2), op
    m.set_launch_threads(10, 2)
    a = m.query_vv_vf()
    m.set_launch_threads(10, 0)
    b = m.query_vv_vf()
    assert all(torch.equal(x, y) for p, q in zip(a, b) for x, y in zip(p, q))


@pytest.mark.parametrize("level,patch_size", [(1, 512), (4, 16), (4, 512), (5, 2048), (5, 16), (6, 16)])
def test_normals_and_edge_weights_of_few_and_many_patches(level, patch_size):
    """Every workgroup size that the patch count chooses, patches from a few
    faces to more than the register rounds. FP32 sums of a few exact-input
    terms: 1e-5 of the largest value."""
    V, F = mg.permute_mesh(*mg.icosphere(level, seed=8, sigma=0.002), seed=8)
    m, x = _mesh(V, F, patch_size)
    l2g = m.array("v_l2g")
    X = np.empty((m.nV, 3))
    X[l2g] = x.cpu().numpy().T
    c = X[F]
    n = np.cross(c[:, 1] - c[:, 0], c[:, 2] - c[:, 0])
    l = ((c - np.roll(c, -1, 1)) ** 2).sum(2)  # corner j to j + 1
    for mode, wt in (("max", 1.0 / (l + np.roll(l, 1, 1))), ("area", np.full(l.shape, 0.5))):
        ref = np.zeros((m.nV, 3))
        np.add.at(ref, F.reshape(-1), (n[:, None, :] * wt[:, :, None]).reshape(-1, 3))
        got = m.vertex_normals(x, mode).cpu().numpy().T
        assert np.abs(got - ref[l2g]).max() <= 1e-5 * np.abs(ref).max()
    cot = {}
    for j in range(3):
        a, b = c[:, (j + 1) % 3] - c[:, j], c[:, (j + 2) % 3] - c[:, j]
        k = (a * b).sum(1) / np.linalg.norm(np.cross(a, b), axis=1)
        for p, q, v in zip(F[:, (j + 1) % 3].tolist(), F[:, (j + 2) % 3].tolist(), k):
            cot[(min(p, q), max(p, q))] = cot.get((min(p, q), max(p, q)), 0.0) + v
    ev = np.sort(m.array("ev").reshape(-1, 2).astype(np.int64)[m.array("e_l2g")], 1)
    w = m.arap_weights(x).cpu().numpy()
    ref = np.array([cot[(a, b)] for a, b in ev.tolist()])
    assert np.abs(w - np.maximum(0.0, 0.5 * ref)).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("name,a,b", [("normals", 40, 64), ("rotations", 28, 85), ("smooth", 50, 100), ("weights", 40, 80),
                                      ("step", 43, 60)])
def test_patches_near_the_lds_limit(name, a, b):
    """One patch that holds a whole torus of 2 a b faces and takes the form
    that needs least LDS, against patches of 512 faces. The row orders differ:
    twice the 1e-5 (rotations 1e-4) of each against FP64."""
    import torch
    V, F = mg.permute_mesh(*mg.torus(a, b), seed=9)
    out = []
    for patch_size in (16384, 512):
        m, x = _mesh(V, F, patch_size)
        assert (m.P == 1) == (patch_size == 16384)
        pose = (x + 0.3 * torch.sin(2.0 * x.flip(0))).contiguous()
        ids = m.array("v_l2g")
        if name == "normals":
            y = m.vertex_normals(x).T
        elif name == "smooth":
            y = m.smooth(x, 0.5, 3).T
        elif name == "weights":
            y, ids = m.arap_weights(x)[:, None], m.array("e_l2g")
        elif name == "step":
            y = m.symdir3_grad_step(m.symdir_rest(x), pose, 1e-3).T
        else:
            y = m.arap_rotations(x, pose, m.arap_weights(x))
        r = np.empty(y.shape)
        r[ids] = y.cpu().numpy()
        out.append(r)
    assert np.abs(out[0] - out[1]).max() <= (2e-4 if name == "rotations" else 2e-5) * np.abs(out[1]).max()


def test_matrix_free_solve_refuses_open_meshes_of_any_patch_size():
    import rxmesh_amd as rx
    V, F = mg.grid(80)
    for patch_size in (512, 32768):
        m, x = _mesh(V, F, patch_size)
        with pytest.raises(rx.RXMError) as e:
            m.mcf_matfree_cg(x, x, 1e-3, max_iter=3)
        assert e.value.code == 6


def _two_streams(V, F):
    """A mesh, its positions and two streams that wait for neither the default stream nor each other."""
    import torch
    m, x = _mesh(V, F, 512)
    torch.cuda.synchronize()
    return m, x, torch.cuda.Stream(), torch.cuda.Stream()


@pytest.mark.parametrize("steps", [0, 4])
def test_ring_plan_built_on_another_stream(steps):
    """A call on one stream builds the multi-step plan (build_vv_plan, or a
    smoothing with `steps` per launch), the next on another smooths over it:
    the bits of single steps."""
    import torch
    V, F = mg.icosphere(7, seed=11, sigma=0.01)
    m, x, a, b = _two_streams(V, F)
    m.set_launch_threads(8, 0)
    ref = m.smooth(x, 0.5, 7)
    n, _, _, _ = _two_streams(V, F)
    out, tmp, out_a, tmp_a = (torch.empty_like(x) for _ in range(4))
    torch.cuda.synchronize()
    if steps:
        n.set_launch_threads(8, steps)
        n.smooth(x, 0.5, 4, out=out_a, tmp=tmp_a, stream=a)
    else:
        n.build_vv_plan(stream=a)
    n.smooth(x, 0.5, 7, out=out, tmp=tmp, stream=b)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)


def test_face_plan_built_on_another_stream():
    """Normals on one stream build the face plan, curvature, gradient and step
    on another use it: the bits of the same calls in order."""
    import torch
    V, F = mg.icosphere(7, seed=12, sigma=0.01)
    m, x, a, b = _two_streams(V, F)
    Mr = m.symdir_rest(x)
    y = (x * 1.1).contiguous()
    torch.cuda.synchronize()
    calls = (lambda q, s: q.gaussian_curvature(y, stream=s), lambda q, s: q.symdir3_grad(Mr, y, stream=s),
             lambda q, s: q.symdir3_grad_step(Mr, y, 1e-3, stream=s))
    for call in calls:
        n, _, _, _ = _two_streams(V, F)
        with torch.cuda.stream(a):
            n.vertex_normals(y, "max")
        with torch.cuda.stream(b):
            got = call(n, None)
        torch.cuda.synchronize()
        with torch.cuda.stream(b):
            want = call(n, None)
        torch.cuda.synchronize()
        assert torch.equal(got[0] if isinstance(got, tuple) else got, want[0] if isinstance(want, tuple) else want)


@pytest.mark.parametrize("planned", [False, True])
def test_smoothing_in_a_captured_graph(planned):
    """Capture with build_vv_plan inside, of a mesh whose VV plan exists
    already (and, `planned`, its multi-step plan): three replays, eager work
    between them, each the bits of the eager smoothing."""
    import torch
    V, F = mg.icosphere(5, seed=13, sigma=0.01)
    m, x = _mesh(V, F, 256)
    ref, tmp = m.smooth(x, 0.5, 4), torch.empty_like(x)  # builds the VV plan
    if planned:
        m.build_vv_plan()
    src, out = x.clone(), torch.empty_like(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.build_vv_plan()
        m.smooth(src, 0.5, 4, out=out, tmp=tmp)
    for k in (1.0, 2.0, 0.5):  # powers of two: the smoothing scales exactly
        src.copy_(x * k)
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref * k)
        assert torch.equal(m.smooth(src, 0.5, 4), ref * k)
        torch.cuda.synchronize()
    m.build_vv_plan()
    assert torch.equal(m.smooth(x, 0.5, 4), ref)


@pytest.mark.parametrize("nu,nw,patch_size", [(16, 16, 8192), (16, 32, 8192), (32, 32, 8192), (25, 41, 8192),
                                              (32, 64, 8192), (3, 683, 8192), (1200, 460, 512), (97, 53, 256)])
def test_vertex_normals_at_the_rounds_of_each_workgroup(nu, nw, patch_size):
    """One patch of 512, 1024, 2048, 2050, 4096 and 4098 faces (a round more or
    less for 256, 512 and 1024 threads, and the form without a face pass), and
    many patches, against FP64. Bound per vertex, from the fp32 evaluation (u the
    unit roundoff): a normal's component is off by at most 4 u |e1| |e2| (two
    products of rounded differences, one subtraction), a weight by 6 u (two
    squared lengths of three terms, a reciprocal of 1 ulp) and a sum of k terms
    by k u: (10 + k) u times the sum of weight |e1| |e2| over its faces."""
    V, F = mg.permute_mesh(*mg.torus(nu, nw), seed=14)
    m, x = _mesh(V, F, patch_size)
    assert (m.P == 1) == (patch_size == 8192) and (patch_size != 512 or m.P > 2048)
    l2g = m.array("v_l2g")
    X = np.empty((m.nV, 3))
    X[l2g] = x.cpu().numpy().T
    c = X[F]
    n = np.cross(c[:, 1] - c[:, 0], c[:, 2] - c[:, 0])
    l = ((c - np.roll(c, -1, 1)) ** 2).sum(2)
    size = np.sqrt(l[:, 0] * l[:, 2])  # |e1| |e2|: edges 0 -> 1 and 2 -> 0
    gather = lambda t: np.bincount(F.reshape(-1), t.reshape(-1), m.nV)  # noqa: E731
    k = gather(np.ones(F.shape))
    for mode, wt in (("max", 1.0 / (l + np.roll(l, 1, 1))), ("area", np.full(l.shape, 0.5))):
        ref = np.stack([gather(n[:, None, j] * wt) for j in range(3)], 1)
        bound = (10 + k) * 2.0 ** -24 * gather(size[:, None] * wt)
        got = m.vertex_normals(x, mode).cpu().numpy().T
        assert (np.abs(got - ref[l2g]) <= bound[l2g][:, None]).all()


def test_automatic_smoothing_of_patches_beyond_several_steps():
    """Two patches of 8000 faces, beyond the plan kernel's tables: one step per
    launch goes over the host-built plan, five do not fit LDS. The automatic
    choice stays with single steps whatever plan was made before."""
    import torch
    import rxmesh_amd as rx
    V, F = mg.torus(80, 100)
    m = rx.Mesh(F, face_patch=(F.min(1) // 100 >= 40).astype(np.uint32))
    assert m.P == 2 and m.info["max_owned_faces"] < 8500
    x = torch.from_numpy(np.ascontiguousarray(V[m.array("v_l2g")].T.astype(np.float32))).cuda()
    m.set_launch_threads(8, 0)
    ref = m.smooth(x, 0.5, 6)
    one = m.smooth(x, 0.5, 1)
    m.set_launch_threads(8, 6)
    assert torch.equal(m.smooth(x, 0.5, 1), one)
    m.build_vv_plan()
    m.set_launch_threads(8, -1)
    assert torch.equal(m.smooth(x, 0.5, 6), ref)


def test_arap_rotations_of_nearly_undecided_covariances():
    """Covariances whose best rotation leads the next one by a gap of 1e-1 to
    1e-5 of the largest singular value (mirrored ones, and such of nearly one
    direction), where the closed form and the sweeps it falls back on meet. R
    against FP64 of the same fp32 input. Bound, u the fp32 unit roundoff: k
    products summed leave S off by (k + 3) u sum w |a| |c|, the 4 x 4 matrix by
    sqrt(3) of that, its eigenvector by that over the gap of its eigenvalues, R
    by 4 times that; the sweeps add 64 u |S| over the gap, the closed form at
    most 1e-5."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(5, seed=15), seed=15)
    m, _ = _mesh(V, F, 512)
    l2g, e_l2g = m.array("v_l2g"), m.array("e_l2g")
    ev = m.array("ev").reshape(-1, 2).astype(np.int64)[e_l2g]  # global endpoints by linear edge
    rng = np.random.default_rng(15)
    w = rng.uniform(0.5, 1.5, m.nE).astype(np.float32)
    ring = [[] for _ in range(m.nV)]
    for k, (i, j) in enumerate(ev.tolist()):
        ring[i].append((j, k))
        ring[j].append((i, k))
    P, X = (rng.normal(size=(m.nV, 3)).astype(np.float32) for _ in range(2))
    free, chosen = np.ones(m.nV, bool), []
    for v in range(m.nV):  # vertices whose rings are disjoint
        ids = [v] + [j for j, _ in ring[v]]
        if free[ids].all():
            free[ids] = False
            chosen.append(v)
    rot = lambda: np.linalg.qr(rng.normal(size=(3, 3)))[0]  # noqa: E731
    for n, v in enumerate(chosen):
        gap, s2 = 10.0 ** -rng.uniform(1, 5), rng.uniform(0.2, 0.9)
        U, W = rot(), rot()
        mirrored = n % 4 != 0
        U[:, 2] *= np.sign(np.linalg.det(U @ W)) * (-1.0 if mirrored else 1.0)
        T = U @ np.diag([1.0, s2, s2 - gap / 2] if mirrored else [1.0, gap / 4, gap / 4]) @ W
        P[v] = X[v] = 0.0
        nb, wt = [j for j, _ in ring[v]], np.array([w[k] for _, k in ring[v]], np.float64)
        a = -P[nb].astype(np.float64)
        X[nb] = -(a @ np.linalg.solve((wt[:, None] * a).T @ a, T))  # sum w a c^T = T
    Pd, Xd = (torch.from_numpy(np.ascontiguousarray(q[l2g].T)).cuda() for q in (P, X))
    R = np.empty((m.nV, 3, 3))
    R[l2g] = m.arap_rotations(Pd, Xd, torch.from_numpy(w).cuda()).cpu().numpy().reshape(-1, 3, 3)
    u, decades = 2.0 ** -24, set()
    for v in chosen:
        nb, wt = [j for j, _ in ring[v]], np.array([w[k] for _, k in ring[v]], np.float64)
        a, c = -P[nb].astype(np.float64), -X[nb].astype(np.float64)
        U, s, Wt = np.linalg.svd((wt[:, None] * a).T @ c)
        sign = np.sign(np.linalg.det(U @ Wt))
        U[:, 2] *= sign
        gap = 2.0 * (s[1] + sign * s[2])
        off = np.sqrt(3.0) * (len(nb) + 3) * (wt * np.linalg.norm(a, axis=1) * np.linalg.norm(c, axis=1)).sum()
        bound = 1e-5 + 4.0 * u * (off + 64.0 * s[0]) / gap
        assert np.abs(R[v] - Wt.T @ U.T).max() <= bound, (v, gap / s[0], bound)
        decades.add(int(np.floor(np.log10(gap / s[0]))))
    assert {-2, -3, -4, -5} <= decades


@pytest.mark.parametrize("share", [1, 7, 900])
@pytest.mark.parametrize("patch_size", [64, 512, 4096])
def test_oriented_rows_of_many_vertices_with_several_fans(share, patch_size):
    """Two closed surfaces and a sheet glued vertex to vertex (two and three
    fans, closed and open, one to most vertices of a patch): oriented VV and
    VE against the oracle, unoriented too."""
    import rxmesh_amd as rx
    from oracle.oracle import OracleMesh
    parts = [mg.torus(60, 40)[1], mg.torus(60, 40)[1] + 2400, mg.grid(60, seed=3)[1] + 4800]
    n = 4800 + int(parts[2].max()) - 4799
    spots = np.random.default_rng(16).permutation((np.arange(0, 58, 2)[:, None] * 40 + np.arange(0, 38, 2)).ravel())[:share]
    glue = np.arange(n)
    glue[spots + 2400] = spots
    third = spots[::3]
    glue[4800 + (third // 40) * 60 + third % 40] = third  # vertices of the sheet, two apart in both directions
    F = np.unique(glue[np.concatenate(parts)], return_inverse=True)[1].reshape(-1, 3).astype(np.uint32)
    F = mg.permute_mesh(np.zeros((int(F.max()) + 1, 3)), F, seed=16)[1]
    m = rx.Mesh(F, patch_size=patch_size)
    assert m.info["is_edge_manifold"] and m.info["is_consistently_oriented"]
    o = OracleMesh(F).set_patches(m.array("face_patch"), m.array("patches_val"), m.array("patches_offset"))
    for op in ("VV", "VE"):
        for oriented in (True, False):
            rp, col = m.query(op, oriented=oriented)
            orp, ocol = o.query(op, oriented=oriented)
            assert np.array_equal(rp.cpu().numpy(), orp) and np.array_equal(col.cpu().numpy()[:len(ocol)], ocol)


@pytest.mark.parametrize("shape", ["cones", "glued", "grid", "sphere"])
@pytest.mark.parametrize("patch_size", [16, 512, 4096])
def test_closed_fans_of_any_valence(shape, patch_size):
    """Which vertices the assembly takes from the face pass: the diagonal and
    mass of the assembled system against FP64 sums over the faces for vertices
    of one closed fan, among them such of 700 faces, boundaries and glued
    vertices. 1e-5 of the largest value, the assembly's bound elsewhere, on
    the vertices of closed fans."""
    import torch
    if shape == "cones":  # closed fans of 700, 30 and 3 faces; the rims are boundaries
        F = np.concatenate([_fan(700, True), _fan(30, True) + 701, _fan(3, True) + 732])
    elif shape == "glued":
        F = np.concatenate([mg.torus(20, 12)[1], mg.torus(20, 12)[1] + 240])
        F = np.unique(np.where(F == 245, 7, F), return_inverse=True)[1].reshape(-1, 3)
    else:
        F = mg.grid(25, seed=4)[1] if shape == "grid" else mg.icosphere(3, seed=4)[1]
    F = F.astype(np.uint32)
    rng = np.random.default_rng(17)
    V = rng.normal(size=(int(F.max()) + 1, 3))
    m, x = _mesh(V, F, patch_size)
    X = np.empty((m.nV, 3))
    X[m.array("v_l2g")] = x.cpu().numpy().T
    rp, col, val, mass = (t.cpu().numpy() for t in m.cot_assemble(x, 0.1))
    nxt = {}  # successor around v, by (v, neighbour)
    for a, b, c in F.tolist():
        for v, p, q in ((a, b, c), (b, c, a), (c, a, b)):
            nxt.setdefault(v, {})[p] = q
    closed = np.zeros(m.nV, bool)
    for v, succ in nxt.items():
        nb = set(succ) | set(succ.values())
        p = s = next(iter(succ))
        n = 0
        while p in succ and n < len(nb):
            p, n = succ[p], n + 1
            if p == s:
                break
        closed[v] = p == s and n == len(nb)
    if shape in ("glued", "sphere"):  # closed surfaces: the matrix-free solve wants every vertex of one closed fan
        import rxmesh_amd as rx
        if shape == "sphere":
            m.mcf_matfree_cg(x, x, 1e-3, max_iter=1)
        else:
            with pytest.raises(rx.RXMError) as e:
                m.mcf_matfree_cg(x, x, 1e-3, max_iter=1)
            assert e.value.code == 6
    assert closed.any() and closed.sum() == {"cones": 3, "glued": 478, "grid": 23 * 23, "sphere": m.nV}[shape]
    c = X[F]
    area = 0.5 * np.linalg.norm(np.cross(c[:, 1] - c[:, 0], c[:, 2] - c[:, 0]), axis=1)
    w, vor = {}, np.zeros(m.nV)
    clamp = lambda t: np.clip(t, -19.1, 19.1)  # noqa: E731
    for j in range(3):
        i0, i1, i2 = j, (j + 1) % 3, (j + 2) % 3
        e1, e2 = c[:, i1] - c[:, i0], c[:, i2] - c[:, i0]
        d0 = (e1 * e2).sum(1)
        d1 = -(e1 * (c[:, i2] - c[:, i1])).sum(1)
        d2 = (e2 * (c[:, i2] - c[:, i1])).sum(1)
        for p, q, t in zip(F[:, i1].tolist(), F[:, i2].tolist(), clamp(d0 / area)):
            w[(min(p, q), max(p, q))] = w.get((min(p, q), max(p, q)), 0.0) + t
        t = np.maximum(0.125 * ((e2 * e2).sum(1) * clamp(d1 / area) + (e1 * e1).sum(1) * clamp(d2 / area)), 0.0)
        t = np.where(d0 < 0, 0.25 * area, np.where((d1 < 0) | (d2 < 0), 0.125 * area, t))
        np.add.at(vor, F[:, i0], t)
    ms = vor / 0.5
    diag = ms.copy()
    for (p, q), t in w.items():
        diag[p] += 0.1 * max(t, 0.0)
        diag[q] += 0.1 * max(t, 0.0)
    l2g = m.array("v_l2g")
    ok = closed[l2g]
    for got, ref in ((mass, ms), (val[rp[:-1]], diag)):
        assert np.abs(got - ref[l2g])[ok].max() <= 1e-5 * np.abs(ref[l2g][ok]).max()


@pytest.mark.parametrize("level,patch_size", [(3, 16), (6, 64), (4, 256), (6, 256), (7, 256), (4, 512), (5, 1024)])
def test_workgroup_sizes_of_small_patches(level, patch_size):
    """Curvature, explicit step and single smoothing steps where the size of the
    patches and their number choose the workgroup: curvature against FP64
    (1e-5 of the angle sums, the angles' 1.4e-7 rad times the valence well
    inside), the others the bits of the general CSR kernels or of every
    workgroup size."""
    import torch
    V, F = mg.permute_mesh(*mg.icosphere(level, seed=18, sigma=0.002), seed=18)
    m, x = _mesh(V, F, patch_size)
    l2g = m.array("v_l2g")
    X = np.empty((m.nV, 3))
    X[l2g] = x.cpu().numpy().T
    c = X[F]
    ang, mix = np.zeros(m.nV), np.zeros(m.nV)
    dots, s = [], np.linalg.norm(np.cross(c[:, 1] - c[:, 0], c[:, 2] - c[:, 0]), axis=1)
    for j in range(3):
        dots.append(((c[:, (j + 1) % 3] - c[:, j]) * (c[:, (j + 2) % 3] - c[:, j])).sum(1))
    obtuse = (dots[0] < 0) | (dots[1] < 0) | (dots[2] < 0)
    length = [((c[:, j] - c[:, (j + 1) % 3]) ** 2).sum(1) for j in range(3)]
    for j in range(3):
        a = (length[(j + 2) % 3] * dots[(j + 1) % 3] + length[j] * dots[(j + 2) % 3]) / (8 * s)
        ang += np.bincount(F[:, j], np.arctan2(s, dots[j]), m.nV)
        mix += np.bincount(F[:, j], np.where(obtuse, np.where(dots[j] < 0, s / 4, s / 8), a), m.nV)
    gc, am = (t.cpu().numpy().astype(np.float64) for t in m.gaussian_curvature(x))
    assert np.abs(am - mix[l2g]).max() <= 1e-5 * mix.max()
    assert np.abs(gc * am - (2 * np.pi - ang)[l2g]).max() <= 1e-5 * 2 * np.pi
    m.set_launch_threads(8, 0)
    assert torch.equal(m.smooth(x, 0.5, 3), m.smooth_csr(m.query("VV"), x, 0.5, 3))
    A = m.cot_assemble(x, 1e-4)
    y = m.mcf_explicit(A, x, 2)
    for threads in (256, 512):
        m.set_launch_threads(0, threads)
        assert torch.equal(m.mcf_explicit(A, x, 2), y)
