"""The mesh functions gather their triangles and add gradients straight to the vertices: every
form of faces and vertices the gather takes gives the same values and gradients, against the
FP64 CPU adjoint scattered to the vertices."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
TOL = 1e-4  # relative to the larger of the component and 5 % of the array's rms, as in test_gpu_autograd


@pytest.mark.parametrize("form", ["int32", "int64", "negative", "cpu", "strided", "in_place", "points_only"])
def test_mesh_forms(qabi, scenes, form):
    from oracle import adjoint as J
    from quarry import autograd as AG

    V, F, tris = scenes.icosphere(levels=2, radius=10.0, noise=0.1, seed=5)
    rng = np.random.default_rng(6)
    q = rng.uniform(-15, 15, (3001, 3)).astype(np.float32)
    rays = scenes.sphere_rays(3001, seed=7)
    up = rng.uniform(-1, 1, 3001).astype(np.float32)
    up[:20] = 0.0
    faces = torch.from_numpy(F).cuda()
    if form in ("int64", "cpu"):
        faces = faces.long().cpu() if form == "cpu" else faces.long()
    if form == "negative":
        faces = torch.where(faces % 3 == 0, faces - V.shape[0], faces)
    base = torch.from_numpy(V).cuda()
    v = (torch.stack([base, base], 2).contiguous()[:, :, 0] if form == "strided" else base.clone()).requires_grad_(
        form != "points_only")
    assert v.is_contiguous() == (form != "strided")
    p = torch.from_numpy(q).cuda().requires_grad_()
    o = torch.from_numpy(rays[:, :3].copy()).cuda().requires_grad_()
    d = torch.from_numpy(rays[:, 3:6].copy()).cuda().requires_grad_()
    d2, idx = AG.closest_point_dist2(p, v, faces)
    t, hit = AG.ray_hit_t(o, d, v, faces)
    if form == "in_place":  # between forward and backward
        with torch.no_grad():
            v.add_(1.0)
    g = torch.from_numpy(up).cuda()
    ins = [p, o, d] + ([v] if v.requires_grad else [])
    got = torch.autograd.grad([d2, t], ins, [g, torch.where(torch.isfinite(t), g, torch.zeros_like(g))])
    prim, hp = idx.cpu().numpy(), hit.cpu().numpy()
    T64 = tris.astype(np.float64)
    cq, ct = J.tri_adjoint(q.astype(np.float64), T64, prim, up.astype(np.float64))
    co, cd, ct2 = J.ray_adjoint(rays[:, :3].astype(np.float64), rays[:, 3:6].astype(np.float64), T64, hp,
                                up.astype(np.float64))
    cV = np.zeros(V.shape)
    for k in range(3):
        np.add.at(cV, F[:, k], (ct + ct2).reshape(-1, 3, 3)[:, k])
    for a, ref in zip(got, (cq, co, cd, cV)):
        a = a.cpu().numpy().astype(np.float64)
        floor = 0.05 * float(np.sqrt(np.mean(ref ** 2)))
        assert np.max(np.abs(a - ref) / np.maximum(np.abs(ref), floor)) < TOL


@pytest.mark.parametrize("levels", [2, 4])  # 320 and 5,120 faces
def test_vertex_gradient_sums_by_triangle(qabi, scenes, levels):
    """Many queries per triangle: the vertex gradients carry the rounding of two short sums
    (queries into corners, corners into vertices), not of one over every query around a
    vertex.  Yardstick: the per-triangle adjoint summed into the vertices in FP64.  The second
    level adds about six FP32 terms: half an ulp each against a first level of 50 to 800, so
    half as much again as the yardstick's error is allowed; a flat sum has two to four times
    that error."""
    import ctypes

    from oracle import adjoint as J
    from quarry import autograd as AG

    A = AG.A
    V, F, tris = scenes.icosphere(levels=levels, radius=10.0, noise=0.1, seed=5)
    rng = np.random.default_rng(levels)
    n = 262144
    q = rng.normal(0, 1, (n, 3))
    q = (q * (rng.uniform(8, 12, (n, 1)) / np.linalg.norm(q, axis=1, keepdims=True))).astype(np.float32)
    up = rng.uniform(0, 1, n).astype(np.float32)
    rays = scenes.sphere_rays(n, seed=7)
    T64 = tris.astype(np.float64)

    def fold(corners):
        out = np.zeros(V.shape)
        for k in range(3):
            np.add.at(out, F[:, k], np.asarray(corners, np.float64).reshape(-1, 3, 3)[:, k])
        return out

    def error(got, want):
        return np.linalg.norm(got - want) / np.linalg.norm(want)

    faces, g = torch.from_numpy(F).cuda(), torch.from_numpy(up).cuda()
    v = torch.from_numpy(V).cuda().requires_grad_()
    t = torch.from_numpy(tris.reshape(-1, 9)).cuda().requires_grad_()

    # closest points
    p = torch.from_numpy(q).cuda()
    d2, idx = AG.closest_point_dist2(p, v, faces)
    got = torch.autograd.grad(d2, v, g)[0].cpu().numpy()
    corners = torch.autograd.grad(AG._ClosestDist2.apply(p, t, A.PRIM_TRI, A.ORDER_MORTON, True, A.BUILDER_LBVH)[0], t,
                                  g)[0].cpu().numpy()
    want = fold(J.tri_adjoint(q.astype(np.float64), T64, idx.cpu().numpy(), up.astype(np.float64))[1])
    here, there = error(got, want), error(fold(corners), want)
    print(f"closest, {F.shape[0]} faces: {here:.2e}, yardstick {there:.2e}", flush=True)
    assert here < 1.5 * there

    # rays, with the yardstick through the C entry points
    o, d = (torch.from_numpy(rays[:, c:c + 3].copy()).cuda() for c in (0, 3))
    th, hit = AG.ray_hit_t(o, d, v, faces)
    gh = torch.where(torch.isfinite(th), g, torch.zeros_like(g))
    got = torch.autograd.grad(th, v, gh)[0].cpu().numpy()
    b = A.Bvh.from_device(A.PRIM_TRI, t.data_ptr(), tris.shape[0], A.BUILDER_LBVH)
    rd = torch.from_numpy(rays).cuda()
    res, hp = torch.empty(n, dtype=torch.int64, device="cuda"), torch.empty(n, dtype=torch.int32, device="cuda")
    gt = torch.zeros_like(t)
    AG._on_stream()
    A.check(A.lib().qr_raycast_save_device(b.h, AG._p(rd), n, AG._p(res), AG._p(hp), A.ORDER_INPUT, 0,
                                           ctypes.byref(ctypes.c_double())))
    A.check(A.lib().qr_adjoint_ray(b.h, AG._p(rd), n, AG._p(res), AG._p(hp), AG._p(gh), None, None, AG._p(gt)))
    want = fold(J.ray_adjoint(rays[:, :3].astype(np.float64), rays[:, 3:6].astype(np.float64), T64, hit.cpu().numpy(),
                              gh.cpu().numpy().astype(np.float64))[2])
    here, there = error(got, want), error(fold(gt.cpu().numpy()), want)
    print(f"rays, {F.shape[0]} faces: {here:.2e}, yardstick {there:.2e}", flush=True)
    assert here < 1.5 * there


@pytest.mark.parametrize("entry", ["closest", "ray"])
def test_mesh_entry_points(qabi, scenes, entry):
    """The C entry points that take faces: the same vertex gradients (added to what is there)
    as the per-triangle ones folded, NULL gradients and no queries taken."""
    import ctypes

    from quarry import autograd as AG

    A, L = AG.A, AG.A.lib()
    V, F, tris = scenes.icosphere(levels=3, radius=10.0, noise=0.1, seed=5)
    n = 5000
    rng = np.random.default_rng(9)
    t, f = torch.from_numpy(tris.reshape(-1, 9)).cuda(), torch.from_numpy(F.astype(np.int32)).cuda()
    g = torch.from_numpy(rng.uniform(-1, 1, n).astype(np.float32)).cuda()
    AG._on_stream()
    b = A.Bvh.from_device(A.PRIM_TRI, t.data_ptr(), tris.shape[0], A.BUILDER_LBVH)
    ms = ctypes.c_double()
    gt, gv = torch.zeros_like(t), torch.ones(V.shape, dtype=torch.float32, device="cuda")
    ga, gb = (torch.empty((n, 3), dtype=torch.float32, device="cuda") for _ in range(2))
    if entry == "closest":
        q = torch.from_numpy(rng.uniform(-15, 15, (n, 3)).astype(np.float32)).cuda()
        res, aux = torch.empty((n, 2), dtype=torch.int32, device="cuda"), torch.empty(n, dtype=torch.int32, device="cuda")
        A.check(L.qr_closest_device(b.h, AG._p(q), n, AG._p(res), A.ORDER_INPUT, 0, ctypes.byref(ms)))
        A.check(L.qr_closest_save_aux(b.h, AG._p(q), n, AG._p(res), AG._p(aux)))

        def tri(m, out):
            return L.qr_adjoint_closest(b.h, AG._p(q), m, AG._p(res), AG._p(aux), AG._p(g), AG._p(ga), AG._p(out))

        def mesh(m, out):
            return L.qr_adjoint_closest_mesh(b.h, AG._p(q), m, AG._p(res), AG._p(aux), AG._p(g), AG._p(f), AG._p(gb),
                                             AG._p(out))
    else:
        q = torch.from_numpy(scenes.sphere_rays(n, seed=3)).cuda()
        res, hp = torch.empty(n, dtype=torch.int64, device="cuda"), torch.empty(n, dtype=torch.int32, device="cuda")
        A.check(L.qr_raycast_save_device(b.h, AG._p(q), n, AG._p(res), AG._p(hp), A.ORDER_INPUT, 0, ctypes.byref(ms)))

        def tri(m, out):
            return L.qr_adjoint_ray(b.h, AG._p(q), m, AG._p(res), AG._p(hp), AG._p(g), AG._p(ga), None, AG._p(out))

        def mesh(m, out):
            return L.qr_adjoint_ray_mesh(b.h, AG._p(q), m, AG._p(res), AG._p(hp), AG._p(g), AG._p(f), AG._p(gb), None,
                                         AG._p(out))
    A.check(tri(n, gt))
    A.check(mesh(n, gv))
    A.check(mesh(n, None))
    A.check(mesh(0, gv))
    assert torch.equal(ga, gb)
    want = np.ones(V.shape)
    for k in range(3):
        np.add.at(want, F[:, k], gt.cpu().numpy().astype(np.float64).reshape(-1, 3, 3)[:, k])
    # a vertex sums some tens of terms of the gradients' size in FP32: 64 half-ulps of them
    assert np.max(np.abs(gv.cpu().numpy() - want)) < 64 * 2 ** -24 * max(1.0, np.abs(want).max())
    out = torch.zeros(V.shape, dtype=torch.float32, device="cuda")
    A.check(L.qr_adjoint_vertices(AG._p(gt), AG._p(f), F.shape[0], AG._p(out)))
    assert np.max(np.abs(out.cpu().numpy() + 1 - want)) < 64 * 2 ** -24 * max(1.0, np.abs(want).max())
    assert L.qr_adjoint_vertices(AG._p(gt), None, F.shape[0], AG._p(out)) != A.QR_OK
    assert L.qr_adjoint_vertices(AG._p(gt), AG._p(f), -1, AG._p(out)) != A.QR_OK
