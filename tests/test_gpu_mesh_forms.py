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
