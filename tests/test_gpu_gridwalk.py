"""Ray walks through the cells of a marching-cubes surface (Bvh.set_grid) against the tree: every
trace gives the same hits, rays that meet two faces at one distance among them, so the deterministic
mode's sums agree face by face, on surfaces that fill the grid differently: a hole, a trench whose
mesh stops a cell short of the periodic faces, a flat surface on a grid plane, noise with faces in
most cells, a grid two nodes wide, odd sizes."""
import numpy as np
import pytest

from oracle import levelset as ol

pytestmark = pytest.mark.gpu


def _phi(name):
    rng = np.random.default_rng(11)
    if name == "hole":
        return ol.init_sdf(7.0, 6.5, 9.75, 0.25, 2.6, 6.0, 3.0, True), 0.25, 0
    if name == "trench":
        return ol.init_sdf(6.0, 1.5, 12.0, 0.15, 1.5, 7.0, 3.0, False), 0.15, 1
    if name == "flat":          # phi exactly 0 on a node plane
        z = np.arange(20)[None, None, :] * 0.25
        return np.broadcast_to(2.5 - z, (17, 13, 20)), 0.25, 1
    if name == "noise":
        return rng.standard_normal((19, 23, 21)) + 0.02 * (10 - np.arange(21)), 0.1, 1
    if name == "thin":          # two nodes along y
        p = ol.init_sdf(4.0, 0.4, 8.0, 0.2, 1.2, 4.0, 2.0, False)
        assert p.shape[1] == 2
        return p, 0.2, 1
    p = ol.init_sdf(6.6, 3.4, 6.2, 0.2, 2.0, 3.0, 2.0, True)
    return p + 0.05 * rng.standard_normal(p.shape), 0.2, 0      # "rough"


NAMES = ["hole", "trench", "flat", "noise", "thin", "rough"]


@pytest.fixture
def det():
    from petch import ops
    ops.set_deterministic(True)
    yield
    ops.set_deterministic(False)


def _surface(name):
    import torch
    from petch import flux, ops
    phi, dx, per = _phi(name)
    dev = torch.device("cuda", 0)
    tphi = torch.from_numpy(np.ascontiguousarray(phi, np.float32)).to(dev)
    mesh = flux.SurfaceMesh(dev).build(tphi, dx)
    L = [n * dx for n in phi.shape]
    return mesh, tphi, dx, ops.make_box(*L, L[2] - dx, per), dev


def _l1(a, b):
    return float((a.double() - b.double()).abs().sum() / b.double().abs().sum().clamp(min=1e-30))


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("n", [1, 63, 4097, 300000])
def test_walk_gives_the_trees_fluxes(name, n, det):
    import torch
    from petch import flux, ops
    from petch.params import PAR
    mesh, phi, dx, box, dev = _surface(name)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    # stickings up to 0.9: the adjoint weighs a path by 1 / (1 - S)
    bare = torch.from_numpy(np.random.default_rng(3).uniform(0.05, 0.9, mesh.nf).astype(np.float32)).to(dev)
    par = dict(PAR, ion_source="powcos", ion_exponent=20.0)
    gn = ops.gas_normals(phi, dx, mesh.centroids, mesh.normals)
    area = mesh.areas

    def fluxes(b):
        src = flux.NEUTRAL_SOURCE
        a, o = ops.trace_neutral_rr_pair(b, box, src, bare, 0.7, n, 5, 1.0, n // 2, 6)
        out = [a.clone(), o.clone(), ops.trace_neutral_rr(b, box, src, bare, 0.3, n, 7).clone()]
        ion = ops.trace_ion_yield(b, box, flux.ion_source(par), flux.ion_params(par), n, 8)
        out += [x.clone() for x in ion]
        out.append(ops.trace_neutral_cap(b, box, src, bare, 0.5, 4, n, 9).clone())
        out.append(ops.trace_redeposition(b, mesh.centroids, gn, area, bare, 0.5, n, 10).clone())
        g = ops.trace_neutral_rr_pair_adjoint(b, box, src, bare, 0.7, n, 5, a.clone(), 1.0, n // 2,
                                              6, o.clone())
        out.append(g.clone())
        assert b.status() == 0
        return out
    for k, (x, y) in enumerate(zip(fluxes(mesh.bvh), fluxes(tree))):
        assert torch.isfinite(x).all()
        if k < 10:
            assert torch.equal(x, y), (name, n, k)
        else:
            # float sums of the adjoint, in any order: 1e-5 of their mass, its terms cancel
            assert _l1(x, y) <= 1e-4, (name, n, k)


@pytest.mark.parametrize("name", NAMES)
def test_walk_gives_the_trees_form_factors(name):
    from petch import ops
    mesh, phi, dx, box, dev = _surface(name)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    gn = ops.gas_normals(phi, dx, mesh.centroids, mesh.normals)
    a = ops.trace_ff(mesh.bvh, box, mesh.centroids, gn, 24, 17)
    b = ops.trace_ff(tree, box, mesh.centroids, gn, 24, 17)
    assert bool((a == b).all())


def test_batch_of_grids_equals_the_single_surfaces(det):
    import torch
    from petch import flux, ops
    from petch._abi import PetchError
    S = [_surface(n) for n in ("hole", "noise", "thin")]
    meshes = [flux.SurfaceMesh(S[0][4]) for _ in S]
    mcs = ops.marching_cubes_batch([(s[1], s[2], m.bufs) for s, m in zip(S, meshes)])
    for m, mc in zip(meshes, mcs):
        m.build_from(*mc, grid=m.bufs.grid)
    ops.bvh_build_batch([m.bvh_item() for m in meshes])
    items = []
    for k, (s, m) in enumerate(zip(S, meshes)):
        assert torch.equal(m.faces, s[0].faces)
        items.append(dict(bvh=m.bvh, box=s[3], bare=torch.full((m.nf,), 0.4, device=s[4]),
                          beta_a=0.7, n_a=20000 + k, seed_a=3, beta_b=1.0, n_b=500, seed_b=4))
    got = ops.trace_neutral_rr_batch(flux.NEUTRAL_SOURCE, items)
    for it, s, (a, o) in zip(items, S, got):
        x, y = ops.trace_neutral_rr_pair(s[0].bvh, it['box'], flux.NEUTRAL_SOURCE, it['bare'], 0.7,
                                         it['n_a'], 3, 1.0, 500, 4)
        assert torch.equal(a, x) and torch.equal(o, y)
    # a surface off its grid is reported, and a rebuilt tree forgets its grid
    m = meshes[0]
    cells, nx, ny, nz, dx = m.grid
    m.bvh.set_grid(m.verts + 0.1 * dx, m.faces, m.grid)
    assert m.bvh.status() == 4
    m.bvh.build(m.verts, m.faces)
    assert m.bvh.status() == 0
    with pytest.raises(PetchError):
        m.bvh.set_grid(m.verts, m.faces, (cells, 1, ny, nz, dx))
    with pytest.raises(PetchError, match="twice"):
        ops.bvh_set_grid_batch([meshes[k].bvh_item() for k in (1, 0, 1)])


@pytest.mark.parametrize("name", NAMES)
def test_walk_answers_ray_queries_as_the_tree(name):
    """Rays from inside, beside and above the grid, off the surface by 1e-4, along the axes and
    from grid points: the same face and, to the bit, the same distance for every ray (both run the
    same triangle test), also where it meets an edge or a vertex exactly."""
    import torch
    from petch import ops
    mesh, phi, dx, box, dev = _surface(name)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    n, g = 400000, torch.Generator().manual_seed(1)
    o = (torch.rand((n, 3), generator=g) * 1.2 - 0.1) * torch.tensor([s * dx for s in phi.shape])
    k = torch.randint(0, mesh.nf, (n // 2,), generator=g)
    o[:n // 2] = mesh.centroids.cpu()[k] + 1e-4 * torch.randn((n // 2, 3), generator=g)
    d = torch.randn((n, 3), generator=g)
    axis = torch.rand(n, generator=g) < 0.1
    d[axis] = torch.eye(3)[torch.randint(0, 3, (int(axis.sum()),), generator=g)] * \
        torch.where(torch.rand((int(axis.sum()), 1), generator=g) < 0.5, 1.0, -1.0)
    node = torch.rand(n, generator=g) < 0.1
    o[node] = torch.round(o[node] / dx) * dx
    o = o.to(dev).contiguous()
    # + 0.0: no -0.0, for which the tree's slab test drops a ray that runs in a box's lower plane
    d = (d / d.norm(dim=1, keepdim=True) + 0.0).to(dev).contiguous()
    for tmax in (1.0e6, 3.3 * dx):
        fa, ta = mesh.bvh.query_ray(o, d, tmax)
        fb, tb = tree.query_ray(o, d, tmax)
        assert int((fb >= 0).sum()) > 1000
        print(name, tmax, int((fa != fb).sum()), int((ta != tb).sum()), flush=True)
        assert torch.equal(fa, fb) and torch.equal(ta, tb)


def _aimed_rays(mesh, phi, dx, kind, n, gen):
    """Rays at vertices and edges of the surface, or that run nearly along a grid plane into one."""
    import torch
    v, f = mesh.verts.cpu(), mesh.faces.cpu().long()
    L = torch.tensor([s * dx for s in phi.shape])
    q = f[torch.randint(0, mesh.nf, (n,), generator=gen)]
    a, b = v[q[:, 0]], v[q[:, 1]]
    u = torch.rand((n, 1), generator=gen)
    target = a + u * (b - a) if kind == "edge" else a
    if kind == "beside":
        # components 1e-2 to 1e-7 of the others on one axis, on half of the rays on two
        d = torch.randn((n, 3), generator=gen)
        ax = torch.randint(0, 3, (n,), generator=gen)
        two = (torch.rand(n, generator=gen) < 0.5).float()
        rows = torch.arange(n)
        d[rows, ax] *= 10 ** (-2 - 5 * torch.rand(n, generator=gen))
        d[rows, (ax + 1) % 3] *= 10 ** (-two * (1 + 5 * torch.rand(n, generator=gen)))
        d = d / d.norm(dim=1, keepdim=True)
        o = target - torch.rand((n, 1), generator=gen) * 0.7 * float(L.max()) * d
    else:
        o = (torch.rand((n, 3), generator=gen) * 1.2 - 0.1) * L
        d = target - o
        d = d / d.norm(dim=1, keepdim=True)
    return o.contiguous(), (d + 0.0).contiguous()


@pytest.mark.parametrize("kind", ["vertex", "edge", "beside"])
@pytest.mark.parametrize("name", NAMES)
def test_rays_at_vertices_edges_and_beside_planes_hit_as_on_the_tree(name, kind):
    """Where two cells meet, a ray can lie on either side of the plane between them by rounding, and
    one nearly along the plane stays there: both cells have to be looked into. The walk's distances
    are the tree's to the bit (one triangle test, one query of the tree for a ray that meets two
    faces at once), and so are the faces."""
    import torch
    from petch import ops
    mesh, phi, dx, box, dev = _surface(name)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    o, d = _aimed_rays(mesh, phi, dx, kind, 400000, torch.Generator().manual_seed(2))
    fa, ta = mesh.bvh.query_ray(o.to(dev), d.to(dev))
    fb, tb = tree.query_ray(o.to(dev), d.to(dev))
    assert int((fb >= 0).sum()) > 100000
    print(name, kind, int((fa != fb).sum()), int((ta != tb).sum()), flush=True)
    assert torch.equal(fa, fb) and torch.equal(ta, tb)


def _doubled(mesh, phi, dx, share):
    """mesh with the faces (a, b, c) of a share of its cells followed by (a, b, their centroid): the
    verts and faces, and the walked and the plain tree over them. A ray that hits the added face
    meets two at one distance, or an ulp apart."""
    import torch
    from petch import ops
    dev = mesh.device
    n = phi.numel()
    cnt = mesh.grid[0][:n].long() & 15
    gen = torch.Generator().manual_seed(4)
    twice = (torch.rand(n, generator=gen).to(dev) < share) & (cnt <= 7)
    new = torch.where(twice, 2 * cnt, cnt)
    first = torch.cumsum(new, 0) - new
    cells = torch.where(cnt > 0, (first << 4) | new, 0).to(torch.int32)
    copies = torch.repeat_interleave(torch.where(twice, 2, 1), cnt)
    faces = torch.repeat_interleave(mesh.faces, copies, dim=0)
    at = torch.cumsum(copies, 0)[copies == 2] - 1
    faces[at, 2] = mesh.nv + torch.arange(len(at), dtype=torch.int32, device=dev)
    verts = torch.cat([mesh.verts, mesh.centroids[copies == 2]]).contiguous()
    nx, ny, nz = phi.shape
    walked = ops.Bvh(dev).build(verts, faces).set_grid(verts, faces, (cells, nx, ny, nz, dx))
    assert walked.status() == 0
    return verts, faces, walked, ops.Bvh(dev).build(verts, faces)


# 3M rays: more ties than the list of a launch takes, so that the tree traces the rays left over
@pytest.mark.parametrize("name,share,n", [("hole", 0.3, 40000), ("trench", 0.05, 40001),
                                          ("flat", 0.5, 4097), ("noise", 0.2, 20000),
                                          ("thin", 0.1, 63), ("rough", 1.0, 20000),
                                          ("hole", 1.0, 3000000)])
def test_rays_that_meet_two_faces_at_once_take_the_trees(name, share, n, det):
    """A tied ray starts over on the tree and deposits what its walk had not: with coincident faces
    ties come at every bounce, and the deterministic sums and the numbers of hits are the tree's to
    the bit, in the batched launches too. (The adjoint's float sums: each adds at most 1e5 terms,
    in any order, 1e5 * 2^-24 of their mass at the very most; 1e-5 of it.)"""
    import torch
    from petch import flux, ops
    from petch.params import PAR
    mesh, phi, dx, box, dev = _surface(name)
    verts, faces, walked, tree = _doubled(mesh, phi, dx, share)
    nf = int(faces.shape[0])
    bare = torch.from_numpy(np.random.default_rng(3).uniform(0.05, 0.9, nf).astype(np.float32)).to(dev)
    par = dict(PAR, ion_source="powcos", ion_exponent=20.0)
    cen, area, nrm = ops.mesh_attrs(verts, faces)
    gn = ops.gas_normals(phi, dx, cen, nrm)
    src, isrc, ipar = flux.NEUTRAL_SOURCE, flux.ion_source(par), flux.ion_params(par)

    def fluxes(b):
        ops.trace_hit_counts(dev)
        a, o = ops.trace_neutral_rr_pair(b, box, src, bare, 0.7, n, 5, 1.0, n // 2, 6)
        out = [a.clone(), o.clone(), ops.trace_neutral_rr(b, box, src, bare, 0.3, n, 7).clone()]
        out += [x.clone() for x in ops.trace_ion_yield(b, box, isrc, ipar, n, 8)]
        out.append(ops.trace_neutral_cap(b, box, src, bare, 0.5, 4, n, 9).clone())
        hits = tuple(int(x) for x in ops.trace_hit_counts(dev))
        out.append(ops.trace_redeposition(b, cen, gn, area, bare, 0.5, n, 10).clone())
        if n < 1000000:
            out.append(ops.trace_ff(b, box, cen, gn, 24, 17).clone())
            items = [dict(bvh=b, box=box, bare=bare, beta_a=0.7, n_a=n // (k + 1), seed_a=3 + k,
                          beta_b=1.0, n_b=n // 2, seed_b=4) for k in range(3)]
            for x, y in ops.trace_neutral_rr_batch(src, items):
                out += [x.clone(), y.clone()]
            items = [dict(bvh=b, box=box, src=isrc, ion=ipar, n=n // (k + 1), seed=3 + k)
                     for k in range(3)]
            for x in ops.trace_ion_yield_batch(items):
                out += [y.clone() for y in x]
            g = ops.trace_neutral_rr_pair_adjoint(b, box, src, bare, 0.7, n, 5, a, 1.0, n // 2, 6, o)
        else:
            g = None
        assert b.status() == 0
        return out, hits, g
    (x, hx, gx), (y, hy, gy) = fluxes(walked), fluxes(tree)
    assert hx == hy and hx[0] >= n // 4
    for k, (p, q) in enumerate(zip(x, y)):
        assert torch.equal(p, q), (k, float((p - q).abs().max()))
    if gx is not None:
        assert float((gx - gy).abs().sum()) <= 1e-5 * float(gy.abs().sum())


@pytest.mark.parametrize("name", NAMES)
def test_rays_from_far_outside_hit_as_on_the_tree(name, det):
    """The rounding of an origin grows with its distance; beyond the grid's reach (about 100 cells,
    or the grid's own length where that is more) a ray is left to the tree: queries, rays that
    start there within a trace, and launches whose source plane lies there."""
    import torch
    from petch import flux, ops
    mesh, phi, dx, box, dev = _surface(name)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    g = torch.Generator().manual_seed(6)
    n, L = 100000, max(phi.shape) * dx
    for far in (2, 10, 100, 1000):
        q = mesh.faces.cpu().long()[torch.randint(0, mesh.nf, (n,), generator=g)]
        u = torch.rand((n, 3, 1), generator=g)
        aim = (mesh.verts.cpu()[q] * (u / u.sum(1, keepdim=True))).sum(1)
        d = torch.randn((n, 3), generator=g)
        d = d / d.norm(dim=1, keepdim=True)
        o = (aim - far * L * d).to(dev).contiguous()
        fa, ta = mesh.bvh.query_ray(o, d.to(dev))
        fb, tb = tree.query_ray(o, d.to(dev))
        assert int((fb >= 0).sum()) > n // 2
        print(name, far, int((fa != fb).sum()), int((ta != tb).sum()), flush=True)
        assert torch.equal(fa, fb) and torch.equal(ta, tb), far
    # form-factor rays from points up to 400 cells off, towards the surface
    q = torch.randint(0, mesh.nf, (mesh.nf,), generator=g).to(dev)
    d = torch.randn((mesh.nf, 3), generator=g).to(dev)
    d = d / d.norm(dim=1, keepdim=True)
    away = torch.linspace(0.0, 400.0, mesh.nf, device=dev)[:, None] * dx
    cen = (mesh.centroids[q] - away * d).contiguous()
    a, b = (ops.trace_ff(t, box, cen, d.contiguous(), 256, 3) for t in (mesh.bvh, tree))
    assert int((b >= 0).sum()) > 100 and torch.equal(a, b)
    bare = torch.full((mesh.nf,), 0.5, device=dev)
    far_box = ops.make_box(*(s * dx for s in phi.shape[:2]), 1e4 * L, 300 * L, 1)
    a, b = (ops.trace_neutral_rr(t, far_box, flux.NEUTRAL_SOURCE, bare, 0.5, 20000, 3)
            for t in (mesh.bvh, tree))
    assert float(b.sum()) > 0 and torch.equal(a, b)


@pytest.mark.parametrize("name", ["hole", "trench"])
def test_traces_in_large_units_equal_the_trees(name, det):
    """With coordinates of thousands, re-emission points 1e-4 off the surface round onto it or below,
    and the next query may meet the same face again, on the walk as on the tree."""
    import torch
    from petch import flux, ops
    from petch.params import PAR
    phi, dx, per = _phi(name)
    dev, dx = torch.device("cuda", 0), dx * 1000.0
    tphi = torch.from_numpy(np.ascontiguousarray(phi * 1000.0, np.float32)).to(dev)
    mesh = flux.SurfaceMesh(dev).build(tphi, dx)
    L = [n * dx for n in phi.shape]
    box = ops.make_box(*L, L[2] - dx, per)
    tree = ops.Bvh(dev).build(mesh.verts, mesh.faces)
    bare = torch.full((mesh.nf,), 0.4, device=dev)
    par = dict(PAR, ion_source="powcos", ion_exponent=20.0)

    def run(b):
        ops.trace_hit_counts(dev)
        out = [ops.trace_neutral_rr(b, box, flux.NEUTRAL_SOURCE, bare, 0.5, 50000, 7).clone(),
               ops.trace_ion_yield(b, box, flux.ion_source(par), flux.ion_params(par), 50000, 8)]
        return out, ops.trace_hit_counts(dev)
    (a, ha), (b, hb) = run(mesh.bvh), run(tree)
    print(name, ha, hb, flush=True)
    assert ha == hb and all(torch.equal(x, y) for x, y in zip(a, b))
