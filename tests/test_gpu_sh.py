"""GPU tests of the SH-PRT render (nwprt_sh_render: RenderEngine::shRender,
Renderer/RenderEngine.cpp:459-486, and __closesthit__SHradiance,
Renderer/device_functions/devicePrograms.cu:312-501) against the FP64
oracle's replay of the same random stream (orc_sh_render).

Bar: on pixels whose first hit is away from edges and ties (oracle margin
>= 1e-4), |gpu - oracle| <= 1e-3 (|oracle| + 1e-2 max): the two differ
only by FP32 rounding (no shadow rays, so no sample can flip)."""
import numpy as np
import pytest

from cases import mesh_scene

pytestmark = pytest.mark.gpu


def _scene(seed, sphere=(48, 24), soup=40):
    s = mesh_scene(seed, sphere=sphere, soup=soup, mirror=False)
    return s  # roughPlastic x 2 + cookTorrance


@pytest.mark.parametrize("seed,w,h,degree,samples,kinds", [(0, 32, 24, 2, 32, None),
                                                           (1, 29, 17, 0, 16, None),
                                                           (2, 24, 16, 8, 8, None),
                                                           (3, 16, 12, 4, 16, (4, 2, 0)),
                                                           (4, 24, 16, 2, 16, (1, 1, 2))])
def test_sh_render_replays_oracle(nw, orc, ctx, seed, w, h, degree, samples, kinds):
    s = _scene(seed, sphere=(16, 8) if degree == 8 else (48, 24), soup=10 if degree == 8 else 40)
    if kinds is not None:
        # DisneyBSDF rows take a plastic-with-sheen and a tinted-metal set
        disney = [(0.0, 0.0, 0.4, 0.5, 0.2, 0.0, 0.7, 0.5, 0.6, 0.3, 1.5),
                  (0.0, 0.9, 0.0, 0.5, 0.5, 0.6, 0.0, 0.5, 0.0, 1.0, 1.45)]
        mats = np.array([nw.material_row(m) for m in s["materials"]], np.float32)
        mats[:3, 7] = kinds
        for i, k in enumerate(kinds):
            if k == 1:
                mats[i, 8:] = disney[i % 2]
        s["materials"] = mats
    rng = np.random.default_rng(seed)
    nc = (degree + 1) ** 2
    nv = len(s["vertices"])
    T = (rng.normal(0, 0.3, (nv, nc, nc, 3)) + np.eye(nc)[None, :, :, None]).astype(np.float32)
    L = rng.normal(0, 1, (nc, 3)).astype(np.float32)
    L[0] = [3.0, 2.5, 2.0]
    view = rng.lognormal(0, 1, (6, 4, 4, 3)).astype(np.float32)
    mesh = ctx.mesh_create(s["vertices"], s["indices"], s["materials"], normals=s["normals"],
                           material_ids=s["material_ids"])
    dT, dL, dv = (nw.DeviceBuffer.from_array(x) for x in (T, L, view))
    out = nw.DeviceBuffer(w * h * 16)
    ctx.sh_render(mesh, np.reshape(s["camera"], (3, 3)), w, h, dT, dL, degree, out,
                  brdf_samples=samples, seed=77 + seed, env_faces=dv, env_n=4)
    ctx.sync()
    got = out.download(np.float32, (w * h, 4)).astype(np.float64)
    want = orc.sh_render(s["vertices"], s["indices"], s["normals"], s["materials"], s["camera"],
                         w, h, T, L, degree, material_ids=s["material_ids"], samples=samples,
                         seed=77 + seed, env_faces=view)
    safe = want["margin"] >= 1e-4
    assert safe.mean() > 0.95
    ref = want["color"]
    top = np.abs(ref[:, :3]).max()
    err = np.abs(got[safe, :3] - ref[safe, :3]) / (np.abs(ref[safe, :3]) + 1e-2 * top)
    assert err.max() <= 1e-3, err.max()
    assert np.all(got[:, 3] == 1.0)
    assert (want["prim"] >= 0).sum() > 0.2 * w * h
    ctx.mesh_destroy(mesh)


@pytest.mark.parametrize("degree", [0, 1, 2, 3])
def test_sh_light_response_forms(nw, orc, ctx, degree):
    """Light response by one wave (degree 0) and four waves a vertex, with a
    vertex count that is no multiple of four and rows no multiple of the
    waves: the oracle's colours."""
    s = _scene(5, sphere=(11, 7), soup=3)
    nv, nc, w, h = len(s["vertices"]), (degree + 1) ** 2, 24, 16
    assert nv % 4
    rng = np.random.default_rng(degree)
    T = rng.normal(0, 0.5, (nv, nc, nc, 3)).astype(np.float32)
    L = rng.normal(0, 1, (nc, 3)).astype(np.float32)
    mesh = ctx.mesh_create(s["vertices"], s["indices"], s["materials"], normals=s["normals"],
                           material_ids=s["material_ids"])
    out = nw.DeviceBuffer(w * h * 16)
    ctx.sh_render(mesh, np.reshape(s["camera"], (3, 3)), w, h, nw.DeviceBuffer.from_array(T),
                  nw.DeviceBuffer.from_array(L), degree, out, brdf_samples=8, seed=5)
    ctx.sync()
    got = out.download(np.float32, (w * h, 4)).astype(np.float64)
    want = orc.sh_render(s["vertices"], s["indices"], s["normals"], s["materials"], s["camera"],
                         w, h, T, L, degree, material_ids=s["material_ids"], samples=8, seed=5)
    safe = want["margin"] >= 1e-4
    ref = want["color"][safe, :3]
    err = np.abs(got[safe, :3] - ref) / (np.abs(ref) + 1e-2 * np.abs(ref).max())
    assert err.max() <= 1e-3, err.max()
    ctx.mesh_destroy(mesh)


@pytest.mark.parametrize("degree,at_end", [(0, True), (2, False)])
def test_sh_render_many_vertices(nw, orc, ctx, degree, at_end):
    """More vertices than a launch of one 256-thread workgroup each could take
    (2^32 threads): the render still runs, with a few of them in use (the last
    ones at degree 0, the first at degree 2)."""
    s = _scene(7, sphere=(16, 8), soup=4)
    used, n, nc, w, h = len(s["vertices"]), (1 << 24) + 5, (degree + 1) ** 2, 24, 16
    rng = np.random.default_rng(2)
    T = rng.normal(0, 1, (used, nc, nc, 3)).astype(np.float32)
    L = rng.normal(0, 1, (nc, 3)).astype(np.float32)
    first = n - used if at_end else 0
    v = np.zeros((n, 3), np.float32)
    nr = np.zeros((n, 3), np.float32)
    nr[:, 2] = 1.0
    v[first:first + used], nr[first:first + used] = s["vertices"], s["normals"]
    ix = s["indices"] + np.int32(first)
    dT = nw.DeviceBuffer(n * nc * nc * 12)
    if at_end:
        full = np.zeros((n, nc, nc, 3), np.float32)
        full[first:] = T
        dT.upload(full)
    else:
        full = None
        dT.zero()
        dT.upload(T)
    print(f"sh_render {n} vertices degree {degree}", flush=True)
    mesh = ctx.mesh_create(v, ix, s["materials"], normals=nr, material_ids=s["material_ids"])
    out = nw.DeviceBuffer(w * h * 16)
    ctx.sh_render(mesh, np.reshape(s["camera"], (3, 3)), w, h, dT, nw.DeviceBuffer.from_array(L),
                  degree, out, brdf_samples=8, seed=9)
    ctx.sync()
    got = out.download(np.float32, (w * h, 4))
    ctx.mesh_destroy(mesh)
    if at_end:
        want = orc.sh_render(v, ix, nr, s["materials"], s["camera"], w, h, full, L, degree,
                             material_ids=s["material_ids"], samples=8, seed=9)
        safe = want["margin"] >= 1e-4
        ref = want["color"][safe, :3]
        err = np.abs(got[safe, :3] - ref) / (np.abs(ref) + 1e-2 * np.abs(ref).max())
        assert err.max() <= 1e-3, err.max()
    else:  # the same vertices alone, where four waves share each
        mesh = ctx.mesh_create(v[:used], ix, s["materials"], normals=nr[:used],
                               material_ids=s["material_ids"])
        small = nw.DeviceBuffer(w * h * 16)
        ctx.sh_render(mesh, np.reshape(s["camera"], (3, 3)), w, h, dT,
                      nw.DeviceBuffer.from_array(L), degree, small, brdf_samples=8, seed=9)
        ctx.sync()
        ref = small.download(np.float32, (w * h, 4))
        ctx.mesh_destroy(mesh)
        assert np.any(ref[:, :3] != ref[0, :3])
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_sh_render_errors(nw, ctx):
    s = mesh_scene(0)  # has a mirror
    T = nw.DeviceBuffer(len(s["vertices"]) * 9 * 9 * 12)
    L = nw.DeviceBuffer(9 * 12)
    out = nw.DeviceBuffer(8 * 8 * 16)
    cam = np.reshape(s["camera"], (3, 3))
    mesh = ctx.mesh_create(s["vertices"], s["indices"], s["materials"], normals=s["normals"],
                           material_ids=s["material_ids"])
    with pytest.raises(nw.NwprtError) as e:
        ctx.sh_render(mesh, cam, 8, 8, T, L, 2, out)
    assert e.value.status == nw.ERR_UNSUPPORTED
    ctx.mesh_destroy(mesh)
    s = mesh_scene(0, mirror=False)
    mesh = ctx.mesh_create(s["vertices"], s["indices"], s["materials"])  # no normals
    with pytest.raises(nw.NwprtError) as e:
        ctx.sh_render(mesh, cam, 8, 8, T, L, 2, out)
    assert e.value.status == nw.ERR_INVALID_ARGUMENT
    ctx.mesh_destroy(mesh)
    mesh = ctx.mesh_create(s["vertices"], s["indices"], s["materials"], normals=s["normals"])
    for kw in ({"degree": 9}, {"degree": -1}, {"brdf_samples": 0}):
        args = {"degree": 2, "brdf_samples": 4}
        args.update(kw)
        with pytest.raises(nw.NwprtError) as e:
            ctx.sh_render(mesh, cam, 8, 8, T, L, args["degree"], out,
                          brdf_samples=args["brdf_samples"])
        assert e.value.status == nw.ERR_INVALID_ARGUMENT
    ctx.mesh_destroy(mesh)
