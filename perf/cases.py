"""Performance cases of the relighting framework: the calls a program that
renders with it makes, over the sizes, precisions and options in real use.

Each case is a dict of plain values; `prepare` builds what a program holds
before the call (scene, environment map, G-buffer, mesh, batch or server in
device memory), `run` is one pass through the public entry points, `exact`
the same result in FP64 with torch alone.

Kinds:
  relight   environment map from new or turned cubemap faces, then a relight
            of the frame (nwprt_envmap_update_faces / _rotated, nwprt_relight)
  two_pass  pass p1 + pass p2 over a resident selection, reference-layout
            scene with the G-buffer's aux inputs (TCNNPass_p1 / TCNNPass_p2)
  batch     jobs of uneven size as one captured graph (nwprt_batch_launch)
  served    requests through the request server until all are done
  denoise   the edge-avoiding filter over a relit frame (nwprt_denoise)
  cast      the G-buffer of a triangle mesh with its direct term
  sh_render the SH-PRT baseline's frame from transfer matrices
  transfer  the SH-PRT baseline's transfer matrices (path tracing)
"""
import math
import random

import numpy as np
import torch

import neural_wavelet_prt_demo_amd as nw
from neural_wavelet_prt_demo_amd import DeviceBuffer, DeviceFrame

LEVELS, GROWTH, BASE, LOG2_T = 16, 1.5, 16, 19
DENOISE_PASSES = 5
PRECISION = {"fp32": nw.PREC_FP32, "fp16": nw.PREC_FP16, "bf16": nw.PREC_BF16,
             "fp8": nw.PREC_FP8}
LUM = (0.212671, 0.715160, 0.072169)


def listed():
    return [
        # A thumbnail or probe frame whose light changes on every call: the
        # smallest relight of the workloads (128 x 128, 6 x 32 x 32 map, K 64).
        # Launches and the selection's latency count, not arithmetic.
        {"name": "probe_bf16", "kind": "relight", "w": 128, "h": 128, "n": 32, "k": 64,
         "prec": "bf16", "env": "faces", "hash": "f32", "background": 0.0},
        # The headline request: full-HD frame, 6 x 128 x 128 map, K 300.
        {"name": "frame_bf16", "kind": "relight", "w": 1920, "h": 1080, "n": 128, "k": 300,
         "prec": "bf16", "env": "faces", "hash": "f16", "background": 0.0},
        # The same request in FP8 with the light turned about the vertical,
        # as 70 % of the served stream's requests ask for.
        {"name": "frame_fp8_rotated", "kind": "relight", "w": 1920, "h": 1080, "n": 128, "k": 300,
         "prec": "fp8", "env": "rotated", "hash": "f16", "background": 0.0},
        # A window of odd size with sky behind the scene, in the reference's
        # own precision and with the drop-in workload's map size and K.
        {"name": "window_fp16", "kind": "relight", "w": 1283, "h": 717, "n": 64, "k": 128,
         "prec": "fp16", "env": "faces", "hash": "f16", "background": 0.3},
        # The plain FP32 form, used where radiance is checked or baked: the
        # precision study's network on a quarter-HD frame.
        {"name": "still_fp32", "kind": "relight", "w": 960, "h": 540, "n": 64, "k": 64,
         "prec": "fp32", "env": "faces", "hash": "f32", "background": 0.05},
        # A reference-layout model (aux inputs from the G-buffer, no
        # projection) through the interactive loop's two passes.
        {"name": "loop_aux_fp16", "kind": "two_pass", "w": 1280, "h": 720, "n": 64, "k": 64,
         "prec": "fp16", "hash": "f16", "background": 0.1},
        # Offline jobs of uneven size and K packed into one graph.
        {"name": "batch_bf16", "kind": "batch", "jobs": 6, "pick": 3, "n": 64, "prec": "bf16"},
        # A burst of requests through the server: turned, fresh and resident
        # maps, full-HD and smaller views.
        {"name": "served_bf16", "kind": "served", "requests": 5, "pick": 4, "n": 128, "k": 300,
         "prec": "bf16"},
        # The filter after the relight at full HD, default five passes.
        {"name": "denoise", "kind": "denoise", "w": 1920, "h": 1080},
        # The step before the relight: primary rays and one direct-light
        # sample per pixel over a quarter of a million triangles.
        {"name": "cast_direct", "kind": "cast", "w": 1920, "h": 1080, "grid": 320, "samples": 1,
         "n": 64},
        # The SH baseline's frame at the reference's tested degree.
        {"name": "sh_frame", "kind": "sh_render", "w": 1920, "h": 1080, "sphere": 192,
         "degree": 8, "samples": 64, "n": 64},
        # The SH baseline's precomputation on a small model.
        {"name": "sh_transfer", "kind": "transfer", "sphere": 64, "degree": 4, "samples": 64},
    ]


def _size(rng, lo, hi, odd=0.5):
    """A size spread over the logarithm of [lo, hi]; odd half the time."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, v | 1) if rng.random() < odd else v


def draw(rng):
    kind = rng.choice(["relight"] * 5 + ["two_pass", "batch", "served", "denoise", "cast",
                                         "sh_render", "transfer"])
    w = _size(rng, 33, 1920)
    h = max(17, min(1080, int(w * rng.uniform(0.4, 1.1))))
    if kind == "relight":
        prec = rng.choice(["fp32", "fp16", "bf16", "bf16", "fp8"])
        n = rng.choice([16, 32, 64, 128])
        if prec == "fp32":  # stills: up to a quarter of full HD
            w, h = min(w, 961), min(h, 541)
        return {"kind": kind, "w": w, "h": h, "n": n, "k": _size(rng, 16, 96 if prec == "fp32" else 300),
                "prec": prec, "env": rng.choice(["faces", "rotated"]),
                "hash": rng.choice(["f16", "f32"]), "background": round(rng.uniform(0.0, 0.5), 3)}
    if kind == "two_pass":
        return {"kind": kind, "w": w, "h": h, "n": rng.choice([32, 64, 128]),
                "k": _size(rng, 16, 128), "prec": rng.choice(["fp16", "bf16"]), "hash": "f16",
                "background": round(rng.uniform(0.0, 0.4), 3)}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(2, 6), "pick": rng.randrange(1000), "n": 64,
                "prec": rng.choice(["bf16", "fp16"])}
    if kind == "served":
        return {"kind": kind, "requests": rng.randint(1, 5), "pick": rng.randrange(1000),
                "n": rng.choice([64, 128]), "k": _size(rng, 32, 300), "prec": "bf16"}
    if kind == "denoise":
        return {"kind": kind, "w": w, "h": h}
    if kind == "cast":
        return {"kind": kind, "w": w, "h": h, "grid": _size(rng, 24, 320),
                "samples": rng.randint(0, 2), "n": rng.choice([32, 64])}
    if kind == "sh_render":
        return {"kind": kind, "w": w, "h": h, "sphere": _size(rng, 24, 192),
                "degree": rng.choice([2, 4, 8]), "samples": rng.choice([16, 64]), "n": 64}
    return {"kind": kind, "sphere": _size(rng, 12, 64), "degree": rng.choice([1, 2, 4]),
            "samples": rng.choice([32, 64])}


# ------------------------------------------------------------------ inputs --

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + stream * 7919) & 0x7FFFFFFF)
    return g


def _normal(seed, stream, shape, std):
    return torch.randn(shape, generator=_gen(seed, stream), device="cuda") * std


def _uniform(seed, stream, shape):
    return torch.rand(shape, generator=_gen(seed, stream), device="cuda")


def _level_table(n_levels=LEVELS):
    """Scale, resolution, dense flag, size and offset of each grid level
    (FP32 scale: exp2(l log2 b) N_min - 1, rounded at each step)."""
    f = np.float32
    lb = f(math.log2(GROWTH))
    out, off = [], 0
    for l in range(n_levels):
        s = f(f(2.0 ** float(f(f(l) * lb))) * f(BASE)) - f(1.0)
        res = int(math.ceil(float(s))) + 1
        dense = res ** 3 <= 1 << LOG2_T
        size = min((res ** 3 + 7) // 8 * 8, 1 << LOG2_T) if dense else 1 << LOG2_T
        out.append((f(s), res, dense, size, off))
        off += size
    return out, off


def _scene_arrays(seed, n, hash_dtype, aux):
    """Trained-network stand-in: hash entries N(0, 0.1), wavelet features
    N(0, 0.1), He-normal layers, LeCun-normal projection (none with aux,
    whose wavelet features are larger, as the reference's layout has it)."""
    _, entries = _level_table()
    std = 0.5 if aux else 0.1
    h = _normal(seed, 1, (entries, 2), std)
    h = h.half() if hash_dtype == "f16" else h
    a = {"hash": h, "wfeat": _normal(seed, 2, (32, 6 * n * n), std),
         "proj": None if aux else _normal(seed, 3, (32, 32), 1 / math.sqrt(32))}
    a["w1"] = _normal(seed, 4, (64, 32), math.sqrt(2 / 32))
    a["w2"] = _normal(seed, 5, (64, 64), math.sqrt(2 / 64))
    a["w3"] = _normal(seed, 6, (64, 64), math.sqrt(2 / 64))
    a["w4"] = _normal(seed, 7, (3, 64), math.sqrt(2 / 64))
    a["waux"] = _normal(seed, 8, (64, 16), math.sqrt(2 / 80)) if aux else None
    return a


def _make_scene(ctx, n, hash_dtype, aux, a):
    desc = nw.config_scene_desc(n, nw.DTYPE_F16 if hash_dtype == "f16" else nw.DTYPE_F32,
                                projection=not aux, aux=aux)
    layers = [a["w1"], a["w2"], a["w3"], a["w4"]] + ([a["waux"]] if aux else [])
    h = a["hash"].cpu().numpy()
    return ctx.scene_create(desc, {
        "hash_table": h.view(np.uint16) if hash_dtype == "f16" else h,
        "wavelet_features": a["wfeat"].cpu().numpy(),
        "projection": None if aux else a["proj"].cpu().numpy(),
        "layers": torch.cat([x.reshape(-1) for x in layers]).cpu().numpy()})


def _faces(seed, n, stream=20):
    """Log-normal radiance with a 3 x 3-texel sun of 1e3 on one face."""
    f = torch.exp(1.5 * _normal(seed, stream, (6, n, n, 3), 1.0))
    r = random.Random(seed * 31 + stream)
    face, row, col = r.randrange(6), r.randrange(1, n - 1), r.randrange(1, n - 1)
    f[face, row - 1:row + 2, col - 1:col + 2] = 1e3
    return f


def _sphere_dirs(u, v):
    z = 1 - 2 * u
    r = torch.sqrt(torch.clamp(1 - z * z, min=0))
    return torch.stack([r * torch.cos(2 * math.pi * v), r * torch.sin(2 * math.pi * v), z], -1)


def _gbuffer(seed, w, h, background, surface=False):
    """G-buffer planes in the reference's encodings.  Positions are uniform in
    the unit cube, or with `surface` those of a rolling surface seen by a
    camera (neighbouring pixels close together)."""
    P = w * h
    if surface:
        y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"),
                              indexing="ij")
        fx, fy = (x.reshape(-1) + 0.5) / w, (y.reshape(-1) + 0.5) / h
        ph = 6.28 * _uniform(seed, 30, (3,))
        z = 0.5 + 0.2 * torch.sin(9 * fx + ph[0]) * torch.cos(7 * fy + ph[1]) \
            + 0.1 * torch.sin(23 * fx + 17 * fy + ph[2])
        pos = torch.stack([fx, fy, z], -1).float()
    else:
        pos = _uniform(seed, 30, (P, 3))
    u = _uniform(seed, 31, (P, 4))
    n = _sphere_dirs(u[:, 0], u[:, 1])
    v = _sphere_dirs(u[:, 2], u[:, 3])
    ndv = (n * v).sum(-1, keepdim=True)
    v = torch.where(ndv < 0, -v, v)
    r = 2 * ndv.abs() * n - v
    m = _uniform(seed, 32, (P, 11))
    one = torch.ones((P, 1), device="cuda")
    return {"position": torch.cat([pos, one], 1), "normal": torch.cat([n * 0.5 + 0.5, one], 1),
            "reflect": torch.cat([r * 0.5 + 0.5, one], 1), "kd": torch.cat([m[:, 0:3], one], 1),
            "ks": torch.cat([m[:, 3:6], one], 1), "direct": torch.cat([m[:, 6:9], one], 1),
            "roughness": 0.05 + 0.95 * m[:, 9],
            "env_flag": (m[:, 10] >= background).to(torch.uint8)}


def _yaw(seed, i=0):
    return random.Random(seed * 17 + i).uniform(0.1, 6.1)


def _plan(case):
    """Jobs of a batch, or requests of a served burst, from the case alone."""
    r = random.Random(case["pick"])
    sizes = [(256, 256), (512, 512), (1280, 720), (1920, 1080)]
    if case["kind"] == "batch":
        return [(*r.choice(sizes), r.choice([32, 64, 128, 300])) for _ in range(case["jobs"])]
    return [(*r.choice([(1920, 1080), (1280, 720), (961, 541)]),
             r.choice(["rotated", "rotated", "fresh", "resident"]))
            for _ in range(case["requests"])]


def _heightfield(seed, grid):
    """A rolling heightfield of grid x grid cells with vertex normals under a
    sphere, three glossy materials."""
    r = random.Random(seed)
    a, b, c = (r.uniform(0.0, 6.28) for _ in range(3))
    xs, zs = np.linspace(-8.0, 8.0, grid + 1), np.linspace(-9.0, 5.0, grid + 1)
    X, Z = np.meshgrid(xs, zs)
    Y = -1.5 + 0.35 * np.sin(0.9 * X + a) * np.cos(0.7 * Z + b) + 0.1 * np.sin(3.1 * X + 2.3 * Z + c)
    dx = 0.315 * np.cos(0.9 * X + a) * np.cos(0.7 * Z + b) + 0.31 * np.cos(3.1 * X + 2.3 * Z + c)
    dz = -0.245 * np.sin(0.9 * X + a) * np.sin(0.7 * Z + b) + 0.23 * np.cos(3.1 * X + 2.3 * Z + c)
    nr = np.stack([-dx, np.ones_like(X), -dz], -1).reshape(-1, 3)
    nr /= np.linalg.norm(nr, axis=1, keepdims=True)
    i0 = (np.arange(grid)[:, None] * (grid + 1) + np.arange(grid)[None, :]).reshape(-1)
    ti = np.concatenate([np.stack([i0, i0 + grid + 1, i0 + 1], 1),
                         np.stack([i0 + 1, i0 + grid + 1, i0 + grid + 2], 1)])
    sv, sn, si = _sphere(max(16, grid // 2), (0.5, 0.2, -2.0), 1.6)
    verts = np.concatenate([np.stack([X, Y, Z], -1).reshape(-1, 3), sv])
    mids = np.concatenate([(np.arange(len(ti)) // 4096) % 2, np.full(len(si), 2)])
    mats = [[0.45, 0.4, 0.3, 0.04, 0.04, 0.04, 0.6, 2], [0.3, 0.45, 0.25, 0.04, 0.04, 0.04, 0.8, 2],
            [0.8, 0.2, 0.2, 0.5, 0.5, 0.5, 0.15, 2]]
    return (verts, np.concatenate([nr, sn]), np.concatenate([ti, si + (grid + 1) ** 2]),
            mids.astype(np.int32), mats)


def _sphere(nu, centre, radius):
    nv = max(4, nu // 2)
    T, PH = np.meshgrid(np.linspace(0, np.pi, nv + 1),
                        np.linspace(0, 2 * np.pi, nu, endpoint=False), indexing="ij")
    n = np.stack([np.sin(T) * np.cos(PH), np.cos(T), np.sin(T) * np.sin(PH)], -1).reshape(-1, 3)
    a = (np.arange(nv)[:, None] * nu + np.arange(nu)[None, :]).reshape(-1)
    b = (np.arange(nv)[:, None] * nu + (np.arange(nu)[None, :] + 1) % nu).reshape(-1)
    idx = np.concatenate([np.stack([a, a + nu, b], 1), np.stack([b, a + nu, b + nu], 1)])
    return np.asarray(centre) + radius * n, n, idx


def _sphere_scene(seed, nu):
    """A glossy sphere over a rough ground quad, with vertex normals."""
    y = 0.2 + 0.1 * random.Random(seed).random()
    sv, sn, si = _sphere(nu, (0.0, y, -2.0), 1.6)
    g = np.array([[-8, -1.6, -9], [8, -1.6, -9], [8, -1.6, 5], [-8, -1.6, 5]])
    idx = np.concatenate([si, np.array([[0, 2, 1], [0, 3, 2]]) + len(sv)])
    mids = np.concatenate([np.zeros(len(si)), np.ones(2)]).astype(np.int32)
    mats = [[0.8, 0.3, 0.2, 0.04, 0.04, 0.04, 0.3, 2], [0.5, 0.5, 0.5, 0.04, 0.04, 0.04, 0.8, 0]]
    return (np.concatenate([sv, g]), np.concatenate([sn, np.tile([0.0, 1.0, 0.0], (4, 1))]), idx,
            mids, mats)


CAMERA = [[0.0, 2.5, 7.5], [0.0, -0.8, -2.0], [0.0, 1.0, 0.0]]


# ------------------------------------------------------------------- state --

_CTX = None


def _context():
    """One context per process, as a renderer holds it."""
    global _CTX
    if _CTX is None:
        _CTX = nw.Context(0)
    return _CTX


class _Raw:
    """A device buffer's memory as torch sees it."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (buf.ptr, False), "version": 2}


_TYPES = {torch.float32: "<f4", torch.int32: "<i4", torch.uint8: "|u1"}


def _view(buf, shape, dtype=torch.float32):
    return torch.as_tensor(_Raw(buf, shape, _TYPES[dtype]), device="cuda")


def _device(t):
    """A DeviceBuffer that holds tensor t."""
    b = DeviceBuffer(t.numel() * t.element_size())
    _view(b, t.shape, t.dtype).copy_(t)
    return b


def _frame(g, w, h):
    f = DeviceFrame(w, h)
    for k, v in g.items():
        _view(f.bufs[k], v.shape, v.dtype).copy_(v)
    return f


def _outputs(frame, rgba8=True):
    P = frame.width * frame.height
    out = {"indirect": _view(frame.out["indirect"], (P, 4)),
           "with_direct": _view(frame.out["indirect_with_direct"], (P, 4))}
    if rgba8:
        out["rgba8"] = _view(frame.out["rgba8"], (P,), torch.int32)
    return out


class _State:
    """Handles of one prepared case; given back when it is dropped."""

    def __init__(self, case):
        self.case, self.ctx = case, _context()
        self.owned = []

    def own(self, kind, handle):
        self.owned.append((kind, handle))
        return handle

    def __del__(self):
        try:
            for kind, handle in reversed(self.owned):
                getattr(self.ctx, kind + "_destroy")(handle)
        except Exception:
            pass


def prepare(case, seed):
    s = _State(case)
    ctx, kind = s.ctx, case["kind"]
    if kind in ("relight", "two_pass"):
        aux = kind == "two_pass"
        s.prec = PRECISION[case["prec"]]
        s.scene = s.own("scene", _make_scene(ctx, case["n"], case["hash"], aux,
                                             _scene_arrays(seed, case["n"], case["hash"], aux)))
        s.frame = _frame(_gbuffer(seed, case["w"], case["h"], case["background"], surface=aux),
                         case["w"], case["h"])
        s.faces = _device(_faces(seed, case["n"]))
        torch.cuda.synchronize()
        s.env = s.own("envmap", ctx.envmap_from_faces(s.faces, case["k"], face_size=case["n"]))
        s.yaw = _yaw(seed)
        s.rgba8 = case["prec"] != "fp8"  # FP8 renders feed the denoiser, not the screen
        s.fo = s.frame.frame_out(rgba8=s.rgba8)
        s.out = _outputs(s.frame, s.rgba8)
    elif kind == "batch":
        a = [_scene_arrays(seed + i, case["n"], "f16", False) for i in range(2)]
        scenes = [s.own("scene", _make_scene(ctx, case["n"], "f16", False, x)) for x in a]
        s.frames, s.keep, jobs = [], [], []
        for j, (w, h, k) in enumerate(_plan(case)):
            f = _frame(_gbuffer(seed + 100 * j, w, h, 0.0), w, h)
            s.keep.append(_device(_faces(seed, case["n"], 20 + j)))
            torch.cuda.synchronize()
            env = s.own("envmap", ctx.envmap_from_faces(s.keep[-1], k, face_size=case["n"]))
            s.frames.append(f)
            jobs.append((scenes[j % 2], env, f))
        s.batch = s.own("batch", ctx.batch_create(jobs, PRECISION[case["prec"]]))
        s.out = [_outputs(f) for f in s.frames]
    elif kind == "served":
        s.scene = s.own("scene", _make_scene(ctx, case["n"], "f16", False,
                                             _scene_arrays(seed, case["n"], "f16", False)))
        s.frames, s.reqs = [], []
        for j, (w, h, env) in enumerate(_plan(case)):
            f = _frame(_gbuffer(seed + 100 * j, w, h, 0.0), w, h)
            d = _device(_faces(seed, case["n"], 20 + j))
            torch.cuda.synchronize()
            if env == "resident":
                e = s.own("envmap", ctx.envmap_from_faces(d, case["k"], face_size=case["n"]))
                s.reqs.append((f, {"env": e}, d))
            elif env == "rotated":
                s.reqs.append((f, {"faces": d, "yaw": _yaw(seed, j), "k": case["k"],
                                   "face_size": case["n"]}, d))
            else:  # a fresh map arrives in host memory
                host = d.download(np.float32, (6, case["n"], case["n"], 3))
                s.reqs.append((f, {"faces": host, "k": case["k"], "face_size": case["n"]}, d))
            s.frames.append(f)
        s.server = s.own("server", ctx.server_create(precision=PRECISION[case["prec"]]))
        s.out = [_outputs(f) for f in s.frames]
    elif kind == "denoise":
        s.bufs = {k: _device(v) for k, v in _denoise_inputs(case, seed).items()}
        s.dst = DeviceBuffer(case["w"] * case["h"] * 16)
        s.out = _view(s.dst, (case["h"], case["w"], 4))
    elif kind == "cast":
        v, nr, ix, mid, mats = _heightfield(seed, case["grid"])
        s.mesh = s.own("mesh", ctx.mesh_create(v, ix, mats, normals=nr, material_ids=mid))
        s.frame = DeviceFrame(case["w"], case["h"])
        P = case["w"] * case["h"]
        for k, b in s.frame.bufs.items():
            dt, c = nw.GBUFFER_FIELDS[k]
            _view(b, (b.nbytes,), torch.uint8).zero_()
        s.faces = _device(_faces(seed, case["n"]))
        s.out = {k: _view(s.frame.bufs[k], (P, c) if c > 1 else (P,),
                          torch.uint8 if dt == np.uint8 else torch.float32)
                 for k, (dt, c) in nw.GBUFFER_FIELDS.items()}
    elif kind == "sh_render":
        v, nr, ix, mid, mats = _sphere_scene(seed, case["sphere"])
        s.mesh = s.own("mesh", ctx.mesh_create(v, ix, mats, normals=nr, material_ids=mid))
        nc = (case["degree"] + 1) ** 2
        # Transfer matrices decay with the band of row and column.
        band = torch.floor(torch.sqrt(torch.arange(nc, device="cuda").float()))
        amp = 0.3 / ((1 + band)[:, None] * (1 + band)[None, :])
        T = torch.randn((len(v), nc * nc, 3), generator=_gen(seed, 40), device="cuda")
        T *= amp.reshape(1, nc * nc, 1)
        s.transfer = _device(T)
        del T
        L = _normal(seed, 41, (nc, 3), 0.2)
        L[0] = torch.tensor([2.0, 1.8, 1.6], device="cuda")
        s.light, s.faces = _device(L), _device(_faces(seed, case["n"]))
        s.dst = DeviceBuffer(case["w"] * case["h"] * 16)
        s.out = _view(s.dst, (case["h"], case["w"], 4))
    else:
        v, nr, ix, mid, mats = _sphere_scene(seed, case["sphere"])
        s.mesh = s.own("mesh", ctx.mesh_create(v, ix, mats, normals=nr, material_ids=mid))
        nc = (case["degree"] + 1) ** 2
        s.basis = DeviceBuffer.from_array(nw.sh_basis_faces(case["degree"], 32))
        s.dst = DeviceBuffer(len(v) * nc * nc * 12)
        s.out = _view(s.dst, (len(v), nc * nc, 3))
    s.seed = seed
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s.case, s.ctx
    kind = case["kind"]
    if kind == "relight":
        if case["env"] == "rotated":
            ctx.envmap_update_rotated(s.env, s.faces, s.yaw)
        else:
            ctx.envmap_update_faces(s.env, s.faces)
        ctx.relight(s.scene, s.env, s.frame, s.prec, out=s.fo)
    elif kind == "two_pass":
        ctx.TCNNPass_p1(s.scene, 0, s.frame, s.prec)
        ctx.TCNNPass_p2(s.scene, s.env, 0, s.frame, s.prec)
    elif kind == "batch":
        ctx.batch_launch(s.batch)
    elif kind == "served":
        for f, req, _ in s.reqs:
            ctx.server_submit(s.server, s.scene, f, **req)
        ctx.server_poll(s.server, wait=2)
    elif kind == "denoise":
        ctx.denoise(s.bufs["color"], s.bufs["normal"], s.bufs["albedo"], s.dst, case["w"],
                    case["h"])
    elif kind == "cast":
        light = {"light_faces": s.faces, "light_n": case["n"],
                 "direct_samples": case["samples"]} if case["samples"] else {}
        ctx.gbuffer_cast(s.mesh, CAMERA, s.frame, env_faces=s.faces, env_n=case["n"],
                         seed=s.seed, **light)
    elif kind == "sh_render":
        ctx.sh_render(s.mesh, CAMERA, case["w"], case["h"], s.transfer, s.light, case["degree"],
                      s.dst, brdf_samples=case["samples"], seed=s.seed, env_faces=s.faces,
                      env_n=case["n"])
    else:
        ctx.sh_compute_transfer(s.mesh, s.basis, 32, case["degree"], s.dst,
                                samples=case["samples"], seed=s.seed)
    return s.out


# --------------------------------------------------------- work, tolerance --

PAIR_FLOPS = 2 * (32 * 64 + 64 * 64 + 64 * 64 + 64 * 3)


def work(case):
    kind = case["kind"]
    _, entries = _level_table()

    def relight(w, h, k, n, hash_bytes, aux=False, out_bytes=36):
        # Each pixel reads its position, flag and direct term (and the aux
        # planes) and writes its outputs; a frame touches at most the whole
        # hash table, or its 8 corners a level.
        P = w * h
        table = min(entries * 2 * hash_bytes, P * LEVELS * 8 * 2 * hash_bytes)
        b = P * (33 + (68 if aux else 0) + out_bytes) + table + k * (32 * 4 + 12) + 6 * n * n * 12
        return b, P * k * (PAIR_FLOPS + (2048 if aux else 0)) + P * LEVELS * 8 * 4

    if kind in ("relight", "two_pass"):
        b, f = relight(case["w"], case["h"], case["k"], case["n"],
                       2 if case["hash"] == "f16" else 4, aux=kind == "two_pass",
                       out_bytes=32 if case["prec"] == "fp8" else 36)
    elif kind == "batch":
        r = [relight(w, h, k, case["n"], 2) for w, h, k in _plan(case)]
        b, f = sum(x[0] for x in r), sum(x[1] for x in r)
    elif kind == "served":
        r = [relight(w, h, case["k"], case["n"], 2) for w, h, _ in _plan(case)]
        b, f = sum(x[0] for x in r), sum(x[1] for x in r)
    elif kind == "denoise":
        # Colour, normal and albedo in, colour out; 25 taps a pass.
        P = case["w"] * case["h"]
        b, f = P * 64, P * DENOISE_PASSES * 25 * 32
    elif kind == "cast":
        # G-buffer planes out, triangles (36 B) and vertex normals in; about
        # one box test a level and a leaf a ray, three rays a sample.
        P, g = case["w"] * case["h"], case["grid"]
        tris = 2 * g * g + 2 * max(16, g // 2) * max(4, max(16, g // 2) // 2)
        rays = P * (1 + 2 * case["samples"])
        b, f = P * (85 + (16 if case["samples"] else 0)) + tris * 48, rays * (20 * math.log2(tris) + 100)
    elif kind == "sh_render":
        nc, P, nu = (case["degree"] + 1) ** 2, case["w"] * case["h"], case["sphere"]
        nv = nu * (max(4, nu // 2) + 1) + 4
        b = nv * nc * nc * 12 + P * 16
        f = nv * nc * nc * 6 + nv * case["samples"] * (nc * 4 + 100) + P * 400
    else:
        nc, nu = (case["degree"] + 1) ** 2, case["sphere"]
        nv = nu * (max(4, nu // 2) + 1) + 4
        paths = nv * case["samples"]
        b = nv * nc * nc * 12 + nc * 6 * 32 * 32 * 12
        f = paths * nc * (nc * 6 + 400) + paths * 1500
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    # Four times the error measured against FP64: two correct forms of one
    # precision differ by no more than that.
    if kind == "two_pass":  # aux inputs carry a large share of the radiance
        return {"fp16": {"rel": 5e-4, "max": 2e-3, "differ": 1e-3},
                "bf16": {"rel": 4e-3, "max": 2e-2, "differ": 1e-2}}[case["prec"]]
    if kind in ("relight", "batch", "served"):
        # `differ`: whole pixels (three packed bytes) on another tone-map step.
        return {"fp32": {"rel": 3e-7, "max": 2e-6, "differ": 1e-4},
                "fp16": {"rel": 1e-5, "max": 5e-5, "differ": 1e-3},
                "bf16": {"rel": 7e-5, "max": 4e-4, "differ": 1e-3},
                "fp8": {"rel": 1e-3, "max": 5e-3}}[case["prec"]]
    if kind == "denoise":
        return {"rel": 6e-7, "max": 6e-6}
    if kind == "sh_render":  # no shadow rays: only a primary ray can flip
        return {"rel": 5e-4, "max": 0.99}
    # A shadow ray or a path within rounding of an edge may take the other
    # side; that sample then differs by its whole value.
    return {"rel": 5e-3, "max": 0.99, "differ": 1e-4}


# ------------------------------------------------------------- FP64 results --

def _haar(faces):
    """Non-standard orthonormal Haar transform of [6][n][n][3] faces, FP64
    scaling values, each coefficient rounded to FP32 once."""
    x = faces.double()
    out = torch.zeros_like(faces)
    while x.shape[1] > 1:
        a, b, c, d = x[:, 0::2, 0::2], x[:, 0::2, 1::2], x[:, 1::2, 0::2], x[:, 1::2, 1::2]
        m = x.shape[1] // 2
        out[:, :m, m:2 * m] = (((a - b) + (c - d)) * 0.5).float()
        out[:, m:2 * m, :m] = (((a + b) - (c + d)) * 0.5).float()
        out[:, m:2 * m, m:2 * m] = (((a - b) - (c - d)) * 0.5).float()
        x = ((a + b) + (c + d)) * 0.5
    out[:, 0, 0] = x[:, 0, 0].float()
    return out


def _select(faces, k):
    """Indices and strengths of the k largest area-weighted luminances, ties
    to the lower index."""
    coef = _haar(faces)
    n = faces.shape[1]
    lum = (coef[..., 0] * LUM[0] + coef[..., 1] * LUM[1]) + coef[..., 2] * LUM[2]
    i = torch.arange(n, device="cuda")
    m = torch.maximum(i[:, None], i[None, :]).clamp(min=1)
    j = torch.floor(torch.log2(m.double() + 0.25))
    score = (lum.abs() * torch.pow(4.0, -j).float()).reshape(-1)
    score = torch.where(score >= 1.17549435e-38, score, torch.zeros_like(score))
    idx = torch.sort(score, descending=True, stable=True).indices[:k]
    return idx, coef.reshape(-1, 3)[idx].double()


def _rotate(faces, yaw):
    """Faces turned about +y, each texel from the nearest source texel; FP32
    direction arithmetic, every operation rounded."""
    n = faces.shape[1]
    g = 2.0 * ((torch.arange(n, device="cuda").float() + 0.5) / n) - 1.0
    v, u = torch.meshgrid(g, g, indexing="ij")
    one = torch.ones_like(u)
    d = [(one, v, u), (-one, v, -u), (u, one, v), (u, -one, -v), (u, v, -one), (-u, v, one)]
    x, y, z = (torch.stack([f[c] for f in d]) for c in range(3))
    cs = torch.tensor(math.cos(yaw), dtype=torch.float32, device="cuda")
    sn = torch.tensor(math.sin(yaw), dtype=torch.float32, device="cuda")
    xs, zs = cs * x - sn * z, sn * x + cs * z
    ax, ay, az = xs.abs(), y.abs(), zs.abs()
    f, m = torch.zeros_like(xs, dtype=torch.long), torch.ones_like(xs)
    uc, vc = torch.zeros_like(xs), torch.zeros_like(xs)
    X, Y, Z = (ax >= ay) & (ax >= az), (ay >= ax) & (ay >= az), (az >= ax) & (az >= ay)
    for face, hit, mm, a, b in ((0, X & (xs > 0), ax, zs, y), (1, X & ~(xs > 0), ax, -zs, y),
                                (2, Y & (y > 0), ay, xs, zs), (3, Y & ~(y > 0), ay, xs, -zs),
                                (4, Z & ~(zs > 0), az, xs, y), (5, Z & (zs > 0), az, -xs, y)):
        f = torch.where(hit, torch.full_like(f, face), f)
        m, uc, vc = torch.where(hit, mm, m), torch.where(hit, a, uc), torch.where(hit, b, vc)
    col = torch.floor(0.5 * (uc / m + 1.0) * n).long().clamp(0, n - 1)
    row = torch.floor(0.5 * (vc / m + 1.0) * n).long().clamp(0, n - 1)
    return faces[f, row, col]


def _hash_features(a, pos):
    """FP64 trilinear hash-grid features [P][32]; grid positions in FP32."""
    table, _ = _level_table()
    out = torch.empty((pos.shape[0], 32), dtype=torch.float64, device="cuda")
    for l, (scale, res, dense, size, off) in enumerate(table):
        p = (pos.double() * float(scale) + 0.5).float()
        fl = torch.floor(p)
        fr = (p - fl).double()
        g = fl.long()
        acc = torch.zeros((pos.shape[0], 2), dtype=torch.float64, device="cuda")
        for c in range(8):
            b = (c & 1, c >> 1 & 1, c >> 2 & 1)
            x, y, z = (g[:, i] + b[i] for i in range(3))
            if dense:
                i = (x + y * res + z * res * res) % size
            else:
                i = (x ^ (y * 2654435761 & 0xFFFFFFFF) ^ (z * 805459861 & 0xFFFFFFFF)) & (size - 1)
            w = torch.ones_like(fr[:, 0])
            for ax in range(3):
                w = w * (fr[:, ax] if b[ax] else 1.0 - fr[:, ax])
            acc += w[:, None] * a["hash"][off + i].double()
        out[:, 2 * l:2 * l + 2] = acc
    return out


def _aux_inputs(g):
    f = lambda k: g[k][:, :3].double()
    r = torch.log(25.0 * g["roughness"].double() + 1.0) / math.log(26.0)
    return torch.cat([f("normal"), f("reflect"), r[:, None], 2 * f("kd") - 1, 2 * f("ks") - 1,
                      torch.ones((r.shape[0], 3), dtype=torch.float64, device="cuda")], 1)


def _relight64(a, g, idx, light, rgba8):
    """Indirect radiance of every pixel in FP64: sum over the selection of
    max(light softplus(MLP(features * wavelet features)), 0)."""
    P, k = g["position"].shape[0], len(idx)
    ind = torch.zeros((P, 4), dtype=torch.float64, device="cuda")
    ind[:, 3] = 1.0
    w1 = a["w1"].double()[None] * a["wfeat"][:, idx].double().t()[:, None, :]  # [k][64][32]
    w2, w3, w4 = (a[x].double().t().contiguous() for x in ("w2", "w3", "w4"))
    hit = torch.nonzero(g["env_flag"]).reshape(-1)
    for p0 in range(0, len(hit), 16384):
        px = hit[p0:p0 + 16384]
        h = _hash_features(a, g["position"][px, :3])
        if a["proj"] is not None:
            h = h @ a["proj"].double().t()
        aux = 0.0
        if a["waux"] is not None:
            ax = _aux_inputs({q: v[px] for q, v in g.items()})
            aux = (ax @ a["waux"].double().t())[:, None, :]
        rgb = torch.zeros((len(px), 3), dtype=torch.float64, device="cuda")
        for k0 in range(0, k, 32):
            w = w1[k0:k0 + 32]
            y = (h @ w.reshape(-1, 32).t()).reshape(len(px), -1, 64).relu_()
            y = ((y.reshape(-1, 64) @ w2).reshape(len(px), -1, 64) + aux).relu_()
            y = (y.reshape(-1, 64) @ w3).relu_()
            t = torch.nn.functional.softplus((y @ w4).reshape(len(px), -1, 3), threshold=40.0)
            rgb += (light[None, k0:k0 + 32] * t).clamp_(min=0).sum(1)
        ind[px, :3] = rgb
    wd = ind.clone()
    wd[:, :3] += g["direct"][:, :3].double()
    out = {"indirect": ind, "with_direct": wd}
    if rgba8:
        out["rgba8"] = None
    return out


def _denoise_inputs(case, seed):
    """A noisy relit frame: smooth radiance times Monte-Carlo-like noise,
    piecewise-constant normals and albedo with edges."""
    w, h = case["w"], case["h"]
    y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"),
                          indexing="ij")
    cells = ((x // 97) + 31 * (y // 61)).reshape(-1) % 256
    base = 0.5 + torch.sin(x * 0.013) * torch.cos(y * 0.017) * 0.4
    noise = torch.exp(0.5 * _normal(seed, 50, (h, w, 3), 1.0))
    n = torch.nn.functional.normalize(_normal(seed, 51, (256, 3), 1.0), dim=1)[cells]
    a = _uniform(seed, 52, (256, 3))[cells]
    one = torch.ones((h, w, 1), device="cuda")
    return {"color": torch.cat([base[..., None] * noise, one], -1).contiguous(),
            "normal": torch.cat([n.reshape(h, w, 3), one], -1).contiguous(),
            "albedo": torch.cat([a.reshape(h, w, 3), one], -1).contiguous()}


def _denoise64(case, seed):
    g = {k: v.double() for k, v in _denoise_inputs(case, seed).items()}
    p = nw.Context.denoise_default_params()
    c, n, a = (g[k][..., :3] for k in ("color", "normal", "albedo"))
    lum = c @ torch.tensor([0.2126, 0.7152, 0.0722], dtype=torch.float64, device="cuda")
    lit = lum[lum > 1e-8]
    kappa = float(torch.exp2(-torch.log2(lit).mean())) if len(lit) else 1.0
    H, W = case["h"], case["w"]
    B3 = (1 / 16, 4 / 16, 6 / 16, 4 / 16, 1 / 16)
    for i in range(p.iterations):
        s = 1 << i
        num, den = torch.zeros_like(c), torch.zeros((H, W, 1), dtype=torch.float64, device="cuda")
        for dy in range(-2, 3):
            for dx in range(-2, 3):
                oy, ox = dy * s, dx * s
                ya, yb, xa, xb = max(0, -oy), min(H, H - oy), max(0, -ox), min(W, W - ox)
                if ya >= yb or xa >= xb:
                    continue
                P = (slice(ya, yb), slice(xa, xb))
                Q = (slice(ya + oy, yb + oy), slice(xa + ox, xb + ox))
                d = kappa ** 2 * 4.0 ** i / p.sigma_color ** 2 * ((c[Q] - c[P]) ** 2).sum(-1) \
                    + ((n[Q] - n[P]) ** 2).sum(-1) / p.sigma_normal ** 2 \
                    + ((a[Q] - a[P]) ** 2).sum(-1) / p.sigma_albedo ** 2
                wt = (B3[dx + 2] * B3[dy + 2] * torch.exp(-d))[..., None]
                num[P] += wt * c[Q]
                den[P] += wt
        c = num / den
    return torch.cat([c, g["color"][..., 3:]], -1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("relight", "two_pass"):
        aux = kind == "two_pass"
        faces = _faces(seed, case["n"])
        if case.get("env") == "rotated":
            faces = _rotate(faces, _yaw(seed))
        idx, light = _select(faces, case["k"])
        return _relight64(_scene_arrays(seed, case["n"], case["hash"], aux),
                          _gbuffer(seed, case["w"], case["h"], case["background"], surface=aux),
                          idx, light, case["prec"] != "fp8")
    if kind == "batch":
        a = [_scene_arrays(seed + i, case["n"], "f16", False) for i in range(2)]
        return [_relight64(a[j % 2], _gbuffer(seed + 100 * j, w, h, 0.0),
                           *_select(_faces(seed, case["n"], 20 + j), k), True)
                for j, (w, h, k) in enumerate(_plan(case))]
    if kind == "served":
        a, out = _scene_arrays(seed, case["n"], "f16", False), []
        for j, (w, h, env) in enumerate(_plan(case)):
            faces = _faces(seed, case["n"], 20 + j)
            if env == "rotated":
                faces = _rotate(faces, _yaw(seed, j))
            out.append(_relight64(a, _gbuffer(seed + 100 * j, w, h, 0.0),
                                  *_select(faces, case["k"]), True))
        return out
    if kind == "denoise":
        return _denoise64(case, seed)
    return None  # ray tracing: brute force over every triangle takes minutes
