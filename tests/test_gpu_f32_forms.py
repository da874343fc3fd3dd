"""The plain FP32 relight's launch shapes: the workgroup's waves splitting the
wavelets (up to 16384 pixels), one wave per 16 pixels (up to 65536) and per
32 pixels.  Sizes around the crossings, ragged tails, odd and small K, with
and without aux inputs."""
import numpy as np
import pytest

from cases import make_case
from conftest import max_rel_err

pytestmark = pytest.mark.gpu

# FP32 products and sums over at most 16 + 64 + 64 + 64 + 32 terms a layer
# chain: about 240 rounding errors of 2^-24 each, 1.5e-5 of the summed
# magnitudes, with a margin for cancellation (the repository's FP32 bar).
TOL_FP32 = 1e-4
SIZES = [1, 15, 17, 64, 1000, 16384, 16385, 65536, 65537 + 30]


@pytest.mark.parametrize("aux,k", [(False, 1), (False, 6), (True, 5)])
def test_f32_shapes_agree_and_match_the_oracle(nw, orc, ctx, aux, k):
    case = make_case(nw, orc, seed=5, width=max(SIZES), height=1, face_size=8, k=k,
                     background=0.2, aux=aux, log2_hashmap_size=12)
    scene = ctx.scene_create(case.desc, case.params)
    env = ctx.envmap_from_faces(case.faces, k)
    idx, st = ctx.envmap_selection(env)
    results = {}
    for p in SIZES:
        g = {name: np.ascontiguousarray(v[:p]) for name, v in case.gbuf.items()}
        frame = nw.DeviceFrame(p, 1, g)
        ctx.relight(scene, env, frame, nw.PREC_FP32)
        ctx.sync()
        results[p] = frame.results()
        at = np.unique(np.concatenate([np.arange(max(0, p - 20), p), np.arange(0, p, 1 + p // 40)]))
        ref, _ = case.oscene.relight(idx, st, g, pixels=at.astype(np.int32))
        err = max_rel_err(ref, results[p]["indirect"][at, :3])
        assert err <= TOL_FP32, (p, err)
    full = results[max(SIZES)]
    for p in SIZES:  # the same pixel, whatever shape computed it
        for name, v in results[p].items():
            assert np.array_equal(v.view(np.uint32), full[name][:p].view(np.uint32)), (p, name)
    ctx.envmap_destroy(env)
    ctx.scene_destroy(scene)


@pytest.mark.parametrize("p", [1000, 20000, 65536 + 77])
def test_f32_tap_leaves_background_rows(nw, orc, ctx, p):
    """The transport tap of each launch shape writes the hit pixels' rows, as
    the oracle has them, and no row of a background pixel (the wrapper clears
    the buffer first), wherever hits and background share a wave."""
    k = 3
    case = make_case(nw, orc, seed=6, width=p, height=1, face_size=8, k=k, background=0.4,
                     log2_hashmap_size=12)
    scene = ctx.scene_create(case.desc, case.params)
    env = ctx.envmap_from_faces(case.faces, k)
    idx, st = ctx.envmap_selection(env)
    frame = nw.DeviceFrame(p, 1, case.gbuf)
    t = ctx.debug_transport(scene, env, frame, 0, p, nw.PREC_FP32)
    hit = case.gbuf["env_flag"].reshape(-1) != 0
    assert 0.5 < hit.mean() < 0.7
    assert not np.any(t[~hit])
    at = np.nonzero(hit)[0][::max(1, p // 50)].astype(np.int32)
    _, _, ref = case.oscene.relight(idx, st, case.gbuf, pixels=at, transport=True)
    assert max_rel_err(ref.reshape(-1, 3), t[at].reshape(-1, 3)) <= TOL_FP32
    ctx.envmap_destroy(env)
    ctx.scene_destroy(scene)
