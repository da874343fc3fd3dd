"""The BF16 / FP16 relight's two workgroup shapes (256 pixels, or 64 pixels
shared by the four waves for small frames and a frame's last partial round):
the same bits as the unsplit variant and as the batch form, at the sizes
where the split changes, ragged tails, odd and small K."""
import numpy as np
import pytest

from cases import make_case
from conftest import max_rel_err

pytestmark = pytest.mark.gpu

ROUND = 131072  # 512 workgroups x 256 pixels
SIZES = [1, 63, 65, 1000, 98304 - 1, 98304 + 1, ROUND, ROUND + 1, ROUND + 4097]


@pytest.mark.parametrize("precision,aux,k,table", [("bf16", False, 1, "f32"),
                                                   ("bf16", False, 7, "f16"),
                                                   ("fp16", False, 10, "f32"),
                                                   ("fp16", True, 6, "f16"),
                                                   ("bf16", True, 3, "f32")])
def test_split_relight_same_bits(nw, orc, ctx, precision, aux, k, table):
    case = make_case(nw, orc, seed=9, width=max(SIZES), height=1, face_size=8, k=k,
                     background=0.1, aux=aux, log2_hashmap_size=12,
                     hash_dtype=nw.DTYPE_F16 if table == "f16" else nw.DTYPE_F32)
    prec = nw.PRECISIONS[precision]
    scene = ctx.scene_create(case.desc, case.params)
    env = ctx.envmap_from_faces(case.faces, k)
    idx, st = ctx.envmap_selection(env)
    for p in SIZES:
        g = {name: np.ascontiguousarray(v[:p]) for name, v in case.gbuf.items()}
        frame, other = nw.DeviceFrame(p, 1, g), nw.DeviceFrame(p, 1, g)
        ctx.relight(scene, env, frame, prec)
        if aux:  # the batch form takes 64 pixels a wave
            batch = ctx.batch_create([(scene, env, other)], prec)
            ctx.batch_launch(batch)
            ctx.sync()
            ctx.batch_destroy(batch)
        else:
            ctx.set_relight_variant(1)  # never split
            ctx.relight(scene, env, other, prec)
            ctx.set_relight_variant(-1)
        ctx.sync()
        a, b = frame.results(), other.results()
        for name in a:
            assert np.array_equal(a[name].view(np.uint32), b[name].view(np.uint32)), (p, name)
        at = np.arange(max(0, p - 70), p).astype(np.int32)
        ref, _ = case.oscene.relight(idx, st, g, pixels=at)
        # The repository's bars for 16-bit operands (2^-8 and 2^-11 relative
        # rounding through four layers).
        assert max_rel_err(ref, a["indirect"][at, :3]) <= {"bf16": 2e-2, "fp16": 5e-3}[precision], p
    ctx.envmap_destroy(env)
    ctx.scene_destroy(scene)


# (rounds of 512 workgroups, workgroups of the rest, K): both sides of every
# line of the rule that splits the rest, and of the default variant's.
EDGES = [(0, 128, 1), (0, 129, 15), (0, 129, 16), (0, 192, 16), (0, 193, 31), (0, 193, 32),
         (0, 256, 32), (0, 257, 7), (0, 257, 8), (0, 320, 8), (0, 321, 23), (0, 321, 24),
         (0, 384, 24), (0, 385, 24), (1, 0, 8), (1, 129, 16), (1, 193, 64), (1, 256, 64),
         (2, 0, 8), (2, 1, 7), (2, 1, 8), (2, 1, 27), (2, 1, 28), (2, 129, 39), (2, 129, 40),
         (2, 257, 23), (2, 257, 24), (2, 321, 39), (2, 321, 40), (5, 64, 9)]


@pytest.mark.parametrize("precision,softplus", [("bf16", True), ("fp16", False)])
def test_split_rule_edges_same_bits(nw, orc, precision, softplus):
    ctx = nw.Context(0)  # nothing tuned
    p_max = max(512 * r + w for r, w, _ in EDGES) * 256
    case = make_case(nw, orc, seed=12, width=p_max, height=1, face_size=8, k=64, background=0.1,
                     log2_hashmap_size=12, softplus=softplus)
    prec = nw.PRECISIONS[precision]
    scene = ctx.scene_create(case.desc, case.params)
    for rounds, wgs, k in EDGES:
        p = (512 * rounds + wgs) * 256 - 3  # the last workgroup is ragged
        env = ctx.envmap_from_faces(case.faces, k)
        assert ctx.selected_relight_variant(prec, k, p) == (
            0 if 8 <= k < 28 and 512 * rounds + wgs > 1024 else 5), (rounds, wgs, k)
        g = {name: np.ascontiguousarray(v[:p]) for name, v in case.gbuf.items()}
        frame, other = nw.DeviceFrame(p, 1, g), nw.DeviceFrame(p, 1, g)
        ctx.relight(scene, env, frame, prec)
        ctx.set_relight_variant(1)  # never split
        ctx.relight(scene, env, other, prec)
        ctx.set_relight_variant(-1)
        ctx.sync()
        a, b = frame.results(), other.results()
        for name in a:
            assert np.array_equal(a[name].view(np.uint32), b[name].view(np.uint32)), (p, k, name)
        idx, st = ctx.envmap_selection(env)
        at = np.unique(np.concatenate([np.arange(max(0, p - 40), p), np.arange(0, p, 1 + p // 20)]))
        ref, _ = case.oscene.relight(idx, st, g, pixels=at.astype(np.int32))
        # The bars of 16-bit operands above, per value for softplus outputs.  A
        # linear output is a sum of 64 signed products that may cancel, so its
        # rounding scales with their magnitudes: the bar is on the largest value.
        err = max_rel_err(ref, a["indirect"][at, :3], floor=1e-3 if softplus else 1.0)
        assert err <= {"bf16": 2e-2, "fp16": 5e-3}[precision], (p, k)
        ctx.envmap_destroy(env)
    ctx.close()


def test_autotune_on_aux_scene_leaves_the_bucket(nw, orc):
    """Every variant of an aux scene is the same kernel, so tuning one names
    the default and keeps what a scene with a choice recorded for the shape."""
    w, h, k = 64, 48, 8
    ctx = nw.Context(0)
    scenes, frames = [], []
    for aux in (False, True):
        case = make_case(nw, orc, seed=3, width=w, height=h, face_size=8, k=k, aux=aux,
                         log2_hashmap_size=12)
        scenes.append(ctx.scene_create(case.desc, case.params))
        frames.append(nw.DeviceFrame(w, h, case.gbuf))
    env = ctx.envmap_from_faces(case.faces, k)
    for prec in (nw.PREC_BF16, nw.PREC_FP16):
        kept, _ = ctx.autotune_relight(scenes[0], env, frames[0], prec)
        assert ctx.selected_relight_variant(prec, k, w * h) == kept
        for _ in range(3):
            best, ms = ctx.autotune_relight(scenes[1], env, frames[1], prec)
            assert best == 5 and ms > 0
            assert ctx.selected_relight_variant(prec, k, w * h) == kept
    ctx.close()
