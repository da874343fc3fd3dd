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
            ctx.set_relight_variant(0)
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
