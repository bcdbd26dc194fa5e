"""Ray lists at the sizes where the order they are traced in changes (2048 rays by tiles, 262,144 by rows): what a ray
returns and is given as its gradient is the same wherever it stands in the list, and the surfels' gradients are the same sums,
replayed from a complete record and traced again behind an incomplete one."""
import pytest
import torch

import dst_scenes as S
from helpers import gpu_trace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks_per_wave", [12.0, 0.01])
@pytest.mark.parametrize("handover", ["off", "always"])
@pytest.mark.parametrize("n", [2047, 2048, 5001, 262143, 262144])
def test_a_ray_is_the_same_anywhere_in_its_list(n, handover, blocks_per_wave):
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    ctx = tracer.optix_context
    sc = S.scene_cube(P=3000, seed=4)
    r = torch.Generator().manual_seed(n)
    o = torch.rand(1, n, 3, generator=r) * 1.6 - 0.8
    d = torch.nn.functional.normalize(torch.randn(1, n, 3, generator=r), dim=-1)
    up = {k: torch.randn(1, n, c, generator=r) for k, c in (("rgb", 3), ("dpt", 1), ("norm", 3))}
    perm = torch.randperm(n, generator=r)
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    if handover == "always":
        ctx.set_handover(2)
    got = []
    for at in (torch.arange(n), perm):
        ctx.record_blocks_per_wave = blocks_per_wave
        out, grads = gpu_trace(tracer, sc, o[:, at], d[:, at], upstream={k: v[:, at] for k, v in up.items()}, build=False)
        got.append((out, grads))
    (a, ga), (b, gb) = got
    p = perm.numpy()
    assert a["rgb"].std() > 0.01
    for k in ("rgb", "dpt", "acc", "norm", "mid"):
        assert (a[k][0][p].view("int32") == b[k][0].view("int32")).all(), k
    for k, g in ga.items():
        if g is None:
            continue
        x, y = (torch.from_numpy(v).double() for v in (g[:, p] if k in ("ray_o", "ray_d") else g, gb[k]))
        # fp32 terms of up to n rays added in doubles a workgroup and in floats beyond: n^0.5 roundings of 6e-8 at most
        assert (x - y).norm() <= 6e-8 * (n ** 0.5 + 16.0) * x.norm() + 1e-12, (k, float((x - y).norm() / x.norm()))
