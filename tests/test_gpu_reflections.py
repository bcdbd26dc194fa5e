"""Reflections of images too large to be recorded ray by ray, against the oracle: per-ray outputs bit-identical, gradients
within the usual bar.  Mid-size images are traced ray by ray from the start (k_row_fwd<RowTiles> with a record, <RowRays>
without), larger ones by tiles, their reflections ray by ray (<RowBeyond>); HANDOVER_OFF has the latter at mid sizes too, so
that the tests below run on both paths.  The oracle follows a window of the image; upstream gradients are zero outside of it,
so that the per-surfel sums are the window's alone."""
import numpy as np
import pytest
import torch

import dst_scenes as S
from helpers import GRAD_REL, assert_forward_exact, assert_gradients, gpu_trace, oracle_scene, upstream

pytestmark = pytest.mark.gpu
H, W = 152, 176          # 418 waves: above the sizes that are recorded ray by ray
PATHS = pytest.mark.parametrize("path", ["rows", "tiles_then_rows"])


def tracer_by(path):
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    if path == "tiles_then_rows":
        tracer.optix_context.set_handover(dst._C.HANDOVER_OFF)
    return tracer


def window_reference(oracle, sc, o, d, aux, rows, cols, **kw):
    ug = upstream(o.shape[0], o.shape[1], aux)
    inside = torch.zeros(o.shape[0], o.shape[1], 1)
    inside[rows, cols] = 1.0
    ug = {k: v * inside for k, v in ug.items()}
    s = oracle_scene(oracle, sc, o[rows, cols].contiguous(), d[rows, cols].contiguous(), **kw)
    ref = oracle.forward(s, oracle.HITS_BVH_LEXI)
    ugn = {k: v[rows, cols].contiguous().numpy() for k, v in ug.items()}
    return ug, ref, oracle.backward(s, ref, ugn, oracle.HITS_BVH_LEXI), oracle.backward(s, ref, ugn, oracle.HITS_BVH_LEXI, noise=True)


def check_window(out, g, ref, refg, refg64, rows, cols, tag):
    assert_forward_exact({k: v[rows, cols] for k, v in out.items() if k != "wet"}, ref)
    got = dict(g)
    for k in ("ray_o", "ray_d"):
        got[k] = g[k][rows, cols]
    assert_gradients(got, refg, refg64, GRAD_REL, tag)


def translucent_corridor(n=720, seed=5):
    """A mirror in front of the camera and, behind the camera, a stack of quads as wide as the view: seven in ten too
    faint to count at all, the others a per cent or two.  A reflected ray meets them all."""
    gen = torch.Generator().manual_seed(seed)
    x = torch.cat([torch.tensor([4.0]), -1.0 - 6.0 * torch.rand(n, generator=gen)])
    means = torch.stack([x, 0.2 * torch.randn(n + 1, generator=gen), 0.2 * torch.randn(n + 1, generator=gen)], dim=-1)
    scales = torch.full((n + 1, 2), 1.6)
    nn = torch.tensor([1.0, 0.0, 0.0]) + torch.cat([torch.zeros(1, 3), 0.05 * torch.randn(n, 3, generator=gen)])
    nn = torch.nn.functional.normalize(nn, dim=-1)
    rotations = torch.stack([1 + nn[:, 2], -nn[:, 1], nn[:, 0], torch.zeros(n + 1)], dim=-1)   # z into the normal
    rotations = torch.nn.functional.normalize(rotations, dim=-1)
    faint = torch.rand(n + 1, generator=gen) < 0.7
    opacities = torch.where(faint, torch.full((n + 1,), 0.003), 0.01 + 0.01 * torch.rand(n + 1, generator=gen))
    opacities[0] = 0.999
    others = 0.1 * torch.rand(n + 1, 2, generator=gen)
    others[0, 0] = 0.9
    sc = {"means3D": means, "scales": scales, "rotations": rotations.contiguous(), "opacities": opacities[:, None].contiguous(),
          "shs": 0.3 * torch.randn(n + 1, 16, 3, generator=gen), "others_precomp": others}
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    return sc


@PATHS
def test_a_long_way_through_translucent_surfels_is_recorded(oracle, path):
    """Some fifty chunks of sixteen entries behind the mirror: the record of the second step has room for them all, is
    complete, and stays the size it is; replay and re-trace both give the oracle's gradients."""
    sc = translucent_corridor()
    o, d = S.pinhole_rays(H, W, 40.0, (0.0, 0.0, 0.0), (1.0, 0.0, 0.0))
    rows, cols = slice(60, 76), slice(70, 94)
    kw = dict(max_trace_depth=1, specular_threshold=0.4)
    ug, ref, refg, refg64 = window_reference(oracle, sc, o, d, 2, rows, cols, **kw)
    assert ref["n_proc"].max() > 16 * 40 and ref["n_con"].mean() > 100
    tracer = tracer_by(path)
    ctx = tracer.optix_context
    sizes = []
    for step in range(4):
        out, g = gpu_trace(tracer, sc, o, d, upstream=ug, build=(step == 0), **kw)
        rec = ctx._record_watch[-1]
        sizes.append(rec.blocks)
        assert rec.complete() == (step > 0), (step, rec.requested_blocks(), rec.blocks)
        assert rec.requested_blocks() > 40 * rec.n_waves / 2
        check_window(out, g, ref, refg, refg64, rows, cols, "step %d " % step)
    assert sizes[1] == sizes[2] == sizes[3]


@PATHS
@pytest.mark.parametrize("depth,aux,mode", [(1, 2, "plain"), (1, 4, "det"), (2, 8, "norec"), (3, 2, "plain"), (3, 4, "colors"),
                                            (1, 3, "colors_det"), (2, 2, "half"), (1, 8, "distortion"), (3, 8, "det"),
                                            (2, 4, "norows")])
def test_reflections_of_mid_size_images(oracle, depth, aux, mode, path):
    from test_gpu_parity import check_case
    sc = S.scene_room(P=12000, seed=depth + aux, aux=aux, half=1.5)
    sc["others_precomp"][:, 0] = sc["others_precomp"][:, 0] * 0.8 + 0.1    # the reference divides by the specular
    if mode.startswith("colors"):
        sc["colors_precomp"] = torch.rand(12000, 3, generator=torch.Generator().manual_seed(3))
        del sc["shs"]
    o, d = S.pinhole_rays(H, W, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15))
    kw = dict(max_trace_depth=depth, specular_threshold=0.0 if depth == 3 else 0.1, bg=(0.3, 0.1, 0.2))
    tracer = tracer_by(path)
    ctx = tracer.optix_context
    tracer.deterministic = mode.endswith("det")
    seen, call = sc, tracer
    if mode == "half":
        from test_gpu_tiles import _HalfSeen
        tracer.sh_half = True
        seen, call = dict(sc, shs=sc["shs"].half().float()), _HalfSeen(tracer, sc["shs"])
    elif mode == "norec":
        ctx.record_max_bytes = 0
    elif mode == "norows":
        ctx.gradient_rows = False
    if mode == "distortion":
        tracer.distortion = True
        out, _ = gpu_trace(tracer, sc, o, d, **kw)
        ref = oracle.forward(oracle_scene(oracle, sc, o, d, **kw), oracle.HITS_BVH_LEXI, compute_dist=True)
        np.testing.assert_array_equal(out["dist"].view(np.uint32), ref["dist"][..., :1].view(np.uint32))
        assert out["dist"].max() > 1e-6
        tracer.distortion = False
    runs = [check_case(oracle, call, seen, o, d, **kw) for _ in range(3 if tracer.deterministic else 2)]
    assert mode == "norec" or ctx._record_watch[-1].complete()
    assert (runs[0][0]["mid"][..., (14 + aux) * depth + 3:(14 + aux) * depth + 6] != 0).any()    # the last bounce is reached
    if tracer.deterministic:
        for k, v in runs[1][0]["grads_gpu"].items():
            assert v is None or np.array_equal(v.view(np.uint32), runs[2][0]["grads_gpu"][k].view(np.uint32)), k
        assert np.array_equal(runs[0][1]["wet"], runs[1][1]["wet"])


@pytest.mark.parametrize("size,depth,aux,det", [(264, 1, 2, False), (264, 3, 8, True), (328, 2, 4, False)])
def test_tiles_then_rows_on_images_beyond_the_small_ones(oracle, size, depth, aux, det):
    """First bounce by tiles, the others by rows, with a record (264x264) and without one (328x328)."""
    import diff_surfel_tracing as dst
    sc = S.scene_room(P=12000, seed=20 + depth, aux=aux, half=1.5)
    sc["others_precomp"][:, 0] = sc["others_precomp"][:, 0] * 0.8 + 0.1
    o, d = S.pinhole_rays(size, size, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15))
    rows, cols = slice(120, 140), slice(100, 124)
    kw = dict(max_trace_depth=depth, specular_threshold=0.1)
    tracer = dst.SurfelTracer()
    tracer.deterministic = det
    ug, ref, refg, refg64 = window_reference(oracle, sc, o, d, aux, rows, cols, **kw)
    for step in range(2):
        out, g = gpu_trace(tracer, sc, o, d, upstream=ug, build=(step == 0), **kw)
        check_window(out, g, ref, refg, refg64, rows, cols, "step %d " % step)
    assert tracer.optix_context._record_watch[-1].complete()
    out, _ = gpu_trace(tracer, sc, o, d, build=False, **kw)
    assert_forward_exact({k: v[rows, cols] for k, v in out.items() if k != "wet"}, ref)


@pytest.mark.parametrize("n", [15, 16, 17, 33, 63, 64, 65, 124, 125, 130, 190, 300])
def test_a_ray_goes_on_from_what_its_last_walk_left(oracle, n):
    """Stacks of n faint quads, some at one depth, in front of a list of rays: chunks that end at the stack's end, kept quads
    that just fit a row's memory or do not, and rays that graze the quads' edges."""
    import diff_surfel_tracing as dst
    from test_gpu_parity import check_case
    gen = torch.Generator().manual_seed(n)
    means = torch.stack([0.02 * torch.randn(n, generator=gen), 0.02 * torch.randn(n, generator=gen),
                         1.0 + torch.floor(12.0 * torch.rand(n, generator=gen)) / 4.0], dim=-1)
    means[::2, 2] += 0.001 * torch.arange(n)[::2]
    rot = torch.zeros(n, 4)
    rot[:, 0] = 1.0
    # (scales unequal: a round quad has no gradient about its normal, only its rounding)
    sc = {"means3D": means, "scales": torch.tensor([[0.1, 0.06]]).repeat(n, 1), "rotations": rot,
          "opacities": 0.01 + 0.05 * torch.rand(n, 1, generator=gen), "shs": 0.3 * torch.randn(n, 16, 3, generator=gen)}
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    o = torch.zeros(1, 96, 3)
    d = torch.nn.functional.normalize(torch.cat([0.12 * torch.randn(1, 96, 2, generator=gen), torch.ones(1, 96, 1)], dim=-1), dim=-1)
    d[0, :16, 0] = 0.3 / 1.0      # past or along the nearest quads' edges
    check_case(oracle, dst.SurfelTracer(), sc, o, d.contiguous())


@pytest.mark.parametrize("n,batches", [(60, 1), (140, 1), (400, 1), (400, 9)])
def test_rays_with_and_without_room_share_a_wave(oracle, n, batches):
    """One ray of every four meets a stack of n quads, more than its row has room to keep where n is large; its neighbours meet
    a dozen or three dozen, or nothing.  Once one ray of a wave has no room, none of the wave's walks keeps anything any more
    until all have ended.  (A list of 2304 rays is traced in an order of its own.)"""
    import diff_surfel_tracing as dst
    from test_gpu_parity import check_case
    gen = torch.Generator().manual_seed(n)
    sizes, x = [n, 12, 36], [0.0, 4.0, 8.0]
    means = torch.cat([torch.stack([x[k] + 0.02 * torch.randn(m, generator=gen), 0.02 * torch.randn(m, generator=gen),
                                    1.0 + 3.0 * torch.rand(m, generator=gen)], dim=-1) for k, m in enumerate(sizes)])
    P = means.shape[0]
    rot = torch.zeros(P, 4)
    rot[:, 0] = 1.0
    sc = {"means3D": means, "scales": torch.tensor([[0.1, 0.06]]).repeat(P, 1), "rotations": rot,
          "opacities": 0.01 + 0.03 * torch.rand(P, 1, generator=gen), "shs": 0.3 * torch.randn(P, 16, 3, generator=gen)}
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    R = 256 * batches
    o = torch.zeros(1, R, 3)
    o[0, :, 0] = torch.tensor(x + [12.0]).repeat(R // 4)
    o[0, :, :2] += 0.02 * torch.randn(R, 2, generator=gen)
    d = torch.nn.functional.normalize(torch.cat([0.01 * torch.randn(1, R, 2, generator=gen), torch.ones(1, R, 1)], dim=-1), dim=-1)
    ref, _ = check_case(oracle, dst.SurfelTracer(), sc, o, d.contiguous())
    proc = ref["n_proc"].reshape(-1, 4)
    assert (proc[:, 0] > 0.5 * n).mean() > 0.9 and (proc[:, 1] <= 12).all() and (proc[:, 3] == 0).all()


@pytest.mark.parametrize("blocks", [16, 17])
def test_a_list_whose_record_is_one_block_short(oracle, blocks):
    """512 rays, 128 waves: their first pieces fill sixteen blocks of the record, the few pieces that two waves ask for
    beyond those lie in a seventeenth, of which nobody gets the first piece.  With sixteen blocks the record has to be
    known to be incomplete, with seventeen it is replayed."""
    import diff_surfel_tracing as dst
    from test_gpu_parity import check_case
    gen = torch.Generator().manual_seed(17)
    n = 40
    means = torch.stack([0.02 * torch.randn(n, generator=gen), 0.02 * torch.randn(n, generator=gen), 1.0 + 0.05 * torch.arange(n)], dim=-1)
    rot = torch.zeros(n, 4)
    rot[:, 0] = 1.0
    sc = {"means3D": means, "scales": torch.tensor([[0.3, 0.2]]).repeat(n, 1), "rotations": rot,
          "opacities": 0.01 + 0.05 * torch.rand(n, 1, generator=gen), "shs": 0.3 * torch.randn(n, 16, 3, generator=gen)}
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    o = torch.zeros(1, 512, 3)
    d = torch.cat([0.02 * torch.randn(1, 512, 2, generator=gen), torch.ones(1, 512, 1)], dim=-1)
    d[:, 8:] *= -1.0      # the first two waves' rays meet everything, the others nothing
    tracer = dst.SurfelTracer()
    ctx = tracer.optix_context
    ctx.record_blocks_per_wave = (blocks - 0.5) / dst._C.HitRecord.layout(1, 512, 0, 1.0)[3]
    ctx.update_record_estimate = lambda: None
    ref, _ = check_case(oracle, tracer, sc, o, torch.nn.functional.normalize(d, dim=-1).contiguous())
    assert (ref["n_proc"].reshape(-1)[:8] > 32).all() and not ref["n_proc"].reshape(-1)[8:].any()
    rec = ctx._record_watch[-1]
    assert rec.blocks == blocks and rec.requested_blocks() == 17 and rec.complete() == (blocks == 17)


def _pairs_of_quads(n, gen, along, apart):
    """`n` pairs of faint quads across the z axis, each pair at one place, the next 0.02 further on (a pair is one leaf group
    of the hierarchy, with a flat box).  Their low x sides lie along the line x = along * z, `apart` from it at random, and they
    end within their Gaussian there, so that every one of them shows."""
    z = 1.0 + 0.02 * torch.arange(n).repeat_interleave(2)
    side = along * z + apart * torch.randn(n, generator=gen).repeat_interleave(2)
    means = torch.stack([side + 0.5, torch.zeros(2 * n), z], dim=-1)
    rot = torch.zeros(2 * n, 4)
    rot[:, 0] = 1.0
    sc = {"means3D": means, "scales": torch.tensor([[0.6, 0.5]]).repeat(2 * n, 1), "rotations": rot,
          "opacities": 0.01 + 0.01 * torch.rand(2 * n, 1, generator=gen), "shs": 0.3 * torch.randn(2 * n, 16, 3, generator=gen)}
    corner = torch.tensor([[-0.5, -0.6, 0.0], [-0.5, 0.6, 0.0], [0.5, -0.6, 0.0], [0.5, 0.6, 0.0]])
    sc["vertices"] = (means[:, None, :] + corner).reshape(-1, 3).contiguous()
    sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])[1]
    return sc


@pytest.mark.parametrize("distance", [3.0, 300.0, 3000.0, 30000.0])
def test_rays_from_far_away_along_the_sides_of_quads(oracle, distance):
    """A chunk's origin carries the rounding of the ray's own, however close to the scene it lies: chunks of a ray that comes
    from thousands of scene sizes away look along lines that far apart, and what one of them passes by another may meet.  The
    first walk keeps more than fits a row's memory, the second one what the others go on from."""
    import diff_surfel_tracing as dst
    gen = torch.Generator().manual_seed(int(distance))
    ulp = distance * 2.0 ** -24
    sc = _pairs_of_quads(80, gen, 0.7, 4.0 * ulp)
    R = 2048
    d = torch.nn.functional.normalize(torch.tensor([0.7, 0.05, 1.0]), dim=0).expand(1, R, 3).contiguous()
    at = torch.stack([0.7 * 2.0 + 4.0 * ulp * torch.randn(R, generator=gen), 0.1 * torch.randn(R, generator=gen), torch.full((R,), 2.0)], dim=-1)
    o = (at.double() - (distance * (1.0 + 0.2 * torch.rand(R, 1, generator=gen))).double() * d[0].double()).float()[None].contiguous()
    s = oracle_scene(oracle, sc, o, d)
    ref = oracle.forward(s, oracle.HITS_BRUTE_LEXI)
    assert (ref["n_proc"] > 40).sum() > R // 8
    out, _ = gpu_trace(dst.SurfelTracer(), sc, o, d)
    assert_forward_exact(out, ref)


@pytest.mark.parametrize("length", [1.0, 1e-3, 1e-5])
def test_short_directions_along_quads_of_one_plane(oracle, length):
    """Directions need not be of length one.  Sixty quads of one plane, met at a slant, and as many of another behind it: which
    of them lie behind a chunk's origin is a matter of the origin's rounding, which does not shrink with the direction."""
    import diff_surfel_tracing as dst
    gen = torch.Generator().manual_seed(7)
    n, R = 120, 1024
    normal = torch.nn.functional.normalize(torch.tensor([-0.6, 0.2, 1.0]), dim=0)
    q = torch.nn.functional.normalize(torch.stack([1 + normal[2], -normal[1], normal[0], torch.tensor(0.0)]), dim=0)   # z into the normal
    sc = {"scales": 0.3 + 0.1 * torch.rand(n, 2, generator=gen), "rotations": q.expand(n, 4).contiguous(),
          "opacities": 0.02 + 0.02 * torch.rand(n, 1, generator=gen), "shs": 0.3 * torch.randn(n, 16, 3, generator=gen)}
    x = torch.nn.functional.normalize(torch.tensor([1.0, 0.0, 0.6]), dim=0)      # in the plane
    y = torch.linalg.cross(normal, x)
    centre = torch.where((torch.arange(n) < n // 2)[:, None], torch.tensor([2.0, 1.0, 2.0]), torch.tensor([3.0, 1.5, 3.0]))
    sc["means3D"] = (centre + 0.1 * torch.randn(n, 1, generator=gen) * x + 0.1 * torch.randn(n, 1, generator=gen) * y).contiguous()
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    o = (0.05 * torch.randn(1, R, 3, generator=gen)).contiguous()
    d = length * torch.nn.functional.normalize(torch.tensor([2.0, 1.0, 2.0]) + 0.1 * torch.randn(1, R, 3, generator=gen), dim=-1)
    s = oracle_scene(oracle, sc, o, d.contiguous())
    ref = oracle.forward(s, oracle.HITS_BRUTE_LEXI)
    assert (ref["n_proc"] > 16).sum() > R // 2
    out, _ = gpu_trace(dst.SurfelTracer(), sc, o, d.contiguous())
    assert_forward_exact(out, ref)
