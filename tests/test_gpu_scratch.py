"""The forward trace's scratch memory (DstParams.scratch): hits evaluated from records of the surfels, and blocks traced in
the order of a cost guessed for them, both of which the call makes first.  Outputs, and what a record lets the backward trace
replay, have to be those of the same call without scratch memory bit for bit, whatever the scales (quotients by them are
formed from their reciprocals in the records, and divided out where that does not hold)."""
import pytest
import torch

import dst_scenes as S
from diff_surfel_tracing import _C

pytestmark = pytest.mark.gpu


RECORD_BYTES = 64   # of a surfel


def layers(vertices):
    """How often the quads cover the surface of the box of their centres."""
    q = vertices.reshape(-1, 4, 3).double()
    area = torch.linalg.cross(q[:, 1] - q[:, 0], q[:, 2] - q[:, 0]).norm(dim=1).sum()
    e = (0.5 * (q.amin(1) + q.amax(1))).amax(0) - (0.5 * (q.amin(1) + q.amax(1))).amin(0)
    return float(area / (2 * (e[0] * e[1] + e[1] * e[2] + e[2] * e[0])))


def blocks_of(o):
    return ((o.shape[0] + 15) // 16) * ((o.shape[1] + 15) // 16)


def both(monkeypatch, tracer, sc, o, d, depth=0, aux=0, training=False, record=False):
    """(outputs with scratch memory, without, bytes of it).  With `record`, behind the outputs the number of blocks that were
    asked for in a hit record, and the rays' gradients as replayed from it."""
    g = {k: v.cuda() for k, v in sc.items()}
    e, bg, eye = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    others = torch.rand(sc["means3D"].shape[0], aux, generator=torch.Generator().manual_seed(3)).cuda() if aux else e
    real, taken, out, (H, W) = _C._scratch, [], [], o.shape[:2]

    def spy(p, keep):
        real(p, keep)
        taken.append(keep["scratch"].numel() if "scratch" in keep else 0)

    args = (True, o.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3, e, others, g["opacities"], g["scales"], 1.0,
            g["rotations"], e, eye, eye, bg, False, False, depth, 0.1)
    if not _C.load_library().dst_trace_scratch_bytes(sc["means3D"].shape[0], H, W):
        pytest.fail("this size has no scratch memory")
    for use in (True, False):
        monkeypatch.setattr(_C, "_scratch", spy if use else lambda p, keep: None)
        rec = _C.HitRecord(H, W, max(1, depth), 16.0, torch.device("cuda")) if record else None
        res = [x for x in _C.trace_surfels(tracer.optix_context, training, *args, hit_record=rec) if x is not None]
        if record:
            gen = torch.Generator().manual_seed(8)
            ups = [torch.randn(x.shape, generator=gen).cuda() for x in res[:6]]
            asked = rec.words[:1].clone()
            assert int(asked) <= rec.blocks
            grads = _C.trace_surfels_backward(tracer.optix_context, *args, *res[:7], *ups, hit_record=rec)[:2]
            assert grads[1].abs().max() > 0
            res[7:7] = [asked.to(torch.int32), *grads]
        out.append(res)
        torch.cuda.synchronize()
    monkeypatch.setattr(_C, "_scratch", real)
    return out[0], out[1], taken[0]


def view(H, W):
    return S.pinhole_rays(H, W, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15))


@pytest.mark.parametrize("H,W,P,makes", [
    # one row and one column of blocks, an odd one, the largest grid whose blocks are ordered; fewer surfels than rays
    (8, 8221, 30011, "both"), (4111, 16, 30011, "both"), (257, 256, 30011, "both"), (1040, 1008, 30011, "both"),
    (1040, 1024, 30011, "records"),                                 # one block row more
    (257, 256, 10007, "records"),                                   # quads that cover the room three times
    (8, 8221, 300000, "order"), (4111, 16, 300000, "order"), (257, 256, 300000, "order"),   # four surfels to a ray and more
])
def test_every_block_is_traced_once(monkeypatch, H, W, P, makes):
    """Outputs, what is recorded and what is replayed from it: the same bits with the blocks' order and the records of the
    surfels, with either alone, and with neither."""
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    sc = S.scene_room(P=P, seed=6, half=1.5)
    o, d = view(H, W)
    assert (layers(sc["vertices"]) > 5.5) == (P != 10007) and layers(sc["vertices"]) > 2.5
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    with_, without, size = both(monkeypatch, tracer, sc, o, d, training=True, record=True)
    assert size == (0 if makes == "order" else RECORD_BYTES * P) + (0 if makes == "records" else 8 * blocks_of(o))
    assert without[0].std() > 0.01
    for a, b in zip(with_[:-1], without[:-1]):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    torch.testing.assert_close(with_[-1], without[-1], rtol=1e-4, atol=1e-4)   # blending weights: sums in another order


@pytest.mark.parametrize("record", [False, True])
@pytest.mark.parametrize("depth,aux", [(0, 0), (0, 3), (0, 8), (1, 2), (1, 8)])
def test_records_change_no_bit(monkeypatch, depth, aux, record):
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    sc = S.scene_room(P=30011, seed=4, half=1.5)
    o, d = view(331, 317)
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    with_, without, size = both(monkeypatch, tracer, sc, o, d, depth, aux, record=record)
    assert size == (RECORD_BYTES * 30011 if aux <= 4 or depth else 0) + 8 * blocks_of(o)
    for a, b in zip(with_, without):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("case", ["eight channels", "rows", "hand-over", "one layer", "options"])
def test_nothing_is_made_that_no_kernel_reads(monkeypatch, case):
    """No memory is taken for it, and where a caller gives all that the size could want, none of it is written."""
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    P = 3000 if case == "one layer" else 30011
    sc = S.scene_room(P=P, seed=4, half=0.4 if case == "one layer" else 1.5)
    assert (layers(sc["vertices"]) < 1.8) == (case == "one layer")
    o, d = view(256, 399) if case == "rows" else view(331, 317)   # 102,144 rays; 104,927
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    if case == "hand-over":
        tracer.optix_context.set_handover(_C.HANDOVER_ALWAYS, 4000)
    if case == "options":
        tracer.optix_context.distortion = True
    read = 8 * blocks_of(o) if case == "eight channels" else 0    # the order
    given = []

    def all_of_it(p, keep):
        size = _C.load_library().dst_trace_scratch_bytes(p.P, p.H, p.W)
        assert size == RECORD_BYTES * P + 8 * blocks_of(o)
        assert _C.load_library().dst_trace_scratch_needed(tracer.optix_context.handle, _C.C.byref(p)) == (0 if p.flags else read)
        given.append(torch.full((size,), 0xA5, dtype=torch.uint8, device="cuda"))
        keep["scratch"], p.scratch = given[0], given[0].data_ptr()

    monkeypatch.setattr(_C, "_scratch", all_of_it)
    g = {k: v.cuda() for k, v in sc.items()}
    e, bg, eye = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    others = torch.rand(P, 8).cuda() if case == "eight channels" else e
    out = _C.trace_surfels(tracer.optix_context, False, True, o.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3, e,
                           others, g["opacities"], g["scales"], 1.0, g["rotations"], e, eye, eye, bg, False, False, 0, 0.0)
    assert out[0].std() > 0.01
    if case == "options":
        assert not given
    else:
        assert bool((given[0][read:] == 0xA5).all())


@pytest.mark.parametrize("factor", [0.0, 1e-42, 1e-20, 2.0 ** -40, 0.99 * 2.0 ** -40, 1.0, 2.0 ** 40, 1.01 * 2.0 ** 40, 1e20, 3e38,
                                    -1.0, float("inf"), float("nan")])
def test_scales_of_any_size(monkeypatch, factor):
    """The quads stay what they are; the scales the trace is given are theirs times `factor`, on every third surfel."""
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    sc = S.scene_room(P=20000, seed=5, half=1.5)
    o, d = view(257, 407)
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    sc["scales"][::3] *= factor
    if factor in (2.0 ** -40, 2.0 ** 40):   # the edges of the reciprocals' range
        sc["scales"][::3] = factor
    sc["means3D"][1::50] = 1e30             # far too large to divide by way of a reciprocal
    with_, without, size = both(monkeypatch, tracer, sc, o, d)
    assert size > RECORD_BYTES * 20000
    for a, b in zip(with_, without):
        same = (a.view(torch.int32) == b.view(torch.int32)) | (torch.isnan(a) & torch.isnan(b))
        assert bool(same.all())


def test_misaligned_scratch_is_refused(monkeypatch):
    import diff_surfel_tracing as dst
    tracer = dst.SurfelTracer()
    sc = S.scene_cube(P=64, seed=0)
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    o, d = S.rays_cube(257, 407)
    called = []

    def shifted(p, keep):
        keep["scratch"] = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
        p.scratch = keep["scratch"].data_ptr() + 64
        called.append(p.scratch)

    monkeypatch.setattr(_C, "_scratch", shifted)
    e, bg, eye = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    g = {k: v.cuda() for k, v in sc.items()}
    with pytest.raises(RuntimeError, match="aligned"):
        _C.trace_surfels(tracer.optix_context, False, True, o.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3,
                         e, e, g["opacities"], g["scales"], 1.0, g["rotations"], e, eye, eye, bg, False, False, 0, 0.0)
    assert called
