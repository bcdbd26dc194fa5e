"""Training steps of one context on two streams in turn, without the host waiting in between: the buffers kept between
calls (records, rows of gradient sums and marks) go from stream to stream, grow with the scene and change with the
mode, and every step's gradients are those of the step on its own.  (Images small enough to share nothing else: ray lists
and images of 1536 blocks and more must not overlap on one context.)"""
import pytest
import torch

import dst_scenes as S
from helpers import GRAD_REL, PARAM_NAMES, assert_same_sums, settings

pytestmark = pytest.mark.gpu
DEV = "cuda"


def step(tracer, st, g, o, d, ug, leaf):
    out = tracer(o, d, g["vertices"], leaf["means3D"], torch.zeros_like(leaf["means3D"]), shs=leaf["shs"],
                 others_precomp=leaf["others_precomp"], opacities=leaf["opacities"], scales=leaf["scales"],
                 rotations=leaf["rotations"], tracer_settings=st)
    names = [k for k in PARAM_NAMES if k in leaf]
    losses = [out[0], out[1], out[2], out[3], out[5]]
    return dict(zip(names, torch.autograd.grad(losses, [leaf[k] for k in names], [ug[k] for k in ("rgb", "dpt", "acc", "norm", "aux")])))


@pytest.mark.parametrize("size,handover", [((48, 64), True), ((152, 176), True), ((152, 176), False)])
def test_two_streams_in_turn(size, handover):
    import diff_surfel_tracing as dst
    H, W = size
    tracer = dst.SurfelTracer()
    if not handover:   # the larger image by tiles
        tracer.optix_context.set_handover(dst._C.HANDOVER_OFF)
    st = settings(dst, H, W, DEV)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    views = [tuple(t.to(DEV) for t in S.rays_cube(H, W, view=v)) for v in range(4)]
    ups = [{k: t.to(DEV) for k, t in S.upstream_grads(H, W, 2, seed=v).items()} for v in range(4)]
    for P in (3000, 7000, 16000):                    # each scene needs larger rows than the one before
        g = {k: v.to(DEV) for k, v in S.scene_cube(P=P, seed=P, aux=2).items()}
        tracer.build_acceleration_structure(g["vertices"], g["faces"], True)
        leaf = {k: g[k].clone().requires_grad_(True) for k in PARAM_NAMES if k in g}
        fresh = dst.SurfelTracer()
        fresh.build_acceleration_structure(g["vertices"], g["faces"], True)
        want = [step(fresh, st, g, *views[v], ups[v], leaf) for v in range(4)]
        torch.cuda.synchronize()
        for det in (False, True, False):
            tracer.deterministic = det
            tracer.optix_context.deterministic_check = False     # (it waits)
            got, noise = [], []
            for v in range(4):
                with torch.cuda.stream(streams[v % 2]):
                    got.append(step(tracer, st, g, *views[v], ups[v], leaf))
                    # what the allocator has free on either stream is taken and written over at once
                    noise.append([torch.full((n,), 7.0, device=DEV) for n in (P * 66, P, P // 4)])
            torch.cuda.synchronize()
            for v in range(4):
                for k in want[v]:
                    assert_same_sums(got[v][k].cpu().numpy(), want[v][k].cpu().numpy(), GRAD_REL, "view %d %s" % (v, k))
            del noise
    tracer.optix_context.release_memory()
    assert not tracer.optix_context._row_pool and not tracer.optix_context._record_pool


@pytest.mark.parametrize("size,depth,handover", [((48, 64), 0, True), ((152, 176), 1, True), ((152, 176), 1, False)])
def test_a_captured_training_step_can_be_replayed(size, depth, handover):
    """Forward and backward recorded into a graph: every replay gives the eager gradients, with eager training steps in
    between, one of them in two halves around the replay (the graph's record and rows are its own).  (Without the hand-over the
    larger image's first bounce is traced by tiles, its reflections by rows.)"""
    import diff_surfel_tracing as dst
    H, W = size
    tracer = dst.SurfelTracer()
    if not handover:
        tracer.optix_context.set_handover(dst._C.HANDOVER_OFF)
    st = settings(dst, H, W, DEV, max_trace_depth=depth, specular_threshold=0.1)
    g = {k: v.to(DEV) for k, v in S.scene_room(P=6000, seed=1, aux=2, half=1.5).items()}
    g["others_precomp"][:, 0] = g["others_precomp"][:, 0] * 0.8 + 0.1
    tracer.build_acceleration_structure(g["vertices"], g["faces"], True)
    o, d = (t.to(DEV) for t in S.pinhole_rays(H, W, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15)))
    o2, d2 = (t.to(DEV) for t in S.pinhole_rays(H, W, 50.0, (0.6, 0.3, 0.15), (-0.9, 0.45, -0.15)))
    ug = {k: t.to(DEV) for k, t in S.upstream_grads(H, W, 2, seed=2).items()}
    leaf = {k: g[k].clone().requires_grad_(True) for k in PARAM_NAMES if k in g}
    own = lambda grads: {k: v.clone() for k, v in grads.items()}  # noqa: E731
    for _ in range(3):                                   # the record's size settles
        want, want2 = own(step(tracer, st, g, o, d, ug, leaf)), own(step(tracer, st, g, o2, d2, ug, leaf))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(tracer, st, g, o, d, ug, leaf)              # warm-up on a side stream, as torch asks before a capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(tracer, st, g, o, d, ug, leaf)
    for k in range(4):
        for t in got.values():
            t.fill_(-7.0)
        out = tracer(o2, d2, g["vertices"], leaf["means3D"], torch.zeros_like(leaf["means3D"]), shs=leaf["shs"],
                     others_precomp=leaf["others_precomp"], opacities=leaf["opacities"], scales=leaf["scales"],
                     rotations=leaf["rotations"], tracer_settings=st)
        graph.replay()
        half = torch.autograd.grad([out[0], out[1], out[2], out[3], out[5]], list(leaf.values()),
                                   [ug[n] for n in ("rgb", "dpt", "acc", "norm", "aux")])
        torch.cuda.synchronize()
        for name, eager in zip(leaf, half):
            assert_same_sums(got[name].cpu().numpy(), want[name].cpu().numpy(), GRAD_REL, "replay %d %s" % (k, name))
            assert_same_sums(eager.cpu().numpy(), want2[name].cpu().numpy(), GRAD_REL, "around replay %d %s" % (k, name))
        if k == 1:
            tracer.optix_context.release_memory()
            torch.cuda.empty_cache()
