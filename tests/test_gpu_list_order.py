"""Ray lists at the sizes where the order they are traced in changes (2048 rays by tiles, 65,536 and 262,144 by rows): what a ray
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


def _pixels(n, seed, cameras=1):
    """n pixels of cameras in a room of half a size of 1.5, in no order"""
    r = torch.Generator().manual_seed(seed)
    parts = []
    for _ in range(cameras):
        eye = torch.rand(3, generator=r) * 2.0 - 1.0
        parts.append(S.pinhole_rays(256, (n // cameras + 256) // 256, 70.0, tuple(eye.tolist()), tuple((-eye + 0.1).tolist())))
    o, d = (torch.cat([p[k].reshape(-1, 3) for p in parts])[None] for k in (0, 1))
    at = torch.randperm(o.shape[1], generator=r)[:n]
    return o[:, at].contiguous(), d[:, at].contiguous()


def _list(kind, n):
    if kind in ("one place", "twenty places"):
        return _pixels(n, 1, 1 if kind == "one place" else 20)
    if kind.startswith("rows of"):   # an image, row after row
        w = int(kind.split()[-1])
        return tuple(x.reshape(1, -1, 3)[:, :n].contiguous() for x in S.pinhole_rays((n + w - 1) // w, w, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15)))
    if kind == "in order":
        a = torch.arange(n) * (6.2831853 / 2048)
        el = torch.floor(torch.arange(n) / 2048.0) * 0.01 - 0.3
        d = torch.stack([a.cos() * el.cos(), a.sin() * el.cos(), el.sin()], 1)[None]
        return torch.zeros(1, n, 3) + 0.1, d.contiguous()
    r = torch.Generator().manual_seed(2)
    return (torch.rand(1, n, 3, generator=r) * 2 - 1) * 1.4, torch.nn.functional.normalize(torch.randn(1, n, 3, generator=r), dim=-1)


def _forward(tracer, sc, o, d, record=None):
    from diff_surfel_tracing import _C
    g = {k: v.cuda() for k, v in sc.items()}
    e, bg, eye = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    return _C.trace_surfels(tracer.optix_context, False, True, o.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3, e, e,
                            g["opacities"], g["scales"], 1.0, g["rotations"], e, eye, eye, bg, False, False, 0, 0.0, hit_record=record)[:7]


@pytest.fixture(scope="module")
def room():
    import diff_surfel_tracing as dst
    sc = S.scene_room(P=20000, seed=3, half=1.5)
    tracer = dst.SurfelTracer()
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    return tracer, sc


@pytest.mark.parametrize("kind,n,sorts", [
    ("one place", 65535, None), ("one place", 65536, True), ("one place", 66560, True), ("one place", 66561, True), ("one place", 300001, True),
    ("twenty places", 100003, True), ("in order", 65536, False),
    ("rows of 256", 65536, False), ("rows of 512", 131072, False), ("rows of 1024", 131072, False), ("rows of 100", 70000, False), ("in order", 262147, False), ("unrelated", 131071, False),
    ("unrelated", 262144, True)])
def test_which_lists_are_sorted(room, kind, n, sorts):
    """The order that the record of a list keeps has every ray once; it is the rays' own for lists that come in order, and
    for unrelated rays that are not very many, and puts rays of nearly the same direction together otherwise."""
    from diff_surfel_tracing import _C
    tracer, sc = room
    o, d = _list(kind, n)
    record = _C.HitRecord(1, n, 1, 1.0, torch.device("cuda"))
    header = _C.HitRecord.layout(1, n, 1, 1.0)[1]
    kept = record.words[header:header + (n + 1) // 2]
    kept.fill_(-1)
    _forward(tracer, sc, o, d, record)
    order = kept.view(torch.int32)[:n].cpu().long()
    if sorts is None:   # too short: nothing is left there
        assert bool((order == -1).all())
        return
    assert torch.equal(order.sort().values, torch.arange(n))
    assert torch.equal(order, torch.arange(n)) == (not sorts)
    if sorts:
        def apart(at):   # from one ray to the next, where they begin and where they go
            return (o[0][at][1:] - o[0][at][:-1]).norm(dim=-1).mean() + (d[0][at][1:] - d[0][at][:-1]).norm(dim=-1).mean()
        assert apart(order) < 0.5 * apart(torch.arange(n))
        if kind == "one place":
            # directions of a key lie within a sixteenth of a 256 x 256 map's side or so of each other
            assert apart(order) < 0.05


@pytest.mark.parametrize("kind", ["one place", "unrelated", "odd"])
def test_order_changes_no_bit(monkeypatch, room, kind):
    """With the order and without; rays that go nowhere or begin nowhere among them."""
    from diff_surfel_tracing import _C
    tracer, sc = room
    n = 262145 if kind == "unrelated" else 70001
    o, d = _list("one place" if kind == "odd" else kind, n)
    if kind == "odd":
        d[0, 5::97] = 0.0
        d[0, 7::193] = float("nan")
        d[0, 11::211, 0] = float("inf")
        o[0, 13::89, 1] = float("nan")
        o[0, 17::83, 2] = float("inf")
        o[0, 19::79] = 1e30
        d[0, 23::71] *= 1e-30
    with_ = _forward(tracer, sc, o, d)
    record = _C.HitRecord(1, n, 1, 8.0, torch.device("cuda"))
    recorded = _forward(tracer, sc, o, d, record)
    monkeypatch.setattr(_C, "_scratch", lambda p, keep, *more: None)
    without = _forward(tracer, sc, o, d)
    record2 = _C.HitRecord(1, n, 1, 8.0, torch.device("cuda"))
    _forward(tracer, sc, o, d, record2)
    assert without[0].std() > 0.01
    for k in range(7):
        for x in (with_[k], recorded[k]):
            a, b = x, without[k]
            assert bool(((a.view(torch.int32) == b.view(torch.int32)) | (torch.isnan(a) & torch.isnan(b))).all()), k
    header = _C.HitRecord.layout(1, n, 1, 8.0)[1]
    order = record2.words[header:header + (n + 1) // 2].view(torch.int32)[:n]
    assert torch.equal(order.cpu(), torch.arange(n, dtype=torch.int32))   # (a record has one in any case: the backward trace reads it)


@pytest.mark.parametrize("surfels,n,record,looks", [(20000, 65535, True, False), (20000, 65536, False, True), (4000, 65536, False, False),
                                                    (4000, 65536, True, True), (4000, 262143, False, False), (4000, 262144, False, True)])
def test_which_lists_are_looked_at(monkeypatch, surfels, n, record, looks):
    """Long ones, in thin scenes (a room covered 1.3 times instead of 6) longer ones where nothing is recorded.  The others
    take no memory for it and come as they are, with the same results."""
    from diff_surfel_tracing import _C
    import diff_surfel_tracing as dst
    sc = S.scene_room(P=surfels, seed=3, half=1.5)
    tracer = dst.SurfelTracer()
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    real, taken = _C._scratch, []

    def spy(p, keep):
        real(p, keep)
        taken.append(bool(p.scratch))

    o, d = _list("one place", n)
    out = []
    for scratch in (spy, lambda p, keep: None):
        monkeypatch.setattr(_C, "_scratch", scratch)
        out.append(_forward(tracer, sc, o, d, _C.HitRecord(1, n, 1, 4.0, torch.device("cuda")) if record else None))
    assert taken in ([], [False]) if not looks else taken == [True]
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def test_deterministic_sums_know_no_order(room):
    """Fixed-point sums of a sorted list: the same bits from run to run, wherever its rays stand."""
    tracer, sc = room
    n = 70001
    o, d = _list("one place", n)
    r = torch.Generator().manual_seed(9)
    up = {k: torch.randn(1, n, c, generator=r) for k, c in (("rgb", 3), ("dpt", 1), ("norm", 3))}
    perm = torch.randperm(n, generator=r)
    tracer.deterministic = True
    try:
        got = []
        for at in (torch.arange(n), torch.arange(n), perm):
            tracer.optix_context.record_blocks_per_wave = 12.0
            got.append(gpu_trace(tracer, sc, o[:, at], d[:, at], upstream={k: v[:, at] for k, v in up.items()}, build=False)[1])
        for other in got[1:]:
            for k, g in got[0].items():
                if g is not None and k not in ("ray_o", "ray_d"):
                    assert (g.view("int32") == other[k].view("int32")).all(), k
    finally:
        tracer.deterministic = False


def test_order_in_a_graph(room):
    """The order is made on the device in every replay: other rays in the captured buffers, other orders."""
    tracer, sc = room
    n = 66000
    lists = [_list("one place", n), _list("in order", n), _pixels(n, 7)]
    o, d = (t.cuda() for t in lists[0])
    g = {k: v.cuda() for k, v in sc.items()}
    eager = [[t.clone() for t in _forward(tracer, g, *x)] for x in lists]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        _forward(tracer, g, o, d)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _forward(tracer, g, o, d)
    for k in (0, 1, 2, 0, 2):
        o.copy_(lists[k][0])
        d.copy_(lists[k][1])
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, eager[k]):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))
        _forward(tracer, g, *(t.cuda() for t in lists[(k + 1) % 3]))   # the program's own work in between
        torch.cuda.synchronize()
