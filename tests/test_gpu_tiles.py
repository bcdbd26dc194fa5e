"""Images traced by tiles of 8x8 rays (the bundle walk) without the tile hand-over, against the oracle: the degenerate
scenes of the random sweep, whose own images are small enough to be traced ray by ray, and the options of the forward
trace.  152 x 176 rays are 418 tiles; HANDOVER_OFF keeps the walk whatever the scene holds."""
import warnings

import numpy as np
import pytest
import torch

import dst_scenes as S
import helpers
from helpers import assert_forward_exact, gpu_trace, oracle_scene
from test_gpu_parity import _with_scales, check_case
from test_gpu_sweep import TRAITS, _apply_trait

pytestmark = pytest.mark.gpu
H, W = 152, 176


def tile_tracer(**options):
    import diff_surfel_tracing as dst
    from diff_surfel_tracing import _C
    t = dst.SurfelTracer()
    t.optix_context.set_handover(_C.HANDOVER_OFF)
    for k, v in options.items():
        setattr(t, k, v)
    return t


def view(kind):
    if kind == "room":
        return S.pinhole_rays(H, W, 70.0, (-0.6, -0.3, 0.15), (0.9, 0.45, -0.15))
    if kind == "lidar":
        return S.pinhole_rays(H, W, 80.0, (0.0, 0.0, 1.8), (30.0, 10.0, 0.0))
    return S.rays_cube(H, W, view=1)


@pytest.mark.parametrize("fine", [False, True])
@pytest.mark.parametrize("trait", sorted(set(TRAITS)))
def test_degenerate_scenes(oracle, monkeypatch, trait, fine):
    """As in the sweep: its shares of elements that may lean on the rounding allowance."""
    seed = 100 * sorted(set(TRAITS)).index(trait) + 7 * fine
    kind = ("cube", "room", "lidar")[seed % 3]
    P = 300 if trait == "samepoint" else 4000
    sc = {"cube": lambda: S.scene_cube(P=P, seed=seed, aux=2), "room": lambda: S.scene_room(P=P, seed=seed, aux=4, half=1.5),
          "lidar": lambda: S.scene_lidar(P=P, seed=seed, aux=0)}[kind]()
    if fine:
        sc = _with_scales(sc, 1.0 / 30.0)
    sc = {k: v.clone() for k, v in sc.items()}
    move, zoom = _apply_trait(sc, trait, torch.Generator().manual_seed(seed + 77))
    o, d = view(kind)
    o = (o * zoom + (0.0 if move is None else move)).contiguous()
    monkeypatch.setattr(helpers, "MAX_LOUD", 1.0)
    monkeypatch.setattr(helpers, "MAX_NOISY", 2e-2)
    monkeypatch.setattr(helpers, "MIN_NOISY", 8)
    tracer = tile_tracer()
    check_case(oracle, tracer, sc, o, d, bg=(0.1, 0.3, 0.2), start_from_first=not fine)
    info = tracer.optix_context.trace_info()
    assert info.handover_active == 0 and info.tiles_handed_over == 0


@pytest.mark.parametrize("aux,colors,sh", [(0, False, 1), (2, True, 3), (3, False, 0), (8, False, 3)])
def test_deterministic_mode(oracle, aux, colors, sh):
    """Fixed-point sums: the oracle's gradients, and the same bits on every run (after the first, which sizes the
    record)."""
    sc = S.scene_room(P=9000, seed=aux, aux=aux, half=1.5)
    if colors:
        sc["colors_precomp"] = torch.rand(9000, 3, generator=torch.Generator().manual_seed(3))
        del sc["shs"]
    tracer = tile_tracer(deterministic=True)
    runs = []
    with warnings.catch_warnings():
        warnings.simplefilter("error", RuntimeWarning)
        for _ in range(3):
            ref, out = check_case(oracle, tracer, sc, *view("room"), **({} if colors else {"sh_degree": sh}))
            runs.append((out["wet"], ref["grads_gpu"]))
    for k, v in runs[1][1].items():
        assert v is None or np.array_equal(v.view(np.uint32), runs[2][1][k].view(np.uint32)), k
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[1][0], runs[2][0])


@pytest.mark.parametrize("det", [False, True])
def test_half_coefficients_and_distortion(oracle, det):
    sc = S.scene_cube(P=8000, seed=4)
    o, d = view("cube")
    seen = dict(sc)
    seen["shs"] = sc["shs"].half().float()               # what the kernels read
    tracer = tile_tracer(sh_half=True, distortion=True, deterministic=det)
    out, _ = gpu_trace(tracer, sc, o, d)
    ref = oracle.forward(oracle_scene(oracle, seen, o, d), oracle.HITS_BVH_LEXI, compute_dist=True)
    assert_forward_exact({**out, "dist": 0 * out["dist"]}, {**ref, "dist": 0 * ref["dist"]})
    np.testing.assert_array_equal(out["dist"].view(np.uint32), ref["dist"][..., :1].view(np.uint32))
    assert out["dist"].max() > 1e-6
    tracer.distortion = False
    check_case(oracle, _HalfSeen(tracer, sc["shs"]), seen, o, d)


class _HalfSeen:
    """The tracer, given the fp32 coefficients where the oracle is given their binary16 values."""

    def __init__(self, tracer, shs):
        self._tracer, self._shs = tracer, shs

    def __getattr__(self, name):
        return getattr(self._tracer, name)

    def __call__(self, *a, shs=None, **k):
        return self._tracer(*a, shs=shs + (self._shs.to(shs.device) - shs.detach()), **k)


@pytest.mark.parametrize("aux,det", [(2, False), (4, True), (8, False)])
@pytest.mark.parametrize("P", [1, 3, 4, 5, 100, 101, 107, 108, 109, 112, 113, 240])
def test_gradient_table_edges(oracle, P, aux, det):
    """One 16x16 block before P faint surfels that all of its rays meet: its table of gradients (112, 108 or 100 rows with two, four or
    eight auxiliary channels, in groups of four) takes few of them, all, or no more than it has rows for."""
    sc = {k: v.clone() for k, v in S.scene_cube(P=P, seed=P, aux=aux).items()}
    gen = torch.Generator().manual_seed(P)
    sc["means3D"] = torch.cat([2.0 + 0.01 * torch.arange(P)[:, None].float(), 0.05 * torch.randn(P, 2, generator=gen)], 1)
    q = torch.tensor([0.7071, 0.0, 0.7071, 0.0]) + 0.05 * torch.randn(P, 4, generator=gen)   # facing along x
    sc["rotations"] = q / q.norm(dim=1, keepdim=True)
    sc["scales"] = 0.5 + 0.2 * torch.rand(P, 2, generator=gen)
    sc["opacities"] = 0.02 + 0.02 * torch.rand(P, 1, generator=gen)
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    o, d = S.pinhole_rays(16, 16, 10.0, (0.0, 0.0, 0.0), (1.0, 0.0, 0.0))
    ref, _ = check_case(oracle, tile_tracer(deterministic=det), sc, o, d)
    assert ref["n_con"].min() >= 0.9 * P   # (a ray in ten is outside some splat)


@pytest.mark.parametrize("aux,det", [(0, False), (3, True), (8, False)])
@pytest.mark.parametrize("P", [63, 64, 65, 129])
def test_closing_edges(oracle, P, aux, det):
    """Sizes around the 64 surfels that the closing kernel takes at a time, every other surfel met by no ray: the oracle's
    gradients, and again from rows that the call before left empty."""
    sc = {k: v.clone() for k, v in S.scene_cube(P=P, seed=P, aux=aux).items()}
    sc["means3D"][1::2, 2] += 50.0
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    tracer = tile_tracer(deterministic=det)
    for _ in range(2):
        ref, _ = check_case(oracle, tracer, sc, *view("cube"))
        assert np.abs(ref["grads_gpu"]["means3D"][0::2]).max() > 0.0 and not ref["grads_gpu"]["means3D"][1::2].any()


@pytest.mark.parametrize("kind,fov", [("cube", 20.0), ("cube", 140.0), ("room", 70.0), ("lidar", 110.0)])
@pytest.mark.parametrize("shrink,shift", [(1.0, 0.0), (1.0 / 30.0, 0.0), (20.0, 0.0), (1.0, 3e4)])
def test_rays_of_one_origin(kind, fov, shrink, shift):
    """Bundles whose rays begin at one place leave out quads by their edges.  With one ray of every tile moved a little
    they do not; the other rays' results have to be the same bit for bit.  Slivers of quads, far from the origin too."""
    from diff_surfel_tracing import _C
    sc = {"cube": lambda: S.scene_cube(P=6000, seed=2), "room": lambda: S.scene_room(P=9000, seed=2, half=1.5),
          "lidar": lambda: S.scene_lidar(P=9000, seed=2, aux=0)}[kind]()
    sc = {k: v.clone() for k, v in sc.items() if k != "others_precomp"}
    sc["scales"] = sc["scales"] * shrink
    sc["scales"][::3, 0] *= 25.0
    sc["means3D"] += shift
    sc["vertices"], sc["faces"] = S.get_triangles(sc["means3D"], sc["scales"], sc["rotations"])
    eye = {"cube": (3.0, 0.2, 0.1), "room": (-0.6, -0.3, 0.15), "lidar": (0.0, 0.0, 1.8)}[kind]
    o, d = S.pinhole_rays(H, W, fov, eye, (0.0, 0.0, 0.0) if kind == "cube" else (1.0, 0.45, 0.15))
    o = o + shift
    moved = o.clone()
    moved[3::8, 5::8] += 1e-3 * (1.0 + abs(shift))
    same = torch.ones(H, W, dtype=torch.bool)
    same[3::8, 5::8] = False
    tracer = tile_tracer()
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    g = {k: v.cuda() for k, v in sc.items()}
    e, bg, eye4 = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    out = [_C.trace_surfels(tracer.optix_context, False, True, x.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3, e, e,
                            g["opacities"], g["scales"], 1.0, g["rotations"], e, eye4, eye4, bg, False, False, 0, 0.0)[:6]
           for x in (o, moved)]
    for a, b in zip(*out):
        assert torch.equal(a.cpu()[same].view(torch.int32), b.cpu()[same].view(torch.int32))


@pytest.mark.parametrize("H_,W_,fov", [(24, 16, 2.0), (40, 48, 35.0), (33, 17, 8.0)])
def test_limb_of_a_sphere(H_, W_, fov):
    """Tiles whose way is full of quads that their edges leave out none of (a bundle that has looked at many for nothing looks at
    edges no more), and tiles beside them that quads are left out for: the same bits with one ray of every tile moved a
    little, for which the edges are not looked at."""
    from diff_surfel_tracing import _C
    sc = S.scene_sphere(P=60000, seed=3)
    # along the tangent from the eye: the limb crosses the image from top to bottom
    o, d = S.pinhole_rays(H_, W_, fov, (4.0, 0.0, 0.0), (0.25, 0.968, 0.0) if fov < 30 else (0.0, 0.0, 0.0))
    moved = o.clone()
    moved[3::8, 5::8] += 1e-3
    same = torch.ones(H_, W_, dtype=torch.bool)
    same[3::8, 5::8] = False
    tracer = tile_tracer()
    tracer.build_acceleration_structure(sc["vertices"].cuda(), sc["faces"].cuda(), rebuild=True)
    g = {k: v.cuda() for k, v in sc.items()}
    e, bg, eye4 = torch.empty(0, device="cuda"), torch.zeros(3, device="cuda"), torch.eye(4, device="cuda")
    out = [_C.trace_surfels(tracer.optix_context, False, True, x.cuda(), d.cuda(), g["vertices"], bg, g["means3D"], g["shs"], 3, e, e,
                            g["opacities"], g["scales"], 1.0, g["rotations"], e, eye4, eye4, bg, False, False, 0, 0.0)[:6]
           for x in (o, moved)]
    assert out[0][2].max() > 0.9
    for a, b in zip(*out):
        assert torch.equal(a.cpu()[same].view(torch.int32), b.cpu()[same].view(torch.int32))
