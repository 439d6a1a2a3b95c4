"""Scene building on the device: the shading records of meshes of many sizes
in one launch, and rebuilding after an edit."""
import dataclasses

import numpy as np
import pytest

import orc
from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from colvillea_amd import _capi as capi
from colvillea_amd.integrator import DiffuseMtl, Entity, TriangleMesh
from test_gpu_edges import _gpu_tables

pytestmark = pytest.mark.gpu


def _pieces():
    """The textured scene with its sphere cut into meshes of 1 triangle to
    just over a block's 256, with and without normals, uvs and tangents, and
    empty meshes first, last and between."""
    desc = scenes.make_textured(width=64, height=48, spp=2, hdri_w=64, hdri_h=32)
    ground, sphere = desc.meshes
    uv = np.stack([sphere.vertices[:, 0], sphere.vertices[:, 1]], 1).astype(np.float32)
    tan = np.cross(sphere.normals, [0.3, 0.8, 0.5]).astype(np.float32)
    empty = TriangleMesh(np.zeros((0, 3)), np.zeros((0, 3)))
    meshes, mesh_of, mtl, xf = [empty, ground], [1], [desc.instance_material[0]], [desc.instance_xform[0]]
    at = 0
    for i, n in enumerate((255, 1, 256, 257, 2, 300, 209)):
        if i in (2, 5):
            meshes.append(empty)
        t = sphere.triangles[at:at + n]
        at += n
        used, idx = np.unique(t, return_inverse=True)
        meshes.append(TriangleMesh(sphere.vertices[used], idx.reshape(-1, 3).astype(np.uint32),
                                   normals=sphere.normals[used] if i % 2 else None, uvs=uv[used] if i % 3 else None,
                                   tangents=tan[used] if i % 4 == 1 else None))
        for k in range(1, 5):
            mesh_of.append(len(meshes) - 1)
            mtl.append(desc.instance_material[1 + (k + i) % 4])
            xf.append(desc.instance_xform[k])
    assert at == len(sphere.triangles)
    meshes.append(empty)
    return dataclasses.replace(desc, meshes=meshes, instance_mesh=mesh_of, instance_material=mtl, instance_xform=np.stack(xf))


def _render(integ, desc):
    integ.resetIterationIndex()
    integ.render(desc.spp)
    return integ.readbackSums(), integ.counters()


def _check(desc, sums, cnt, tables):
    osums, ocnt = orc.Scene(desc, tables=tables).render("f32", samples=(0, desc.spp))
    D = desc.max_depth + 1
    for k in ("rays", "hits", "shadow", "visible"):
        assert np.array_equal(cnt[k][:D], ocnt[k][:D]), (k, cnt[k][:D], ocnt[k][:D])
    # the parity tests' bound: float32 path sums against the oracle's
    assert np.mean((sums - osums) ** 2 / (osums ** 2 + 1e-2)) < 1e-12


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
def test_shading_records_of_many_meshes(width):
    desc = _pieces()
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, desc.width, desc.height) as integ:
        integ.setBVHWidth(width)
        upload_scene(integ, desc)
        sums, cnt = _render(integ, desc)
        _check(desc, sums, cnt, _gpu_tables(integ, desc))


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
def test_rebuild_after_an_edit(width):
    """A mesh replaced by one of another size (every later mesh's records
    move), then an instance moved: each the scene built anew."""
    desc = _pieces()
    k = 4  # the piece of 1 triangle
    other = dataclasses.replace(desc.meshes[-2])
    edited = dataclasses.replace(desc, meshes=desc.meshes[:k] + [other] + desc.meshes[k + 1:])
    moved = edited.instance_xform.copy()
    moved[5:9, 1, 3] += 0.7
    moved = dataclasses.replace(edited, instance_xform=moved)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, desc.width, desc.height) as integ:
        integ.setBVHWidth(width)
        upload_scene(integ, desc)
        _render(integ, desc)
        integ.rebuildBLAS([k], [edited.meshes[k]])
        for d in (edited, moved):
            integ.buildTLAS([d.meshes[m] for m in d.instance_mesh], list(range(len(d.instance_mesh))), d.instance_xform)
            sums, cnt = _render(integ, d)
            _check(d, sums, cnt, _gpu_tables(integ, d))


def _hits(integ, rays):
    n = len(rays)
    t, b, inst, prim = np.zeros(n, np.float32), np.zeros((n, 2), np.float32), np.zeros(n, np.uint32), np.zeros(n, np.uint32)
    capi.check(capi.lib().clhip_trace_batch(integ.ctx, capi.fptr(rays), n, capi.fptr(t), capi.fptr(b), capi.uptr(inst),
                                            capi.uptr(prim)), integ.ctx)
    return t, b, inst, prim


def test_packed_nodes_of_large_trees_and_of_moved_instances():
    """Trees of more nodes than are packed at a time: hits equal those of
    the other tree width (which is not packed), for a first build, moved
    instances, more instances (the node array grows) and fewer."""
    side = 301
    g = np.linspace(-4.0, 4.0, side, dtype=np.float32)
    x, z = np.meshgrid(g, g, indexing="ij")
    y = (0.3 * np.sin(3.0 * x) * np.cos(2.0 * z)).astype(np.float32)
    i = np.arange((side - 1) * side).reshape(side - 1, side)[:, :-1].ravel()
    tri = np.concatenate([np.stack([i, i + 1, i + side], 1), np.stack([i + 1, i + side + 1, i + side], 1)]).astype(np.uint32)
    mesh = TriangleMesh(np.stack([x.ravel(), y.ravel(), z.ravel()], 1), tri)
    ball = scenes.icosphere(2)
    rng = np.random.default_rng(3)
    n = 50000
    o = rng.uniform(-5.0, 5.0, (n, 3))
    d = rng.uniform(-6.0, 6.0, (n, 3)) * [1.0, 0.1, 1.0] - o  # a third aim past the terrain
    rays = np.concatenate([o, np.zeros((n, 1)), d / np.linalg.norm(d, axis=1, keepdims=True), np.full((n, 1), 3e38)],
                          1).astype(np.float32)
    ctx = []
    for width in (4, 8):
        integ = Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8)
        integ.setBVHWidth(width)
        integ.buildMaterials([DiffuseMtl((0.5, 0.5, 0.5))])
        integ.buildGeometryEntities([Entity(0)] * 71)
        integ.buildBLAS([mesh, ball])
        ctx.append(integ)
    try:
        for balls, seed in ((1, 0), (1, 1), (70, 2), (3, 3), (70, 4)):
            r = np.random.default_rng(seed)
            xf = np.concatenate([scenes.IDENTITY[None]] + [scenes.translate_scale(r.uniform(-3, 3, 3), r.uniform(0.1, 0.6))[None]
                                                           for _ in range(balls)]).astype(np.float32)
            out = []
            for integ in ctx:
                integ.buildTLAS([mesh] + [ball] * balls, list(range(balls + 1)), xf)
                out.append(_hits(integ, rays))
            assert 0.2 < (out[0][0] > 0).mean() < 0.95 and np.any(out[0][2] == balls)
            for a, b in zip(*out):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (balls, seed)
        nodes = (ctx[0].counters()["scene_bytes"] - 48 * (len(tri) + len(ball.triangles))) // 80
        assert nodes > 32768, nodes
    finally:
        for integ in ctx:
            integ.close()
