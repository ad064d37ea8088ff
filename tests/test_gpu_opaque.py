"""Walks without look-ups of transparent voxels (scenes whose voxels are all
opaque) and how the passes deal their work to the waves, against the FP32 oracle
and against each other, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from doonengine_amd import scenes
from doonengine_amd.volume import Batch, Volume
from test_gpu_batch import assert_same
from test_gpu_parity import draw_gpu, load_scene, oracle_scene, run_frame_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_direct", [0, 1, 24])
def test_material_turns_transparent_and_back(gpu, n_direct):
    """Materials change without an upload of voxels: the passes follow at once."""
    sc = scenes.config_small(seed=21)
    sc.materials[1].specular, sc.materials[1].shininess = 0.5, 20
    o = oracle.load("f32")
    vol = load_scene(sc)
    vol.v.numDirectRays = n_direct
    for f, opacity in enumerate((1.0, 0.4, 1.0, float(np.nextafter(np.float32(1), np.float32(2))))):
        vol.materials[0]["opacity"] = opacity
        run_frame_and_compare(vol, sc, o, f, 200.0 + f / 60.0, sc.width, sc.height)
    vol.close()


@pytest.mark.parametrize("ignore_first", [False, True])
def test_unused_transparent_material_changes_nothing(gpu, ignore_first):
    """A transparent material that no voxel holds, then one that a far voxel holds
    (the general walk, meeting no transparent voxel): same draw and rays."""
    sc = scenes.config_small(seed=22)
    a = load_scene(sc)
    a.set_material(200, opacity=0.3)
    far = scenes.config_small(seed=22)
    z, y, x = np.argwhere((far.normal_words >> 24) != 255)[0]
    far.normal_words[z, y, x] = (far.normal_words[z, y, x] & 0x00FFFFFF) | (200 << 24)
    b = load_scene(far)
    b.set_material(200, opacity=0.3)
    b.materials[200]["opacity"] = 1.0
    rng = np.random.default_rng(3)
    org = (rng.random((1000, 3)) * sc.map_size).astype(np.float32)
    d = rng.standard_normal((1000, 3)).astype(np.float32)
    pa, pb = draw_gpu(a, sc)[1], draw_gpu(b, far)[1]
    ra, rb = (v.cast_rays(org, d, ignore_first) for v in (a, b))
    b.materials[200]["opacity"] = 0.3
    o = oracle.load("f32")
    s, _ = oracle_scene(o, b, far)
    for u, v in ((pa, pb), (ra, rb)):
        for f in ("voxelIndex", "mapSteps", "voxelSteps"):
            assert np.array_equal(u[f], v[f]), f
    run_frame_and_compare(b, far, o, 0, 300.0, far.width, far.height)
    a.close()
    b.close()


def test_batch_with_one_transparent_volume(gpu):
    """The batch takes the general walk while any volume needs it, and its graph is
    captured again when that changes."""
    def build():
        vols = []
        for i in range(3):
            sc = scenes.batch_scene(i, max_grid=8)
            v = Volume(sc.map_size, min_chunks=64)
            sc.apply(v)
            v.v.numDirectRays = 16
            v.request_all()
            v.sync()
            vols.append(v)
        return vols

    va, vb = build(), build()
    batch = Batch(vb)
    for f, opacity in enumerate((1.0, 0.5, 0.5, 1.0, 1.0)):
        for v in (va[1], vb[1]):
            v.materials[0]["opacity"] = opacity
        for v in va + vb:
            v.mark_visible(100)
            v.sync()
        for v in va:
            v.update_lighting(1, 1000, 10.0 + f)
        batch.update_lighting(1, 1000, 10.0 + f)
        assert_same(va, vb, f"frame {f}")
    batch.close()
    for v in va + vb:
        v.close()


@pytest.mark.parametrize("visible", [1, 2, 7, 100000])
@pytest.mark.parametrize("n_direct", [1, 5, 16, 33, 64])
def test_direct_rays_in_parts_of_requests(gpu, n_direct, visible):
    """Few requests: a single volume's direct rays go to the waves in parts of a
    request, a batch's in whole requests."""
    sc = scenes.batch_scene(4, max_grid=8)
    vols = []
    for _ in range(2):
        v = Volume(sc.map_size, min_chunks=64)
        sc.apply(v)
        v.v.numDirectRays = n_direct
        v.request_all()
        v.sync()
        v.mark_visible(visible)
        v.sync()
        vols.append(v)
    batch = Batch(vols[1:])
    for f in range(2):
        vols[0].update_lighting(1, 1000, 20.0 + f)
        batch.update_lighting(1, 1000, 20.0 + f)
        assert_same(vols[:1], vols[1:], f"frame {f}")
        for v in vols:
            v.mark_visible(visible)
            v.sync()
    batch.close()
    for v in vols:
        v.close()


@pytest.mark.parametrize("n", [1, 63, 64, 257, 4099])
def test_ray_batches_against_oracle(gpu, n):
    """Rays that start anywhere, outside the map too."""
    sc = scenes.config_small(seed=23)
    vol = load_scene(sc)
    rng = np.random.default_rng(n)
    org = ((rng.random((n, 3)) * 1.2 - 0.1) * sc.map_size).astype(np.float32)
    d = (rng.standard_normal((n, 3)) + 1e-4).astype(np.float32)
    o = oracle.load("f32")
    s, _ = oracle_scene(o, vol, sc)
    vol.counters(2, reset=True)
    for first in (False, True):
        r = vol.cast_rays(org, d, first)
        want, _ = o.cast_rays(s, org, d, ignore_first=first)
        for f in ("hit", "voxelIndex", "mapSteps", "voxelSteps"):
            assert np.array_equal(r[f], want[f]), f
        assert np.array_equal(r["pos"].view(np.uint32), want["pos"].view(np.uint32))
        assert np.array_equal(r["normal"].view(np.uint32) & 0x7FFFFFFF, want["normal"].view(np.uint32) & 0x7FFFFFFF)
        c = vol.counters(2, reset=True)
        assert c["rays"] == n and c["hits"] == int(want["hit"].sum())
        assert c["mapSteps"] == int(want["mapSteps"].sum()) and c["voxelSteps"] == int(want["voxelSteps"].sum())
    vol.close()


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("chunks", [(16, 8, 8), (41, 5, 5), (32, 16, 32), (33, 16, 32)])
def test_visible_requests_at_launch_edges(gpu, chunks, split):
    """1024 tiles (one block), one more, the most that one launch takes, and more."""
    rng = np.random.default_rng(chunks[0])
    X, Y, Z = (8 * c for c in chunks)
    nw = np.full((Z, Y, X), 0xFFFFFFFF, np.uint32)
    for _ in range(3):                                     # chunks of 1..3 request words and empty ones
        at = rng.random((Z // 8, Y // 8, X // 8)) < 0.4
        cell = rng.random((8, 8, 8)) < 0.1
        nw[np.kron(at, np.ones((8, 8, 8), bool)) & np.tile(cell, (Z // 8, Y // 8, X // 8))] = 0x0080FF80
    vol = Volume(chunks, min_chunks=chunks[0] * chunks[1] * chunks[2])
    vol.set_material(0)
    vol.set_dense(nw, np.where(nw == 0xFFFFFFFF, 0, 0x80808000).astype(np.uint32))
    vol.request_all()
    vol.sync()
    o = oracle.load("f32")
    for _ in range(split):
        vol.mark_visible(chunks[0] * chunks[1] * chunks[2])
        before, c, _ = vol.export_state()
        vol.sync(split=split)
        req = vol.fetch_requests()
        assert np.array_equal(req, o.visible_requests(before, c, split=split, frame=int(vol.v.frameNum)))
        after, _, _ = vol.export_state()
        assert np.array_equal(after[:, 1], before[:, 1] + 1)
    assert len(req) > 0
    vol.close()
