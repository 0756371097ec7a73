"""Walks over the device-built 4-wide tree against the counting kernels, which walk the
reference's rows: ray batches with the same primitives and distance bits, any-hits against
the host build of the rows' walk, frames bit for bit.  Batches on scenes of fewer than 1,024
triangles walk the rows whatever the tree, so the batch tests' scenes are padded past that;
the frames are of the small scenes themselves, whose trees one workgroup or a few levels
build.  Scenes that the builder refuses (a caller's boxes that are not the triangles' own,
"identical", whose tree is deeper than it goes) give the rows' results too."""
import numpy as np
import pytest

from tests import wide_rays
from zillumgl_amd import render, scene

pytestmark = pytest.mark.gpu
SCENES = wide_rays.scenes()


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    return wide_rays.Probe(tmp_path_factory.mktemp("wide"))


def _compare(probe, ps, n, r=None):
    r = wide_rays.rays(ps, n) if r is None else r
    ctx = render.Context(0)
    try:
        ctx.upload(ps)
        prim, t, b = ctx.trace_closest(r)
        ref = ctx.trace_closest(r, counted=True)
        np.testing.assert_array_equal(prim, ref[0])
        np.testing.assert_array_equal(t.view(np.int32), ref[1].view(np.int32))
        np.testing.assert_array_equal(b, ref[2])
        tm = wide_rays.limits(ps, r.shape[1])
        probe.build(ps)
        want, _, _ = probe.trace(r, tm, rows_only=True)
        np.testing.assert_array_equal(ctx.trace_any(r, tm), want >= 0)
    finally:
        ctx.close()


@pytest.mark.parametrize("name", sorted(SCENES))
def test_batches_equal_the_rows(probe, name):
    ps = scene.pack(wide_rays.padded(SCENES[name]))
    assert ps.indices.shape[0] >= 2048
    _compare(probe, ps, 20000)


@pytest.mark.parametrize("name", ["cornell", "materials", "caustics", "tessellated", "soup1", "soup2", "soup3", "soup4",
                                  "soup5", "soup300", "duplicates", "identical", "slivers"])
def test_frames_equal_the_rows(name):
    ps = scene.pack(SCENES[name], bvh="device")
    ctx = render.Context(0)
    try:
        frames = []
        for count in (False, True):
            ctx.upload(ps)
            ctx.clear()
            ctx.render(0, 0, 16, 1, 5, count_bytes=count)
            frames.append(ctx.read_frame())
        assert np.isfinite(frames[1]).all()
        np.testing.assert_array_equal(frames[0].view(np.int32), frames[1].view(np.int32))
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [1000, 100003])
def test_batch_sizes(probe, n):
    ps = scene.pack(scene.config5(32, 32, n=20, env_size=(8, 4)))  # above the rule's 1,024 triangles
    _compare(probe, ps, n)


@pytest.mark.parametrize("name,scale,turned", wide_rays.LARGE)
def test_rays_nearly_in_a_triangles_plane(probe, name, scale, turned):
    ps = scene.pack(wide_rays.scaled(wide_rays.padded(SCENES[name]), scale, turned))
    r = wide_rays.grazing(ps, 100000)
    _compare(probe, ps, 0, np.concatenate([r, wide_rays.flattened(r)], 1))


@pytest.mark.parametrize("name", ["cornell", "duplicates"])
def test_tables_of_different_trees(probe, name):
    _compare(probe, wide_rays.loose(scene.pack(wide_rays.padded(SCENES[name]))), 100000)


def test_boxes_larger_than_their_triangles(probe):
    ps = scene.pack(scene.config5(32, 32, n=20, env_size=(8, 4)))
    ps.bounds = (ps.bounds + np.array([-1, -1, -1, 1, 1, 1], np.float32) * np.float32(0.05)).astype(np.float32)
    _compare(probe, ps, 5000)
