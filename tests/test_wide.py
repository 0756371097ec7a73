"""The walk over the 4-wide tree (zillumgl_amd/csrc/zgl_wide.h), built for the host, against
the oracle's walk over the reference's rows (src/shader/intersection.glsl:367-427): the
same primitive and the same distance bits for every ray, whether the wide walk vouches for
its hit or hands the ray to the rows; any-hits against the rows."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests import wide_rays
from zillumgl_amd import scene

SCENES = wide_rays.scenes()


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    return wide_rays.Probe(tmp_path_factory.mktemp("wide"))


@pytest.mark.parametrize("name", sorted(SCENES))
def test_wide_walk_equals_the_rows(probe, name):
    ps = scene.pack(SCENES[name])
    assert probe.build(ps) > 0
    r = wide_rays.rays(ps, 20000)
    prim, t, st = probe.trace(r)
    ref_prim, ref_t, _, _ = orc.trace_closest(ps, r)
    np.testing.assert_array_equal(prim, ref_prim)
    np.testing.assert_array_equal(t.view(np.int32), ref_t.view(np.int32))
    assert st[0] > 0.5 * r.shape[1]  # the wide tree was walked
    tm = wide_rays.limits(ps, r.shape[1])
    occ, _, _ = probe.trace(r, tm)
    ref, _, _ = probe.trace(r, tm, rows_only=True)
    np.testing.assert_array_equal(occ >= 0, ref >= 0)


@pytest.mark.parametrize("name", ["cornell", "duplicates", "materials"])
def test_tables_of_different_trees(probe, name):
    ps = wide_rays.loose(scene.pack(SCENES[name]))
    assert probe.build(ps) > 0
    r = wide_rays.rays(ps, 100000)
    prim, t, _ = probe.trace(r)
    ref_prim, ref_t, _ = probe.trace(r, rows_only=True)
    np.testing.assert_array_equal(prim, ref_prim)
    np.testing.assert_array_equal(t.view(np.int32), ref_t.view(np.int32))


def test_ordinary_rays_hardly_ever_need_the_rows(probe):
    ps = scene.pack(SCENES["spheres"])
    probe.build(ps)
    r = wide_rays.rays(ps, 40000)[:, :10000]  # from surfaces, in random directions
    _, _, st = probe.trace(r)
    assert st[1] + st[5] < 0.01 * r.shape[1]
