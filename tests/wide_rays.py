"""Scenes and rays for the tests of the walk over the 4-wide tree, and the host build of
that walk (tests/native/wide_probe.cpp)."""
import copy
import ctypes as C
import os
import subprocess

import numpy as np

from zillumgl_amd import scene

HERE = os.path.dirname(os.path.abspath(__file__))


class Probe:
    def __init__(self, folder):
        out = os.path.join(str(folder), "wide_probe.so")
        subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-Wno-unknown-pragmas",
                        "-shared", "-fPIC", os.path.join(HERE, "native", "wide_probe.cpp"), "-o", out], check=True)
        self.lib = C.CDLL(out)
        self.lib.probe_wide_build.restype = C.c_int64

    def build(self, ps):
        """Slots of the packed scene's wide tree (0: none)."""
        p = lambda a, t: a.ctypes.data_as(C.POINTER(t))
        return self.lib.probe_wide_build(p(ps.vertices, C.c_float), p(ps.indices, C.c_int32),
                                         C.c_int64(ps.indices.shape[0]), p(ps.bounds, C.c_float),
                                         p(ps.hit_table, C.c_int32))

    def margins(self):
        """rel, slack, grow, growRel, reach and the number of planes of the built tree."""
        out = (C.c_float * 6)()
        self.lib.probe_wide_margins(out)
        return list(out)

    def trace(self, rays, tmax=None, rows_only=False):
        """Closest hits (prim, t), or any-hits with tmax: prim >= 0 where occluded; and the
        walk's statistics (see the source)."""
        p = lambda a, t: a.ctypes.data_as(C.POINTER(t))
        r = np.ascontiguousarray(rays, np.float32)
        n = r.shape[1]
        tm = np.zeros(n, np.float32) if tmax is None else np.ascontiguousarray(tmax, np.float32)
        prim, t, st = np.empty(n, np.int32), np.empty(n, np.float32), np.zeros(9, np.int64)
        self.lib.probe_wide_trace(p(r, C.c_float), C.c_int64(n), p(tm, C.c_float), int(tmax is not None),
                                  int(rows_only), p(prim, C.c_int32), p(t, C.c_float), p(st, C.c_int64))
        return prim, t, st


def _mesh(v, f):
    n = np.tile(np.array([0, 0, 1], np.float32), (len(v), 1))
    return scene.Mesh(np.asarray(v, np.float32), n, np.asarray(f, np.uint32), None)


def scenes():
    """name -> SceneDesc: the workloads' geometry at small sizes, and trees at the edges of
    what the wide tree takes (one to five triangles, coplanar duplicates, identical
    centroids deeper than its builder goes, coordinates far from the origin, tiny and
    large ones, slivers)."""
    rng = np.random.default_rng(3)
    out = {"cornell": scene.config1(32, 32), "materials": scene.config_materials(32, 32),
           "caustics": scene.config3(32, 32), "tessellated": scene.config5(32, 32, n=9, env_size=(8, 4)),
           "spheres": scene.config2(32, 32, n_spheres=6, subdiv=3, env_size=(16, 8))}

    def soup(v, name):
        d = scene.config1(32, 32)
        m = len(v) // 3
        d.objects = [(_mesh(v, np.arange(3 * m).reshape(-1, 3)), scene.Material())]
        d.lights = []
        out[name] = d
    for n in (1, 2, 3, 4, 5):
        soup(rng.uniform(0, 1, (3 * n, 3)), f"soup{n}")
    soup(rng.uniform(0, 1, (900, 3)) * 0.2 + np.repeat(rng.uniform(0, 1, (300, 3)), 3, 0), "soup300")
    flat = np.concatenate([np.array([[x, y, 0], [x + 1, y, 0], [x, y + 1, 0]], np.float64)
                           for x in range(6) for y in range(6)])
    soup(np.concatenate([flat, flat, flat + [0, 0, 2]]), "duplicates")
    soup(np.tile(rng.uniform(0, 1, (3, 3)), (400, 1)), "identical")
    base = rng.uniform(0, 1, (600, 3)) * 0.3 + np.repeat(rng.uniform(0, 1, (200, 3)), 3, 0)
    soup(base + [1000, -500, 200], "far")
    soup(base * 1e-4, "tiny")
    soup(base * 3e5, "large")
    thin = base.copy()
    thin[2::3] = thin[0::3] * 0.5 + thin[1::3] * 0.5 + rng.normal(size=(200, 3)) * 1e-5
    soup(thin, "slivers")
    return out


def padded(d, n=33):
    """The scene with a patch of 2 n^2 small triangles in its middle: more triangles than the
    batch kernels' rule for walking the rows."""
    out = copy.copy(d)
    p = np.concatenate([np.asarray(m.positions, np.float64) for m, _ in d.objects])
    lo, hi = p.min(0), p.max(0)
    at = lambda x, y, z: tuple(lo + (hi - lo) * np.array([x, y, z]))
    patch = scene.grid_patch(at(0.4, 0.45, 0.5), at(0.5, 0.45, 0.52), at(0.5, 0.55, 0.54), at(0.4, 0.55, 0.52),
                             (0, 0, 1), n, 0, n, 0, n)
    out.objects = list(d.objects) + [(patch, scene.Material())]
    return out


def loose(ps):
    """The packed scene with tables of different trees: the inner rows of table 0 all get the
    root's box, the other tables keep theirs."""
    ps = copy.copy(ps)
    table = ps.hit_table.copy()
    first = table.reshape(6, -1, 3)[0]
    first[first[:, 1] < 0, 0] = first[0, 0]
    ps.hit_table = table
    return ps


def scaled(d, k, turned=False):
    """The scene k times as large, turned about two axes if asked (no face stays in a plane of
    constant x, y or z)."""
    c, s, e, f = np.cos(0.6), np.sin(0.6), np.cos(0.9), np.sin(0.9)
    turn = np.array([[c, -s, 0], [s, c, 0], [0, 0, 1]]) @ np.array([[1, 0, 0], [0, e, -f], [0, f, e]]) if turned else np.eye(3)

    def moved(mesh):
        m = copy.copy(mesh)
        m.positions = np.ascontiguousarray(((np.asarray(mesh.positions, np.float64) @ turn.T) * k).astype(np.float32))
        return m
    out = copy.copy(d)
    out.objects = [(moved(m), x) for m, x in d.objects]
    out.lights = [(moved(m), x) for m, x in d.lights]
    return out


def grazing(ps, n, seed=7):
    """Rays nearly in the plane of a triangle, 1e-7 to 0.1 off it, from on it, in front of it
    or behind: the FP32 distance of such a hit is far off, and can lie in front of the
    triangle's own box."""
    g = np.random.default_rng(seed)
    t = ps.vertices[ps.indices[g.integers(0, len(ps.indices), n)]].astype(np.float64)
    o = (t * g.dirichlet([1, 1, 1], n)[..., None]).sum(1)
    ab, ac = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    unit = lambda v: v / np.maximum(np.linalg.norm(v, axis=1), 1e-30)[:, None]
    normal, along = unit(np.cross(ab, ac)), unit(ab)
    a = g.uniform(0, 2 * np.pi, n)[:, None]
    d = along * np.cos(a) + np.cross(normal, along) * np.sin(a)
    d = unit(d + normal * (10 ** g.uniform(-7, -1, n) * g.choice([-1, 1], n))[:, None])
    size = np.linalg.norm(ps.vertices.max(0).astype(np.float64) - ps.vertices.min(0))
    o += d * (g.choice([0, 1e-4], n) - g.choice([0, 0, 0.1, 0.3], n) * size)[:, None]
    return np.ascontiguousarray(np.concatenate([o.T, d.T]).astype(np.float32))


def flattened(r, seed=3):
    """The rays with one component of their directions below 1e-6."""
    g = np.random.default_rng(seed)
    r, n = r.copy(), r.shape[1]
    r[3 + g.integers(0, 3, n), np.arange(n)] = g.choice([0, 1e-7, -9e-7, 1e-20], n)
    r[3:] /= np.maximum(np.linalg.norm(r[3:].astype(np.float64), axis=0), 1e-9).astype(np.float32)
    return r


# scene, scale, turned: sizes at which walks that drop subtrees at a fixed distance beyond
# the hit, or test a flattened ray's box on all three axes, return other hits than the rows
LARGE = [("cornell", 10, False), ("cornell", 100, True), ("materials", 555, True), ("caustics", 1000, True),
         ("tessellated", 100, False), ("tessellated", 555, True), ("spheres", 100, False), ("duplicates", 10, True)]


def rays(ps, n, seed=1):
    """Rays the walks meet and rays made to be awkward: from surfaces, at vertices and along
    edges, with components that vanish or nearly do, nearly axis-parallel, unnormalised,
    from far away, not finite."""
    g = np.random.default_rng(seed)
    lo, hi = ps.vertices.min(0).astype(np.float64), ps.vertices.max(0).astype(np.float64)
    o = g.uniform(lo, hi, (n, 3))
    d = g.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    k, m = n // 4, n // 40
    pick = lambda c: ps.vertices[ps.indices[g.integers(0, len(ps.indices), c)]].astype(np.float64)
    on = (pick(k) * g.dirichlet([1, 1, 1], k)[..., None]).sum(1)
    o[:k] = on + d[:k] * 1e-4
    w = g.dirichlet([1, 1, 1], k)
    w[:, 0] = 0
    w[:k // 3] = [0, 0, 1]
    w /= w.sum(1)[:, None]
    to = (pick(k) * w[..., None]).sum(1) - o[k:2 * k]
    d[k:2 * k] = to / np.maximum(np.linalg.norm(to, axis=1), 1e-30)[:, None]
    s = 2 * k
    for a in range(3):
        d[s:s + m, a] = g.choice([0.0, -0.0, 1e-7, -9e-7, 1.1e-6, 1e-20], m)
        s += m
    e = np.zeros((3 * m, 3))
    e[np.arange(3 * m), g.integers(0, 3, 3 * m)] = g.choice([-1.0, 1.0], 3 * m)
    d[s:s + 3 * m] = e + g.choice([0, 1e-7, 1e-4, 1e-3, 2e-3], (3 * m, 3)) * g.normal(size=(3 * m, 3))
    s += 3 * m
    d[2 * k:s] /= np.linalg.norm(d[2 * k:s], axis=1)[:, None]
    d[s:s + m] *= g.choice([1e-3, 0.4, 0.6, 1.5, 40.0], (m, 1))
    s += m
    o[s:s + m] *= g.choice([3.0, 30.0, 1e6], (m, 1))
    s += m
    d[s] = 0
    d[s + 1] = np.nan
    o[s + 2] = np.inf
    d[s + 3] = [0.5, 0, 0]
    return np.ascontiguousarray(np.concatenate([o.T, d.T]).astype(np.float32))


def limits(ps, n, seed=2):
    """Any-hit limits: spread over the scene, none, negative, zero, infinite, NaN."""
    g = np.random.default_rng(seed)
    size = float(np.linalg.norm(ps.vertices.max(0).astype(np.float64) - ps.vertices.min(0)))
    t = g.uniform(0, 0.7 * size, n).astype(np.float32)
    t[::5] = 1e8
    t[:4] = [-1.0, 0.0, np.inf, np.nan]
    return t
