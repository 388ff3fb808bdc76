"""Host geometry of the element products (pm_patches.cpp), compiled alone for
the CPU."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import oracle as O
from poromec_amd import problem as P

CSRC = Path(__file__).resolve().parents[1] / "poromec_amd" / "csrc"
WRAP = r"""
#include "pm_patches.h"
#include <cstring>
extern "C" int element_patches(int numel, int nen, int nnodev, const int *ix, const int *id,
                               const double *x, int L, int *ord, int *ps) {
  std::vector<int> o, p;
  pm_element_patches(numel, nen, nnodev, ix, id, x, L, o, p);
  std::memcpy(ord, o.data(), o.size() * sizeof(int));
  std::memcpy(ps, p.data(), p.size() * sizeof(int));
  return (int)p.size() - 1;
}
extern "C" int parallelepiped(const int *v, const double *x) { return pm_is_parallelepiped(v, x); }
"""


@pytest.fixture(scope="module")
def patches(tmp_path_factory):
    d = tmp_path_factory.mktemp("patches")
    (d / "wrap.cpp").write_text(WRAP)
    so = d / "patches.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-pthread", f"-I{CSRC}",
                    str(d / "wrap.cpp"), str(CSRC / "pm_patches.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


def _parallelepiped(lib, ix, x):
    v = np.ascontiguousarray(ix[:8], np.int32)
    x = np.ascontiguousarray(x, np.float64)
    return bool(lib.parallelepiped(v.ctypes.data_as(C.c_void_p), x.ctypes.data_as(C.c_void_p)))


def _patches(lib, nx, ny, nz, x, lanes):
    """(ord, ps) of a box of vertex-numbered Q1/Q1 elements at coordinates x."""
    ix = np.ascontiguousarray(P.box_mesh(nx, ny, nz)[0])
    idm = np.arange(1, 4 * len(x) + 1, dtype=np.int32)
    x = np.ascontiguousarray(x, np.float64)
    ord_, ps = np.zeros(len(ix), np.int32), np.zeros(len(ix) + 1, np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    n = lib.element_patches(len(ix), 8, len(x), p(ix), p(idm), p(x), lanes, p(ord_), p(ps))
    return ord_, ps[: n + 1]


SHEAR = np.array([[1.0, 0.2, -0.1], [0.15, 0.8, 0.25], [-0.2, 0.1, 1.2]])


@pytest.mark.parametrize("aspect", [1.0, 100.0, 1e4])
def test_parallelepipeds_of_any_aspect(patches, aspect):
    """A vertex moved by d along an edge h changes each of the four bilinear
    and trilinear parts by d / 4h of the edge's own linear part (4 h)."""
    ix, x = P.box_mesh(1, 1, 1, h=(1.0, 1.0, 1.0 / aspect))
    assert _parallelepiped(patches, ix[0], x)
    assert _parallelepiped(patches, ix[0], x[:, [2, 0, 1]])
    assert _parallelepiped(patches, ix[0], x @ SHEAR.T)
    for axis, h in ((0, 1.0), (1, 1.0), (2, 1.0 / aspect)):
        for k in (0, 7):  # a vertex at the origin and one that is not
            for f, ok in ((0.5, True), (2.0, False)):
                y = x.copy()
                y[ix[0, 6] - 1 if k == 0 else ix[0, 0] - 1, axis] += f * 4e-12 * h
                assert _parallelepiped(patches, ix[0], y) == ok, (axis, k, f)
    flat = x.copy()
    flat[:, 2] = 0.0
    assert not _parallelepiped(patches, ix[0], flat)
    flat[0, 0] = np.nan
    assert not _parallelepiped(patches, ix[0], flat)


@pytest.mark.parametrize("nen", [20, 8])
@pytest.mark.parametrize("aspect", [1.0, 100.0, 1e4])
def test_accepted_elements_have_the_parallelepipeds_matrix(patches, aspect, nen):
    """What is accepted has the matrix of its parallelepiped: with J (I + E),
    E one row of at most three parts of 1e-12, ||E|| < 6e-12, and K moves by
    at most (2 + sqrt 3) ||E|| of its norm: 2e-11."""
    def matrix(x):
        d = P.column_deck(1, 1, 1, nen=nen)
        d.x[:] = x
        d.idv[:] = 0
        st = O.build_structure(d)
        m = O.OracleModel(d, st)
        m.assemble(isw=2, lhs=True, rhs=False)
        return np.concatenate([m.ad, np.sqrt(2.0) * m.al[: st["nad"]]])

    ix, x = P.box_mesh(1, 1, 1, h=(1.0, 1.0, 1.0 / aspect))
    k0 = matrix(x)
    accepted = 0
    for axis in range(3):
        for e in np.arange(-18.0, -5.0, 0.5):
            y = x.copy()
            y[ix[0, 6] - 1, axis] = 10.0 ** e  # the vertex at the origin
            if _parallelepiped(patches, ix[0], y):
                accepted += 1
                assert np.linalg.norm(matrix(y) - k0) <= 2e-11 * np.linalg.norm(k0), (axis, e)
    assert accepted >= 3


@pytest.mark.parametrize("lanes", [16, 64])
def test_patches_are_bricks_at_any_offset(patches, lanes):
    """The patches of a mesh at map coordinates are those of the same mesh at
    the origin: full, and bricks of 4 x 4 x 4 (4 x 2 x 2) cells."""
    n, h = 16, 0.25
    _, x = P.box_mesh(n, n, n, h=(h, h, h))
    ord0, ps0 = _patches(patches, n, n, n, x, lanes)
    assert np.array_equal(np.sort(ord0), np.arange(n ** 3))
    assert np.array_equal(ps0, np.arange(0, n ** 3 + 1, lanes))
    for a, b in zip(ps0[:-1], ps0[1:]):
        cell = ord0[a:b, None] // np.array([1, n, n * n]) % n
        assert np.prod(cell.max(0) - cell.min(0) + 1) == lanes
    ord1, ps1 = _patches(patches, n, n, n, x + np.array([7.0e6, -7.0e6, 2.0e3]), lanes)
    assert np.array_equal(ord0, ord1) and np.array_equal(ps0, ps1)


# operator new fails in one call: the `at`-th that is made while `patches` runs
# on the calling thread (at < 0: on any other thread)
ALLOC = r"""
#include <atomic>
#include <cstdlib>
#include <new>
#include <thread>
static std::atomic<int> g_at{0};
static std::atomic<bool> g_on{false};
static std::thread::id g_caller;
void *operator new(std::size_t n) {
  if (g_on.load()) {
    const bool caller = std::this_thread::get_id() == g_caller;
    if (g_at.load() < 0 ? !caller : caller && g_at.fetch_sub(1) == 1) throw std::bad_alloc();
  }
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

#include "pm_patches.h"
#include <cstdio>
int main(int argc, char **argv) {
  const int n = 60, nv = n + 1, numel = n * n * n;
  std::vector<int> ix((size_t)numel * 21, 0), id((size_t)nv * nv * nv * 4), ord, ps, ref, rps;
  std::vector<double> x((size_t)nv * nv * nv * 3);
  for (size_t i = 0; i < id.size(); i++) id[i] = (int)i + 1;
  for (int i = 0; i < nv * nv * nv; i++) {
    x[3 * (size_t)i] = i % nv;
    x[3 * (size_t)i + 1] = i / nv % nv;
    x[3 * (size_t)i + 2] = i / nv / nv;
  }
  for (int e = 0; e < numel; e++)
    for (int k = 0; k < 8; k++)
      ix[(size_t)e * 21 + k] = 1 + (e % n + (k & 1)) + nv * ((e / n % n + (k >> 1 & 1)) +
                                                             nv * (e / n / n + (k >> 2)));
  auto run = [&](std::vector<int> &o, std::vector<int> &p) {
    pm_element_patches(numel, 8, nv * nv * nv, ix.data(), id.data(), x.data(), 64, o, p);
  };
  run(ref, rps);
  g_caller = std::this_thread::get_id();
  int refused = 0;
  for (int at = -1; at < 64; at++) {
    if (at == 0) continue;
    g_at = at;
    g_on = true;
    try {
      run(ord, ps);
      g_on = false;
      if (ord != ref || ps != rps) return 1;
    } catch (const std::bad_alloc &) {  // pm_affine_setup keeps the stored matrix
      g_on = false;
      refused++;
    }
  }
  std::printf("%d refused\n", refused);
  return 0;
}
"""


def test_patches_without_memory(tmp_path):
    """Memory may end anywhere while patches are made: the call comes back, with
    the patches or std::bad_alloc, and the process stays."""
    (tmp_path / "alloc.cpp").write_text(ALLOC)
    exe = tmp_path / "alloc"
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", f"-I{CSRC}",
                    str(tmp_path / "alloc.cpp"), str(CSRC / "pm_patches.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr)
