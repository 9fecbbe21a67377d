"""The device tree at the edges of its construction: trees of one node, sizes
around the blocks of 1024 particles that nodes are counted in, leaves larger
than the window compared in LDS, and coincident particles (cells that cannot
be split at the deepest level).  Everything must equal the host tree's."""
import numpy as np
import pytest
import torch

from research_codes_amd.tree import DeviceTree, HostTree, morton_order

pytestmark = pytest.mark.gpu


def _points(kind, n, rng):
    x = rng.random((3, n))
    if kind == "clumped":                  # a quarter of them at three places
        for k in range(3):
            x[:, k * n // 12:(k + 1) * n // 12] = rng.random((3, 1))
    if kind == "line":                     # one octant pair per level: long chains of single children
        x = np.stack([0.5 ** (1.0 + 18.0 * rng.random(n))] * 3)
    return x


@pytest.mark.parametrize("kind", ["uniform", "clumped", "line"])
@pytest.mark.parametrize("n,n_leaf,n_group", [(1, 8, 16), (2, 1, 1), (8, 8, 16), (9, 8, 8), (1023, 8, 16), (1024, 8, 32),
                                              (1025, 8, 64), (2049, 1, 8), (3000, 512, 600), (3000, 513, 16),
                                              (5000, 8, 7)])
def test_tree_equals_host(kind, n, n_leaf, n_group):
    rng = np.random.default_rng(n + n_leaf)
    x, y, z = _points(kind, n, rng)
    perm = morton_order(x, y, z)
    x, y, z = (np.ascontiguousarray(a[perm]) for a in (x, y, z))
    m, eps2, h = rng.uniform(0.5, 1.5, n), rng.uniform(1e-5, 1e-3, n), rng.uniform(0.02, 0.3, n)
    d = lambda a: torch.from_numpy(a).cuda()   # noqa: E731
    ht = HostTree(x, y, z, m, eps2, n_leaf, n_group)
    dt = DeviceTree(*map(d, (x, y, z, m, eps2)), n_leaf, n_group)
    try:
        for again in range(2):             # built, and built again into the same buffers
            assert dt.n_node == ht.n_node and dt.n_walk == ht.n_walk
            assert np.array_equal(dt.i_off.cpu().numpy(), ht.i_off)
            for k, v in ht.moments().items():
                assert np.array_equal(dt.moments()[k].cpu().numpy(), v), k
            for name, hl, dl in (("gather", ht.gather(h), dt.gather(d(h))), ("symmetry", ht.symmetry(h), dt.symmetry(d(h))),
                                 ("long", ht.long(0.5), dt.long(0.5))):
                for a, b in zip(hl, dl):
                    assert np.array_equal(a, b.cpu().numpy()), (name, again)
            dt._src = None
            dt.rebuild(*map(d, (x, y, z, m, eps2)), n_leaf, n_group)
    finally:
        ht.close()
        dt.close()


@pytest.mark.parametrize("n", [1024, 1025, 8192, 8193])
def test_offsets_of_one_particle_walks(n):
    """As many walks as particles, around the sizes where the scan of their
    counts gives a thread another walk and where it changes its kernel."""
    rng = np.random.default_rng(n)
    x, y, z = rng.random((3, n))
    perm = morton_order(x, y, z)
    x, y, z = (np.ascontiguousarray(a[perm]) for a in (x, y, z))
    m, eps2, h = np.full(n, 1.0 / n), np.full(n, 1e-4), rng.uniform(0.01, 0.05, n)
    d = lambda a: torch.from_numpy(a).cuda()   # noqa: E731
    ht = HostTree(x, y, z, m, eps2, 1, 1)
    dt = DeviceTree(*map(d, (x, y, z, m, eps2)), 1, 1)
    try:
        assert dt.n_walk == ht.n_walk == n
        for name, hl, dl in (("gather", ht.gather(h), dt.gather(d(h))), ("symmetry", ht.symmetry(h), dt.symmetry(d(h))),
                             ("long", ht.long(0.7), dt.long(0.7))):
            for a, b in zip(hl, dl):
                assert np.array_equal(a, b.cpu().numpy()), name
    finally:
        ht.close()
        dt.close()


@pytest.mark.parametrize("kind", ["uniform", "clumped", "line"])
@pytest.mark.parametrize("n,n_leaf,n_group", [(5000, 513, 64), (5000, 2500, 16), (5000, 4999, 5000), (5000, 5000, 64),
                                              (5000, 9000, 1)])
def test_large_leaves_equal_host(kind, n, n_leaf, n_group):
    """Leaves beyond the windows held in LDS, up to more than there are particles."""
    test_tree_equals_host(kind, n, n_leaf, n_group)


@pytest.mark.parametrize("n,n_leaf,n_group,theta", [(30000, 8, 16, 0.5), (30000, 8, 64, 1.0), (6000, 1, 8, 0.3)])
def test_steep_profile_equals_host(n, n_leaf, n_group, theta):
    """Particles spread evenly over four decades of radius: walks at the edge
    hold the whole centre in their search boxes and keep more entries pending
    than the first stack holds.  Built three times: such walks are met, known
    and (with a list that has none between) forgotten again."""
    rng = np.random.default_rng(n + n_group)
    x, y, z = rng.standard_normal((3, n)) * 10.0 ** rng.uniform(-4.0, 0.0, n)
    perm = morton_order(x, y, z)
    x, y, z = (np.ascontiguousarray(a[perm]) for a in (x, y, z))
    m, eps2 = rng.uniform(0.5, 1.5, n), np.full(n, 1e-8)
    h = 0.2 * np.sqrt(x * x + y * y + z * z)
    d = lambda a: torch.from_numpy(a).cuda()   # noqa: E731
    ht = HostTree(x, y, z, m, eps2, n_leaf, n_group)
    dt = DeviceTree(*map(d, (x, y, z, m, eps2)), n_leaf, n_group)
    try:
        want = (ht.gather(h), ht.symmetry(h), ht.long(theta))
        for again in range(3):
            for name, hl, dl in zip(("gather", "symmetry", "long"), want,
                                    (dt.gather(d(h)), dt.symmetry(d(h)), dt.long(theta))):
                for a, b in zip(hl, dl):
                    assert np.array_equal(a, b.cpu().numpy()), (name, again)
            for a, b in zip(ht.long(3.0), dt.long(3.0)):
                assert np.array_equal(a, b.cpu().numpy()), again
    finally:
        ht.close()
        dt.close()
