"""Walk tables with walks of no particles (first, between others, last) give
the other walks' results bit for bit (products: to the order of their atomic
sums), whatever lists the empty walks have."""
import numpy as np
import pytest
import torch

from research_codes_amd import _lib as L
from research_codes_amd.device import FP64, MIXED, Context, Walks

pytestmark = pytest.mark.gpu

SIZES, LENGTHS = [3, 70], [130, 65]
N = sum(SIZES)


def _walks(empties):
    rng = np.random.default_rng(2)
    lists = [rng.integers(0, N, k) for k in LENGTHS]
    sizes = list(SIZES)
    if empties:
        sizes = [0, 3, 0, 0, 70, 0]
        lists = [lists[0][:5], lists[0], lists[1][:0], lists[1], lists[1], lists[0]]
    off = np.concatenate([[0], np.cumsum([len(v) for v in lists])])
    i_off, idx = np.concatenate([[0], np.cumsum(sizes)]), np.concatenate(lists)
    return Walks(i_off, off, idx, off, idx)


def _fields(names, seed):
    rng = np.random.default_rng(seed)
    f = {k: torch.from_numpy(rng.uniform(0.5, 1.5, N)).cuda() for k in names if k != "id"}
    if "id" in names:
        f["id"] = torch.arange(N, dtype=torch.int32, device="cuda")
    return f


def _out(names):
    t = {k: torch.zeros(N, dtype=torch.float64, device="cuda") for k in names}
    if "np" in names:
        t["np"], t["itr"] = t["np"].long(), t["itr"].to(torch.uint8)
    return t


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_functors(precision):
    d = dict(_fields(L.DENS_SRC, 1), ksr=_fields(("k",), 8)["k"] * 0.4, rs=_fields(("k",), 8)["k"] * 0.5)
    h, g = _fields(L.HYDRO_SRC, 2), _fields(L.GRAV_SRC, 4)
    got = []
    with Context(0, eta=0.5, hmax=4.0) as ctx:
        for empties in (False, True):
            w, out = _walks(empties), (_out(L.DENS_OUT), _out(L.HYDRO_OUT), _out(L.GRAV_OUT), _out(L.GRAV_OUT))
            ctx.density(w, d, d, out[0], precision)
            ctx.hydro(w, h, h, out[1], precision)
            for uniform in (False, True):
                ctx.set_params(uniform_softening=uniform)
                ctx.gravity(w, g, g, out[2 + uniform], ps=g, precision=precision)
            got.append(out)
    for a, b in zip(*got):
        for k in a:
            assert torch.equal(a[k], b[k]), k


def test_products():
    d = dict(_fields(L.DENS_SRC, 1), ksr=_fields(("k",), 8)["k"] * 0.4)
    h, g = _fields(L.HYDRO_SRC, 2), _fields(L.GRAV_SRC, 4)
    cot = _fields("01234", 5)
    st = torch.cuda.current_stream().cuda_stream
    got = []
    with Context(0, eta=0.5, hmax=4.0) as ctx:
        for empties in (False, True):
            w, gd, gh = _walks(empties), _out(L.DENS_GRAD), _out(L.HYDRO_GRAD)
            ctx.density_vjp(w, d, _fields(L.DENS_COT, 6), gd)
            ctx.hydro_vjp(w, h, _fields([k for k in L.HYDRO_OUT if k != "vsmx"], 7), gh)
            s = L.GravSrc(**{k: v.data_ptr() for k, v in g.items()})
            g3, n3 = (torch.zeros(N, 3, dtype=torch.float64, device="cuda") for _ in range(2))
            L.check(L.lib().sphk_gravity_vjp_packed_dev(
                ctx.handle, w.n_walk, w.i_off.data_ptr(), w.j_off.data_ptr(), w.j_idx.data_ptr(), s, w.s_off.data_ptr(),
                w.s_idx.data_ptr(), s, s, 0.01, *(c.data_ptr() for c in cot.values()), g3.data_ptr(), n3.data_ptr(), st), "vjp")
            got.append({**{"d" + k: v for k, v in gd.items()}, **{"h" + k: v for k, v in gh.items()}, "g3": g3, "n3": n3})
    for k, a in got[0].items():
        # sums of at most a few hundred terms in another order
        assert float((a - got[1][k]).abs().max()) <= 1e-12 * float(a.abs().max()), k
