"""Lists that end at the last position an offset can name (2^31 - 1): the
tiles after a list's end and the other waves' tiles lie beyond it.  Every
functor and product must give what the same lists give at the start of an
index array."""
import numpy as np
import pytest
import torch

from research_codes_amd import _lib as L
from research_codes_amd.device import FP64, MIXED, Context, Walks

pytestmark = pytest.mark.gpu

SIZES = [3, 40, 70]
LENGTHS = [513, 1, 70]       # several tiles of several waves; one record; a whole tile and a part of one
TOP = 2 ** 31 - 1


@pytest.fixture(scope="module")
def lists():
    rng = np.random.default_rng(3)
    n = sum(SIZES)
    i_off = torch.from_numpy(np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int32)).cuda()
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(LENGTHS)]).astype(np.int32)).cuda()
    idx = torch.from_numpy(rng.integers(0, n, sum(LENGTHS)).astype(np.int32)).cuda()
    far = torch.zeros(TOP, dtype=torch.int32, device="cuda")
    far[TOP - idx.numel():] = idx
    far_off = (off.long() + (TOP - idx.numel())).to(torch.int32)
    yield i_off, (off, idx), (far_off, far)
    del far
    torch.cuda.empty_cache()


def _fields(names, n, seed):
    rng = np.random.default_rng(seed)
    f = {k: torch.from_numpy(rng.uniform(0.5, 1.5, n)).cuda() for k in names if k != "id"}
    if "id" in names:
        f["id"] = torch.arange(n, dtype=torch.int32, device="cuda")
    return f


def _same(run, lists, exact=True):
    """run(walks) -> outputs, for the lists at both places."""
    i_off, near, far = lists
    a, b = run(Walks(i_off, *near)), run(Walks(i_off, *far))
    for k in a:
        if exact:
            assert torch.equal(a[k], b[k]), k
        else:   # sums by atomics: any order of a few hundred terms
            assert float((a[k] - b[k]).abs().max()) <= 1e-12 * float(a[k].abs().max()), k


@pytest.mark.parametrize("known", [True, False])     # the number of i-particles: several waves per walk, or one
@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_functors(lists, precision, known):
    n = sum(SIZES)
    st = torch.cuda.current_stream().cuda_stream

    def zeros(names):
        t = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in names}
        if "np" in names:
            t["np"], t["itr"] = t["np"].long(), t["itr"].to(torch.uint8)
        return t

    def call(name, ctx, w, ins, out_cls, out):
        n_i = (n,) if known else ()
        L.check(getattr(L.lib(), f"sphk_{name}_dev" + ("_n" if known else ""))(
            ctx.handle, w.n_walk, *n_i, w.i_off.data_ptr(), w.j_off.data_ptr(), w.j_idx.data_ptr(), *ins,
            out_cls(**{k: v.data_ptr() for k, v in out.items()}), precision, st), name)
        return out

    def src(cls, f):
        return cls(**{k: v.data_ptr() for k, v in f.items()})

    d = dict(_fields(L.DENS_SRC, n, 1), **{k: torch.full((n,), 0.4, dtype=torch.float64, device="cuda")
                                           for k in ("ksr", "rs")})
    h, g = _fields(L.HYDRO_SRC, n, 2), _fields(L.GRAV_SRC, n, 4)
    with Context(0, eta=0.5, hmax=4.0) as ctx:
        _same(lambda w: call("density", ctx, w, (src(L.DensSrc, d),) * 2, L.DensOut, zeros(L.DENS_OUT)), lists)
        _same(lambda w: call("hydro", ctx, w, (src(L.HydroSrc, h),) * 2, L.HydroOut, zeros(L.HYDRO_OUT)), lists)
        for uniform in (False, True):
            ctx.set_params(uniform_softening=uniform)

            def gravity(w):       # the lists as particles and again as nodes
                s = src(L.GravSrc, g)
                return call("gravity", ctx, w, (s, w.j_off.data_ptr(), w.j_idx.data_ptr(), s, s), L.GravOut,
                            zeros(L.GRAV_OUT))
            _same(gravity, lists)


def test_products(lists):
    n = sum(SIZES)
    st = torch.cuda.current_stream().cuda_stream
    d = dict(_fields(L.DENS_SRC, n, 1), **{k: torch.full((n,), 0.4, dtype=torch.float64, device="cuda")
                                           for k in ("ksr", "rs")})
    h, g = _fields(L.HYDRO_SRC, n, 2), _fields(L.GRAV_SRC, n, 4)
    cot = _fields(("0", "1", "2", "3", "4"), n, 5)
    with Context(0, eta=0.5, hmax=4.0) as ctx:
        def density(w):
            grad = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in L.DENS_GRAD}
            ctx.density_vjp(w, d, _fields(L.DENS_COT, n, 6), grad)
            return grad
        _same(density, lists, exact=False)

        def hydro(w):
            grad = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in L.HYDRO_GRAD}
            ctx.hydro_vjp(w, h, _fields([k for k in L.HYDRO_OUT if k != "vsmx"], n, 7), grad)
            return grad
        _same(hydro, lists)

        def gravity(w):
            s = L.GravSrc(**{k: v.data_ptr() for k, v in g.items()})
            g3, n3 = torch.zeros(n, 3, dtype=torch.float64, device="cuda"), torch.zeros(n, 3, dtype=torch.float64, device="cuda")
            L.check(L.lib().sphk_gravity_vjp_packed_dev(
                ctx.handle, w.n_walk, w.i_off.data_ptr(), w.j_off.data_ptr(), w.j_idx.data_ptr(), s, w.j_off.data_ptr(),
                w.j_idx.data_ptr(), s, s, 0.01, *(c.data_ptr() for c in cot.values()), g3.data_ptr(), n3.data_ptr(), st), "vjp")
            return dict(g=g3, n=n3)
        _same(gravity, lists, exact=False)
