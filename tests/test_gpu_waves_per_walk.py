"""The functors with several waves per walk (few or long walks): the sums do
not depend on the number of waves, so the first walks of a table launched
alone must equal, bit for bit, the same walks within a table padded with
empty-list walks to a number and mean length that take fewer waves."""
import numpy as np
import pytest
import torch

from research_codes_amd import _lib as L
from research_codes_amd.device import FP64, MIXED, Context, Walks

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 9, 32, 33, 64, 70]                    # i-particles, more than a wave among them
LENGTHS = [0, 1, 63, 64, 65, 255, 256, 257, 513, 2050]  # records: no tile, its edges, more rounds than waves


def _table(rng, n_rec, lengths):
    i_off = np.concatenate([[0], np.cumsum(SIZES)])
    off = np.concatenate([[0], np.cumsum(lengths)])
    idx = np.concatenate([rng.integers(0, n_rec, k) for k in lengths])
    return i_off, off, idx


def _padded(i_off, off, n_walk, per):
    """The same walks, then walks of `per` particles with an empty list each."""
    more = n_walk - (len(i_off) - 1)
    last = int(i_off[-1])
    return (np.concatenate([i_off, last + per * (1 + np.arange(more))]), np.concatenate([off, np.full(more, off[-1])]))


# (walks, particles of a padding walk): 8, 4 or 2 waves; 4 or 2; 2; 1
TABLES = [(len(SIZES), 0), (5500, 20), (5500, 10), (5500, 1)]


@pytest.mark.parametrize("list_cap", [192, 256])
@pytest.mark.parametrize("precision", [MIXED, FP64])
@pytest.mark.parametrize("radius", [0.25, 0.45, 0.9])    # few, more than 12 steps a lane, nearly all records members
@pytest.mark.parametrize("grown", [False, True])         # H beyond the search radius: full sweeps take over
def test_density_does_not_depend_on_waves(precision, list_cap, radius, grown):
    rng = np.random.default_rng(int(100 * radius))
    lengths = [1, 64, 65, 130, 192, 193, 256, 257][:len(SIZES)]
    n = sum(SIZES)
    n_all = n + 20 * 5500
    f = {k: torch.from_numpy(rng.uniform(0.0, 1.0, n_all)).cuda() for k in L.DENS_SRC}
    f["id"] = torch.arange(n_all, dtype=torch.int32, device="cuda")
    f["ksr"] = f["ksr"] * 0.0 + radius
    f["rs"] = 1.1 * f["ksr"]
    i_off, j_off, j_idx = _table(rng, n, lengths)
    out = []
    with Context(0, eta=3.0 if grown else 0.3, hmax=10.0) as ctx:
        ctx.set_params(list_cap=list_cap)
        for n_walk, per in TABLES:
            io, jo = _padded(i_off, j_off, n_walk, per)
            o = {k: torch.zeros(n_all, dtype=torch.float64, device="cuda") for k in ("dens", "divv", "rotv", "grdh", "ksr")}
            o["np"] = torch.zeros(n_all, dtype=torch.int64, device="cuda")
            o["itr"] = torch.zeros(n_all, dtype=torch.uint8, device="cuda")
            ctx.density(Walks(io, jo, j_idx), f, f, o, precision)
            out.append({k: v[:n].cpu() for k, v in o.items()})
    for o in out[1:]:
        for k, v in o.items():
            assert torch.equal(v.view(torch.int64) if v.dtype == torch.float64 else v,
                               out[0][k].view(torch.int64) if v.dtype == torch.float64 else out[0][k]), k
    if not grown:
        return
    assert int(out[0]["itr"].sum()) > 0


@pytest.mark.parametrize("precision", [MIXED, FP64])
@pytest.mark.parametrize("shift", range(len(LENGTHS)))
@pytest.mark.parametrize("functor", ["hydro", "uniform", "general"])
def test_results_do_not_depend_on_waves(precision, shift, functor):
    rng = np.random.default_rng(shift)
    lengths = [LENGTHS[(k + shift) % len(LENGTHS)] for k in range(len(SIZES))]
    spj = [LENGTHS[(k + 3 * shift + 1) % len(LENGTHS)] for k in range(len(SIZES))]
    n = sum(SIZES)
    n_all = n + 20 * 5500
    f = {k: torch.from_numpy(rng.uniform(0.1, 1.0, n_all)).cuda() for k in L.HYDRO_SRC}
    f["id"] = torch.arange(n_all, dtype=torch.int32, device="cuda")
    f["eps2"] = torch.from_numpy(np.full(n_all, 0.01) if functor == "uniform" else rng.uniform(0.01, 0.1, n_all)).cuda()
    i_off, j_off, j_idx = _table(rng, n, lengths)
    _, s_off, s_idx = _table(rng, n, spj)
    out = []
    with Context(0) as ctx:
        ctx.set_params(uniform_softening=functor == "uniform")
        for n_walk, per in TABLES:
            io, jo = _padded(i_off, j_off, n_walk, per)
            _, so = _padded(i_off, s_off, n_walk, per)
            if functor == "hydro":
                o = {k: torch.zeros(n_all, dtype=torch.float64, device="cuda") for k in L.HYDRO_OUT}
                ctx.hydro(Walks(io, jo, j_idx), f, f, o, precision)
            else:
                o = {k: torch.zeros(n_all, dtype=torch.float64, device="cuda") for k in L.GRAV_OUT}
                src = {k: f[k] for k in L.GRAV_SRC}
                ctx.gravity(Walks(io, jo, j_idx, so, s_idx), src, src, o, ps=src, precision=precision)
            out.append({k: v[:n].cpu() for k, v in o.items()})
    for o in out[1:]:
        for k, v in o.items():
            assert torch.equal(v, out[0][k]), k
    assert float(sum(v.abs().sum() for v in out[0].values())) > 0.0


@pytest.mark.parametrize("list_cap", [192, 256])
@pytest.mark.parametrize("known,n_walk", [(True, 8192), (True, 8193), (False, 12288), (False, 12289)])
def test_density_does_not_depend_on_occupancy(list_cap, known, n_walk):
    """Around the numbers of walks up to which a mixed launch of one wave per
    walk takes more registers (the mean number of particles known, or not)."""
    rng = np.random.default_rng(31)
    lengths = [1, 64, 65, 130, 192, 193, 256, 257]
    n, n_all = sum(SIZES), sum(SIZES) + n_walk
    f = {k: torch.from_numpy(rng.uniform(0.0, 1.0, n_all)).cuda() for k in L.DENS_SRC}
    f["id"] = torch.arange(n_all, dtype=torch.int32, device="cuda")
    f["ksr"] = f["ksr"] * 0.0 + 0.45
    f["rs"] = 1.1 * f["ksr"]
    i_off, j_off, j_idx = _table(rng, n, lengths)
    out = []
    with Context(0, eta=0.3, hmax=10.0) as ctx:
        ctx.set_params(list_cap=list_cap)
        for tables in ((i_off, j_off), _padded(i_off, j_off, n_walk, 1)):
            w = Walks(*tables, j_idx)
            o = {k: torch.zeros(n_all, dtype=torch.float64, device="cuda") for k in ("dens", "divv", "rotv", "grdh", "ksr")}
            o["np"] = torch.zeros(n_all, dtype=torch.int64, device="cuda")
            o["itr"] = torch.zeros(n_all, dtype=torch.uint8, device="cuda")
            if known:
                ctx.density(w, f, f, o, MIXED)
            else:
                s, d = (c(**{k: v.data_ptr() for k, v in t.items()}) for c, t in ((L.DensSrc, f), (L.DensOut, o)))
                L.check(L.lib().sphk_density_dev(ctx.handle, w.n_walk, w.i_off.data_ptr(), w.j_off.data_ptr(),
                                                 w.j_idx.data_ptr(), s, s, d, MIXED, torch.cuda.current_stream().cuda_stream), "density")
            out.append({k: v[:n].cpu() for k, v in o.items()})
    for k, v in out[0].items():     # bit for bit (NaN where a walk's list holds none of its neighbours)
        bits = (lambda a: a.view(torch.int64)) if v.dtype == torch.float64 else (lambda a: a)
        assert torch.equal(bits(v), bits(out[1][k])), k


@pytest.mark.parametrize("n_walk", [3072, 3073])
def test_hydro_does_not_depend_on_occupancy(n_walk):
    """Around the number of walks up to which an FP64 launch of one wave per
    walk takes more registers, against the several waves of a small table."""
    rng = np.random.default_rng(37)
    n, n_all = sum(SIZES), sum(SIZES) + n_walk
    f = {k: torch.from_numpy(rng.uniform(0.1, 1.0, n_all)).cuda() for k in L.HYDRO_SRC}
    f["id"] = torch.arange(n_all, dtype=torch.int32, device="cuda")
    i_off, j_off, j_idx = _table(rng, n, LENGTHS[:len(SIZES)])
    out = []
    with Context(0) as ctx:
        for tables in ((i_off, j_off), _padded(i_off, j_off, n_walk, 1)):
            o = {k: torch.zeros(n_all, dtype=torch.float64, device="cuda") for k in L.HYDRO_OUT}
            ctx.hydro(Walks(*tables, j_idx), f, f, o, FP64)
            out.append({k: v[:n].cpu().view(torch.int64) for k, v in o.items()})
    for k in out[0]:
        assert torch.equal(out[0][k], out[1][k]), k
