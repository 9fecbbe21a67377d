"""Hydro and gravity with several waves per walk (launches of few walks): the
sums do not depend on the number of waves, so the first walks of a table
launched alone (few walks) must equal, bit for bit, the same walks within a
table padded with empty-list walks to a size that takes fewer waves."""
import numpy as np
import pytest
import torch

from research_codes_amd import _lib as L
from research_codes_amd.device import FP64, MIXED, Context, Walks, empty_out

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 9, 32, 33, 64, 70]                    # i-particles, more than a wave among them
LENGTHS = [0, 1, 63, 64, 65, 255, 256, 257, 513, 2050]  # records: no tile, its edges, more rounds than waves


def _table(rng, n_rec, lengths):
    i_off = np.concatenate([[0], np.cumsum(SIZES)])
    off = np.concatenate([[0], np.cumsum(lengths)])
    idx = np.concatenate([rng.integers(0, n_rec, k) for k in lengths])
    return i_off, off, idx


def _padded(i_off, off, n_walk):
    """The same walks, then walks of one particle (the last) with an empty list each: they write that particle only."""
    more = n_walk - (len(i_off) - 1)
    last = int(i_off[-1])
    return (np.concatenate([i_off, last + 1 + np.arange(more)]), np.concatenate([off, np.full(more, off[-1])]))


@pytest.mark.parametrize("precision", [MIXED, FP64])
@pytest.mark.parametrize("shift", range(len(LENGTHS)))
@pytest.mark.parametrize("functor", ["hydro", "uniform", "general"])
def test_results_do_not_depend_on_waves(precision, shift, functor):
    rng = np.random.default_rng(shift)
    lengths = [LENGTHS[(k + shift) % len(LENGTHS)] for k in range(len(SIZES))]
    spj = [LENGTHS[(k + 3 * shift + 1) % len(LENGTHS)] for k in range(len(SIZES))]
    n = sum(SIZES)
    n_all = n + 23100
    f = {k: torch.from_numpy(rng.uniform(0.1, 1.0, n_all)).cuda() for k in L.HYDRO_SRC}
    f["id"] = torch.arange(n_all, dtype=torch.int32, device="cuda")
    f["eps2"] = torch.from_numpy(np.full(n_all, 0.01) if functor == "uniform" else rng.uniform(0.01, 0.1, n_all)).cuda()
    i_off, j_off, j_idx = _table(rng, n, lengths)
    _, s_off, s_idx = _table(rng, n, spj)
    out = []
    with Context(0) as ctx:
        ctx.set_params(uniform_softening=functor == "uniform")
        # sizes on both sides of every line: 8 / 4 / 2 / 1 waves
        for n_walk in (len(SIZES), 1600, 2100, 4100, 5000, 6600, 23100):
            io, jo = _padded(i_off, j_off, n_walk)
            _, so = _padded(i_off, s_off, n_walk)
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
