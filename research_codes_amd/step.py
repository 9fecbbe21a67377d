"""Device-resident SPH step: the reference's calcSPHKernel and KDK loop with
the particle state in HBM and every O(N) and O(N*list) pass on the GPU.

Order of one force evaluation (sph_yamauchi/run/main.cpp:293-358):
  density (h-iteration, grad-h, div/curl)  -> state dens/divv/rotv/grdh/ksr
  EOS + Balsara                            (hdr_hgas.hpp:318-344, hdr_sph.hpp:79-89)
  softening eps2, tree gravity, write-back (hdr_gravity.hpp:107-137, 346-423)
  hydro EPI prep, hydro, write-back, acc sum, alpha-dot
                                           (hdr_hydro.hpp, hdr_sph.hpp:95-97, hdr_hgas.hpp:750-762)
The walk lists come from the device tree (sphk_dtree.h; tree="device") or
the host tree (sphk_tree.h; tree="host"), which build identical lists; they
are inputs of the step, not part of it.

The density smoothing-length retry loop (hdr_density.hpp:369-415) is in
`converge_density`: particles whose H_3 exceeds their search radius get
rs *= 1.1 and a fresh gather list, and keep the results of the pass in
which they converged (their rs then set to 0, as the reference does).
"""
from __future__ import annotations

import ctypes as C
import time

import numpy as np
import torch

from . import _lib as L
from ._lib import check, lib, raw_stream
from .device import FP64, MIXED, Context, Walks, _mk, to_device
from .tree import DeviceTree, HostTree, morton_order, morton_order_dev, permute_dev

KSRH = 1.936492


def phys(**kw) -> L.Phys:
    d = dict(ninv=1.0 / 1.5, ksrh=KSRH, G=1.0, alpha_max=2.0, alpha_min=0.1, alphu_max=0.0,
             alphu_min=0.0, eps_u=0.0, c_dt=0.1, dt_max=10.0, eps_const=0.0)
    d.update(kw)
    return L.Phys(**d)


class SPHSystem:
    """Particle state on the device plus the current walk lists."""

    def __init__(self, p: dict, ctx: Context, eta: float = 1.6, eps: float | None = None,
                 theta: float = 0.5, n_group: int = 16, n_leaf: int = 8,
                 precision: int = MIXED, hmax: float | None = None, phys_params=None,
                 device="cuda", tree: str = "device", segments=None):
        if tree not in ("device", "host"):
            raise ValueError("tree must be 'device' or 'host'")
        self.tree = tree
        self.ctx = ctx
        self.dev = device
        self.eta = eta
        self.eps = eps
        self.theta = theta
        # walk group size per list kind (an int applies to all three)
        self.n_group = (dict(n_group) if isinstance(n_group, dict)
                        else {"dens": n_group, "hydro": n_group, "grav": n_group})
        self.n_leaf = n_leaf
        self.precision = precision
        self.phys = phys_params or phys()
        # a constant softening leaves the potential independent of H: the
        # gravity write-back then sets the grad-h softening term eta to 0
        self.phys.eps_const = 0.0 if eps is None else float(eps)
        # independent systems (an ensemble of runs): particle counts of
        # consecutive blocks of p; each is Morton-sorted and gets its own tree
        n_all = len(p["x"])
        counts = [n_all] if segments is None else [int(c) for c in segments]
        if sum(counts) != n_all or min(counts) < 1:
            raise ValueError("segments must be positive counts summing to the particle number")
        self.seg = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
        perm = np.concatenate([morton_order(p["x"][a:b], p["y"][a:b], p["z"][a:b]) + a
                               for a, b in zip(self.seg[:-1], self.seg[1:])])
        self.n = n = len(perm)
        f64 = dict(dtype=torch.float64, device=device)
        # the state fields are the rows of one (fields, n) array: a reorder
        # permutes them all in one gather
        self._sbuf = torch.zeros(len(L.STATE_FIELDS), n, **f64)
        self.s = {k: self._sbuf[q] for q, k in enumerate(L.STATE_FIELDS)}
        for k in ("m", "x", "y", "z", "vx", "vy", "vz", "uene", "ksr", "alph", "alphu"):
            self.s[k].copy_(torch.from_numpy(np.ascontiguousarray(p[k][perm], np.float64)))
        self.id = to_device(np.ascontiguousarray(p["id"][perm], np.int32), device)
        self.istar = to_device(np.ascontiguousarray(p.get("istar", np.zeros(n, np.int32))[perm],
                                                    np.int32), device)
        self.rs = torch.zeros(n, **f64)
        self.np_ = torch.zeros(n, dtype=torch.int64, device=device)
        self.itr = torch.zeros(n, dtype=torch.uint8, device=device)
        self.eps2 = torch.zeros(n, **f64)
        self.hprep = {k: torch.zeros(n, **f64) for k in ("hinv", "presc", "bswt_half", "thrm")}
        self.gout = {k: torch.zeros(n, **f64) for k in L.GRAV_OUT}
        self.hout = {k: torch.zeros(n, **f64) for k in L.HYDRO_OUT}
        self.time = 0.0
        self.dt = self.phys.dt_max
        if hmax is None:
            hmax = self.system_size() if len(counts) == 1 else 1e30
        self.hmax = float(hmax)
        self.last_perm = None
        # a constant softening makes every eps2 equal: one rsqrt per gravity pair
        ctx.set_params(eta=eta, ksrh=KSRH, hmax=hmax, uniform_softening=eps is not None)
        self.lists = {}
        self.list_build_s = 0.0
        self._dtrees = {}     # device trees per (segment, group size), rebuilt in place
        self._ss = L.State(**{k: self.s[k].data_ptr() for k in L.STATE_FIELDS})

    # ---------------------------------------------------------- H_max (glue)
    def _com(self, star: int):
        sel = (self.istar == star).to(torch.float64)
        m = self.s["m"] * sel
        M = m.sum()
        return M, [(m * self.s[c]).sum() / M for c in ("x", "y", "z")]

    def system_size(self) -> float:
        """calcSystemSize (hdr_util.hpp:93-113, FlagBinary 0): distance between
        the centres of mass of star 0 and star 1; unbounded for one star."""
        M0, c0 = self._com(0)
        M1, c1 = self._com(1)
        if float(M0) == 0.0 or float(M1) == 0.0:
            return 1e30
        return float(torch.sqrt(sum((a - b) ** 2 for a, b in zip(c0, c1))))

    def update_hmax(self) -> float:
        """calcKernelSupportRadiusMaximum (hdr_util.hpp:489-505): density-
        weighted RMS distance of all particles from star 0's centre of mass."""
        _, c0 = self._com(0)
        d = self.s["dens"]
        r2 = sum((self.s[c] - x0) ** 2 for c, x0 in zip(("x", "y", "z"), c0))
        h = float(torch.sqrt((d * r2).sum() / d.sum()))
        self.ctx.set_params(hmax=h)
        self.hmax = h
        return h

    # ------------------------------------------------------------------ lists
    def _host(self, *keys):
        return [self.s[k].cpu().numpy() for k in keys]

    def _segments(self):
        return list(zip(self.seg[:-1].tolist(), self.seg[1:].tolist()))

    def resort(self):
        """Re-establish Morton order after particles moved (permutes the state;
        each segment of an ensemble on its own).  The permutation applied is
        kept in `last_perm` (None when the order did not change)."""
        self.last_perm = None
        if self.tree == "device":
            x, y, z = self.s["x"], self.s["y"], self.s["z"]
            pt = torch.cat([morton_order_dev(x[a:b], y[a:b], z[a:b]) + a for a, b in self._segments()])
            if bool((pt == torch.arange(self.n, device=pt.device)).all()):
                return
        else:
            x, y, z = self._host("x", "y", "z")
            perm = np.concatenate([morton_order(x[a:b], y[a:b], z[a:b]) + a for a, b in self._segments()])
            if np.array_equal(perm, np.arange(self.n, dtype=perm.dtype)):
                return
            pt = torch.from_numpy(perm.astype(np.int64)).to(self.dev)
        self.last_perm = pt.long()
        if self.tree == "device":
            # every state row and per-particle array in one gather and one copy back
            cols = [self._sbuf[q] for q in range(self._sbuf.shape[0])]
            cols += [self.id, self.istar, self.rs, self.np_, self.itr, self.eps2]
            self._perm_work = permute_dev(pt.to(torch.int32), cols, getattr(self, "_perm_work", None))
            return
        self._sbuf.copy_(self._sbuf[:, self.last_perm])
        for t in (self.id, self.istar, self.rs, self.np_, self.itr, self.eps2):
            t.copy_(t[pt])

    def build_lists(self, kinds=("dens", "hydro", "grav")):
        t0 = time.perf_counter()
        if "grav" in kinds:
            self._softening()
        self._build_lists_segments(kinds)
        torch.cuda.current_stream().synchronize()   # this stream only: a gravity pass may run beside it
        self.list_build_s = time.perf_counter() - t0

    def _tree(self, a: int, b: int, g: int):
        """Tree over particles [a, b) with walk group size g."""
        s = self.s
        if self.tree == "device":
            args = (s["x"][a:b], s["y"][a:b], s["z"][a:b], s["m"][a:b], self.eps2[a:b], self.n_leaf, g)
            t = self._dtrees.get((a, b, g))
            if t is None:
                t = self._dtrees[(a, b, g)] = DeviceTree(*args)
            else:
                t.rebuild(*args)
            return t
        x, y, z, m = (s[k][a:b].cpu().numpy() for k in ("x", "y", "z", "m"))
        return HostTree(x, y, z, m, self.eps2[a:b].cpu().numpy(), self.n_leaf, g)

    def _build_lists_segments(self, kinds):
        """Lists per segment (one tree each, device or host), their indices
        shifted to the segment's place and concatenated into one walk table
        per functor: an ensemble runs in one launch per functor."""
        s = self.s
        dev = torch.device(self.dev)

        def t32(a):
            return a if isinstance(a, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(a)).to(dev)

        parts = {k: [] for k in kinds}
        moms = []
        dev_tree = self.tree == "device"
        for a, b in self._segments():
            trees = {}
            try:
                def tree_for(kind):
                    g = self.n_group[kind]
                    if g not in trees:
                        trees[g] = self._tree(a, b, g)
                    return trees[g]
                if "dens" in kinds:
                    t = tree_for("dens")
                    rs = self.rs[a:b] if dev_tree else self.rs[a:b].cpu().numpy()
                    parts["dens"].append((a, t.i_off, *t.gather(rs)))
                if "hydro" in kinds:
                    t = tree_for("hydro")
                    h = s["ksr"][a:b] if dev_tree else s["ksr"][a:b].cpu().numpy()
                    parts["hydro"].append((a, t.i_off, *t.symmetry(h)))
                if "grav" in kinds:
                    t = tree_for("grav")
                    parts["grav"].append((a, t.i_off, *t.long(self.theta)))
                    moms.append({k: t32(v) for k, v in t.moments().items()})
            finally:
                if not dev_tree:
                    for t in trees.values():
                        t.close()
        for kind, pl in parts.items():
            if len(pl) == 1:
                a, i_off, *rest = pl[0]
                self.lists[kind] = Walks(t32(i_off), *map(t32, rest))
                continue
            i_off, j_off, j_idx, s_off, s_idx = [], [], [], [], []
            jb = sb = nb = 0
            for (a, io, *rest), mom in zip(pl, moms if kind == "grav" else [None] * len(pl)):
                io = t32(io)
                jo, ji = t32(rest[0]), t32(rest[1])
                i_off.append(io[:-1] + a)
                j_off.append(jo[:-1] + jb)
                j_idx.append(ji + a)
                jb += int(jo[-1])
                if kind == "grav":
                    so, si = t32(rest[2]), t32(rest[3])
                    s_off.append(so[:-1] + sb)
                    s_idx.append(si + nb)
                    sb += int(so[-1])
                    nb += int(mom["m"].numel())
            tail = lambda v: torch.tensor([v], dtype=torch.int32, device=dev)   # noqa: E731
            args = [torch.cat(i_off + [tail(self.n)]), torch.cat(j_off + [tail(jb)]), torch.cat(j_idx)]
            if kind == "grav":
                args += [torch.cat(s_off + [tail(sb)]), torch.cat(s_idx)]
            self.lists[kind] = Walks(*args)
        if "grav" in kinds:
            self.mom = moms[0] if len(moms) == 1 else {k: torch.cat([m[k] for m in moms]) for k in moms[0]}

    def autotune_groups(self, candidates=(8, 16, 32), reps: int = 3, precision=None):
        """Pick, per list kind, the walk group size with the fastest kernel
        (for density also the LDS list capacity, 192 or 256).

        Each candidate rebuilds that kind's lists and times `reps` launches
        of its functor (HIP events on the launch stream).  Leaves the best
        lists and settings in place; returns ({kind: size, "dens_list_cap":
        cap}, {kind: {candidate: ms}})."""
        n = self.n
        tmp = {k: torch.empty(n, dtype=torch.float64, device=self.dev)
               for k in ("dens", "divv", "rotv", "grdh", "ksr")}
        tmp["np"] = torch.empty(n, dtype=torch.int64, device=self.dev)
        tmp["itr"] = torch.empty(n, dtype=torch.uint8, device=self.dev)
        run = {"dens": lambda: self.density(out=tmp, precision=precision),
               "hydro": lambda: self.hydro(precision),
               "grav": lambda: self.gravity(precision)}
        def timed(fn):
            fn()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(reps):
                fn()
            e1.record()
            torch.cuda.synchronize()
            return e0.elapsed_time(e1) / reps

        best, table = {}, {}
        for kind in ("dens", "hydro", "grav"):
            table[kind] = {}
            for g in candidates:
                self.n_group[kind] = g
                self.build_lists((kind,))
                if kind == "dens":   # the density kernel's list capacity too
                    for cap in (192, 256):
                        self.ctx.set_params(list_cap=cap)
                        table[kind][f"{g}/{cap}"] = timed(run[kind])
                else:
                    table[kind][str(g)] = timed(run[kind])
            key = min(table[kind], key=table[kind].get)
            if kind == "dens":
                g, cap = (int(v) for v in key.split("/"))
                self.ctx.set_params(list_cap=cap)
                best["dens_list_cap"] = cap
            else:
                g = int(key)
            best[kind] = g
            self.n_group[kind] = g
            self.build_lists((kind,))
        return best, table

    # ---------------------------------------------------------------- kernels
    _st = staticmethod(raw_stream)

    def _softening(self):
        check(lib().sphk_softening_dev(self.ctx.handle, self.n, self.s["ksr"].data_ptr(), KSRH,
                                       0.0 if self.eps is None else float(self.eps),
                                       self.eps2.data_ptr(), self._st()), "sphk_softening_dev")

    def dens_src(self):
        s = self.s
        return dict(id=self.id, m=s["m"], x=s["x"], y=s["y"], z=s["z"], vx=s["vx"], vy=s["vy"],
                    vz=s["vz"], ksr=s["ksr"], rs=self.rs)

    def density(self, out: dict | None = None, precision=None):
        """One density functor pass over the current gather lists."""
        s = self.s
        src = self.dens_src()
        if out is None:
            out = dict(dens=s["dens"], divv=s["divv"], rotv=s["rotv"], grdh=s["grdh"],
                       ksr=s["ksr"], np=self.np_, itr=self.itr)
        self.ctx.density(self.lists["dens"], src, src, out,
                         self.precision if precision is None else precision)
        return out

    def converge_density(self, expand: float = 1.1, max_rounds: int = 100, jump: bool = False,
                         full_lists: bool = False, rounds_out: list | None = None):
        """calcDensityKernel (hdr_density.hpp:369-415) with device list rebuilds.

        rs = 1.1 ksr; each round rebuilds the gather lists and runs the density
        functor.  A particle still retrying (rs != 0) whose H_3 exceeds rs
        retries with rs *= 1.1; otherwise its results are kept (copyFromForce,
        hdr_density.hpp:24-31) and its rs set to 0, so later rounds' lists
        serve only the particles still retrying.  The loop ends when no
        particle retried.  jump=True grows rs to max(1.1 rs, 1.1 H_3) instead
        of 1.1 rs (set-up of a star far from the fixed point only: fewer
        rounds, not the reference's schedule).

        full_lists=True leaves each particle's rs at the value it converged
        with and, when more than one round ran, rebuilds the gather lists
        with them, so that the density functor can be re-run on the converged
        state (the reference leaves rs = 0).  rounds_out (a list) receives
        each round's gather lists and the mask of the particles that took that
        round's results: a particle whose intermediate H outgrew rs has
        results that depend on its round's list.  Returns the number of
        rounds; raises if particles still retry after max_rounds (the
        reference loops without a bound).
        """
        n = self.n
        s = self.s
        self.rs.copy_(expand * s["ksr"])
        rs_conv = torch.zeros_like(self.rs) if full_lists else None
        tmp = {k: torch.empty(n, dtype=torch.float64, device=self.dev)
               for k in ("dens", "divv", "rotv", "grdh", "ksr")}
        tmp["np"] = torch.empty(n, dtype=torch.int64, device=self.dev)
        tmp["itr"] = torch.empty(n, dtype=torch.uint8, device=self.dev)
        flag = torch.zeros(1, dtype=torch.int32, device=self.dev)
        tmp_out = _mk(L.DensOut, L.DENS_OUT, tmp)
        for rnd in range(1, max_rounds + 1):
            self.build_lists(("dens",))
            self.density(out=tmp)
            if rounds_out is not None:
                rounds_out.append((self.lists["dens"], (self.rs != 0.0) & (tmp["itr"] == 0)))
            # the round's bookkeeping in one kernel, one host read
            check(lib().sphk_density_commit_dev(self.ctx.handle, n, self._ss, tmp_out, self.np_.data_ptr(),
                                                self.rs.data_ptr(),
                                                None if rs_conv is None else rs_conv.data_ptr(), float(expand),
                                                int(bool(jump)), flag.data_ptr(), self._st()),
                  "sphk_density_commit_dev")
            if int(flag.item()) == 0:
                break
        else:
            raise RuntimeError(f"density did not converge in {max_rounds} rounds")
        self.itr.zero_()
        if full_lists:
            self.rs.copy_(rs_conv)
            if rnd > 1:
                self.build_lists(("dens",))
        return rnd

    def relax_h(self, passes: int = 3) -> int:
        """Run the smoothing-length retry loop `passes` times, each starting
        from the previous H, so H reaches the fixed point of the three-pass
        iteration (set-up only; the reference starts from relaxed stars, and
        this uses the jump schedule of converge_density)."""
        rounds = 0
        for _ in range(passes):
            rounds += self.converge_density(jump=True)
        return rounds

    def eos_balsara(self):
        check(lib().sphk_eos_balsara_dev(self.ctx.handle, self.n, self._ss, self.phys, self._st()),
              "sphk_eos_balsara_dev")

    def gravity(self, precision=None):
        self._softening()
        s = self.s
        src = dict(m=s["m"], x=s["x"], y=s["y"], z=s["z"], eps2=self.eps2)
        # under a constant softening the softening-gradient sum does not enter
        gout = {k: v for k, v in self.gout.items() if k != "eta"} if self.phys.eps_const > 0 else self.gout
        self.ctx.gravity(self.lists["grav"], src, src, gout, ps=self.mom,
                         precision=self.precision if precision is None else precision)
        go = L.GravOut(**{k: gout[k].data_ptr() if k in gout else None for k in L.GRAV_OUT})
        check(lib().sphk_gravity_writeback_dev(self.ctx.handle, self.n, self._ss, self.phys, go,
                                               self._st()), "sphk_gravity_writeback_dev")

    def hydro_src(self):
        s, h = self.s, self.hprep
        return dict(id=self.id, m=s["m"], x=s["x"], y=s["y"], z=s["z"], vx=s["vx"], vy=s["vy"],
                    vz=s["vz"], hinv=h["hinv"], pres=s["pres"], presc=h["presc"],
                    bswt=h["bswt_half"], dens=s["dens"], vsnd=s["vsnd"], alph=s["alph"],
                    alphu=s["alphu"], thrm=h["thrm"], eta=s["eta"])

    def hydro(self, precision=None):
        h = self.hprep
        check(lib().sphk_hydro_prep_dev(self.ctx.handle, self.n, self._ss, h["hinv"].data_ptr(),
                                        h["presc"].data_ptr(), h["bswt_half"].data_ptr(),
                                        h["thrm"].data_ptr(), self._st()), "sphk_hydro_prep_dev")
        src = self.hydro_src()
        self.ctx.hydro(self.lists["hydro"], src, src, self.hout,
                       self.precision if precision is None else precision)
        ho = L.HydroOut(**{k: self.hout[k].data_ptr() for k in L.HYDRO_OUT})
        check(lib().sphk_hydro_writeback_dev(self.ctx.handle, self.n, self._ss, self.phys, ho,
                                             self._st()), "sphk_hydro_writeback_dev")

    def capture_force(self, precision=None):
        """Record one force evaluation (density, EOS, gravity, hydro and their
        write-backs, 10 kernel launches) on the current lists into a HIP graph
        and return it: `graph.replay()` re-runs the step on the state arrays
        in place.  The lists and state tensors must stay the ones captured;
        kernel timing is switched off while capturing."""
        timing = getattr(self.ctx, "_timing", False)
        self.ctx.timing(False)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            self.force(precision)            # warm-up outside the graph
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            self.force(precision)
        torch.cuda.synchronize()
        self.ctx.timing(timing)
        return g

    def force(self, precision=None, overlap: bool = True):
        """One force evaluation on resident lists (no list rebuild, no retry).

        Under a constant softening the gravity functor and its write-back
        read nothing the density pass and the EOS write: with overlap they run
        on a second stream beside them (the two kernels share the GPU where
        either leaves it idle), joined before the hydro prep, which needs
        both.  overlap=False runs the four in order on one stream (each
        kernel's own duration is then measurable)."""
        if not (overlap and self.phys.eps_const > 0):
            self.density(precision=precision)
            self.eos_balsara()
            self.gravity(precision)
        else:
            cur = torch.cuda.current_stream()
            side = self._side_stream()
            side.wait_stream(cur)
            with torch.cuda.stream(side):
                self.gravity(precision)
            self.density(precision=precision)
            self.eos_balsara()
            cur.wait_stream(side)
        self.hydro(precision)

    def _side_stream(self):
        """A second stream (default priority) for the gravity functor."""
        if getattr(self, "_side", None) is None:
            self._side = torch.cuda.Stream(device=torch.cuda.current_stream().device)
        return self._side

    # ------------------------------------------------------------ integrator
    def diagnostics(self) -> dict:
        out = (C.c_double * 6)()
        check(lib().sphk_diagnostics(self.ctx.handle, self.n, self._ss, self.phys, out, self._st()),
              "sphk_diagnostics")
        return dict(energy=out[0], momentum=np.array(out[1:4]), dt_min=out[4], mass=out[5])

    def snapshot(self) -> dict:
        """Host copy of the particle state in id order (for the writers in
        research_codes_amd.formats)."""
        order = torch.argsort(self.id.long())
        p = {k: v[order].cpu().numpy() for k, v in self.s.items()}
        p["id"] = self.id[order].cpu().numpy().astype(np.int64)
        p["istar"] = self.istar[order].cpu().numpy().astype(np.int64)
        p["np"] = self.np_[order].cpu().numpy()
        return p

    def unbound_mass(self, k: float = 20.0, star: int = -1) -> dict:
        """Unbound mass (analysis/unbound_mass/unbound_mass.py:10-28) of the
        current state, hard threshold and smoothed with slope k; star >= 0
        restricts to one star."""
        out = (C.c_double * 6)()
        check(lib().sphk_unbound_mass_dev(self.ctx.handle, self.n, self._ss, self.istar.data_ptr(),
                                          int(star), float(k), out, self._st()), "sphk_unbound_mass_dev")
        return dict(v_cg=np.array(out[0:3]), unbound=out[3], unbound_smooth=out[4], mass=out[5])

    def next_dt(self, dt_min_particle: float, dt_floor: float = 1e-16) -> float:
        """Power-of-two timestep adjustment of main.cpp:241-273."""
        dtc = min(self.phys.dt_max, dt_min_particle)
        dt = self.dt
        if dt > dtc:
            while dt > dtc:
                dt *= 0.5
                if dt <= dt_floor:
                    raise FloatingPointError(f"timestep underflow at t={self.time}: {dtc}")
        elif 2.0 * dt <= dtc and 2.0 * dt <= self.phys.dt_max:
            dt2 = 2.0 * dt
            if self.time - int(self.time / dt2) * dt2 == 0.0:
                dt *= 2.0
        return dt

    def initialize(self, record: dict | None = None):
        """startSimulation's first force evaluation (hdr_hgas.hpp:1335-1378)."""
        hmax = self.hmax
        rounds = [] if record is not None else None
        self.converge_density(rounds_out=rounds)
        self.eos_balsara()
        self.build_lists(("hydro", "grav"))
        self.gravity()
        self.hydro()
        if record is not None:
            record.update(perm=None, hmax=hmax, dens=self.lists["dens"], dens_rounds=rounds,
                          hydro=self.lists["hydro"], id=self.id.clone(), **self._grav_record())
        self.update_hmax()

    def _grav_record(self) -> dict:
        """The gravity step's long lists and its tree's node ranges (one run;
        an ensemble records nothing here)."""
        if len(self.seg) != 2 or self.tree != "device":
            return {}
        t = self._dtrees.get((0, self.n, self.n_group["grav"]))
        if t is None:
            return {}
        nd = t.nodes()
        return dict(grav=self.lists["grav"], gnode_begin=nd["begin"], gnode_end=nd["end"])

    def kdk(self, dt: float | None = None, record: dict | None = None):
        """One loopSimulation step (hdr_hgas.hpp:1499-1539) with a fixed list
        rebuild per step.  dt overrides the power-of-two timestep rule (a
        fixed schedule, e.g. for finite-difference sensitivities).  `record`
        (a dict) receives the step's reorder, H_max, lists and particle ids
        (in the reordered order).  Returns the diagnostics before the step.
        (Gravity on a second stream beside the density retry loop measured
        slower: the list walks and the retry loop's host reads leave it little
        idle GPU, and the walks slow down beside it.)"""
        d = self.diagnostics()
        self.dt = self.next_dt(d["dt_min"]) if dt is None else float(dt)
        dt = self.dt
        hmax = self.hmax
        check(lib().sphk_predict_dev(self.ctx.handle, self.n, self._ss, dt, self._st()),
              "sphk_predict_dev")
        self.resort()
        rounds = [] if record is not None else None
        self.converge_density(rounds_out=rounds)
        self.eos_balsara()
        self.build_lists(("hydro", "grav"))
        self.gravity()
        self.hydro()
        if record is not None:
            record.update(perm=self.last_perm, hmax=hmax, dens=self.lists["dens"], dens_rounds=rounds,
                          hydro=self.lists["hydro"], id=self.id.clone(), **self._grav_record())
        self.update_hmax()
        check(lib().sphk_correct_dev(self.ctx.handle, self.n, self._ss, dt, self._st()),
              "sphk_correct_dev")
        self.time += dt
        return d
