"""Many independent reconstructions of uneven sizes advanced together (no
counterpart in the reference, which reconstructs one object per run).

Each instance keeps its own ``Solver`` (operators sized for it) and its own
stream.  An ADMM iteration advances every instance in lock-step: the
ptychography CG's heavy launches -- the fused gradient and each line-search
sweep -- are made as one grouped launch for all instances
(``pt_ptycho_grad_group`` / ``pt_ptycho_linesearch_sweep_group``: every instance's
overlap-add tiles in one grid), and the rest of each instance's iteration
runs on its own stream, so small instances overlap on the device.  Without
grouping, the iteration can also be captured as one HIP graph per iteration
(``graph``).
Results are bit-identical to running each instance alone (the grouped
kernels do per instance exactly what the single launches do; within an
instance the order of operations is unchanged).
"""
import torch

from . import _lib
from ._dev import stream
from .solver import Solver, run_ptycho_request


class BatchSolver:
    def __init__(self, solvers, tune=False, tune_cache=None):
        """solvers: one Solver per instance.  tune: pick each instance's
        USFFT launch shapes with the autotuner (sizes on the register line
        FFT have none to tune; instances of one size share
        the cached result; ``tune_cache``: the tuner's JSON file, default its
        own); the shapes are kept in ``self.tuning``."""
        self.solvers = list(solvers)
        self.streams = [torch.cuda.Stream() for _ in self.solvers]
        # the grouped ptychography phase's stream (the same one eagerly and
        # under capture: the library's per-stream workspaces are sized by the
        # eager iterations)
        self.hub = torch.cuda.Stream()
        self.histories = [[] for _ in self.solvers]
        self.tuning = []
        if tune:
            from . import autotune
            kw = {} if tune_cache is None else {"cache": tune_cache}
            self.tuning = [autotune.tune_solver(slv, **kw)[0] for slv in self.solvers]

    @classmethod
    def from_args(cls, args_list, **kw):
        """args_list: Solver constructor argument tuples, one per instance."""
        return cls((Solver(*a) for a in args_list), **kw)

    def admm(self, datas, states, alpha, piter, titer, niter, model, lagr_every=0,
             graph=False, rho=0.5, tau=0.5, callback=None, m0=0, grouped=True):
        """Run niter ADMM iterations on every instance.  states: per instance
        dicts with h, e, psi, phi, lamd, mu, u (the reference's initial guess
        or a previous state, which may also carry rho, tau and Ru).  m0 is the
        index of the first iteration (the first two iterations of a run take
        piter + 32 ptychography CG steps).  grouped: the ptychography CG's
        heavy launches of the small instances (fewer than GROUP_TILES
        overlap-add tiles, where launches count more than overlap) as grouped
        launches; every other instance makes its own launches on its
        stream.  graph (with grouped=False):
        from the third iteration on, one iteration of the whole batch is
        captured as a HIP graph and replayed (eager launches measured faster
        on MI355X with ROCm 7).  Returns [(u, psi)] and keeps each solver's
        ``state``/``history``.  ``callback(m, i, u)`` is called after every
        iteration m for every instance i with its live u buffer."""
        if graph and grouped:
            # the capture of the grouped iteration (its ptychography phase on
            # the hub stream) ended in a host crash inside the HIP runtime's
            # capture end; the cause is not known, so it is not offered
            raise ValueError("BatchSolver.admm: graph capture is available with grouped=False "
                             "only")
        cur = torch.cuda.current_stream()
        ctxs, ds = [], []
        for slv, data, st, s in zip(self.solvers, datas, states, self.streams):
            s.wait_stream(cur)
            with torch.cuda.stream(s):
                ds.append(slv._dev_data(data))
                ctxs.append(slv._admm_setup(st["h"], st["e"], st["psi"], st["phi"], st["lamd"],
                                            st["mu"], st["u"], st.get("rho", rho),
                                            st.get("tau", tau), st.get("Ru"), piter, titer))
            slv.history = []
        graph_obj = None
        run = dict(piter=piter, titer=titer, alpha=alpha, model=model, grouped=grouped)
        for m in range(m0, m0 + niter):
            if graph and m >= 2 and m > m0:
                if graph_obj is None:
                    for s in self.streams:
                        s.synchronize()
                    graph_obj = torch.cuda.CUDAGraph()
                    cap = torch.cuda.Stream()
                    with torch.cuda.graph(graph_obj, stream=cap):
                        for s in self.streams:
                            s.wait_stream(cap)
                        self._step(ctxs, ds, m, **run)
                        for s in self.streams:
                            cap.wait_stream(s)
                # the replay runs on `cur`: order it after every instance
                # stream's previous work, and the reads of this iteration's
                # history (on the instance streams) after it
                for s in self.streams:
                    cur.wait_stream(s)
                graph_obj.replay()
                for s in self.streams:
                    s.wait_stream(cur)
            else:
                self._step(ctxs, ds, m, **run)
            for i, (slv, ctx, d, s) in enumerate(zip(self.solvers, ctxs, ds, self.streams)):
                with torch.cuda.stream(s):
                    slv._admm_record(ctx, d, m, piter, titer, alpha, model, lagr_every, False,
                                     niter)
                    if callback is not None:
                        callback(m, i, ctx["S"]["u"])
        out = []
        for slv, ctx, s in zip(self.solvers, ctxs, self.streams):
            cur.wait_stream(s)
            slv._admm_finish(ctx, m0 + niter)
            out.append((ctx["S"]["u"], ctx["S"]["psi"]))
        return out

    def _step(self, ctxs, ds, m, piter, titer, alpha, model, grouped):
        """Enqueue ADMM iteration m of every instance."""
        pit = piter + (m < 2) * 32      # solver.py:315
        mdl = _lib.PT_MODEL[model]
        gens = [slv._admm_iter_gen(ctx["S"], ctx["blk"], ctx["H"], d, pit, titer, alpha)
                for slv, ctx, d in zip(self.solvers, ctxs, ds)]
        sel = [i for i in range(len(gens)) if grouped and self._small(i)]
        # instances not grouped: the whole iteration on their own streams
        for i in range(len(gens)):
            if i in sel:
                continue
            with torch.cuda.stream(self.streams[i]):
                for req in gens[i]:
                    run_ptycho_request(req, mdl, stream())
        if not sel:
            return
        # the ptychography subproblem of the grouped instances on one stream,
        # its heavy launches grouped (the instances run the same schedule, so
        # they reach each request together); then the rest of each
        # instance's iteration on its own stream
        gens = [gens[i] for i in sel]
        streams = [self.streams[i] for i in sel]
        n = len(gens)
        hub = self.hub
        for s in streams:
            hub.wait_stream(s)
        with torch.cuda.stream(hub):
            st = stream()
            reqs = [next(g) for g in gens]
            while reqs[0][0] != "end":
                kinds = {(r[0], r[2] if r[0] == "ls" else 0) for r in reqs}
                if len(kinds) != 1:
                    raise RuntimeError(f"BatchSolver: instances out of step ({kinds})")
                kind, ng = kinds.pop()
                if kind == "grad":
                    arr = (_lib.GradArgs * n)(*[r[1] for r in reqs])
                    _lib.call("pt_ptycho_grad_group", arr, n, mdl, st)
                else:
                    arr = (_lib.LinesearchArgs * n)(*[r[1] for r in reqs])
                    sw = (_lib.SweepArgs * n)(*[r[3][:3] for r in reqs])
                    _lib.call("pt_ptycho_linesearch_sweep_group", arr, sw, n, ng, *reqs[0][3][3:],
                              mdl, st)
                reqs = [next(g) for g in gens]
            if any(r[0] != "end" for r in reqs):
                raise RuntimeError("BatchSolver: instances out of step")
        for g, s in zip(gens, streams):
            s.wait_stream(hub)
            with torch.cuda.stream(s):
                for req in g:
                    run_ptycho_request(req, mdl, stream())

    # 16 x 16-pixel tiles of the object's angles below which an instance is
    # grouped: its own launches are then so short that fewer of them gain more than
    # the instances gain by overlapping on their streams.  ms per iteration of the
    # whole batch, grouped / on streams: 16 of 48^3 (648 tiles) 13.9 / 17.5, 16 of
    # 64^3 (1536) 15.8 / 17.9, 8 of 72^3 (2187) 10.0 / 10.1, 8 of 80^3 (3000) 12.0 /
    # 11.2, 16 of 96^3 (5184) 33.8 / 29.0, 4 of 192^3 54.5 / 49.9.
    GROUP_TILES = 2048

    def _small(self, i):
        """whether instance i takes part in the grouped launches"""
        slv = self.solvers[i]
        return slv.ntheta * slv.nz * slv.n / 256 < self.GROUP_TILES
