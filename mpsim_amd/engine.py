"""Per-device executor: builds descriptor tables and calls libmpsx.

Every arithmetic step of the MPS path goes through here to the HIP library;
there is no other implementation to fall back on.
"""
from __future__ import annotations

import ctypes
import threading
import warnings
from collections import OrderedDict
from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np

from . import _native as nat

MAX_OPS = 65535  # descriptors per grouped launch (grid y / x limits of the kernels)


def _matrix_addr(x, rows: int, cols: int, ld: int, what: str, seen: dict) -> int:
    """Device address of a rows x cols matrix with row stride `ld` stored in
    a contiguous complex64 tensor at an element offset (x = tensor or
    (tensor, offset)); raises if any element would fall outside it. seen:
    (address, tensor) of the tensors the call has found matrices inside of so far
    (many products share one); holding them, an id stays one tensor's."""
    t, off = x if isinstance(x, tuple) else (x, 0)
    n = t.numel()
    if not (rows and cols):
        return nat.ptr(t) + 8 * off if n else 0
    if cols > ld or off < 0 or off + (rows - 1) * ld + cols > n:
        raise ValueError(f"gemm operand {what}: {rows}x{cols} (ld {ld}) at offset {off} "
                         f"exceeds a tensor of {n} elements")
    if t is not x:
        known = seen.get(id(t))
        if known is not None:
            return known[0] + 8 * off
    if t.element_size() != 8:
        raise ValueError(f"gemm operand {what} must be complex64")
    p = nat.ptr(t)
    if t is not x:
        seen[id(t)] = (p, t)
    return p + 8 * off


def _gemm_rows(ops: Sequence[dict]) -> List[tuple]:
    """Descriptor rows of a grouped product, every matrix checked to lie
    inside its tensor."""
    rows, seen = [], {}
    for o in ops:
        m, n, k, fl = int(o["m"]), int(o["n"]), int(o["k"]), int(o.get("flags", 0))
        lda, ldb, ldc = o["lda"], o["ldb"], o["ldc"]
        # stored shapes: op(A) = A^H means A is stored k x m, else m x k
        ra, ca = (k, m) if fl & nat.GEMM_CONJ_A else (m, k)
        rb, cb = (n, k) if fl & nat.GEMM_CONJ_B else (k, n)
        pa = _matrix_addr(o["A"], ra, ca, lda, "A", seen)
        pb = _matrix_addr(o["B"], rb, cb, ldb, "B", seen)
        pc = _matrix_addr(o["C"], m, n, ldc, "C", seen)
        al = complex(o.get("alpha", 1.0))
        rows.append((pa, pb, pc, m, n, k, lda, ldb, ldc, al.real, al.imag, fl, 0))
    return rows


SPLIT_ROWS = 128  # default split_rows: rows from which a problem counts toward splitting a call


def _rows(it) -> int:
    """Rows of the working matrix: the side orthogonalised (d*chi_l, or
    d*chi_r when S is absorbed left)."""
    if isinstance(it, SplitItem):
        m, n = it.mat.shape
        return n if it.absorb_left else m
    return it.a.shape[1] * (it.b.shape[2] if it.absorb_left else it.a.shape[0])


def _cost(it) -> float:
    """Relative Jacobi work of one problem: rows^2 * row length."""
    if isinstance(it, SplitItem):
        m, n = it.mat.shape
    else:
        m, n = it.a.shape[0] * it.a.shape[1], it.b.shape[1] * it.b.shape[2]
    c, r = (n, m) if it.absorb_left else (m, n)
    return float(c) * c * r


@dataclass
class SvdConfig:
    """Jacobi SVD knobs (see mpsx_svd_opts in include/mpsx.h)."""
    block: int = 0          # 0 = library default
    max_sweeps: int = 0
    check_every: int = 1
    inner_sweeps: int = 0
    tol: float = 0.0
    block_switch: int = 0   # 0 = library default (64 rows)
    unconverged: int = 0    # device address of an int32 non-convergence counter, or 0
    fp32: bool = False      # FP32 working matrix (faster, ~1e-6 relative error per update)
    method: int = 0         # 0: Gram method for FP64 32-row pivots; 1: one-sided everywhere
    fp32_sweeps: int = 0    # Gram method: > 0 adds an FP32 phase of at most this many sweeps
    precondition: int = 0   # Householder QR before the Gram method: 0 none, 1 saturated bonds, 2 all

    def to_c(self) -> nat.SvdOpts:
        return nat.SvdOpts(self.block, self.max_sweeps, self.check_every, self.inner_sweeps,
                           self.tol, self.block_switch, 1 if self.fp32 else 0,
                           self.unconverged or None, self.method, self.fp32_sweeps,
                           self.precondition)


@dataclass(slots=True)
class TwoSiteItem:
    a: "object"            # torch [chi_l, d, chi_m]
    b: "object"            # torch [chi_m, d, chi_r]
    gate: "object"         # torch complex64 [d^2, d^2] on device
    k: int
    absorb_left: bool = False
    want_s: bool = False


@dataclass
class SplitItem:
    """A plain M x N matrix to factorise like a two-site theta."""
    mat: "object"          # torch complex64 [M, N], contiguous
    k: int
    absorb_left: bool = False
    want_s: bool = False


class TwoSiteResult:
    """Factors of one update; `discarded` is a device float64 scalar view."""
    __slots__ = ("a_out", "b_out", "s", "_disc", "_i")

    def __init__(self, a_out, b_out, s, disc, i):
        self.a_out, self.b_out, self.s, self._disc, self._i = a_out, b_out, s, disc, i

    @property
    def discarded(self):
        return self._disc[self._i]


class Engine:
    """Owns the device, a gate cache and a grow-only workspace."""

    _engines: Dict[int, "Engine"] = {}
    _late_words: Dict[int, object] = {}  # per device, held until the process ends
    _lock = threading.Lock()

    def __init__(self, dev):
        import torch
        self.torch = torch
        self.lib = nat.load()
        self.dev = nat.device(dev)
        self._ws = None
        self._gates: "OrderedDict[bytes, object]" = OrderedDict()
        from .tune import tuned_config, tuned_engine, tuned_rounds
        self.svd = tuned_config()
        self.last_sweeps = 0
        # concurrent groups of a split call (at most the 4 hardware queues a
        # process gets), the problems of >= split_rows rows a call needs to
        # be split, and that row count; from the stored tuning when there is
        # one (SPLIT_ROWS and 4 ways otherwise)
        self.split_ways, self.split_min, self.split_rows = tuned_engine()
        self._cus = torch.cuda.get_device_properties(self.dev).multi_processor_count
        # the same two numbers for methods that iterate in rounds, while the rule is
        # the stored one
        self._split_stored = (self.split_min, self.split_rows)
        self._split_rounds = tuned_rounds()
        self._wss: list = []        # workspaces of the helper streams' groups
        self._helpers: list = []    # (stream, single-thread executor) per helper group
        self._keep: list = []       # device tables of the last call, alive until the next
        # Calls share the workspaces and return while their kernels run: one call is
        # enqueued at a time, and a call on another stream than the last one's
        # waits for that to end.
        self._enqueue = threading.RLock()
        # set by a kernel (pinned host memory) when a problem did not converge in a
        # call that had returned by then; report() says so
        idx = self.dev.index if self.dev.index is not None else 0
        self._late_word = self._late_words.setdefault(
            idx, torch.zeros(1, dtype=torch.int32, pin_memory=True))
        self._late_ptr = self._late_word.data_ptr()
        self._late = ctypes.c_int32.from_address(self._late_ptr)
        self._used = None           # stream of the last call
        self._used_handle = -1
        self._used_end = None       # event: the last call's end on that stream

    @classmethod
    def get(cls, dev=None) -> "Engine":
        d = nat.device(dev)
        idx = d.index if d.index is not None else 0
        with cls._lock:
            eng = cls._engines.get(idx)
            if eng is None:
                eng = cls(d)
                cls._engines[idx] = eng
            return eng

    # ------------------------------------------------------------ helpers
    @property
    def stream(self) -> int:
        return nat.stream_handle(self.dev)

    def workspace(self, nbytes: int, slot: int = 0):
        """Grow-only device workspace; slot g > 0 serves the g-th helper
        stream of split calls."""
        while len(self._wss) < slot:
            self._wss.append(None)
        cur = self._wss[slot - 1] if slot else self._ws
        if cur is None or cur.numel() < nbytes:
            grow = max(nbytes, 0 if cur is None else int(cur.numel() * 1.25))
            if cur is not None and self._used is not None:
                # its memory returns to the stream it was allocated on, which need
                # not be the one that worked on it last (and that this one follows)
                cur.record_stream(self._used)
            cur = self.torch.empty(max(grow, 1024), dtype=self.torch.uint8, device=self.dev)
            if slot:
                self._wss[slot - 1] = cur
            else:
                self._ws = cur
        return cur

    def _take_workspaces(self, cur) -> None:
        """Orders the stream `cur` behind the last call's work in the workspaces.
        An event behind every call costs the stream a few us, so one on the
        default stream, which outlives the engine, is recorded only when another
        stream takes over."""
        last = self._used
        if last is not None:
            if not last.cuda_stream:
                self._leave_workspaces(last)
            cur.wait_event(self._used_end)
        self._used, self._used_handle = cur, int(cur.cuda_stream)

    def _leave_workspaces(self, cur) -> None:
        if self._used_end is None:
            self._used_end = self.torch.cuda.Event()
        self._used_end.record(cur)

    def report(self) -> None:
        """Warns (NotConvergedWarning) if the SVD of an update whose kernels have
        ended did not converge after its call had returned. Every two-site call
        and host() look; a caller that waits by other means may."""
        if self._late.value:
            self._late.value = 0
            warnings.warn("the SVD of an earlier two-site update has not converged",
                          nat.NotConvergedWarning, stacklevel=3)

    def host(self, t) -> np.ndarray:
        """The tensor on the host (waits for the current stream)."""
        out = t.cpu().numpy()
        self.report()
        return out

    def gate(self, mat: np.ndarray):
        """Device complex64 copy of a gate matrix (cached by content)."""
        m = np.ascontiguousarray(np.asarray(mat, dtype=np.complex64))
        key = m.tobytes() + bytes(str(m.shape), "ascii")
        g = self._gates.get(key)
        if g is None:
            g = self.torch.from_numpy(m.copy()).to(self.dev)
            self._gates[key] = g
            if len(self._gates) > 8192:
                self._gates.popitem(last=False)
        else:
            self._gates.move_to_end(key)
        return g

    # ------------------------------------------------------------ one-site
    def one_site(self, items: Sequence[Tuple[object, object, object]]) -> None:
        """items: (tensor_in, tensor_out, gate_dev [d, d]); out may be in."""
        if not items:
            return
        rows = []
        for a, out, g in items:
            cl, d, cr = a.shape
            pa = nat.ptr(a)
            rows.append((pa, pa if out is a else nat.ptr(out), nat.ptr(g), cl, cr, d, 0))
        self.one_site_rows(rows)

    def one_site_rows(self, rows: Sequence[tuple]) -> None:
        """Grouped one-site launch from ready descriptor rows
        (a, out, gate, chi_l, chi_r, d, 0) with device addresses."""
        if not rows:
            return
        tab = np.array(rows, dtype=nat.SITE_OP)
        stream = self.stream
        if len(rows) <= nat.SITE_NOW:
            code = self.lib.mpsx_apply_one_site_now(stream, tab.ctypes.data, len(rows))
            if code != nat.MPSX_EINVAL:  # refused (a capture) before anything was launched
                nat.check(code)
                return
        dtab = nat.put_table(tab, self.dev, stream)
        nat.check(self.lib.mpsx_apply_one_site(stream, tab.ctypes.data, dtab.data_ptr(),
                                               len(rows)))
        del dtab

    # ------------------------------------------------------------ two-site
    def _prepare_two_site(self, items: Sequence[TwoSiteItem], cfg, slot: int = 0,
                          workspace: bool = True, stream: Optional[int] = None):
        """Outputs, planned host table, device table and workspace (None with
        workspace=False) of one library call (allocations on the calling
        thread's current stream)."""
        torch = self.torch
        n = len(items)
        # shapes and input pointers (one pass), then every output carved out of
        # one allocation and the descriptor table filled column by column
        cls_, ds, cms, crs, ks, pa, pb, pg, fl = ([] for _ in range(9))
        gate_ptr: Dict[int, int] = {}  # a batch shares few gate tensors
        for it in items:
            if isinstance(it, SplitItem):
                cl, cr = it.mat.shape
                d, cm = 1, 0
                pa.append(nat.ptr(it.mat)); pb.append(0); pg.append(0)
            else:
                cl, d, cm = it.a.shape
                cm2, d2, cr = it.b.shape
                if cm != cm2 or d != d2:
                    raise ValueError(f"site tensors do not share a bond: {tuple(it.a.shape)} {tuple(it.b.shape)}")
                g = gate_ptr.get(id(it.gate))
                if g is None:
                    g = gate_ptr[id(it.gate)] = nat.ptr(it.gate)
                pa.append(nat.ptr(it.a)); pb.append(nat.ptr(it.b)); pg.append(g)
            cls_.append(cl); ds.append(d); cms.append(cm); crs.append(cr); ks.append(it.k)
            fl.append(1 if it.absorb_left else 0)
        cl_a, d_a, cr_a, k_a = (np.asarray(x, dtype=np.int64) for x in (cls_, ds, crs, ks))
        na = cl_a * d_a * k_a
        nb = k_a * d_a * cr_a
        ns = np.array([it.k if it.want_s else 0 for it in items], dtype=np.int64)
        # one allocation per update holds a_out, b_out and S (complex64 slots at
        # 32-element boundaries; S as float32 pairs), so a surviving site tensor
        # pins only its own update's memory
        la = (na + 31) // 32 * 32
        lb = (nb + 31) // 32 * 32
        length = la + lb + (ns + 1) // 2
        disc = torch.empty(n, dtype=torch.float64, device=self.dev)
        bufs = [torch.empty(max(int(m), 1), dtype=torch.complex64, device=self.dev)
                for m in length.tolist()]
        ptr0 = np.array([b.data_ptr() for b in bufs], dtype=np.int64)  # fresh, contiguous
        tab = np.zeros(n, dtype=nat.TWO_SITE_OP)
        tab["a"], tab["b"], tab["gate"] = pa, pb, pg
        tab["a_out"] = np.where(na > 0, ptr0, 0)
        tab["b_out"] = np.where(nb > 0, ptr0 + 8 * la, 0)
        tab["s_out"] = np.where(ns > 0, ptr0 + 8 * (la + lb), 0)
        tab["discarded"] = int(disc.data_ptr()) + 8 * np.arange(n, dtype=np.int64)
        tab["chi_l"], tab["chi_m"], tab["chi_r"] = cls_, cms, crs
        tab["d"], tab["k"], tab["flags"] = ds, ks, fl
        outs: List[TwoSiteResult] = []
        for i, buf in enumerate(bufs):
            cl, d, cr, k = cls_[i], ds[i], crs[i], ks[i]
            a_out = buf.as_strided((cl, d, k), (d * k, k, 1), 0)
            b_out = buf.as_strided((k, d, cr), (d * cr, cr, 1), int(la[i]))
            s = (buf.view(torch.float32).as_strided((k,), (1,), 2 * int(la[i] + lb[i]))
                 if ns[i] else None)
            outs.append(TwoSiteResult(a_out, b_out, s, disc, i))
        nbytes = ctypes.c_size_t(0)
        nat.check(self.lib.mpsx_two_site_plan(tab.ctypes.data, n, ctypes.byref(cfg),
                                              ctypes.byref(nbytes)))
        ws = self.workspace(nbytes.value, slot) if workspace else None
        dtab = nat.put_table(tab, self.dev, self.stream if stream is None else stream)
        return outs, tab, dtab, ws

    def _run_two_site(self, tab, dtab, ws, cfg, stream: int) -> int:
        """The library call itself (blocking while it polls convergence; report()
        covers what it does not poll); returns the sweeps it ran."""
        sweeps = ctypes.c_int(0)
        code = self.lib.mpsx_two_site_async(stream, tab.ctypes.data, dtab.data_ptr(), len(tab),
                                            ctypes.byref(cfg), ws.data_ptr(), ws.numel(),
                                            ctypes.byref(sweeps), self._late_ptr)
        if code == nat.MPSX_ENOTCONV:
            warnings.warn(nat.load().mpsx_last_error().decode(), nat.NotConvergedWarning)
        else:
            nat.check(code)
        return sweeps.value

    def two_site(self, items: Sequence[TwoSiteItem], svd: Optional[SvdConfig] = None
                 ) -> List[TwoSiteResult]:
        """Batched two-site updates on the current stream. A call with at
        least `split_min` problems of `split_rows` or more rows runs as
        `split_ways` groups of equal work concurrently, group 0 on the current
        stream and each other group from its own worker thread on its own
        helper stream: the latency-bound pivot eigensolves of one group then
        overlap the matrix-core phases of the others. Each problem's
        arithmetic is the same either way. Calls on other streams and from other
        threads are ordered: the workspaces are the engine's."""
        if len(items) == 0:
            return []
        self.report()
        with self._enqueue:
            cur = self.torch.cuda.current_stream(self.dev)
            stream = int(cur.cuda_stream)
            if stream != self._used_handle:
                self._take_workspaces(cur)
            try:
                return self._two_site(items, svd, cur, stream)
            finally:
                if stream:
                    self._leave_workspaces(cur)

    def _split_rule(self, cfg) -> Tuple[int, int]:
        """(split_min, split_rows) of a call. The direct solver's chain of steps leaves
        most of the device idle, so its calls are split early. Rounds fill it from
        about 256 rows on: 12 problems of 300 rows take 16.0 ms in one group and 19.7 in
        four (one-sided; FP32 14.1 and 17.3, mixed 11.2 and 12.2), 8 of 384 22.3 and
        27.5."""
        rule = (self.split_min, self.split_rows)
        if rule == self._split_stored and (cfg.method or cfg.rotation_fp32 or cfg.fp32_sweeps > 0 or cfg.block == 8):
            return self._split_rounds
        return rule

    def _fills(self, rows: Sequence[int]) -> bool:
        """Whether the direct solver's groups for the problems of more than 512 rows (a
        workgroup, on a compute unit of its own, for every 16 rows) fill the device:
        one launch is then the fastest (8 of 1024 rows 17.6 ms, 19 to 23 in four
        launches; 11 of 900 21.4 and 26). Not beside larger problems, whose rounds the
        other launches fill (5 of 1024 and 3 of 1200 rows: 73 ms, 69 in four)."""
        return max(rows) <= 1024 and sum(-(-r // 16) for r in rows if r > 512) >= self._cus

    def _two_site(self, items: Sequence[TwoSiteItem], svd: Optional[SvdConfig], cur, stream: int
                  ) -> List[TwoSiteResult]:
        n = len(items)
        cfg = (svd or self.svd).to_c()
        self._keep = []
        split_min, split_rows = self._split_rule(cfg)
        ways = max(1, min(int(self.split_ways), n))
        rows = [_rows(it) for it in items] if ways > 1 and cfg.check_every else []
        if not rows or sum(r >= split_rows for r in rows) < split_min or (
                split_rows < 512 and self._fills(rows)):
            outs, tab, dtab, ws = self._prepare_two_site(items, cfg, stream=stream)
            self._keep = [dtab]
            self.last_sweeps = self._run_two_site(tab, dtab, ws, cfg, stream)
            return outs
        # groups of equal estimated work (rows^2 * row length per problem),
        # largest problems first, each to the least loaded group
        order = sorted(range(n), key=lambda i: -_cost(items[i]))
        grp = [[] for _ in range(ways)]
        load = [0.0] * ways
        for i in order:
            g = min(range(ways), key=lambda x: load[x])
            grp[g].append(i)
            load[g] += _cost(items[i])
        grp = [sorted(g) for g in grp if g]
        preps = []
        for slot, g in enumerate(grp):
            c = cfg if slot == 0 else (svd or self.svd).to_c()
            preps.append((c,) + self._prepare_two_site([items[i] for i in g], c, slot, stream=stream))
        self._keep = [p[3] for p in preps]
        torch = self.torch
        from concurrent.futures import ThreadPoolExecutor
        while len(self._helpers) < len(grp) - 1:
            self._helpers.append((torch.cuda.Stream(self.dev), ThreadPoolExecutor(max_workers=1)))
        fork = torch.cuda.Event()
        fork.record(cur)
        dev = self.dev
        futs = []
        for slot in range(1, len(grp)):
            hs, pool = self._helpers[slot - 1]
            hs.wait_event(fork)  # inputs and outputs are ready on the helper stream
            c, outs_g, tab, dtab, ws = preps[slot]

            def run(c=c, tab=tab, dtab=dtab, ws=ws, hs=hs):
                torch.cuda.set_device(dev)
                return self._run_two_site(tab, dtab, ws, c, int(hs.cuda_stream))

            futs.append(pool.submit(run))
        c, _, tab, dtab, ws = preps[0]
        sweeps = [self._run_two_site(tab, dtab, ws, c, int(cur.cuda_stream))]
        sweeps += [f.result() for f in futs]
        for slot in range(1, len(grp)):
            join = torch.cuda.Event()
            join.record(self._helpers[slot - 1][0])
            cur.wait_event(join)
        self.last_sweeps = max(sweeps)
        outs: List[TwoSiteResult] = [None] * n
        for g, p in zip(grp, preps):
            for j, i in enumerate(g):
                outs[i] = p[1][j]
        return outs

    # ------------------------------------------------------------ gemm
    def gemm(self, ops: Sequence[dict]) -> None:
        """ops: dicts with A, B, C, m, n, k, lda, ldb, ldc, flags, alpha
        (complex). A, B and C are complex64 tensors, or (tensor, element
        offset) pairs for a matrix that starts inside a tensor. Every matrix
        is checked to lie inside its tensor before anything is launched."""
        if not ops:
            return
        if len(ops) > MAX_OPS:  # one launch takes at most MAX_OPS products
            for s in range(0, len(ops), MAX_OPS):
                self.gemm(ops[s:s + MAX_OPS])
            return
        self._launch_gemm(_gemm_rows(ops), (len(ops),))

    def _launch_gemm(self, rows: List[tuple], counts: Sequence[int]) -> None:
        """Grouped products one after the other from one table: the first counts[0]
        rows, the next counts[1], ..."""
        tab = np.array(rows, dtype=nat.GEMM_OP)
        stream = self.stream
        dtab = nat.put_table(tab, self.dev, stream)
        h, d = tab.ctypes.data, dtab.data_ptr()
        for c in counts:
            nat.check(self.lib.mpsx_gemm(stream, h, d, c))
            h += c * tab.itemsize
            d += c * tab.itemsize
        self._last_gemm_table = dtab

    # ------------------------------------------------------------ scale
    def scale(self, tensors: Sequence[object], factor: complex, conj: bool = False) -> None:
        if not tensors:
            return
        tab = np.zeros(len(tensors), dtype=nat.SCALE_OP)
        f = complex(factor)
        for i, t in enumerate(tensors):
            tab[i] = (nat.ptr(t), t.numel(), f.real, f.imag, 1 if conj else 0, 0)
        stream = self.stream
        dtab = nat.put_table(tab, self.dev, stream)
        nat.check(self.lib.mpsx_scale(stream, tab.ctypes.data, dtab.data_ptr(), len(tensors)))
        self._last_scale_table = dtab


class GemmChain:
    """Grouped products that depend on one another (the sweeps of the read-outs), in
    the order they are added: their descriptors travel together, one table for many
    launches, up to what one launch of mpsx_put carries. The operands of products
    not yet launched are kept alive, up to KEEP_BYTES of results. flush() launches
    the rest."""

    TABLE_ROWS = 40         # 3840 bytes of descriptors
    KEEP_BYTES = 64 << 20

    def __init__(self, eng: Engine):
        self.eng = eng
        self._rows: List[tuple] = []
        self._counts: List[int] = []
        self._ops: list = []
        self._bytes = 0

    def gemm(self, ops: Sequence[dict]) -> None:
        if not ops:
            return
        if len(ops) > MAX_OPS:
            for s in range(0, len(ops), MAX_OPS):
                self.gemm(ops[s:s + MAX_OPS])
            return
        if self._rows and len(self._rows) + len(ops) > self.TABLE_ROWS:
            self.flush()
        ops = list(ops)
        rows = _gemm_rows(ops)
        self._rows += rows
        self._counts.append(len(rows))
        self._ops.append(ops)
        self._bytes += 8 * sum(r[3] * r[4] for r in rows)
        if self._bytes > self.KEEP_BYTES:
            self.flush()

    def flush(self) -> None:
        if not self._rows:
            return
        self.eng._launch_gemm(self._rows, self._counts)
        self._rows, self._counts, self._ops, self._bytes = [], [], [], 0
