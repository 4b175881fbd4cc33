"""The MI355X backend: Anvil's kernel IR as one .hip file, compiled into a gfx950 shared library.

This is the HIP counterpart of the reference's CUDA backend (anvil/backend/cuda.py:636-663), with
the same plugin interface:

    generate(prog, seed=0, library=False) -> str        the whole .hip source
    build(source, lib_path)                              hipcc --offload-arch=gfx950 ... -shared
    load(prog, seed=0, library=False) -> HipLibrary      generate + build (cached) + ctypes

and a C ABI that the reference's library mode defines (aarch64.py:141-142, 162-167; pyapi.py:
266-296): `int anvil_entry(void)` and the `anvil_input<k>` / `anvil_output<k>` pointer slots, plus
`int anvil_main(void)` for a whole program (what `anvil run` executes).

How the program runs on the GPU:
  - every device buffer lives in one hipMalloc'ed arena, at offsets from a lifetime plan in which
    temporaries that are never live together share bytes (hip_analysis.plan_arena);
  - each IR kernel, or a run of kernels over the same rows, becomes one HIP kernel with a schedule
    chosen for its shape (hip_kernels: map, serial, rows, split; hip_gemm: fp32 MFMA products with
    the kernel's own statements as the epilogue);
  - loop counters and the scalars computed only from them stay on the host and reach kernels as
    arguments (hip_analysis.host_scalars), so a training loop enqueues work without waiting;
  - the host waits for the device only where it needs a device value (a print, an `if` on a device
    scalar, a data file, a checkpoint) and then reports the first bounds fault a kernel latched.

Generation is deterministic: the same program gives the same bytes, so built libraries are cached
by the hash of their source.
"""
from __future__ import annotations

import ctypes
import hashlib
import os
import shutil
import subprocess
import tempfile
import threading

from .. import ir
from ..ir import F32, I32, Buffer, KernelStmt
from . import hip_analysis as A
from . import hip_gemm
from . import hip_cost
from . import hip_kernels as HK
from .hip_emit import Emitter, Scope, c_string, ctype, flit, ilit, sanitize

HERE = os.path.dirname(os.path.abspath(__file__))
RUNTIME_DIR = os.path.join(HERE, "hip_rt")
ARCH = "gfx950"
FAULT_CODES = 254            # distinct fault messages with a code of their own
GENERIC_FAULT = "index out of bounds"


class HipToolchainError(Exception):
    pass


def runtime_source(attn_train: bool = False, split: bool = False, attn: bool = False) -> str:
    """anvil_rt.h and anvil_hip.h (and the MFMA templates; the split products', the attention's and
    the training attention's when a plan uses them), inlined: a generated file stands alone."""
    def read(name):
        with open(os.path.join(RUNTIME_DIR, name)) as f:
            return f.read().replace("#pragma once\n", "")
    rt = read("anvil_rt.h")
    dev = read("anvil_hip.h").replace('#include "anvil_rt.h"', rt)
    gemm_path = os.path.join(RUNTIME_DIR, "anvil_mfma.h")
    if os.path.exists(gemm_path):
        dev += "\n" + read("anvil_mfma.h")
        if split or attn:
            dev += "\n" + read("anvil_split.h")
        if attn:
            dev += "\n" + read("anvil_attn.h")
        if attn_train:
            dev += "\n" + read("anvil_attn_train.h")
    return dev


# ----------------------------------------------------------------------------- host-side scope

class HostScope(Scope):
    """A scalar kernel computed on the host from host scalars and constants."""

    device = False

    def __init__(self, gen):
        self.gen = gen

    def var(self, v):
        raise AssertionError("a host kernel has no loop variables")

    def buf(self, b):
        r = b.root
        if r.kind == "const" and r.init is not None:
            return f"anvil_init{r.id}"
        raise AssertionError(f"host kernel reads device buffer {r.name}")

    def host_scalar(self, b):
        if b.root.id in self.gen.hosts:
            return f"anvil_h{b.root.id}"
        return None

    def rand_index(self):
        return "0"

    def stream(self):
        return "0u"

    def seed(self):
        return "anvil_hs.seed"

    def fault(self, message):
        return self.gen.fault(message)


# ----------------------------------------------------------------------------- the generator

def source_line(span) -> str:
    """`file.anvil:line` of a span (the reference's Span or a fixture's recorded location)."""
    if span is None:
        return ""
    try:
        loc = span.location()
    except Exception:
        return ""
    parts = loc.rsplit(":", 2)
    return f"{os.path.basename(parts[0])}:{span.line}" if len(parts) == 3 and span.line is not None else ""


def profile_row(p) -> str:
    """The reference's --profile row text for a launch (aarch64.py:877-881): its name in 6 columns,
    what it computes (the labels of its IR kernels joined by '+') cut to 34, its first source line."""
    label = "+".join(k.label or "kernel" for k in p.kernels) or p.kind
    loc = next((source_line(k.span) for k in p.kernels if source_line(k.span)), "")
    return f"{p.name:<6} {label[:34]:<34} {loc}"


def packs_of(plan) -> list:
    """The operand copies (hip_conv.PackPlan) that must run before `plan` or one of its parts."""
    return [p.pack for p in getattr(plan, "parts", [plan]) if getattr(p, "pack", None) is not None]


class HipGen:
    def __init__(self, prog: ir.Program, seed: int = 0, library: bool = False, emulate: bool = False,
                 graphs: bool = False, check: str | None = None):
        # --check: one launch per IR kernel, in program order, each followed by a scan of what it
        # wrote (no fusion, no reordering, no graphs: the first bad value is pinned to one kernel)
        self.check = check
        if check:
            graphs = False
        # temporaries that are a cheap elementwise function of another buffer: recomputed where
        # they are read (the CPU build too, so the CPU tests run the rewritten program)
        if not check and os.environ.get("ANVIL_HIP_REMAT", "1") != "0":
            prog = A.rematerialize(prog)
        if not emulate and not check and os.environ.get("ANVIL_HIP_SINK", "1") != "0":
            prog = A.sink_scalar_kernels(prog)
        if not emulate and not check and os.environ.get("ANVIL_HIP_GATHER_FWD", "1") != "0":
            from . import hip_gemm
            prog = hip_gemm.forward_gather_copies(prog, A.host_scalars(prog))
        # the loop variables the passes add take ids after the program's own
        self.ids = A.IdSource(prog)
        if not check and os.environ.get("ANVIL_HIP_IMPLICIT_CONV", "1") != "0":
            from . import hip_conv
            prog = hip_conv.forward_im2col_copies(prog, self.ids)
        self.prog = prog
        self.seed = seed & 0xFFFFFFFF
        self.library = library
        self.emulate = emulate
        self.hosts = A.host_scalars(prog)
        self.readers = A.all_readers(prog)
        self.attn_train: dict = {}          # first kernel id -> (plan, statements) of a training-attention chain
        self.graphs = graphs
        self.dev_hosts = self.device_visible_hosts() if graphs else set()
        self.hsd = {bid: i for i, bid in enumerate(sorted(self.dev_hosts))}
        self.twins: dict = {}             # host kernel id -> its device twin plan
        self.segments: list = []          # C functions of graph segments
        self.by_id = {b.root.id: b.root for b in prog.buffers}
        self.faults: list[str] = []          # message of latch code i + 1
        self.fault_codes: dict = {}           # message -> latch code
        self.tables: list[str] = []
        self.plans: list = []
        self.plan_of: dict = {}           # first kernel id -> plan (a run of kernels shares one)
        self.ahead: dict = {}             # first kernel id -> (plan, statements) planned before its turn
        self.group_of: dict = {}          # kernel id -> the launch (plan) it is part of
        self.part_of: dict = {}           # kernel id -> the kernel (plan) of that launch it is a stage of
        self.device_bufs: dict[int, Buffer] = {}
        self.mirrored: dict[int, Buffer] = {}
        self.ckpts: list[str] = []
        self.n_labels = 0
        self.gemm = None
        if not emulate:
            try:
                from . import hip_gemm
                self.gemm = hip_gemm
            except ImportError:
                self.gemm = None

    def device_visible_hosts(self) -> set:
        """Host scalars kernels read, and (closing over the host's scalar kernels that compute
        them) everything those are computed from: the device keeps its own copy of these."""
        out: set = set()
        host_ks = []
        for k in ir.all_kernels(self.prog):
            if A.is_host_kernel(k, self.hosts):
                host_ks.append(k)
            else:
                out |= {b.id for b in A.kernel_reads(k) if b.id in self.hosts}
        grown = True
        while grown:
            grown = False
            for k in host_ks:
                if {st.buf.root.id for st in k.stores} & out:
                    more = {b.id for b in A.kernel_reads(k) if b.id in self.hosts} - out
                    if more:
                        out |= more
                        grown = True
        return out

    def hsd_slot(self, b) -> int:
        r = b.root
        if r.id not in self.hsd:
            raise AssertionError(f"host scalar {r.name} is read on the device but has no device copy")
        return self.hsd[r.id]

    def twin_of(self, k):
        """The device twin of a host kernel that computes device-visible scalars, or None."""
        if not self.graphs or not ({st.buf.root.id for st in k.stores} & self.dev_hosts):
            return None
        t = self.twins.get(k.id)
        if t is None:
            t = self.twins[k.id] = HK.TwinPlan(self, k, f"tw{k.id}")
            self.plans.append(t)
        return t

    # ------------------------------------------------------------------ small helpers
    def fault(self, message: str) -> int:
        """The latch code (1, 2, ...) kernels report `message` by. The runtime's text table has 256
        entries (code 0 is no fault), so once FAULT_CODES messages have codes, a new message shares
        the generic bounds message's code (which then takes one more entry if it had none)."""
        codes = self.fault_codes
        if message not in codes and len(codes) >= FAULT_CODES:
            message = GENERIC_FAULT
        if message not in codes:
            self.faults.append(message)
            codes[message] = len(self.faults)
        return codes[message]

    def label(self, hint: str) -> str:
        self.n_labels += 1
        return f"{hint}{self.n_labels}"

    def table(self, ctype_: str, items) -> str:
        name = self.label("anvil_tab")
        self.tables.append(f"static const {ctype_} {name}[] = {{{', '.join(items) or '0'}}};")
        return name

    def strings(self, strs) -> str:
        return self.table("char *const", [c_string(s) for s in strs])

    def is_host(self, b) -> bool:
        return b.root.id in self.hosts

    def dev(self, b) -> str:
        """Host code: the device pointer of a buffer."""
        r = b.root
        self.device_bufs.setdefault(r.id, r)
        return f"anvil_b{r.id}"

    def mirror(self, b) -> str:
        r = b.root
        self.dev(r)
        self.mirrored.setdefault(r.id, r)
        return f"anvil_mir{r.id}"

    def host_view(self, b) -> str:
        """Host code: a host pointer holding b's current contents (fetching it if needed)."""
        r = b.root
        if self.is_host(r):
            return f"(&anvil_h{r.id})"
        return f"(({ctype(r.dtype)} *)anvil_fetch(&{self.mirror(r)}))"

    def scalar_value(self, b) -> str:
        r = b.root
        if self.is_host(r):
            return f"anvil_h{r.id}"
        return f"anvil_read_{'i32' if r.dtype == I32 else 'f32'}({self.dev(r)})"

    # ------------------------------------------------------------------ planning kernels
    def plan_run(self, stmts: list, i: int):
        """The plan for the kernel at stmts[i] and how many statements it takes."""
        if self.check:
            return self.plan_one(stmts, i)
        if not self.emulate and os.environ.get("ANVIL_HIP_ATTN", "1") != "0":
            from . import hip_attn, hip_attn_train
            at = hip_attn.match(self, stmts, i)
            if at is not None:
                return at, 6
            got = hip_attn_train.match(self, stmts, i)
            if got is not None:
                return got
        from . import hip_conv
        from . import hip_rowpro
        got = hip_conv.match_dgrad(self, stmts, i) or hip_rowpro.match(self, stmts, i) or self.row_block(stmts, i)
        if got is not None:
            return got
        return self.plan_one(stmts, i)

    def row_block(self, stmts: list, i: int):
        """A RowBlockPlan for the chain of row-by-row kernels starting at stmts[i], if the chain
        would otherwise take two launches or more."""
        if self.emulate or os.environ.get("ANVIL_HIP_ROWBLOCK", "1") == "0":
            return None
        k = stmts[i].kernel
        if not k.domain or not 64 <= k.domain[0].extent <= 4096:
            return None
        prior = {b.id for st in stmts[:i] if isinstance(st, KernelStmt) for b in A.kernel_writes(st.kernel)}
        rb = HK.RowBlockBuilder(k.domain[0].extent, prior)
        j = i
        while j < len(stmts) and isinstance(stmts[j], KernelStmt) and rb.fits(stmts[j].kernel, self.hosts):
            j += 1
        if j - i < 2:
            return None
        # only a chain: some stage reads what an earlier one wrote (independent kernels are
        # better served side by side, each with its own schedule)
        written: set = set()
        chained = False
        for kk in rb.kernels:
            if {b.id for b in A.kernel_reads(kk)} & written:
                chained = True
            written |= {b.id for b in A.kernel_writes(kk)}
        if not chained:
            return None
        launches, t = 0, i
        while t < j:
            p, used = self.plan_one(stmts, t)
            if (p.kind == "gemm" and p.s.K >= 64) or p.kind == "split":
                # a real product, or a strided reduction: it keeps its schedule, and the chain, if
                # long enough, stops before it
                if os.environ.get("ANVIL_HIP_ROWBLOCK_CUT", "1") == "0" or t - i < 2:
                    return None
                j = t
                rb = HK.RowBlockBuilder(k.domain[0].extent, prior)
                for kk in [st.kernel for st in stmts[i:j]]:
                    if not rb.fits(kk, self.hosts):
                        return None
                break
            launches += 1
            t += used
        if launches < 2:
            return None
        return HK.RowBlockPlan(self, rb.kernels, f"k{k.id}", rb.R, before=rb.before), j - i

    def plan_one(self, stmts: list, i: int):
        k = stmts[i].kernel
        name = f"k{k.id}"
        parallel = A.parallel_safe(k)
        if not parallel:
            return HK.SerialPlan(self, k, name), 1
        if k.red is None:
            scat = HK.scatter_targets(k)
            if scat is not None:
                return HK.GatherSumPlan(self, k, name, *scat), 1
            rows = None if self.emulate or self.check else HK.index_scatter(k)
            if rows is not None and os.environ.get("ANVIL_HIP_INDEX_SCATTER", "1") != "0":
                return HK.IndexScatterPlan(self, k, name, *rows), 1
            plan = HK.MapPlan(self, k, name)
            if self.check or os.environ.get("ANVIL_HIP_MAP_FUSE", "1") == "0":
                return plan, 1
            return plan, 1 + self.absorb_followers(plan, stmts, i + 1)
        if self.gemm is not None:
            g = self.gemm.match(self, k, name)
            if g is not None:
                if os.environ.get("ANVIL_GEMM_FUSE", "1") == "0" or self.check:   # no epilogue fusion
                    g.settle()
                    return g, 1
                used = 1 + self.absorb_followers(g, stmts, i + 1)
                g.settle()
                return g, used
        pool = HK.PoolPlan.match(self, k)
        if pool is not None:
            return pool, 1
        sl = HK.slice_count(k, self.emulate)
        if sl > 1:
            return HK.SlicePlan(self, k, name, sl), 1
        ty = HK.split_ways(k, self.emulate)
        if ty > 1:
            return HK.SplitPlan(self, k, name, ty), 1
        if k.red.op in ("argmax", "argmin") or any(st.accumulate for st in k.stores):
            return HK.RowsPlan(self, [k], name, HK.rows_lanes(k, self.emulate), self.emulate), 1
        gb = HK.GroupBuilder(k)
        j = i + 1
        while (not self.check and j < len(stmts) and isinstance(stmts[j], KernelStmt)
               and gb.fits(stmts[j].kernel, self.hosts)):
            gb.add(stmts[j].kernel)
            j += 1
        plan = HK.RowsPlan(self, gb.kernels, name, HK.rows_lanes(k, self.emulate), self.emulate)
        self.mark_dead_stores(plan)
        return plan, j - i

    def exit_if(self, st) -> bool:
        """An `if` on a host scalar whose only effect is to leave the loop (or iteration)."""
        return (isinstance(st, ir.If) and st.cond.root.id in self.hosts and not st.orelse.stmts
                and len(st.then.stmts) == 1 and isinstance(st.then.stmts[0], (ir.Break, ir.Continue)))

    def can_fixup(self, plan) -> bool:
        """May the K splits of this launch (products, alone or side by side with other parts) add
        their partial tiles in their own last workgroup per tile? If so, mark them. Only with
        $ANVIL_GEMM_FIXUP=1: the device-wide release and acquire around the count (an L2 write-back
        by every workgroup, an L2 invalidation by each tile's last) measured slower than the second
        launch they save (C5 184.3 -> 208.7 us per step, C4 at T = 256 1376 -> 1408 us)."""
        split = [p for p in getattr(plan, "parts", [plan]) if getattr(p, "kslices", 1) > 1]
        if (not split or any(p.kind != "gemm" for p in split) or getattr(plan, "two_launches", False)
                or self.emulate or self.check or os.environ.get("ANVIL_GEMM_FIXUP", "0") != "1"):
            return False
        for p in split:
            p.fixup = True
            p.__dict__.pop("_source", None)             # (an LDS or barrier check may have made it)
        plan.__dict__.pop("_source", None)
        return True

    def place_pack(self, pack, seg, ind):
        """Launch operand copy `pack` before the plan that reads it: as one more part of the launch
        just before (seg's last entry), when that launch runs right before it, is not a serial or
        lone kernel, has no second launch, does not write what the copy reads and has room for a
        part; else alone."""
        pack.own = None
        prev = seg[-1] if seg and seg[-1][0] == "launch" else None
        P = prev[2] if prev is not None else None
        ok = (P is not None and P in self.plans and not self.emulate and not self.check
              and os.environ.get("ANVIL_HIP_SIDE", "1") != "0"
              and P.kind not in ("serial", "pack") and not getattr(P, "alone", False)
              and getattr(P, "exit", None) is None and getattr(P, "kslices", 1) == 1
              and not getattr(P, "two_launches", False) and not getattr(P, "joined", None)
              and len(getattr(P, "parts", [P])) < int(os.environ.get("ANVIL_HIP_SIDE_PARTS", "8"))
              and pack.src.root.id not in {b.root.id for k in P.kernels for b in A.kernel_writes(k)})
        if ok:
            q = pack.with_threads(P.grid()[1])
            if P.kind == "fused":
                new = HK.FusedPlan(self, P.parts + [q], P.name, P.hoisted)
                new.joined_reads = set(P.joined_reads)
            else:
                new = HK.FusedPlan(self, [P, q], "f" + P.name, list(getattr(P, "hoisted", [])))
            self.plans[self.plans.index(P)] = new
            for key, val in list(self.plan_of.items()):
                if val[0] is P:
                    self.plan_of[key] = (new, val[1])
            for key, val in list(self.group_of.items()):
                if val is P:
                    self.group_of[key] = new
            seg[-1] = ("launch", self.launch(new, ind), new)
            return
        pack.own = pack
        self.plans.append(pack)
        seg.append(("launch", self.launch(pack, ind), pack))

    def side_by_side(self, stmts, i, plan, used):
        """Join the launches after `plan` that are independent of it (and of each other) into one
        FusedPlan. Host scalar kernels between them then run before the launch: only if no part
        before them reads what they write. Parts must agree on the workgroup size (a split kernel
        is re-planned to it) unless they have no barrier; their LDS adds up.

        The scan may cross one `if (host scalar) break;` (a step limit checked after the batch is
        gathered): the launch then goes after the check, and the leaving path launches the parts
        that came before the check on their own, so they run exactly when they did."""
        if self.emulate or self.check or os.environ.get("ANVIL_HIP_SIDE", "1") == "0" or getattr(plan, "alone", False):
            return plan, used
        ids = lambda bs: {b.root.id for b in bs}

        def rw(p):
            r, w = set(), set()
            for k in p.kernels:
                r |= ids(A.kernel_reads(k))
                w |= ids(A.kernel_writes(k))
            return r, w
        parts = [plan]
        hoisted = list(getattr(plan, "hoisted", []))
        reads, writes = rw(plan)
        threads = plan.grid()[1]
        j = i + used
        taken = used
        between: list = []
        exit_at = None      # (the if, parts before it, host kernels hoisted before it, the ones after it)
        most = int(os.environ.get("ANVIL_HIP_SIDE_PARTS", "8"))
        while j < len(stmts) and len(parts) < most:
            st = stmts[j]
            if (exit_at is None and not self.graphs and self.exit_if(st)
                    and os.environ.get("ANVIL_HIP_EXIT", "1") != "0"):
                exit_at = (st, len(parts), list(hoisted), list(between))
                between = []
                j += 1
                continue
            if not isinstance(st, KernelStmt):
                break
            k = st.kernel
            if A.is_host_kernel(k, self.hosts):
                between.append(k)
                j += 1
                continue
            cand, cused = self.plan_run(stmts, j)
            if cand.kind in ("serial", "fused") or getattr(cand, "alone", False) or packs_of(cand):
                break                                   # (an operand copy must run before the plan)
            if getattr(cand, "kslices", 1) > 1 and exit_at is not None:
                break                                   # its second launch follows the fused one
            # (a shared tile beside another product has its LDS and registers for both, fewer workgroups to a CU
            # than its own allow: a call of a layer's backward, 2000 x 1000 x 600, 71.4 us apart, 85.5 side by
            # side; a decoder layer's step of 16 x 256 x 256 319 and 314)
            gemms = [p for p in parts + [cand] if p.kind in ("gemm", "conv-dgrad")]
            if len(gemms) > 1 and any(getattr(p, "sched", "") == "tile" for p in gemms):
                break
            moved = between + list(getattr(cand, "hoisted", []))
            if {st2.buf.root.id for h in moved for st2 in h.stores} & reads:
                break
            cr, cw = rw(cand)
            if cw & (reads | writes) or cr & writes:
                break
            t = max(threads, cand.grid()[1])
            fixed = []
            for p in parts + [cand]:
                if p.grid()[1] == t or HK.barrier_free(p):
                    fixed.append(p)
                elif p.kind == "split" and t % p.TY == 0:
                    q = HK.SplitPlan(self, p.k, p.name, p.TY, threads=t)
                    q.skip_stores = p.skip_stores
                    fixed.append(q)
                else:
                    break
            if len(fixed) < len(parts) + 1:
                break
            if HK.fused_lds(fixed) > 96 * 1024:
                break
            parts, threads = fixed, t
            hoisted += moved
            between = []
            reads |= cr
            writes |= cw
            j += cused
            taken = j - i
        if exit_at is not None and any(getattr(p, "kslices", 1) > 1 for p in parts):
            return plan, used                           # the leaving path would need the second launch too
        if exit_at is not None and len(parts) == exit_at[1]:
            hoisted = exit_at[2]                        # nothing joined past the check: stop before it
            exit_at = None
        if len(parts) == 1:
            return plan, used
        if exit_at is None:
            return HK.FusedPlan(self, parts, "f" + plan.name, hoisted), taken
        st, n_pre, before, pre_hosts = exit_at
        pre = parts[:n_pre]
        pre_plan = pre[0] if len(pre) == 1 else HK.FusedPlan(self, pre, "e" + plan.name, [])
        pre_hoist = before + pre_hosts
        post_hoist = hoisted[len(before):]
        fused = HK.FusedPlan(self, parts, "f" + plan.name, pre_hoist + post_hoist)
        fused.exit = (st, pre_plan, pre_hoist, post_hoist)
        return fused, taken

    def join_second(self, stmts, j, first, second) -> bool:
        """Does `second` (the launch that adds a K split's partial tiles or a reduction's slices,
        then runs the kernel's statements: a weight update) run side by side with the next launch,
        the one for stmts[j], instead of alone? Only if what lies between is host scalar kernels
        that write nothing the first launch's kernels read (nor do the next launch's hoisted ones),
        no data passes between the two launches, and their lanes and LDS fit one launch. The next
        launch's parts come first in the grid, the second launch's workgroups after them; the
        buffers the first launch's kernels read are noted as read by the joined launch, so that
        their bytes stay theirs up to it. The next statement's plan is made here and kept for its
        turn either way."""
        if (self.emulate or self.check or os.environ.get("ANVIL_HIP_SIDE", "1") == "0"
                or os.environ.get("ANVIL_HIP_JOIN", "1") == "0" or second.streams or getattr(second, "alone", False)):
            return False
        between = []
        while j < len(stmts) and isinstance(stmts[j], KernelStmt) and A.is_host_kernel(stmts[j].kernel, self.hosts):
            between.append(stmts[j].kernel)
            j += 1
        if j >= len(stmts) or not isinstance(stmts[j], KernelStmt):
            return False
        k = stmts[j].kernel
        if k.id in self.plan_of or k.id in self.ahead:
            return False
        nxt, used = self.plan_run(stmts, j)
        nxt, used = self.side_by_side(stmts, j, nxt, used)
        self.ahead[k.id] = (nxt, used)
        if (nxt.kind == "serial" or getattr(nxt, "alone", False) or getattr(nxt, "exit", None) is not None
                or getattr(nxt, "two_launches", False) or packs_of(nxt)):
            return False
        ids = lambda bs: {b.root.id for b in bs}
        sr, sw = set(), set()
        for kk in first.kernels:
            sr |= ids(A.kernel_reads(kk))
            sw |= ids(A.kernel_writes(kk))
        nr, nw = set(), set()
        for kk in nxt.kernels:
            nr |= ids(A.kernel_reads(kk))
            nw |= ids(A.kernel_writes(kk))
        moved = between + list(getattr(nxt, "hoisted", []))
        if {st.buf.root.id for h in moved for st in h.stores} & sr or sw & (nr | nw) or sr & nw:
            return False
        parts = list(nxt.parts) if nxt.kind == "fused" else [nxt]
        parts += list(second.parts) if second.kind == "fused" else [second]
        t = max(p.grid()[1] for p in parts)
        if any(p.grid()[1] != t and not HK.barrier_free(p) for p in parts):
            return False
        if HK.fused_lds(parts) > 96 * 1024:
            return False
        joined = HK.FusedPlan(self, parts, nxt.name if nxt.kind == "fused" else "f" + nxt.name,
                              list(getattr(nxt, "hoisted", [])))
        joined.joined_reads = {b for kk in first.kernels for b in A.kernel_reads(kk)}
        self.ahead[k.id] = (joined, used)
        return True

    def absorb_followers(self, plan, stmts, j) -> int:
        """Elementwise kernels right after a product (past host-only scalar kernels, which are then
        computed before the launch) that can run in its epilogue; returns the statements taken."""
        taken = 0
        hoist = []
        k = plan.kernels[0]
        reads_k = {b.id for b in A.kernel_reads(k)}
        while j + taken < len(stmts) and isinstance(stmts[j + taken], KernelStmt):
            e = stmts[j + taken].kernel
            if A.is_host_kernel(e, self.hosts):
                if {st.buf.root.id for st in e.stores} & reads_k:
                    break
                hoist.append(e)
                taken += 1
                continue
            prior = [(f, fm) for f, fm, _ in getattr(plan, "followers", [])]
            how = hip_gemm.follower(k, e, self.hosts, prior)
            if how is None or plan.absorb(e, how) is False:
                break
            taken += 1
            plan.hoisted = list(getattr(plan, "hoisted", [])) + hoist
            hoist = []
            if len(plan.kernels) >= 3:
                break
        taken -= len(hoist)                             # host kernels after the last follower stay put
        if len(plan.kernels) > 1:
            self.mark_dead_stores(plan)
        return taken

    def mark_dead_stores(self, plan):
        """Stores of a row group whose buffer only the group reads (from registers) are dropped."""
        if len(plan.kernels) < 2:
            return
        readers_in: dict[int, int] = {}
        for k in plan.kernels:
            for b in A.kernel_reads(k):
                readers_in[b.id] = readers_in.get(b.id, 0) + 1
        if plan.kind in ("gemm", "map"):
            k = plan.kernels[0]
            for i, st in enumerate(k.stmts):
                if not isinstance(st, ir.Store):
                    continue
                b = st.buf.root
                if b.kind not in A.SHARED_KINDS or self.is_host(b) or getattr(b, "heap", False):
                    continue
                # dead: the product itself does not read it, and only its followers (from registers) do
                if b not in A.kernel_reads(k) and self.readers.get(b.id, 0) == readers_in.get(b.id, 0):
                    plan.skip_stores.add((k.id, i))
            return
        for k in plan.kernels:
            cm = plan.canon_map(k)
            _, inner = plan.stage_vars(k)
            for i, st in enumerate(k.stmts):
                if not isinstance(st, ir.Store):
                    continue
                b = st.buf.root
                if b.kind not in A.SHARED_KINDS or self.is_host(b) or getattr(b, "heap", False):
                    continue
                if self.readers.get(b.id, 0) != readers_in.get(b.id, 0):
                    continue
                key = HK.canon_key(st.buf, st.offset, cm)
                element = k.red is None and bool(inner)
                if key is None or (element and key not in plan.cache_arrays):
                    continue
                plan.skip_stores.add((k.id, i))

    # ------------------------------------------------------------------ host code
    def block(self, blk: ir.Block, ind: str, in_loop: bool = False, tail=None) -> list[str]:
        """Host code of a block. In a loop body, each straight run of kernels (device launches and
        the host's scalar kernels) becomes a graph segment. `tail`: launch lines to run at the end
        of the block (a loop counter's twin), put inside the last segment when it ends the block;
        self.tail_used says whether that happened."""
        out = []
        seg: list = []                  # (kind, lines, plan) of the pending run
        stmts = blk.stmts
        self.tail_used = False

        def flush(last: bool):
            if not seg:
                return
            if last and tail is not None and in_loop and self.graphs:
                seg.append(("twin", tail, None))
                self.tail_used = True
            launches = sum(1 for kind, _, _ in seg if kind != "host")
            rand = any(p is not None and p.streams for _, _, p in seg)
            if in_loop and self.graphs and launches >= 2 and not rand:
                out.extend(self.segment(seg, ind))
            else:
                for _, lines, _ in seg:
                    out.extend(lines)
            seg.clear()

        i = 0
        while i < len(stmts):
            st = stmts[i]
            if isinstance(st, KernelStmt):
                k = st.kernel
                if A.is_host_kernel(k, self.hosts):
                    seg.append(("host", self.host_kernel(k, ind), None))
                    twin = self.twin_of(k)
                    if twin is not None:
                        seg.append(("twin", self.launch(twin, ind), twin))
                    if self.check:
                        seg.append(("host", self.check_lines(k, ind), None))
                    i += 1
                    continue
                plan = self.plan_of.get(k.id)
                if plan is None:
                    if k.id in self.ahead:
                        plan, used = self.ahead.pop(k.id)       # planned by join_second
                    else:
                        plan, used = self.plan_run(stmts, i)
                        plan, used = self.side_by_side(stmts, i, plan, used)
                    if getattr(plan, "exit", None) is not None:
                        self.plans.append(plan.exit[1])
                    for pack in packs_of(plan):
                        self.place_pack(pack, seg, ind)
                    self.plans.append(plan)
                    self.plan_of[k.id] = (plan, used)
                    for part in getattr(plan, "parts", [plan]):
                        for kk in part.kernels:
                            self.group_of[kk.id] = plan
                            self.part_of[kk.id] = part
                else:
                    plan, used = plan
                    for pack in packs_of(plan):
                        if pack.own:                    # (a copy fused into an earlier launch runs there)
                            seg.append(("launch", self.launch(pack.own, ind), pack.own))
                exit_ = getattr(plan, "exit", None)
                if exit_ is not None:
                    # the host's scalar kernels before the check, the check (whose leaving path
                    # launches what came before it), the ones after it, then the whole launch
                    st_if, pre_plan, pre_hoist, post_hoist = exit_
                    for hk in pre_hoist:
                        seg.append(("host", self.host_kernel(hk, ind), None))
                    leave = "break;" if isinstance(st_if.then.stmts[0], ir.Break) else "continue;"
                    seg.append(("host", [f"{ind}if ({self.scalar_value(st_if.cond)} != 0) {{"]
                                + self.launch(pre_plan, ind + "    ") + [f"{ind}    {leave}", f"{ind}}}"], None))
                    for hk in post_hoist:
                        seg.append(("host", self.host_kernel(hk, ind), None))
                else:
                    for hk in getattr(plan, "hoisted", []):
                        seg.append(("host", self.host_kernel(hk, ind), None))
                        twin = self.twin_of(hk)
                        if twin is not None:
                            seg.append(("twin", self.launch(twin, ind), twin))
                split = getattr(plan, "kslices", 1) > 1 or getattr(plan, "two_launches", False)
                if split and not hasattr(plan, "reduce_plan"):
                    # a K split across workgroups: its sum; or the plan's own second launch. The sum
                    # joins the next launch when it can (else, with $ANVIL_GEMM_FIXUP=1, the product
                    # adds its partial tiles in its own last workgroup per tile)
                    plan.reduce_plan = plan.second()
                    plan.reduce_plan.joined = self.join_second(stmts, i + used, plan, plan.reduce_plan)
                    if not plan.reduce_plan.joined and self.can_fixup(plan):
                        plan.fixup = True
                    elif not plan.reduce_plan.joined:
                        self.plans.append(plan.reduce_plan)
                seg.append(("launch", self.launch(plan, ind), plan))
                if split and not plan.reduce_plan.joined and not getattr(plan, "fixup", False):
                    seg.append(("launch", self.launch(plan.reduce_plan, ind), plan.reduce_plan))
                if self.check:
                    for kk in plan.kernels:
                        seg.append(("host", self.check_lines(kk, ind), None))
                i += used
                continue
            flush(False)
            out += self.stmt(st, ind)
            i += 1
        flush(True)
        if tail is not None and not self.tail_used:
            out.extend(tail)
            self.tail_used = True
        return out

    def check_lines(self, k: ir.Kernel, ind: str) -> list[str]:
        """--check after kernel k: each f32 tensor it wrote (the caller's arrays aside), with the
        tensors it read as the inputs the report counts nans and infinities in (aarch64.py:459-481)."""
        written = []
        for st in k.stores:
            b = st.buf.root
            if b.dtype == F32 and b.kind not in ir.EXTERN_KINDS and not getattr(b, "heap", False) and b not in written:
                written.append(b)
        if not written:
            return []
        reads: set = set()
        for e in k.exprs():
            for ld in ir.loads_in(e):
                reads.add(ld.buf.root)
        for st in k.stores:
            if st.accumulate:
                reads.add(st.buf.root)
            for g in st.offset.gathers():
                reads.add(g.load.buf.root)
        inputs = [b for b in sorted(reads, key=lambda b: b.id)
                  if b.dtype == F32 and b not in written and b.kind not in ir.EXTERN_KINDS
                  and not getattr(b, "heap", False) and b.numel > 0]
        desc = c_string(getattr(k, "desc", None) or self.describe(k))
        mode = 2 if self.check == "inf" else 1

        def where(b):
            return (f"&anvil_h{b.id}", 1) if self.is_host(b) else (self.dev(b), 0)
        out = []
        for b in written:
            name = f"`{b.name}` ({b.dtype}{list(b.shape)})" if b.shape else f"`{b.name}` (an f32 scalar)"
            ptr, host = where(b)
            ins = [f"{{{where(x)[0]}, {x.numel}LL, {where(x)[1]}, {c_string('`' + x.name + '`')}}}" for x in inputs]
            dims = ", ".join(f"{d}LL" for d in b.shape) or "0LL"
            out.append(f"{ind}{{   // --check {b.name}")
            out.append(f"{ind}    static const long long dims_[] = {{{dims}}};")
            out.append(f"{ind}    static const anvil_check_input ins_[] = {{{', '.join(ins) or '{NULL, 0LL, 0, NULL}'}}};")
            out.append(f"{ind}    anvil_check({ptr}, {b.numel}LL, {mode}, {host}, {c_string(name)}, dims_, {len(b.shape)}, "
                       f"{desc}, ins_, {len(inputs)});")
            out.append(f"{ind}}}")
        return out

    @staticmethod
    def describe(k: ir.Kernel) -> str:
        """Where a kernel comes from (aarch64.py:82-89), when the program did not record it."""
        head = f"  made by `{k.label or 'a computation'}`"
        line = ""
        span = k.span
        if span is not None and span.location():
            head += f" at {span.location()}"
            text = getattr(span, "src", None)
            if text is None and getattr(span, "file", None) is not None:
                text = span.file.line_text(span.line).strip()      # a front-end span (source.py)
            if text:
                line = "\n      " + text
        return f"{head}:{line}\n  computing ({k.name}):  {ir.fmt_kernel(k)}"

    def segment(self, seg: list, ind: str) -> list[str]:
        """A graph segment: a function that records the run (host kernels, twins, launches) and one
        that does only the host's part, for replays."""
        n = len(self.segments)
        rec = [f"static void anvil_seg{n}_record(void) {{"]
        host = [f"static void anvil_seg{n}_host(void) {{"]
        for kind, lines, _ in seg:
            rec.extend(lines)
            if kind == "host":
                host.extend(lines)
            else:
                host.extend(line for line in lines if line.startswith("@@dirty "))
        self.segments.append(rec + ["}"] + host + ["}"])
        return [f"{ind}anvil_segment_run(&anvil_seg{n}, anvil_seg{n}_record, anvil_seg{n}_host);"]

    def host_kernel(self, k: ir.Kernel, ind: str) -> list[str]:
        lines = [f"{ind}{{   // {k.name}: on the host"]
        em = Emitter(HostScope(self), lines, ind + "    ")
        for st in k.stmts:
            if isinstance(st, ir.Let):
                em.let(st)
                continue
            val = em.store_value(st)
            em.emit(f"anvil_h{st.buf.root.id} = {val};")
            em.reset_memo()
        lines.append(f"{ind}}}")
        return lines

    def launch(self, plan, ind: str) -> list[str]:
        out = [f"{ind}{{   // {plan.label}"]
        streams = []
        for n, _ in enumerate(plan.streams):
            out.append(f"{ind}    const uint32_t s{n} = anvil_hs.stream++;")
            streams.append(f"s{n}")
        if not hasattr(plan, "_source"):
            plan._source = plan.source()
        site = self.plans.index(plan)
        blocks, threads = plan.grid()
        args = plan.launch_args(streams)
        for b in plan.bufs.values():
            self.dev(b)
        go = "ANVIL_GO3" if isinstance(blocks, tuple) else "ANVIL_GO"
        grid = ", ".join(str(x) for x in blocks) if isinstance(blocks, tuple) else str(blocks)
        out.append(f"{ind}    anvil_prof_enter({site});")
        out.append(f"{ind}    {go}({plan.name}, {grid}, {threads}, {', '.join(args)});")
        out.append(f"{ind}    anvil_prof_leave();")
        for b in sorted(plan.writes(), key=lambda b: b.id):
            out.append(f"@@dirty {b.id} {ind}    ")
        out.append(f"{ind}}}")
        return out

    def stmt(self, st, ind: str) -> list[str]:
        if isinstance(st, ir.For):
            return self.for_(st, ind)
        if isinstance(st, ir.While):
            out = [f"{ind}while (1) {{"] + self.block(st.cond_block, ind + "    ", in_loop=True)
            out.append(f"{ind}    if ({self.scalar_value(st.cond)} == 0) break;")
            return out + self.block(st.body, ind + "    ", in_loop=True) + [f"{ind}}}"]
        if isinstance(st, ir.If):
            out = [f"{ind}if ({self.scalar_value(st.cond)} != 0) {{"] + self.block(st.then, ind + "    ")
            if st.orelse.stmts:
                out += [f"{ind}}} else {{"] + self.block(st.orelse, ind + "    ")
            return out + [f"{ind}}}"]
        if isinstance(st, ir.Break):
            return [f"{ind}break;"]
        if isinstance(st, ir.Continue):
            return [f"{ind}continue;"]
        if isinstance(st, ir.Print):
            return self.print_(st, ind)
        if isinstance(st, ir.Check):
            loc = f"{st.span.location()}: " if st.span is not None and st.span.location() else ""
            terms = [f"{c}LL * (long long){self.scalar_value(t.buf)}" for t, c in st.value.terms.items()
                     if isinstance(t, ir.ScalarRef)]
            v = " + ".join([f"{st.value.const}LL"] + terms)
            return [f"{ind}{{ const long long v_ = {v};",
                    f"{ind}  if (v_ < {st.lo}LL || v_ > {st.hi}LL) {{ anvil_sync(); "
                    f"anvil_bad_value({c_string(loc + st.message)}, v_); }} }}"]
        if isinstance(st, ir.RTCall):
            return [ind + line for line in self.rtcall(st)]
        raise NotImplementedError(type(st).__name__)

    def for_(self, st: ir.For, ind: str) -> list[str]:
        c = st.counter.root
        start = str(st.start) if isinstance(st.start, int) else f"(long long){self.scalar_value(st.start)}"
        stop = str(st.stop) if isinstance(st.stop, int) else f"(long long){self.scalar_value(st.stop)}"
        name = c_string(c.name)
        out = [f"{ind}{{", f"{ind}    const long long stop_ = {stop};"]
        if self.is_host(c):
            tail = None
            step_twin = ""
            if c.id in self.dev_hosts:
                slot = self.hsd_slot(c)
                out.append(f"{ind}    ANVIL_GO(anvil_twin_set, 1, 64, anvil_hsd, {slot}, (int)({start}));")
                tail = [f"{ind}        ANVIL_GO(anvil_twin_step, 1, 64, anvil_hsd, {slot}, {st.step});"]
                body_has_continue = any(isinstance(x, ir.Continue) for b in ir.walk_blocks(st.body) for x in b.stmts)
                if body_has_continue:
                    step_twin = f"ANVIL_GO(anvil_twin_step, 1, 64, anvil_hsd, {slot}, {st.step}), "
                    tail = None
            out.append(f"{ind}    for (anvil_h{c.id} = (int)({start}); anvil_h{c.id} < stop_; {step_twin}anvil_h{c.id} += {st.step}) {{")
            out.append(f"{ind}        anvil_mark({name});")
            out += self.block(st.body, ind + "        ", in_loop=True, tail=tail)
            out.append(f"{ind}    }}")
        else:
            d = self.dev(c)
            out.append(f"{ind}    for (long long c_ = {start}; c_ < stop_; c_ = (long long)anvil_read_i32({d}) + {st.step}) {{")
            out.append(f"{ind}        anvil_write_i32({d}, (int)c_);")
            out.append(f"@@dirty {c.id} {ind}        ")
            out.append(f"{ind}        anvil_mark({name});")
            out += self.block(st.body, ind + "        ", in_loop=True)
            out.append(f"{ind}    }}")
        out.append(f"{ind}}}")
        return out

    def print_(self, st: ir.Print, ind: str) -> list[str]:
        """A print statement: its text assembled in one buffer, written to stdout (or stderr) in one
        call (the interpreter's exec_print, interp.py:213-239)."""
        f = "stderr" if st.err else "stdout"
        out = [f"{ind}anvil_sync();"]
        if st.err:
            out.append(f"{ind}fflush(stdout);")
        out.append(f"{ind}{{ anvil_text t_ = {{NULL, 0, 0}};")
        for it in list(st.items) + [ir.PrintItem("text", st.end)]:
            if it.kind == "text":
                if it.text:
                    out.append(f"{ind}  anvil_text_str(&t_, {c_string(it.text)});")
            elif it.kind == "scalar":
                b = it.buf.root
                v = f"{self.host_view(b)}[0]"
                if it.fmt:
                    isint = b.dtype == I32 or it.fmt.endswith("d")
                    val = f"(int){v}" if isint else f"anvil_fmt_arg({v})"
                    out.append(f"{ind}  anvil_text_fmt(&t_, {c_string(it.fmt)}, {val});")
                elif b.dtype == I32:
                    out.append(f"{ind}  anvil_text_fmt(&t_, \"%d\", {v});")
                else:
                    out.append(f"{ind}  anvil_text_f32(&t_, {v});")
            elif it.kind == "tensor":
                b = it.buf.root
                dims = self.table("long", [str(d) for d in b.shape])
                out.append(f"{ind}  anvil_text_tensor(&t_, {self.host_view(b)}, {1 if b.dtype == I32 else 0}, "
                           f"{len(b.shape)}, {dims});")
            elif it.kind == "pick":
                tab = self.strings(it.choices)
                out.append(f"{ind}  anvil_text_pick(&t_, (int){self.host_view(it.buf)}[0], {tab}, {len(it.choices)});")
            elif it.kind == "chars":
                out.append(f"{ind}  anvil_text_chars(&t_, (const int *){self.host_view(it.buf)}, {it.buf.numel});")
            else:
                raise NotImplementedError(it.kind)
        out.append(f"{ind}  anvil_text_write(&t_, {f}); }}")
        return out

    def writable(self, b, full: bool) -> str:
        """Host code: prepare b's mirror for a host write (the caller commits it afterwards)."""
        return f"(({ctype(b.root.dtype)} *)anvil_begin_write(&{self.mirror(b)}, {1 if full else 0}))"

    def rtcall(self, st: ir.RTCall) -> list[str]:
        a, n = st.args, st.name
        b = a.get("buf")
        if n == "seed":
            return [f"anvil_hs.seed = {a['value'] & 0xFFFFFFFF}u; anvil_hs.stream = 0;"]
        if n == "skip_rand":
            return ["anvil_hs.stream++;"]
        if n == "exit":
            return ["anvil_sync();", "fflush(stdout);", f"exit({int(a['value'])});"]
        if n in ("iota", "iota_once"):
            return [f"anvil_fill_iota((int *){self.writable(b, True)}, {b.numel}L); anvil_commit(&{self.mirror(b)});"]
        if n == "shuffle":
            if self.is_host(b):
                return [f"anvil_fisher_yates(&anvil_h{b.root.id}, {b.numel}L);"]
            return [f"anvil_fisher_yates((int *){self.writable(b, False)}, {b.numel}L); anvil_commit(&{self.mirror(b)});"]
        if n == "clock":
            return ["anvil_sync();", f"{self.writable(b, True)}[0] = (float)(anvil_seconds() - anvil_hs.t0); "
                    f"anvil_commit(&{self.mirror(b)});"]
        if n == "sleep":
            return ["anvil_sync();", "fflush(stdout);",
                    f"{{ const float s_ = {self.host_view(b)}[0]; if (s_ > 0) usleep((useconds_t)(s_ * 1e6f)); }}"]
        if n == "nonzero":
            src = a["src"]
            return [f"anvil_find_nonzero((const int *){self.host_view(src)}, {src.numel}L, (int *){self.writable(b, True)}, "
                    f"{b.numel}L); anvil_commit(&{self.mirror(b)});"]
        if n == "load_idx":
            return ["anvil_sync();", f"anvil_read_idx({c_string(a['path'])}, {self.writable(b, True)}, {b.numel}L, "
                    f"{a['header']}L, {1 if b.dtype == I32 else 0}); anvil_commit(&{self.mirror(b)});"]
        if n == "load_csv":
            return ["anvil_sync();", f"anvil_read_csv({c_string(a['path'])}, (float *){self.writable(b, True)}, "
                    f"{b.numel}L, {a['skip']}L); anvil_commit(&{self.mirror(b)});"]
        if n == "load_bytes":
            return ["anvil_sync();", f"anvil_read_bytes({c_string(a['path'])}, (int *){self.writable(b, True)}, "
                    f"{b.numel}L); anvil_commit(&{self.mirror(b)});"]
        if n == "load_npy":
            return ["anvil_sync();", f"anvil_read_npy({c_string(a['path'])}, {self.writable(b, True)}, {b.numel}L, "
                    f"{a['offset']}L, {a['kind']}, {a['size']}); anvil_commit(&{self.mirror(b)});"]
        if n == "save_npy":
            tab = self.table("unsigned char", [str(x) for x in a["header"]])
            return ["anvil_sync();", f"anvil_write_npy({c_string(a['path'])}, {tab}, {len(a['header'])}L, "
                    f"{self.host_view(b)}, {4 * b.numel}L);"]
        if n == "input":
            return ["anvil_sync();", f"if (anvil_read_number((float *){self.writable(b, True)})) goto anvil_end;",
                    f"anvil_commit(&{self.mirror(b)});"]
        if n == "show":
            return ["anvil_sync();", f"anvil_show_grid((const int *){self.host_view(b)}, {a['rows']}L, {a['cols']}L, "
                    f"{self.strings(a['glyphs'])}, {len(a['glyphs'])});"]
        if n in ("save", "load"):
            tab = self.label("anvil_ckpt")
            bufs = a["bufs"]
            self.ckpts.append((tab, bufs))
            out = ["anvil_sync();"]
            if n == "save":
                out.append(f"{{ anvil_ckpt_entry e_[] = {{{', '.join(f'{{(void *){self.host_view(x)}, {ir.ckpt_key(x.root)}ULL}}' for x in bufs)}}};")
                out.append(f"  anvil_ckpt_save({c_string(a['path'])}, e_, {len(bufs)}L); }}")
                return out
            out.append(f"{{ anvil_ckpt_entry e_[] = {{{', '.join(f'{{(void *){self.writable(x, False)}, {ir.ckpt_key(x.root)}ULL}}' for x in bufs)}}};")
            out.append(f"  const float ok_ = anvil_ckpt_load({c_string(a['path'])}, e_, {len(bufs)}L);")
            for x in bufs:
                out.append(f"  anvil_commit(&{self.mirror(x)});")
            if self.is_host(b):
                out.append(f"  anvil_h{b.root.id} = ok_; }}")
            else:
                out.append(f"  {self.writable(b, True)}[0] = ok_; anvil_commit(&{self.mirror(b)}); }}")
            return out
        raise NotImplementedError(n)

    # ------------------------------------------------------------------ the file
    def generate(self) -> str:
        body = self.block(self.prog.main, "    ")
        kernels_src = [p._source if hasattr(p, "_source") else p.source() for p in self.plans]
        # device buffers: every buffer a kernel or the host touches on the device
        for p in self.plans:
            for b in p.bufs.values():
                self.device_bufs.setdefault(b.id, b)
        externs = [b for b in self.prog.buffers if b.root is b and b.kind in ir.EXTERN_KINDS]
        for b in externs:
            self.dev(b)
        for b in self.prog.buffers:
            r = b.root
            if r.init is not None and r.id in self.device_bufs:
                self.mirror(r)
        HSD_ID = 900_000_003
        self.device_bufs[HSD_ID] = A.new_buffer(HSD_ID, "host_scalars.device_copy", (max(1, len(self.hsd)),), I32,
                                                "scratch")
        dev = sorted(self.device_bufs.values(), key=lambda b: b.id)
        share = os.environ.get("ANVIL_HIP_SHARE", "1") != "0"
        plan = A.plan_arena(self.prog, dev, self.full_writer, share=share, fused=self.fused_group,
                            extra=self.extra_reads)
        self.arena = plan
        # the no-allocation entry: the caller brings the arguments and results, so its scratch
        # holds only the other buffers (same lifetime sharing)
        extern_ids = {b.id for b in externs}
        inner = [b for b in dev if b.id not in extern_ids]
        splan = A.plan_arena(self.prog, inner, self.full_writer, share=share, fused=self.fused_group,
                             extra=self.extra_reads)
        src = self.prog.source
        name = src.display_path() if src is not None and hasattr(src, "display_path") else "<program>"
        out = [f"// Generated by anvil (HIP backend) from {name} for MI355X ({ARCH}).",
               f"// Build: hipcc --offload-arch={ARCH} {' '.join(f for f in HIP_FLAGS if f != '-w')} prog.hip -o prog.so -lz",
               "", runtime_source(any(p.kind.startswith("attention-train") for p in self.plans),
                              any("anvil_mm_tile_split<" in text or "anvil_mm_tile_shared<" in text for text in kernels_src),
                              any(p.kind == "attention" for p in self.plans)), "",
               "// ---------------------------------------------------------------- buffers"]
        for b in dev:
            where = f"arena + {plan.offsets[b.id]}"
            out.append(f"static {ctype(b.dtype)} *anvil_b{b.id};   // {b.kind} {b.name}{list(b.shape)} at {where}")
        for bid in sorted(self.hosts):
            b = self.by_id[bid]
            out.append(f"static {ctype(b.dtype)} anvil_h{bid};   // host scalar {b.name}")
        for b in sorted(self.mirrored.values(), key=lambda b: b.id):
            out.append(f"static anvil_mirror anvil_mir{b.id};")
        out.append("static uint32_t *anvil_hsd;   // device copies of host scalars: " +
                   ", ".join(f"[{i}] {self.by_id[bid].name}" for bid, i in sorted(self.hsd.items(), key=lambda t: t[1])))
        for n in range(len(self.segments)):
            out.append(f"static anvil_segment anvil_seg{n};")
        need = splan.size if inner else 0
        out += ["// scratch of anvil_entry_noalloc: every buffer but the arguments and results, at the",
                "// offsets of the same lifetime plan; one copy per GPU, held until the process ends",
                f"static const long long anvil_scratch_need = {need}LL;",
                f"ANVIL_SCRATCH_ARRAY(anvil_scratch, {need if 0 < need <= SCRATCH_MAX else 256});"]
        for b in self.prog.buffers:
            r = b.root
            if r is b and r.init is not None:
                vals = ", ".join(flit(float(v)) if r.dtype == F32 else ilit(int(v)) for v in r.init)
                out.append(f"static const {ctype(r.dtype)} anvil_init{r.id}[] = {{{vals}}};")
        out += [""] + self.tables
        out += ["", "// ---------------------------------------------------------------- kernels"]
        out += kernels_src
        out += ["", "// ---------------------------------------------------------------- profiling sites"]
        sites = []
        for p in self.plans:
            fl, by = hip_cost.plan_cost(p)
            sites.append(f"{{{c_string(p.name + ' ' + p.kind + ': ' + p.label)}, 0.0, 0, {float(fl)!r}, {float(by)!r}, "
                         f"{c_string(profile_row(p))}}}")
        sites = sites or ['{"none", 0.0, 0, 0.0, 0.0, ""}']
        out.append(f"static anvil_site anvil_site_table[] = {{{', '.join(sites)}}};")
        out += ["", "// ---------------------------------------------------------------- set-up"]
        out.append("// what the host needs, whichever entry runs first (allocates nothing)")
        out.append("static void anvil_setup_host(void) {")
        out.append("    static int done = 0;")
        out.append("    if (done) return;")
        out.append("    done = 1;")
        for i, m in enumerate(self.faults, 1):
            out.append(f"    anvil_fault_text[{i}] = {c_string(m)};")
        out.append("    anvil_sites = anvil_site_table;")
        out.append(f"    anvil_nsites = {len(self.plans)};")
        out.append(f"    anvil_hs.seed0 = {self.seed}u;")
        out.append("}")
        out.append("static void anvil_setup(void) {")
        out.append("    if (anvil_dev.ready) return;")
        out.append("    anvil_setup_host();")
        out.append(f"    anvil_device_open({plan.size});")
        for b in dev:
            out.append(f"    anvil_b{b.id} = ({ctype(b.dtype)} *)(anvil_dev.arena + {plan.offsets[b.id]});")
        out.append(f"    anvil_hsd = (uint32_t *)anvil_b{HSD_ID};")
        for b in sorted(self.mirrored.values(), key=lambda b: b.id):
            out.append(f"    anvil_mirror_init(&anvil_mir{b.id}, (void **)&anvil_b{b.id}, {max(4, 4 * b.numel)});")
        out.append("}")
        out += ["", "// the state a run starts from: zeroed memory, constants uploaded, seed and stream reset",
                "static void anvil_fresh(void) {",
                "    anvil_arena_zero();"]
        for b in dev:
            r = b
            if r.init is not None:
                out.append(f"    memcpy(anvil_mir{r.id}.host, anvil_init{r.id}, sizeof anvil_init{r.id});")
                out.append(f"    anvil_commit(&anvil_mir{r.id});")
        for b in sorted(self.mirrored.values(), key=lambda b: b.id):
            if b.init is None:
                out.append(f"    anvil_mir{b.id}.valid = 0;")
        for bid in sorted(self.hosts):
            out.append(f"    anvil_h{bid} = 0;")
        out += ["    anvil_hs.seed = anvil_hs.seed0;", "    anvil_hs.stream = 0;", "    anvil_hs.t0 = anvil_seconds();", "}"]
        def undirty(lines):
            res = []
            for line in lines:
                if line.startswith("@@dirty "):
                    _, bid, ind = line.split(" ", 2)
                    if int(bid) in self.mirrored:
                        res.append(f"{ind}anvil_mir{bid}.valid = 0;")
                    continue
                res.append(line)
            return res
        if self.segments:
            out += ["", "// ---------------------------------------------------------------- graph segments"]
            for fn in self.segments:
                out += undirty(fn)
        out += ["", "// ---------------------------------------------------------------- the program",
                "static int anvil_program(void) {"]
        for line in body:
            if line.startswith("@@dirty "):
                _, bid, ind = line.split(" ", 2)
                if int(bid) in self.mirrored:
                    out.append(f"{ind}anvil_mir{bid}.valid = 0;")
                continue
            out.append(line)
        out += ["    goto anvil_end;", "anvil_end:", "    anvil_sync();", "    fflush(stdout);", "    return 0;", "}"]
        out += self.abi(externs, plan)
        out += self.abi_noalloc(externs, dev, splan, need, HSD_ID)
        return "\n".join(out) + "\n"

    def abi_noalloc(self, externs, dev, splan, need, hsd_id) -> list[str]:
        """anvil_entry_noalloc: one call of the function on the caller's device buffers and stream,
        with every other buffer in the library's static `anvil_scratch` array; no allocation of any
        kind (no hipMalloc, pinned host memory, events or graphs). Refused (a negative status and a
        message on stderr, nothing run) when an argument's size differs from the compiled shape, when
        the scratch would exceed SCRATCH_MAX, or when the program keeps host copies of device
        buffers (prints, data files, checkpoints) or runs --check, which allocate."""
        def slot(b):
            return int(b.name[len(b.kind):]) if b.name[len(b.kind):].isdigit() else None
        ins = [(slot(b), b) for b in externs if b.kind == "input"]
        outs = [(slot(b), b) for b in externs if b.kind == "output"]
        n_in = 1 + max([k for k, _ in ins if k is not None], default=-1)
        n_out = 1 + max([k for k, _ in outs if k is not None], default=-1)
        why = None
        if any(k is None for k, _ in ins + outs):
            why = "its arguments are not numbered input<k>/output<k> slots"
        elif self.mirrored:
            why = "the program keeps host copies of device buffers (prints, data files, checkpoints)"
        elif self.check:
            why = "it was built with --check"
        extern_ids = {b.id for b in externs}
        out = ["",
               "// No allocation: the caller's device buffers and stream, the other buffers in anvil_scratch.",
               "// Calls that overlap on one GPU share its anvil_scratch and race: serialize them.",
               "static void anvil_bind_scratch(char *base) {"]
        for b in dev:
            if b.id not in extern_ids:
                out.append(f"    anvil_b{b.id} = ({ctype(b.dtype)} *)(base + {splan.offsets[b.id]});")
        out.append(f"    anvil_hsd = (uint32_t *)anvil_b{hsd_id};")
        out += ["}", 'extern "C" {',
                "int anvil_entry_noalloc(void *const *inputs, const long long *input_bytes, int n_inputs,",
                "                        void *const *outputs, const long long *output_bytes, int n_outputs,",
                "                        void *stream) {"]
        if why is not None:
            out += [f"    (void)inputs; (void)input_bytes; (void)n_inputs; (void)outputs; (void)output_bytes;",
                    f"    (void)n_outputs; (void)stream;",
                    f"    return anvil_refuse(-4, {c_string('this library cannot run without allocating: ' + why + '; use anvil_entry_device')});",
                    "}", "}", ""]
            return out
        out += [f"    if (n_inputs != {n_in} || n_outputs != {n_out})",
                f'        return anvil_refuse(-1, "takes {n_in} inputs and {n_out} outputs, got %d and %d", n_inputs, n_outputs);',
                f"    if (anvil_scratch_need > ANVIL_SCRATCH_MAX)",
                f'        return anvil_refuse(-3, "needs %lld bytes of scratch, more than its maximum of %lld (use anvil_entry_device)", anvil_scratch_need, ANVIL_SCRATCH_MAX);']
        for side, arr, sizes, items in (("input", "inputs", "input_bytes", ins), ("output", "outputs", "output_bytes", outs)):
            for k, b in sorted(items, key=lambda t: t[0]):
                out.append(f"    if ({arr}[{k}] == NULL || {sizes}[{k}] != {4 * b.numel}LL)")
                out.append(f'        return anvil_refuse(-2, "{side} {k} must be a device buffer of {4 * b.numel} bytes ({b.dtype}{list(b.shape)}), got %lld bytes at %p", {sizes}[{k}], {arr}[{k}]);')
        out += ["    anvil_fault_t *fault = NULL;",
                "    char *base = anvil_scratch_here(&fault);",
                "    if (base == NULL) return anvil_refuse(-5, \"cannot find its scratch array on the current device\");",
                "    anvil_setup_host();",
                "    const anvil_device_state saved = anvil_dev;",
                "    uint32_t *keep_hsd = anvil_hsd;"]
        for b in dev:
            out.append(f"    {ctype(b.dtype)} *keep{b.id} = anvil_b{b.id};")
        out += ["    anvil_noalloc_begin(stream, fault);",
                "    anvil_bind_scratch(base);"]
        for k, b in ins:
            out.append(f"    anvil_b{b.id} = ({ctype(b.dtype)} *)inputs[{k}];")
        for k, b in outs:
            out.append(f"    anvil_b{b.id} = ({ctype(b.dtype)} *)outputs[{k}];")
        out += ["    anvil_zero_scratch(base, anvil_scratch_need);     // every call starts from zeroed scratch",
                "    const int prof = anvil_prof.on, suspended = anvil_graphs.suspended;",
                "    anvil_prof.on = 0;",
                "    anvil_graphs.suspended = 1;",
                "    anvil_hs.seed = anvil_hs.seed0; anvil_hs.stream = 0;",
                "    const int rc = anvil_program();",
                "    anvil_prof.on = prof;",
                "    anvil_graphs.suspended = suspended;",
                "    anvil_dev = saved;",
                "    anvil_hsd = keep_hsd;"]
        for b in dev:
            out.append(f"    anvil_b{b.id} = keep{b.id};")
        out += ["    return rc;", "}", "}", ""]
        return out

    def fused_group(self, k):
        """(launch key, buffers k's own kernel writes) when k is one of several IR kernels of a launch."""
        plan = self.group_of.get(k.id)
        if plan is None or len(plan.kernels) < 2:
            return None
        part = self.part_of[k.id]
        if len(part.kernels) < 2:
            return id(plan), set()          # alone in its part: its reads are its own inputs
        if not hasattr(part, "_writes"):
            part._writes = part.writes()
        return id(plan), part._writes

    def extra_reads(self, st) -> set:
        """Buffers a launch reads beyond the IR kernels it replaces (noted at its first kernel)."""
        if not isinstance(st, KernelStmt):
            return set()
        plan = self.group_of.get(st.kernel.id)
        if plan is None or not plan.kernels or plan.kernels[0] is not st.kernel or not hasattr(plan, "extra_reads"):
            return set()
        return plan.extra_reads()

    def full_writer(self, st, b) -> bool:
        if isinstance(st, KernelStmt):
            plan = self.plan_of.get(st.kernel.id)
            k = st.kernel
            if plan is not None:
                plan = plan[0]
                if hasattr(plan, "full_writes"):
                    return b.id in plan.full_writes()
                if any((k.id, i) in plan.skip_stores for i, s in enumerate(k.stmts)
                       if isinstance(s, ir.Store) and s.buf.root is b):
                    return False
            return A._full_write(k, b)
        if isinstance(st, ir.RTCall):
            return st.name in A.RT_FULL_WRITES and st.args.get("buf") is not None and st.args["buf"].root is b
        return False

    def buffer_table(self) -> list[str]:
        """anvil_buffer_read(id, dst, bytes): a buffer's current contents, for tests and tools."""
        out = ["int anvil_buffer_read(int id, void *dst, long long bytes) {", "    switch (id) {"]
        for b in sorted({x.root.id: x.root for x in self.prog.buffers}.values(), key=lambda b: b.id):
            n = 4 * max(1, b.numel)
            if self.is_host(b):
                out.append(f"    case {b.id}: if (bytes < 4) return -2; memcpy(dst, &anvil_h{b.id}, 4); return 4;")
            elif b.id in self.device_bufs:
                out.append(f"    case {b.id}: if (bytes < {n}) return -2; anvil_to_host(dst, anvil_b{b.id}, {n}); return {n};")
        out += ["    default: return -1;", "    }", "}"]
        return out

    def abi(self, externs, plan) -> list[str]:
        ins = sorted([b for b in externs if b.kind == "input"], key=lambda b: b.name)
        outs = sorted([b for b in externs if b.kind == "output"], key=lambda b: b.name)
        out = ["", "// ---------------------------------------------------------------- C ABI", 'extern "C" {']
        for b in ins + outs:
            out.append(f"void *anvil_{sanitize(b.name)} = NULL;")
            out.append(f"void *anvil_d{sanitize(b.name)} = NULL;")
        out += [
            "int anvil_init(void) { anvil_setup(); anvil_fresh(); return 0; }",
            "int anvil_main(void) {",
            "    anvil_setup();",
            "    anvil_fresh();",
            "    return anvil_program();",
            "}",
            "int anvil_entry(void) {",
            "    if (!anvil_dev.ready) { anvil_setup(); anvil_fresh(); }",
            "    anvil_hs.seed = anvil_hs.seed0; anvil_hs.stream = 0;"]
        for b in ins:
            out.append(f"    if (anvil_{sanitize(b.name)}) anvil_to_device(anvil_b{b.id}, anvil_{sanitize(b.name)}, {4 * b.numel});")
            if b.id in self.mirrored:
                out.append(f"    anvil_mir{b.id}.valid = 0;")
        out.append("    const int rc = anvil_program();")
        for b in outs:
            out.append(f"    if (anvil_{sanitize(b.name)}) anvil_to_host(anvil_{sanitize(b.name)}, anvil_b{b.id}, {4 * b.numel});")
        out += ["    return rc;", "}",
                "// the same call with device pointers in the anvil_d<slot> variables: no copies",
                "int anvil_entry_device(void) {",
                "    if (!anvil_dev.ready) { anvil_setup(); anvil_fresh(); }",
                "    anvil_device_barrier();",
                "    anvil_graphs.suspended = 1;",
                "    anvil_hs.seed = anvil_hs.seed0; anvil_hs.stream = 0;"]
        for b in ins + outs:
            out.append(f"    {ctype(b.dtype)} *keep{b.id} = anvil_b{b.id};")
            out.append(f"    if (anvil_d{sanitize(b.name)}) anvil_b{b.id} = ({ctype(b.dtype)} *)anvil_d{sanitize(b.name)};")
            if b.id in self.mirrored:
                out.append(f"    anvil_mir{b.id}.valid = 0;")
        out.append("    const int rc = anvil_program();")
        out.append("    anvil_graphs.suspended = 0;")
        for b in ins + outs:
            out.append(f"    anvil_b{b.id} = keep{b.id};")
            if b.id in self.mirrored:
                out.append(f"    anvil_mir{b.id}.valid = 0;")
        out += ["    return rc;", "}"]
        out += self.buffer_table()
        out += [f"long long anvil_arena_bytes(void) {{ return {plan.size}LL; }}",
                f"long long anvil_arena_unshared_bytes(void) {{ return {plan.size - plan.placed_bytes + plan.shared_bytes}LL; }}",
                f"const char *anvil_target(void) {{ return {c_string('emulate' if self.emulate else ARCH)}; }}",
                "}",
                ""]
        return out


# ----------------------------------------------------------------------------- plugin API

def generate(prog: ir.Program, seed: int = 0, library: bool = False, emulate: bool = False,
             graphs: bool | None = None, check: str | None = None) -> str:
    """The .hip source of a program (library=True: a function lowered by pyapi.lower, called
    through anvil_entry with the input/output slots). emulate=True: a CPU build of the same
    program for testing the generator on a machine without a GPU. graphs=True: loop bodies are
    captured into HIP graphs and replayed (default: $ANVIL_HIP_GRAPHS, else off — on MI355X with
    ROCm 7.2 eager launches measured faster for the C2 training step). check="nan" | "inf": the
    reference's `--check` (cli.py:44-45): after each kernel, stop at the first nan (or infinity) it
    wrote and say which computation made it."""
    if graphs is None:
        graphs = os.environ.get("ANVIL_HIP_GRAPHS", "0") == "1"
    if check not in (None, "nan", "inf"):
        raise ValueError(f"check must be None, 'nan' or 'inf', not {check!r}")
    return HipGen(prog, seed=seed, library=library, emulate=emulate, graphs=graphs, check=check).generate()


SCRATCH_MAX = 64 << 20      # bytes: the largest anvil_scratch a library holds (ANVIL_SCRATCH_MAX)


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise HipToolchainError("hipcc not found (ROCm is needed to build for MI355X; set $HIPCC)")


# -amdgpu-mfma-vgpr-form: matrix-core accumulators in ordinary VGPRs. With the compiler's own choice
# the attention kernel kept its output tiles in AGPRs and copied all 64 of them out and back on every
# key tile around the (VALU) softmax rescale: 272 register moves per 128 MFMAs. No generated kernel
# spills with it.
HIP_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-munsafe-fp-atomics", "-w",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-mllvm", "-amdgpu-mfma-vgpr-form"]


def build(source: str, lib_path: str, emulate: bool = False) -> None:
    """Compile a generated file into a shared library at lib_path (atomically)."""
    d = tempfile.mkdtemp(prefix="anvil-hip-")
    try:
        src = os.path.join(d, "prog.hip")
        with open(src, "w") as f:
            f.write(source)
        tmp = os.path.join(d, "prog.so")
        if emulate:
            cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
            if cxx is None:
                raise HipToolchainError("no C++ compiler for the CPU build")
            cmd = [cxx, "-O1", "-std=c++17", "-fwrapv", "-w", "-ffp-contract=off", "-DANVIL_EMULATE", "-fPIC",
                   "-shared", "-x", "c++", src, "-o", tmp, "-lz"]
        else:
            cmd = [hipcc(), f"--offload-arch={ARCH}"] + HIP_FLAGS + [src, "-o", tmp, "-lz"]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise HipToolchainError(f"{os.path.basename(cmd[0])} failed:\n{r.stderr[-4000:]}")
        os.makedirs(os.path.dirname(os.path.abspath(lib_path)), exist_ok=True)
        shutil.move(tmp, lib_path + ".tmp")
        os.replace(lib_path + ".tmp", lib_path)
    finally:
        shutil.rmtree(d, ignore_errors=True)


def cache_dir() -> str:
    """Where built libraries are kept: $ANVIL_CACHE, else the package's own _libs directory (so
    libraries built on one machine travel with the source tree)."""
    d = os.environ.get("ANVIL_CACHE") or os.path.join(os.path.dirname(HERE), "_libs")
    os.makedirs(d, exist_ok=True)
    return d


def library_path(source: str, emulate: bool = False) -> str:
    key = hashlib.sha256(source.encode()).hexdigest()[:20]
    return os.path.join(cache_dir(), f"anvil-{key}{'-cpu' if emulate else ''}.so")


_BUILD_LOCK = threading.Lock()


def compile_source(source: str, emulate: bool = False, rebuild: bool = False) -> str:
    lib = library_path(source, emulate)
    with _BUILD_LOCK:
        if rebuild or not os.path.exists(lib):
            build(source, lib, emulate=emulate)
    return lib


class HipLibrary:
    """A loaded generated library and its C ABI."""

    def __init__(self, path: str, source: str | None = None):
        self.path = path
        self.source = source
        self.lib = ctypes.CDLL(path)
        for fn in ("anvil_main", "anvil_entry", "anvil_entry_device", "anvil_init", "anvil_sync_device",
                   "anvil_profile_count", "anvil_marks_count", "anvil_marks_window"):
            getattr(self.lib, fn).restype = ctypes.c_int
        self.lib.anvil_profile_ms.restype = ctypes.c_double
        self.lib.anvil_profile_ms.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_calls.restype = ctypes.c_long
        self.lib.anvil_profile_calls.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_flops.restype = ctypes.c_double
        self.lib.anvil_profile_flops.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_bytes.restype = ctypes.c_double
        self.lib.anvil_profile_bytes.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_label.restype = ctypes.c_char_p
        self.lib.anvil_profile_label.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_where.restype = ctypes.c_char_p
        self.lib.anvil_profile_where.argtypes = [ctypes.c_int]
        self.lib.anvil_profile_enable.argtypes = [ctypes.c_int]
        self.lib.anvil_marks_select.argtypes = [ctypes.c_char_p]
        self.lib.anvil_marks_window.argtypes = [ctypes.c_int, ctypes.c_int]
        self.lib.anvil_marks_elapsed_ms.restype = ctypes.c_double
        self.lib.anvil_marks_elapsed_ms.argtypes = [ctypes.c_int, ctypes.c_int]
        self.lib.anvil_arena_bytes.restype = ctypes.c_longlong
        self.lib.anvil_target.restype = ctypes.c_char_p
        self.lock = threading.Lock()

    def slot(self, name: str) -> ctypes.c_void_p:
        return ctypes.c_void_p.in_dll(self.lib, f"anvil_{name}")

    def main(self) -> int:
        return self.lib.anvil_main()

    def profile(self) -> list[tuple[str, float, int, float, float]]:
        """Per launch site: (label, total ms, launches, FLOPs per launch, bytes per launch)."""
        self.lib.anvil_sync_device()
        n = self.lib.anvil_profile_count()
        return [(self.lib.anvil_profile_label(i).decode(), self.lib.anvil_profile_ms(i),
                 self.lib.anvil_profile_calls(i), self.lib.anvil_profile_flops(i),
                 self.lib.anvil_profile_bytes(i)) for i in range(n)]


def load(prog: ir.Program, seed: int = 0, library: bool = False, emulate: bool = False,
         rebuild: bool = False, graphs: bool | None = None) -> HipLibrary:
    src = generate(prog, seed=seed, library=library, emulate=emulate, graphs=graphs)
    return HipLibrary(compile_source(src, emulate=emulate, rebuild=rebuild), src)
