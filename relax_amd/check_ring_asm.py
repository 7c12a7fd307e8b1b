"""Build-time checks of the generated code: of ``csrc/q4g32_gemv_list.hip`` and ``csrc/q4g32_batch_list.hip``, and of the
tiled GEMMs.

The compute wavefronts of the one-row list and of lists of more than 16 rows load their weight stream with inline-assembly
loads into a ring of registers and wait for them by hand, so the compiler does not know that those registers are
in flight between a load and its wait.  The source makes every read of a ring register an asm
statement that depends on the wait; what is left to chance is register allocation (a copy or a
spill of a ring register inserted between load and wait would read it too early).  This script
compiles the file to assembly and verifies, in the kernel's text, that

* every ring register (destination of a ``global_load_* ... nt`` or ``buffer_load_* ... nt`` instruction) is read only by the
  instructions the source uses for it (``v_and_or_b32``, ``v_lshrrev_b32 .., 8 | 16, ..``, ``v_cvt_f32_f16``,
  and the cross-lane ``v_mov_b32_dpp`` of the batch kernel's lane exchange, which the compiler never
  generates by itself), never by a plain move, a store or anything else, and
* each ring slot keeps one register in the prologue and in the loop (no renaming copies).

What the text cannot show is a slot abandoned on the way out of the loop: its load is still in flight, and
a register the compiler reuses behind the loop would receive the data on top of its new value.  The
sources therefore wait for all loads (``s_waitcnt vmcnt(0)``) where the ring's loop ends.

Registers that the compiler also uses for short-lived temporaries while a slot is empty are
recognised by being written by another instruction first.

Kernels of these files with non-temporal loads, in whatever form, and those of ``held_gemm.h`` must also be free of register spills (no ``scratch_*`` instruction).

A second check (``check_asm_results``) covers what inline assembly costs besides: the compiler does
not keep the hardware's wait states between an inline-assembly VALU result and an MFMA or DPP
instruction that reads it.

``check_direct_loads_drained``, of the tiled GEMMs: no result is staged in LDS before every direct load to it has landed.

``check_empty_descriptors``, of the tiled GEMMs and of lists of several rows: the loads past the end lie outside their
descriptors however the range check counts a scalar offset.
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCES = ("q4g32_gemv_list.hip", "q4g32_batch_list.hip")
# the kernel with activations in registers (held_gemm.h)
HELD_SOURCES = ("gptq.hip", "q4g32_skinny.hip")
# the tiled GEMMs (mfma_gemm_lds.h)
DIRECT_LOAD_SOURCES = ("gemm_256.hip", "gptq.hip", "intb_gemm.hip", "q4g32_gemm.hip", "q4n32.hip")
# kernels of SOURCES whose loads past the end have a scalar offset
GUARDED_KERNELS = {"q4g32_batch_list.hip": ("q4g32_batch_list_kernel", "q4g32_batch_rows_kernel")}
ALLOWED_READERS = ("v_and_or_b32", "v_lshrrev_b32", "v_cvt_f32_f16", "v_mov_b32_dpp")


_COMPILERS = " (waited for by the compiler)"  # behind a non-temporal load outside of inline assembly


def _is_ring_load(l: str) -> bool:
    """A load of the weight stream that is waited for by hand: a non-temporal load in inline assembly."""
    return l.startswith(("global_load_", "buffer_load_")) and l.endswith(" nt")


def _regs(tok: str):
    """'v[4:7]' -> {4,5,6,7}; 'v12' -> {12}; anything else -> empty."""
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"v(\d+)", tok)
    return {int(m.group(1))} if m else set()


def _check_function(body: list[str]) -> list[str]:
    errors = []
    ring = set()
    for l in body:
        if _is_ring_load(l):
            ring |= _regs(l.split()[1].rstrip(","))
    if not ring:
        return []
    # walk the text; a ring register is "loaded" after a ring load wrote it and until something else writes it
    loaded = set()
    for l in body:
        parts = l.replace(",", " ").split()
        op, ops = parts[0], parts[1:]
        if _is_ring_load(l):
            loaded |= _regs(ops[0])
            continue
        if not ops:
            continue
        stores = ("global_store", "ds_write", "buffer_store", "scratch_store", "global_atomic", "ds_add")
        writes = _regs(ops[0]) if not op.startswith(("s_",) + stores) else set()
        reads = set()
        for t in (ops if not writes else ops[1:]):
            reads |= _regs(t)
        if op.startswith(stores):
            reads |= _regs(ops[0])
        hit = reads & loaded
        if hit and not op.startswith(ALLOWED_READERS):
            errors.append(f"ring register(s) {sorted(hit)} read by `{l}`")
        if op.startswith("v_lshrrev_b32") and hit and ops[1] not in ("8", "16"):
            errors.append(f"unexpected shift of a ring register: `{l}`")
        loaded -= writes  # now a temporary of the compiler
    return errors


HAZARD_WINDOW = 3  # instructions: the hardware wants up to 2 wait states, one instruction may be a zero-cycle s_nop


def check_asm_results(asm_text: str) -> list[str]:
    """The compiler inserts the wait states between a VALU result and an MFMA or DPP instruction that reads it
    only when it issued the VALU instruction itself: the text of an inline-assembly statement is opaque to its
    hazard recognizer.  So no register written inside an ASMSTART / ASMEND block may be read by a v_mfma* or
    *_dpp instruction within the next HAZARD_WINDOW instructions, unless an s_nop of the block itself follows
    the write (loads are exempt: their results are waited for with s_waitcnt)."""
    errors = []
    recent = []  # (instructions ago, set of registers) written by inline assembly
    in_asm = False
    for raw in asm_text.splitlines():
        t = raw.strip()
        if t.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if t.startswith(";;#ASMEND"):
            in_asm = False
            continue
        l = t.split(";")[0].strip()
        if not l or l.startswith(".") or l.endswith(":"):
            if l.endswith(":") and not l.startswith("."):
                recent = []
            continue
        parts = l.replace(",", " ").split()
        op, ops = parts[0], parts[1:]
        if in_asm and op.startswith("s_nop"):
            recent = []  # the statement brings its own wait states
            continue
        reads_all = set()
        for tok in ops[1:] if ops else []:
            reads_all |= _regs(tok)
        if (op.startswith("v_mfma") or op.endswith("_dpp") or "_dpp " in l) and not in_asm:
            for age, regs in recent:
                hit = regs & (reads_all | (_regs(ops[0]) if op.endswith("_dpp") else set()))
                if hit:
                    errors.append(f"`{l}` reads v{sorted(hit)} written by inline assembly {age} instruction(s) before")
        recent = [(a + 1, r) for a, r in recent if a + 1 < HAZARD_WINDOW]
        if in_asm and ops and op.startswith("v_") and not op.startswith("v_cmp"):
            recent.append((0, _regs(ops[0])))
    return errors


def _functions(asm_text: str, labels: bool = False):
    """(name, instructions) of every function of the file, with its local labels if asked for."""
    functions, cur, in_asm = [], None, False
    for raw in asm_text.splitlines():
        t = raw.strip()
        in_asm = t.startswith(";;#ASMSTART") or (in_asm and not t.startswith(";;#ASMEND"))
        l = raw.split(";")[0].strip()
        if not l:
            continue
        if not in_asm and l.endswith(" nt"):
            l += _COMPILERS
        if l.endswith(":") and not l.startswith("."):  # a function label
            cur = []
            functions.append((l[:-1], cur))
        elif l.startswith(".Lfunc_end"):
            cur = None
        elif cur is not None and (l.startswith(".LBB") if l.endswith(":") else not l.startswith(".")):
            if labels or not l.endswith(":"):
                cur.append(l)
    return functions


def _spills(body: list[str]) -> list[str]:
    """These kernels are written to fit their register budget.  A spill anywhere in them (also in a service
    wavefront's path: one extra branch there once sent 64 load registers through scratch memory and
    cost the 4-linear step 3 of 21 us) is a regression the tests do not show."""
    spills = [l for l in body if l.startswith(("scratch_load", "scratch_store"))]
    return [f"{len(spills)} scratch accesses (register spills), the first: `{spills[0]}`"] if spills else []


def check_held(asm_text: str) -> list[str]:
    """Every ``held_gemm_kernel`` of the file: up to all 256 registers, and no spill."""
    kernels = [body for name, body in _functions(asm_text) if "held_gemm_kernel" in name]
    return [e for body in kernels for e in _spills(body)] if kernels else ["no held_gemm_kernel found"]


def check(asm_text: str) -> list[str]:
    """Checks every kernel of the file on its own (register names mean nothing across kernels)."""
    errors, with_ring = [], 0
    for _, body in _functions(asm_text):
        if any(_is_ring_load(l) or l.endswith(_COMPILERS) for l in body):
            with_ring += any(_is_ring_load(l) for l in body)
            errors += _check_function(body)
            errors += _spills(body)
    if with_ring == 0:
        return ["no ring loads found (expected global_load_* / buffer_load_* ... nt in the kernel)"]
    return errors


def _blocks(body: list[str]):
    """Basic blocks of a function's text as (instructions, indices of the blocks behind it)."""
    blocks, labels = [[]], {}
    for l in body:
        if l.endswith(":"):
            if blocks[-1]:
                blocks.append([])
            labels[l[:-1]] = len(blocks) - 1
        else:
            blocks[-1].append(l)
            if l.startswith(("s_branch", "s_cbranch", "s_endpgm", "s_setpc")):
                blocks.append([])
    out = []
    for i, b in enumerate(blocks):
        succ = []
        if b and b[-1].startswith(("s_branch", "s_cbranch")):
            succ.append(labels[b[-1].split()[1]])
        if i + 1 < len(blocks) and not (b and b[-1].startswith(("s_branch", "s_endpgm", "s_setpc"))):
            succ.append(i + 1)
        out.append((b, succ))
    return out


def _is_direct_load(l: str) -> bool:
    """A load from memory to LDS."""
    return l.startswith("global_load_lds_") or (l.startswith("buffer_load_") and l.endswith(" lds"))


def check_direct_loads_drained(asm_text: str) -> list[str]:
    """The tiled GEMMs keep direct loads (memory to LDS) in flight all through their K loop, past its end too, and then stage
    the results in the same LDS.  Such a load is nobody's register, so the compiler puts no wait in front of a write to the
    place it fills; and it may fill a place where another wavefront writes.  So in every ``gemm_lds_kernel``, on every
    way from such a load to a ``ds_write``, there must be an ``s_waitcnt vmcnt(0)`` and an ``s_barrier`` behind it."""
    CLEAN, DRAINED, PENDING = 0, 1, 2
    errors, kernels = [], 0
    for name, body in _functions(asm_text, labels=True):
        if "gemm_lds_kernel" not in name or not any(_is_direct_load(l) for l in body):
            continue
        kernels += 1
        blocks = _blocks(body)
        entry = [CLEAN] * len(blocks)
        todo, seen, bad = [0], set(), set()
        while todo:
            i = todo.pop()
            seen.add(i)
            state = entry[i]
            for l in blocks[i][0]:
                if _is_direct_load(l):
                    state = PENDING
                elif l.startswith("s_waitcnt") and "vmcnt(0)" in l and state == PENDING:
                    state = DRAINED
                elif l.startswith("s_barrier") and state == DRAINED:
                    state = CLEAN
                elif l.startswith("ds_write") and state != CLEAN:
                    bad.add((l, state))
            for j in blocks[i][1]:
                if state > entry[j] or j not in seen:
                    entry[j] = max(state, entry[j])
                    todo.append(j)
        for l, state in sorted(bad)[:3]:
            errors.append(f"{name}: `{l}` with direct loads " + ("on their way" if state == PENDING else "of other wavefronts on their way"))
    if kernels == 0:
        return ["no direct loads found (expected global_load_lds_* or buffer_load_* ... lds in a gemm_lds_kernel)"]
    return errors


_SGPRS = re.compile(r"(?:s(\d+)|s\[(\d+):(\d+)\])$")
_BUFFER_LOAD = re.compile(r"buffer_load_\w+ .*s\[\d+:\d+\], (\S+)(?: offen.*)?$")


def _sgprs(operand: str) -> range:
    m = _SGPRS.match(operand)
    if not m:
        return range(0)
    return range(int(m[1]), int(m[1]) + 1) if m[1] else range(int(m[2]), int(m[3]) + 1)


def check_empty_descriptors(asm_text: str, kernel: str = "gemm_lds_kernel") -> list[str]:
    """Past the last step of K the tiled GEMMs load against a buffer descriptor of 0 bytes, and the lists of several rows
    past the last piece of a row.  If the range check subtracts the scalar offset from the bytes of the descriptor, such a load
    lies outside only with a scalar offset that the descriptor holds.  So in every function of that name the scalar
    offset of a buffer load is 0, or a register that on every way to the load was last written by a choice between an
    offset and 0 (or by an AND with the mask of what there is)."""
    errors, loads = [], 0

    def after(block, guarded, bad):
        guarded = set(guarded)
        for l in block:
            m = _BUFFER_LOAD.match(l)
            if m:
                if m[1] != "0" and not (m[1][0] == "s" and guarded.issuperset(_sgprs(m[1]))):
                    bad.add(l)
                continue
            op, _, rest = l.partition(" ")
            operands = [o.strip() for o in rest.split(",")]
            written = set(_sgprs(operands[0]))
            masked = (op == "s_cselect_b32" and "0" in operands[1:]) or op == "s_and_b32"
            copied = op == "s_mov_b32" and (operands[1] == "0" or (_sgprs(operands[1]) and guarded.issuperset(_sgprs(operands[1]))))
            guarded = guarded | written if masked or copied else guarded - written
        return guarded

    for name, body in _functions(asm_text, labels=True):
        if kernel not in name or not any(_BUFFER_LOAD.match(l) for l in body):
            continue
        blocks = _blocks(body)
        entry = [None] * len(blocks)
        entry[0] = set()
        todo = [0]
        while todo:
            i = todo.pop()
            out = after(blocks[i][0], entry[i], set())
            for j in blocks[i][1]:
                joined = out if entry[j] is None else entry[j] & out
                if joined != entry[j]:
                    entry[j] = joined
                    todo.append(j)
        bad = set()
        for (block, _), guarded in zip(blocks, entry):
            if guarded is not None:
                after(block, guarded, bad)
        loads += sum(1 for l in body if _BUFFER_LOAD.match(l))
        for l in sorted(bad)[:3]:
            errors.append(f"{name}: `{l}` may have a scalar offset against an empty descriptor")
    if loads == 0:
        return [f"no buffer loads found in a {kernel}"]
    return errors


def _assembly(hipcc: str, flags, name: str) -> str:
    with tempfile.TemporaryDirectory() as td:
        out = os.path.join(td, "k.s")
        subprocess.check_call([hipcc, *flags, "-S", "--cuda-device-only", os.path.join(HERE, "csrc", name), "-o", out],
                              stderr=subprocess.DEVNULL)
        with open(out) as f:
            return f.read()


def check_source(hipcc: str, flags, name: str) -> None:
    """Raises if the code generated for one of SOURCES, HELD_SOURCES or DIRECT_LOAD_SOURCES is not as it has to be."""
    text = _assembly(hipcc, flags, name)
    if name in SOURCES + HELD_SOURCES:
        found = check_asm_results(text)
        if found:
            raise RuntimeError(f"{name}: an inline-assembly result reaches an MFMA / DPP instruction without wait states:\n  "
                               + "\n  ".join(found[:20]))
    if name in HELD_SOURCES:
        found = check_held(text)
        if found:
            raise RuntimeError(f"{name}: registers of a kernel with the activations in them are spilled:\n  " + "\n  ".join(found[:20]))
    if name in DIRECT_LOAD_SOURCES:
        found = check_direct_loads_drained(text)
        if found:
            raise RuntimeError(f"{name}: LDS is written while direct loads to it may be on their way:\n  " + "\n  ".join(found[:20]))
        found = check_empty_descriptors(text)
        if found:
            raise RuntimeError(f"{name}: a load past the last step may touch memory:\n  " + "\n  ".join(found[:20]))
    if name not in SOURCES:
        return
    errs = check(text)
    past = [e for k in GUARDED_KERNELS.get(name, ()) for e in check_empty_descriptors(text, k)]
    if past:
        raise RuntimeError(f"{name}: a load past the end may touch memory:\n  " + "\n  ".join(past[:20]))
    if errs:
        raise RuntimeError(f"{name}: the generated code touches in-flight ring registers:\n  " + "\n  ".join(errs[:20]))


if __name__ == "__main__":
    from relax_amd import build as _b  # noqa: E402

    for _name in sorted({*SOURCES, *HELD_SOURCES, *DIRECT_LOAD_SOURCES}):
        _b.check_asm(_name)
    print("ring registers, direct loads: ok")
