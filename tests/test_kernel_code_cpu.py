"""What the kernels' inline assembly relies on and the compiler does not check, read
from the machine code of the library as it is built (llvm-objdump; no GPU)."""

import functools
import re
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

from small_q_attention_amd import build as sqa_build

OBJDUMP = Path("/opt/rocm/lib/llvm/bin/llvm-objdump")
_LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// 0*([0-9A-F]+):.*?(?:<.*\+0x([0-9a-f]+)>)?$")


@functools.lru_cache(maxsize=1)
def kernels():
    """``{symbol: [(address, mnemonic, operands, branch target or None)]}`` of the library."""
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    if sqa_build.is_stale():
        sqa_build.build()
    out = {}
    with tempfile.TemporaryDirectory() as tmp:
        lib = Path(tmp) / "lib.so"
        shutil.copy(sqa_build.LIB_PATH, lib)
        subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=tmp, check=True,
                       capture_output=True)
        for code in sorted(Path(tmp).glob("lib.so.*amdgcn*")):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code.name], cwd=tmp,
                                  check=True, capture_output=True, text=True).stdout
            body = None
            for line in text.splitlines():
                head = re.match(r"^([0-9a-f]+) <(\S+)>:$", line)
                if head:
                    start, body = int(head.group(1), 16), []
                    out[head.group(2)] = body
                    continue
                m = _LINE.match(line)
                if m and body is not None:
                    to = start + int(m.group(4), 16) if m.group(4) else None
                    body.append((int(m.group(3), 16), m.group(1), m.group(2), to))
    assert any("sqa_partial_kernel" in k for k in out)
    return out


def _loads_into_lds(op, args):
    return op.startswith("global_load_lds") or (op.startswith("buffer_load") and
                                                args.split()[-1] == "lds")


def _scalars(text):
    """Numbers of the scalar registers named in an operand list."""
    regs = {int(n) for n in re.findall(r"\bs(\d+)\b", text)}
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(lo), int(hi) + 1))
    return regs


def test_loads_into_lds_keep_their_wait_states():
    """A load into LDS takes its LDS address from m0 and its base from scalar registers:
    one wait state after a scalar write of m0, five after a vector instruction's write of
    a scalar register it reads. The compiler keeps them for its own instructions and does
    not look into inline assembly."""
    seen = 0
    for name, code in kernels().items():
        for i, (_, op, args, _) in enumerate(code):
            if not _loads_into_lds(op, args):
                continue
            seen += 1
            reads, states = _scalars(args), 0
            for _, prev, pargs, _ in reversed(code[max(0, i - 5):i]):
                dest = pargs.split(",")[0]
                if prev.startswith("s_") and dest == "m0":
                    assert states >= 1, f"{name}: {op} right after {prev} m0"
                if prev.startswith("v_"):
                    assert states >= 5 or not reads & _scalars(dest), f"{name}: {prev} {pargs}"
                states += 1 + (int(pargs, 0) if prev == "s_nop" else 0)
                if states >= 5:
                    break
    assert seen > 0


_LOADS = {("KvNative", 64): 6, ("KvNative", 128): 8, ("KvNative", 256): 16,
          ("KvFp8", 64): 5, ("KvFp8", 128): 6, ("KvFp8", 256): 8}  # per page and head


def _partial_kernels():
    """``(symbol, code, pages of the ring, load instructions per page of a wave, whether it
    has a page loop)`` (without one: splits of a ring in one step)."""
    for name, code in kernels().items():
        m = re.search(r"sqa_partial_kernelILi\d+ELi(\d+)ELi\d+ELi\d+ELi(\d+)ENS0_\d+Elem\w+?"
                      r"ENS0_\d+(Kv[A-Za-z0-9]+?)ILi\d+EEELi(\d)ELb\dELb(\d)E", name)
        if m:
            pages, hd, kv, heads = int(m.group(1)), int(m.group(2)), m.group(3), int(m.group(4))
            yield name, code, pages, _LOADS[kv, hd] * heads, m.group(5) == "0"


def test_the_page_loop_never_drains_its_ring():
    """In a turn of the page loop the wave waits for the pages it is about to use, with
    the others in flight. A ring register moved elsewhere at the turn's end waits for a
    load just issued instead."""
    for name, code, pages, loads, loop in _partial_kernels():
        if not loop:
            continue
        at = {ins[0]: i for i, ins in enumerate(code)}
        turns = []
        for i, (addr, _, _, to) in enumerate(code):
            if to is not None and to <= addr and to in at:
                body = code[at[to]:i + 1]
                n = sum(op.startswith("buffer_load") for _, op, _, _ in body)
                if n == pages * loads and not any(op.startswith("global_store")
                                                  for _, op, _, _ in body):
                    turns.append(body)
        assert turns, name
        waits = [int(w) for _, op, args, _ in min(turns, key=len) if op == "s_waitcnt"
                 for w in re.findall(r"vmcnt\((\d+)\)", args)]
        # One page is used per step, two where the step takes a pair of pages or
        # computes the next page's scores ahead.
        least = (pages - (2 if pages > 2 else 1)) * loads
        assert waits and min(waits) >= least, f"{name}: waits {waits}, {least} loads in flight"


def test_the_wait_for_a_piece_s_rows_counts_the_loads_behind_them():
    """A piece begins by waiting until no more vector loads are in flight than a full ring
    has: its Q and mask words, copied into LDS before the ring's pages were requested, are
    there then. The count is written in the source; the instructions are the compiler's."""
    for name, code, pages, loads, _ in _partial_kernels():
        ops = [op for _, op, _, _ in code]
        assert ops.count("s_barrier") == 1, name
        barrier = ops.index("s_barrier")
        copies = [i for i, op in enumerate(ops[:barrier]) if op.startswith("global_load_lds")]
        assert copies, name
        behind = ops[copies[-1]:barrier]
        assert sum(op.startswith("buffer_load") for op in behind) == pages * loads, name
        # The six-bit counter's 63 waits for at least as much.
        want = f"vmcnt({min(pages * loads, 63)})"
        assert any(op == "s_waitcnt" and args.strip() == want
                   for _, op, args, _ in code[barrier:]), f"{name}: no {want} behind the barrier"


def test_the_arguments_on_the_way_to_the_first_load_come_in_one_trip():
    """The main kernel asks for the arguments it needs first at once. The order of the
    argument record decides whether the compiler can (a register of an unused word taken
    for a later load splits the trip in two)."""
    for name, code, _, _, _ in _partial_kernels():
        waits = 0
        for _, op, args, _ in code:
            waits += op == "s_waitcnt" and "lgkmcnt" in args
            if op.startswith("global_load") or (op.startswith("s_load") and "s[0:1]" not in args):
                break
        assert waits == 1, f"{name}: {waits} trips"
