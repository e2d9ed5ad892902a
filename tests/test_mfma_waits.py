"""The LDS ring of the MFMA tiles, checked in the compiled code.

mfma_tile_q (hx_mfma.hpp) fills its A ring with buffer loads that write LDS and waits for a chunk by the number of
vector-memory instructions issued after it.  That count holds only if the compiler keeps the loads of different
chunks apart and drops none, which no run shows reliably (a late load reads what the LDS held before).  So every
path through every tile of the built library is followed here: at the barrier ahead of chunk b, the A loads of the
chunks 0..b have to be complete."""
import re
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "helios_glm53flash_amd" / "libhx_exl3.so"
LLVM = Path("/opt/rocm/llvm/bin")
KERNELS = ("linear_mfma_kernel", "grouped_gu_kernel", "grouped_gemm_kernel")
VMEM = ("buffer_load", "buffer_store", "global_load", "global_store", "scratch_", "flat_", "global_atomic",
        "buffer_atomic")


def tile_kernels(lib, tmp):
    """name -> basic blocks of every tile kernel: {address: ([op, ..], [successor, ..])}; op: 'A' (load into LDS),
    'V' (another vector-memory instruction), 'B' (barrier) or the n of a wait for at most n outstanding."""
    obj = tmp / "lib.so"
    obj.write_bytes(Path(lib).read_bytes())
    subprocess.run([LLVM / "llvm-objdump", "--offloading", obj], check=True, capture_output=True, cwd=tmp)
    out = {}
    for co in sorted(tmp.glob("*gfx950*")):
        p = subprocess.run([LLVM / "llvm-objdump", "-d", co], stdout=subprocess.PIPE, text=True, check=True)
        for part in re.split(r"\n(?=[0-9a-f]{16} <)", p.stdout):
            name = re.match(r"[0-9a-f]{16} <(\w+)>:", part)
            if name and any(k in name.group(1) for k in KERNELS):
                out[name.group(1)] = blocks(part.splitlines()[1:])
    return out


def blocks(lines):
    code = []  # (address, op, branch target, falls through)
    pc = 0     # what a far branch adds to: s_getpc_b64, s_add_u32 of a literal, s_addc_u32, s_setpc_b64
    for s in lines:
        m = re.match(r"\s*(\S+)\s*(.*?)\s*// ([0-9A-F]+): ([0-9A-F]{8})", s)
        if not m:
            continue
        name, args, at, word = m.group(1), m.group(2), int(m.group(3), 16), int(m.group(4), 16)
        op = target = None
        through = name not in ("s_branch", "s_endpgm", "s_setpc_b64")
        if name.startswith(VMEM):
            op = "A" if name.startswith("buffer_load") and re.search(r"\blds\b", args) else "V"
        elif name == "s_waitcnt" and "vmcnt" in args:
            op = int(re.search(r"vmcnt\((\d+)\)", args).group(1))
        elif name == "s_barrier":
            op = "B"
        elif name == "s_branch" or name.startswith("s_cbranch"):
            off = word & 0xffff
            target = at + 4 + 4 * (off - 0x10000 if off & 0x8000 else off)
        elif name == "s_getpc_b64":
            pc = at + 4
        elif name == "s_add_u32" and pc:
            lit = int(args.split(",")[-1], 0)
            far, pc = pc + (lit - (1 << 32) if lit >> 31 else lit), 0
        elif name == "s_setpc_b64":
            target = far
        code.append((at, op, target, through))
    starts = {code[0][0]} | {t for _, _, t, _ in code if t} | {b[0] for a, b in zip(code, code[1:]) if a[2] or not a[3]}
    out, cur = {}, None
    for at, op, target, through in code:
        if at in starts:
            if cur is not None:
                out[cur][1].append(at)
            cur = at
            out[cur] = ([], [])
        if cur is None:
            continue
        if op is not None:
            out[cur][0].append(op)
        if target:
            out[cur][1].append(target)
        if not through:
            cur = None
    return out


def compact(bb):
    """The blocks with runs of blocks that do nothing skipped over: successors are blocks with ops."""
    def reach(label, seen):
        if label in seen:
            return set()
        seen.add(label)
        if bb[label][0]:
            return {label}
        return set().union(*[reach(s, seen) for s in bb[label][1]]) if bb[label][1] else set()
    return {k: (v[0], sorted(set().union(*[reach(s, set()) for s in v[1]]) if v[1] else set()))
            for k, v in bb.items() if v[0]}


def check(bb):
    """Follows every path of every tile from its first A load to the wait that drains the ring; returns the number
    of tiles and the tiles at fault, with the A loads of a chunk, the chunk and the loads that may be late."""
    bb = compact(bb)
    entries = []  # blocks whose A loads come before any barrier: the prologue of a tile
    for k, (ops, _) in bb.items():
        head = ops[:ops.index("B")] if "B" in ops else ops
        if "A" in head and not in_loop(bb, k):
            entries.append(k)
    bad = []
    for e in entries:
        na = per_step(bb, e)
        late = follow(bb, e, na)
        if late:
            bad.append((e, na) + late)
    return len(entries), bad


def in_loop(bb, k):
    """Whether k can reach itself without meeting a wait for everything (a tile ends with one)."""
    todo, seen = list(bb[k][1]), set()
    while todo:
        s = todo.pop()
        if s == k:
            return True
        if s in seen or drains(bb[s][0]):
            continue
        seen.add(s)
        todo += bb[s][1]
    return False


def drains(ops):
    return any(a == 0 and b == "B" for a, b in zip(ops, ops[1:]))


def per_step(bb, e):
    """A loads between the first two barriers of the tile, on the path that has the most (the main loop)."""
    best, todo, seen = 0, [(e, 0, 0, 0)], set()
    while todo:
        k, i, bars, n = todo.pop()
        if (k, i, bars, n) in seen:
            continue
        seen.add((k, i, bars, n))
        for j, op in enumerate(bb[k][0][i:], i):
            if op == "B":
                bars += 1
                if bars == 2:
                    best = max(best, n)
                    break
            elif op == "A" and bars == 1:
                n += 1
        else:
            todo += [(s, 0, bars, n) for s in bb[k][1]]
    return best


def follow(bb, e, na):
    todo, seen = [(e, (), 0, 0)], set()
    while todo:  # block, outstanding ops (oldest first), A loads issued less those due by now, barriers (0, 1: some)
        k, out, spare, begun = todo.pop()
        if (k, out, spare) in seen:
            continue
        seen.add((k, out, spare))
        ops, done = bb[k][0], False
        for i, op in enumerate(ops):
            if op in ("A", "V"):
                out = (out + (op,))[-63:]
                spare += op == "A"
            elif op == "B":
                spare -= na
                if out.count("A") > spare:
                    return spare, out.count("A")
                if begun and not out.count("A") and ops[i - 1] == 0:
                    done = True  # the drained ring: the tile's loads are over
                    break
                begun = 1
            else:
                out = out[len(out) - op:] if op < len(out) else out
        if not done:
            todo += [(s, out, spare, begun) for s in bb[k][1]]
    return None


@pytest.mark.skipif(not (LLVM / "llvm-objdump").exists(), reason="no llvm-objdump")
def test_every_chunk_is_complete_at_its_barrier(tmp_path):
    if not LIB.exists():
        import __graft_entry__
        __graft_entry__.build()
    kernels = tile_kernels(LIB, tmp_path)
    tiles = 0
    for name, bb in kernels.items():
        n, bad = check(bb)
        tiles += n
        assert not bad, f"{name}: {bad}"
    print(len(kernels), "kernels,", tiles, "tiles")
    assert tiles >= 100


@pytest.mark.parametrize("order,ok", [("ATATAT", True), ("ATTTAA", False)])
def test_checker_on_a_ring_of_three(order, ok):
    """A ring of 3 chunks of one A load and one other: the prologue's loads chunk by chunk, or the A loads last, so
    that a wait for 4 outstanding leaves chunk 1's in flight at the barrier ahead of it."""
    ops = [{"A": "A", "T": "V"}[c] for c in order]
    bb = {"entry": (ops + [4, "B"], ["loop"]), "loop": (["A", "V", 4, "B"], ["loop", "end"]), "end": ([0, "B"], [])}
    assert (check(bb)[1] == []) == ok
