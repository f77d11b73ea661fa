"""The gfx950 instructions of the built library, for CPU tests of what only the compiled kernels show."""
import re
import subprocess
from functools import lru_cache
from pathlib import Path

LIB = Path(__file__).resolve().parent.parent / "nebula_amd" / "lib" / "libnebula_hq.so"
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


@lru_cache(maxsize=None)
def kernels(tmp: Path) -> dict:
    """Mangled kernel name -> its instructions [(address, opcode, operands, branch target or None)];
    tmp: a folder for the code objects."""
    lib = tmp / LIB.name
    lib.write_bytes(LIB.read_bytes())
    subprocess.run([str(OBJDUMP), "--offloading", lib.name], cwd=tmp, check=True, capture_output=True)
    out = {}
    for obj in sorted(tmp.glob("*gfx950")):
        text = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True,
                              text=True).stdout
        code, base = None, 0
        for line in text.splitlines():
            head = re.match(r"([0-9a-f]+) <(\w+)>:", line)
            if head:
                code, base = out.setdefault(head[2], []), int(head[1], 16)
                continue
            m = re.match(r"\t(\S+) ?(.*?)\s*// 0*([0-9A-F]+):(?:.*<\w+?(?:\+0x([0-9a-f]+))?>)?", line)
            if m and code is not None:
                to = base + int(m[4] or "0", 16) if "branch" in m[1] else None
                code.append((int(m[3], 16), m[1], m[2], to))
    return out


def unlanded_copies(code) -> list:
    """Addresses at which a wavefront meets others (s_barrier, or an arrival count in LDS) while one
    of its own copies from memory into LDS may still be in flight: the others would read the stage
    too early. Memory operations retire in issue order, so what matters is the fewest issued after
    the youngest such copy over all paths (None: no copy in flight), held against each wait's count."""
    at = {a: i for i, (a, *_) in enumerate(code)}
    state = {0: None}  # instruction -> operations behind the copy; the smaller, the worse
    work, bad = [0], set()
    while work:
        i = work.pop()
        addr, op, args, to = code[i]
        y = state[i]
        if op.startswith(("buffer_load", "buffer_store", "buffer_atomic", "global_", "flat_", "scratch_")):
            y = 0 if " lds" in args or "_lds" in op else y if y is None else min(y + 1, 64)
        elif op == "s_waitcnt" and y is not None:
            n = re.search(r"vmcnt\((\d+)\)", args)
            if n and y >= int(n[1]):
                y = None
        elif op in ("s_barrier", "ds_add_u32") and y is not None:
            bad.add(addr)
        succ = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if to is not None:
            succ.append(at[to])
        for j in succ:
            if j >= len(code):
                continue
            if j not in state or (y is not None and (state[j] is None or y < state[j])):
                state[j] = y
                work.append(j)
    return sorted(bad)
