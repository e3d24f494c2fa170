"""Whether the built extension keeps the distances that products.hip's matrix instructions need.

Those of its largest tiles are written in inline assembly, so that the compiler neither sees how long their results take nor
that they read registers early. What must hold is therefore looked for in the machine code, along every path of a kernel:

* no other instruction touches a result's registers within AFTER wait states of the product that writes it: this
  instruction (four passes) needs 7, one of eight passes 11;
* no product reads a register that a vector instruction has written within BEFORE wait states ahead of it;
* no product reads another's result but as its own sum, the whole of it, at least SAME wait states later.

A wait state is an instruction, or one of those that s_nop stands for. ``setup.py`` runs this behind each build.
"""

import os
import re
import shutil
import subprocess
import tempfile

AFTER, BEFORE, SAME = 11, 2, 3
_LINE = re.compile(r"^\s+(\S+)\s*(.*?)\s*//\s*([0-9A-F]+):(?:.*<[^>+]*(?:\+0x([0-9a-f]+))?>)?")
_REGISTERS = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _registers(text):
    return {(m[1], i) for m in _REGISTERS.finditer(text) for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)}


def _kernels(listing):
    name, lines = None, []
    for line in listing.splitlines():
        start = re.match(r"^([0-9a-f]+) <(.*)>:", line)
        if start:
            if name:
                yield name, at, lines
            name, at, lines = start[2], int(start[1], 16), []
        else:
            m = _LINE.match(line)
            if m:
                lines.append((m[1], m[2], int(m[3], 16), m[4]))
    if name:
        yield name, at, lines


def problems(listing, wanted):
    """Lines of what is too near in the kernels whose name has ``wanted``, and the number of products looked at."""
    found, seen = [], 0
    for name, start, lines in _kernels(listing):
        if wanted not in name:
            continue
        at = {address: i for i, (_, _, address, _) in enumerate(lines)}
        follow = []
        for i, (op, _, _, target) in enumerate(lines):
            after = [] if op in ("s_branch", "s_endpgm") or i + 1 == len(lines) else [i + 1]
            if op == "s_branch" or op.startswith("s_cbranch"):
                after.append(at[start + int(target or "0", 16)])
            follow.append(after)

        def near(i, states):
            """Instructions behind the i-th with fewer than ``states`` wait states between, with their number."""
            best, todo = {}, [(j, 0) for j in follow[i]]
            while todo:
                j, passed = todo.pop()
                if passed >= states or best.get(j, states) <= passed:
                    continue
                best[j] = passed
                op, args = lines[j][:2]
                todo += [(k, passed + (int(args) + 1 if op == "s_nop" else 1)) for k in follow[j]]
            return best

        for i, (op, args, address, _) in enumerate(lines):
            product = op.startswith("v_mfma")
            if not product and not op.startswith("v_"):
                continue
            operands = re.split(r",\s*", args)
            if product:
                seen += 1
                result = _registers(operands[0])
                for j, passed in near(i, AFTER).items():
                    other, text = lines[j][:2]
                    if not result & _registers(text):
                        continue
                    parts = re.split(r",\s*", text)
                    own = other == op and parts[0] == parts[3] == operands[0] and not result & _registers(" ".join(parts[1:3]))
                    if not own or passed < SAME:
                        found.append(f"{name} {address:x}: {op} {args}, {passed} states on: {other} {text}")
            else:
                written = _registers(args if "swap" in op else operands[0])
                for j, passed in near(i, BEFORE).items() if written else ():
                    if lines[j][0].startswith("v_mfma") and written & _registers(lines[j][1]):
                        found.append(f"{name} {address:x}: {op} {args}, {passed} states on: {lines[j][0]} {lines[j][1]}")
    return found, seen


def listing(extension, wanted, objdump):
    """The machine code of the extension's part that has kernels of this name."""
    with tempfile.TemporaryDirectory() as folder:
        copy = os.path.join(folder, "extension.so")
        shutil.copy(extension, copy)
        subprocess.run([objdump, "--offloading", copy], check=True, stdout=subprocess.DEVNULL, cwd=folder)
        for part in sorted(os.listdir(folder)):
            path = os.path.join(folder, part)
            if part.endswith("gfx950"):
                with open(path, "rb") as f:
                    if wanted.encode() in f.read():
                        return subprocess.run([objdump, "-d", path], check=True, capture_output=True, text=True).stdout
    return ""


def objdump():
    path = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
    return path if os.path.exists(path) else None


# product_kernel<true, true, 256, ...>: the tiles whose products are inline assembly
WANTED = "14product_kernelILb1ELb1ELi256E"


def check(extension):
    """Raises where a distance is too short, or where the products are not found. Without the disassembler nothing is looked at."""
    tool = objdump()
    if tool is None:
        print(f"{extension}: no llvm-objdump, the distances of products.hip's matrix instructions are not checked")
        return
    found, seen = problems(listing(extension, WANTED, tool), WANTED)
    if found or seen < 256 + 128:
        raise RuntimeError("\n".join([f"{extension}: matrix instructions too near their operands ({seen} looked at)"] + found[:20]))
    print(f"{extension}: {seen} matrix instructions of products.hip keep their distances")
