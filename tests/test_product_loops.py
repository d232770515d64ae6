"""The main loops of the products by tiles, as they were compiled: their only wait for
memory is the counted one, which lets the loads of the units ahead stay on their way.
(A register that is spilled around such a loop puts waits for everything into it.)"""
import glob
import os
import re
import subprocess

import pytest

import polyrl_amd

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def main_loops(text):
    """(name, instructions) of every kernel's innermost loops with products."""
    for kernel in re.finditer(r"^[0-9a-f]+ <(\S*(?:product|parts|linear)_kernel\S*)>:\n"
                              r"(.*?)(?=^$|\Z)", text, re.S | re.M):
        name, code = kernel.group(1), []
        for line in kernel.group(2).splitlines():
            m = re.match(r"\s+(.*?)\s*// ([0-9A-F]+):", line)
            if m:
                code.append((int(m.group(2), 16), m.group(1), line))
        at = {a: i for i, (a, _, _) in enumerate(code)}
        loops = []
        for i, (_, ins, line) in enumerate(code):
            m = re.search(r"<\S+\+0x([0-9a-f]+)>$", line)
            if m and re.match(r"s_c?branch", ins):
                to = at.get(code[0][0] + int(m.group(1), 16))
                if to is not None and to < i:
                    loops.append((to, i))
        for a, b in loops:
            if any(a <= c and d <= b and (c, d) != (a, b) for c, d in loops):
                continue
            body = [ins for _, ins, _ in code[a:b + 1]]
            if any(ins.startswith("v_mfma") for ins in body):
                yield name, body


def test_waits(tmp_path):
    built = glob.glob(os.path.join(os.path.dirname(polyrl_amd.__file__), "_hip.*.so"))
    if not built or not os.path.exists(OBJDUMP):
        pytest.skip("no built extension or no disassembler")
    os.symlink(built[0], tmp_path / "hip.so")
    subprocess.run([OBJDUMP, "--offloading", "hip.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    seen = set()
    for part in sorted(tmp_path.glob("hip.so.*gfx950")):
        names = subprocess.run([OBJDUMP, "-t", part], check=True, text=True,
                               stdout=subprocess.PIPE).stdout
        if not re.search("(product|parts|linear)_kernelI", names):
            continue
        text = subprocess.run([OBJDUMP, "-d", part], check=True, text=True,
                              stdout=subprocess.PIPE).stdout
        for name, body in main_loops(text):
            form = re.search(r"(product_kernelILb[01]ELi\d|parts_kernelILi\dELi\d"
                             r"|linear_kernelILi\dELN\S*?KindE\d)", name).group(1)
            seen.add(form)
            waits = [ins for ins in body if "vmcnt" in ins]
            assert len(waits) == 1 and "vmcnt(0)" not in waits[0], (form, waits)
            assert not any("scratch" in ins for ins in body), form
    # forms: weights' and input gradients, sums of two and three, four kinds of forward
    # products (with what is kept from 6 row parts on)
    assert len(seen) == 4 + 6 + 3 * 6 + 3, sorted(seen)
