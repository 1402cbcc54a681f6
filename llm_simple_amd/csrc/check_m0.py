"""Checks that nothing but the kernels' own assembly uses M0.

The tile loads of flash_prefill.hip and matmul_tile.hip write M0, the LDS address of a load, in one assembly statement and use
it in the three loads after.  The compiler does not see that: it must need M0 for nothing itself in between.  In the built code
every instruction of these kernels that names M0 has to be one that they wrote:

    s_add_u32 m0, ...   s_nop 0                          for the loads that follow
    s_mov_b32 m0, sN    s_nop 0    global_load_lds_...   for the load of the same statement

  check_m0.py OBJECT...     objects or libraries with gfx950 code; exits with 1 if an instruction is neither
"""
import glob
import os
import re
import shutil
import subprocess
import sys
import tempfile

KERNELS = ("flash_prefill_kernel", "matmul_tile_kernel")
OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")


def foreign_uses(listing):
    """(uses of M0 in the kernels, those that are none of the two forms: kernel and instruction) of a disassembly."""
    kernel, code, uses, foreign = None, [], 0, []
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if head:
            kernel = head.group(1) if any(k in head.group(1) for k in KERNELS) else None
        elif kernel and line.startswith("\t"):
            code.append((kernel, " ".join(line.split("//")[0].split())))
    for i, (kernel, text) in enumerate(code):
        if not re.search(r"\bm0\b", text):
            continue
        uses += 1
        after = [t for _, t in code[i + 1:i + 3]]
        own = re.match(r"s_add_u32 m0, s\d+, ", text) and after[:1] == ["s_nop 0"]
        own = own or (re.match(r"s_mov_b32 m0, s\d+$", text) and after[:1] == ["s_nop 0"]
                      and after[1:] and after[1].startswith("global_load_lds_"))
        if not own:
            foreign.append((kernel, text))
    return uses, foreign


def listings(path):
    with tempfile.TemporaryDirectory() as tmp:
        copy = os.path.join(tmp, os.path.basename(path))
        shutil.copy(path, copy)
        subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True)  # writes beside its input
        for part in sorted(glob.glob(copy + ".*gfx950")):
            yield subprocess.run([OBJDUMP, "-d", part], check=True, capture_output=True, text=True).stdout


def check(path):
    uses, foreign = 0, []
    for listing in listings(path):
        u, f = foreign_uses(listing)
        uses, foreign = uses + u, foreign + f
    return uses, foreign


def main(paths):
    bad = False
    for path in paths:
        uses, foreign = check(path)
        for kernel, text in foreign:
            print("%s: %s: M0 used outside of the tile loads: %s" % (path, kernel, text), file=sys.stderr)
        if not uses:
            print("%s: no tile load found" % path, file=sys.stderr)
        bad = bad or foreign or not uses
    return 1 if bad else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
