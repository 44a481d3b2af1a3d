"""Check of the built gfx950 code: no vector instruction before a join's exec restore.

Where the lanes of a wavefront come together again, the block starts with the instruction that
restores their mask (s_or_b64 exec, or a saveexec form).  The register allocator of the compiler
the library is built with (clang 22, ROCm 7.2) can put the spill of a vector register in front of
it when copies of scalar registers stand there already.  Such a spill stores for the lanes that
are active in front of the restore, after a loop over lanes for none at all, and every later
reload returns what the scratch memory held.  One build of the fused multi-network kernel lost two
coefficients of its logarithm that way and returned wrong abundances without any error; whether a
build does depends on its register pressure, so every build is checked.

A block counts as a join if a branch on an empty mask (s_cbranch_execz) leads to it right after
the mask was narrowed, or if it follows a loop's branch on a non-empty one (s_cbranch_execnz): its
first instructions may run with no lane active, so a vector instruction that only some lanes were to
skip cannot be there.  (The compiler also writes branches that are never taken as s_cbranch_execz,
behind no change of the mask: their targets are ordinary code.)

    python3 isa_check.py lib/libnnet_mi355x.so     lists the findings, exit status 1 if any
"""
import os
import re
import subprocess
import sys
import tempfile

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")

_FUNC = re.compile(r"^([0-9a-f]+) <(\S+)>:$")
_INS = re.compile(r"^\t(\S+)(?: (.*?))?\s*// ([0-9A-F]+):[0-9A-F ]*(?:<([^>+]+)(?:\+0x([0-9a-f]+))?>)?$")
# vector instructions whose effect does not depend on the active lanes
_ANY_LANES = re.compile(r"v_(readlane|writelane|readfirstlane|mfma|nop)")
# a join gives lanes back: the mask of the branch it ends, or the other side of an if / else
_RESTORE = re.compile(r"s_or_b64 exec, exec,|s_mov_b64 exec,|s_(or|andn2)_saveexec_b64")
# the mask loses lanes (an else: what its saveexec form gave back, less the other side)
_NARROW = re.compile(r"s_(and|andn2|xor)_b64 exec,|s_(and|andn2)_saveexec_b64")
_VECTOR = re.compile(r"(v|scratch|global|flat|ds|buffer)_")


def _kernels(text):
    """(name, [(address, opcode, operands, branch target)]) of each function of a disassembly."""
    name, ins, base = None, [], {}
    for line in text.splitlines():
        m = _FUNC.match(line)
        if m:
            if ins:
                yield name, ins
            name, ins = m.group(2), []
            base[name] = int(m.group(1), 16)
            continue
        m = _INS.match(line)
        if m:
            target = base.get(m.group(4), 0) + int(m.group(5) or "0", 16) if m.group(4) else None
            ins.append((int(m.group(3), 16), m.group(1), m.group(2) or "", target))
    if ins:
        yield name, ins


def findings(text):
    """[(function, address, instruction)] of the misplaced instructions in a disassembly, and the
    number of joins looked at."""
    found, joins = [], 0
    for name, ins in _kernels(text):
        starts, narrowed = set(), False
        targets = {t for _, _, _, t in ins if t is not None}
        for k, (a, op, args, target) in enumerate(ins):
            if a in targets:
                narrowed = False
            if _NARROW.match(f"{op} {args}"):
                narrowed = True
            elif _RESTORE.match(f"{op} {args}"):
                narrowed = False
            elif op == "s_cbranch_execz" and narrowed:
                starts.add(target)
            elif op == "s_cbranch_execnz" and narrowed and k + 1 < len(ins):
                nxt = ins[k + 1]
                starts.add(nxt[3] if nxt[1] == "s_branch" else nxt[0])
            if op.startswith(("s_cbranch", "s_branch", "s_setpc")):
                narrowed = False
        at = {a: k for k, (a, _, _, _) in enumerate(ins)}
        for s in sorted(starts):
            joins += 1
            seen = []
            for a, op, args, _ in ins[at[s]:]:
                if _RESTORE.match(f"{op} {args}"):
                    found += [(name, x, i) for x, i in seen]
                    break
                if "saveexec" in op or (op.startswith("s_") and args.startswith("exec")):
                    break  # the next, narrower branch
                if op.startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")):
                    break
                if _VECTOR.match(op) and not _ANY_LANES.match(op):
                    seen.append((a, f"{op} {args}"))
    return found, joins


def disassemble(lib):
    """The disassembly of every gfx950 code object in the library."""
    out = []
    with tempfile.TemporaryDirectory() as tmp:
        link = os.path.join(tmp, "lib.so")
        os.symlink(os.path.abspath(lib), link)
        subprocess.run([OBJDUMP, "--offloading", link], check=True, cwd=tmp, capture_output=True)
        objects = sorted(f for f in os.listdir(tmp) if f.endswith("gfx950"))
        if not objects:
            raise RuntimeError(f"no gfx950 code object in {lib}")
        for f in objects:
            out.append(subprocess.run([OBJDUMP, "-d", os.path.join(tmp, f)], check=True, capture_output=True,
                                      text=True).stdout)
    return "\n".join(out)


def main(lib):
    if not os.path.exists(OBJDUMP):
        print(f"isa_check: {OBJDUMP} not there, {lib} not checked")
        return 0
    found, joins = findings(disassemble(lib))
    for name, address, ins in found:
        print(f"isa_check: {name}: {address:#x}: {ins}: in front of the restore of the lane mask")
    print(f"isa_check: {lib}: {joins} joins, {len(found)} misplaced vector instructions")
    return 1 if found else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1]))
