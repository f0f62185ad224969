"""Rules of the gfx950 code that the compiler cannot check, because the instructions come from
inline assembly: read from the assembly of the built library's own code objects (no GPU)."""
import os
import re
import shutil
import subprocess

from kata_amd.build import LIB

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _assembly(tmp_path):
    """The instruction lines of every gfx950 code object in the library, in order."""
    so = shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", so], check=True, capture_output=True)
    lines = []
    for f in sorted(os.listdir(tmp_path)):
        if f.endswith("gfx950"):
            r = subprocess.run([OBJDUMP, "-d", str(tmp_path / f)], check=True, capture_output=True, text=True)
            lines += [l.split("//")[0].strip() for l in r.stdout.splitlines() if l.startswith("\t")]
    return lines


def test_wait_state_between_m0_and_lds_copy(tmp_path):
    """An instruction that writes M0 and a copy into LDS, whose LDS address is M0, need one wait
    state between them; the hazard recogniser does not look into inline assembly."""
    asm = _assembly(tmp_path)
    copies = [i for i, l in enumerate(asm) if re.match(r"(global|buffer)_load.*\blds\b|global_load_lds_", l)]
    assert len(copies) > 100                       # the GEMMs' loops are full of them
    bad = [f"{asm[i - 1]} ; {asm[i]}" for i in copies if re.match(r"s_\w+ m0\b", asm[i - 1])]
    assert not bad, f"{len(bad)} of {len(copies)}: {bad[0]}"


def test_wait_states_between_vector_sgpr_write_and_lds_copy(tmp_path):
    """A copy whose base address is in SGPRs needs five wait states after a vector instruction that
    wrote one of them (a readlane of a spilled address, say); s_nop n is n + 1 of them."""
    asm = _assembly(tmp_path)
    bad = []
    for i, l in enumerate(asm):
        m = re.match(r"global_load_lds_\w+ v\d+, s\[(\d+):(\d+)\]", l)
        states = 0
        for j in range(i - 1, max(i - 6, -1), -1) if m else ():
            if states >= 5:
                break
            w = re.match(r"v_\w+ s(?:\[(\d+):(\d+)\]|(\d+))", asm[j])
            if w:
                lo, hi = int(w[1] or w[3]), int(w[2] or w[3])
                if lo <= int(m[2]) and hi >= int(m[1]):
                    bad.append(f"{asm[j]} ; {l}")
            n = re.match(r"s_nop (\d+)", asm[j])
            states += int(n[1]) + 1 if n else 1
    assert not bad, f"{len(bad)}: {bad[0]}"
