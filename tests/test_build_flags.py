"""The library's Makefile rebuilds its objects when the compiler, its flags or
the Makefile change: in a copy of the folder, with a stand-in compiler."""
import os
import shutil
import subprocess
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("make") is None, reason="no make")
def test_objects_follow_flags(tmp_path):
    csrc = tmp_path / "anchorwave_amd" / "csrc"
    shutil.copytree(os.path.join(ROOT, "anchorwave_amd", "csrc"), csrc, ignore=shutil.ignore_patterns("build"))
    shutil.copytree(os.path.join(ROOT, "include"), tmp_path / "include")
    log = tmp_path / "log"
    compilers = []
    for name in ("cc1", "cc2"):
        cc = tmp_path / name
        cc.write_text(f"""#!/bin/sh
echo "$@" >> {log}
while [ $# -gt 0 ]; do [ "$1" = -o ] && touch "$2"; shift; done
""")
        cc.chmod(0o755)
        compilers.append(str(cc))

    def compiled(*args):
        log.write_text("")
        subprocess.run(["make", "-C", str(csrc), *args], check=True, capture_output=True)
        return sum(" -c " in line for line in log.read_text().splitlines())

    first = compiled(f"HIPCC={compilers[0]}")
    assert first == len(list(csrc.glob("*.hip")) + list(csrc.glob("*.cpp")))
    assert compiled(f"HIPCC={compilers[0]}") == 0
    assert compiled(f"HIPCC={compilers[0]}", "ARCH=gfx942") == first
    assert compiled(f"HIPCC={compilers[0]}", "ARCH=gfx942") == 0
    assert compiled(f"HIPCC={compilers[1]}", "ARCH=gfx942") == first
    makefile = csrc / "Makefile"
    later = time.time() + 10
    os.utime(makefile, (later, later))
    assert compiled(f"HIPCC={compilers[1]}", "ARCH=gfx942") == first
    # and one source alone
    later += 10
    os.utime(csrc / "ksw2_api.cpp", (later, later))
    for obj in (csrc / "build").iterdir():
        os.utime(obj, (later - 5, later - 5))
    assert compiled(f"HIPCC={compilers[1]}", "ARCH=gfx942") == 1
