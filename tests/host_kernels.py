"""Compiles device code of iron_amd/csrc for the CPU (tests/cpu_block: one block at a
time, a fiber per thread) and runs a C++ main over it."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "iron_amd" / "csrc"
CPU_BLOCK = ROOT / "tests" / "cpu_block"
CLANG = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and Path(c).exists()), None)


def device_part(name, until="host side", close="}\n"):
    """A .hip file up to its host side: kernels and what they use, namespace closed."""
    text = (CSRC / name).read_text()
    return text[:text.index(until)].rsplit("\n", 1)[0] + "\n" + close


def definition(name, what):
    """One function, kernel or constant of a .hip file, from its template line on."""
    text = (CSRC / name).read_text()
    m = re.search(r"^(?:template [^\n]*\n)?[^\n;{}]*\b" + re.escape(what) + r"\b\s*(?:=[^\n]*;|\([^;{]*\{)", text, re.M)
    assert m, f"{what} not found in {name}"
    if m.group(0).endswith(";"):
        return m.group(0) + "\n"
    depth, i = 1, m.end()
    while depth:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        i += 1
    return text[m.start():i] + "\n"


def _no_launches(text):
    """Host launch statements become plain calls (main launches through the header)."""
    return re.sub(r"<<<.*?>>>", "", text, flags=re.S)


def build(tmp_path, source, main, *flags):
    """An executable of main() over the device source."""
    if CLANG is None:
        pytest.skip("no clang++")
    src, exe = tmp_path / "k.cpp", tmp_path / "k"
    for h in CSRC.glob("*.hpp"):
        (tmp_path / h.name).write_text(_no_launches(h.read_text().replace("../../include", str(ROOT / "include"))))
    src.write_text(_no_launches(source) + main)
    r = subprocess.run([CLANG, "-std=c++20", "-O1", "-w", *flags, f"-I{CPU_BLOCK}", str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


def run(exe, *args, timeout=120):
    """The numbers main() prints; fails the test on a nonzero exit."""
    r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-2000:]}{r.stderr[-2000:]}"
    return [float(v) for v in r.stdout.split()]
