"""Host-side pin of the end flags of a GMRES cycle.

A launch that carries a Hessenberg update (or a cycle's start) writes the flags
in its first workgroup while its others read them: what they read must not be
what it writes, or the wavefronts of one workgroup could disagree before a
barrier.  tests/native/cycle_flags_check.cpp drives the functions of
vivlasov1d_amd/csrc/gmres_dev.h through histories of solves and asserts that
every launch's answer is unchanged by its own writes and right.  Planted
mistakes (the flag of the same launch, a restart that reads the reason, the
wrong parity) in a copy of the header are each reported."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vivlasov1d_amd", "csrc")


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    pytest.skip("hipcc not available")


def _run(tmp_path, edit=None):
    for d in ("vivlasov1d_amd/csrc", "tests/native", "include"):
        (tmp_path / d).mkdir(parents=True)
    for name in ("gmres_dev.h", "vv1d_internal.h", "wave_ops.h", "tile_index.h"):
        text = open(os.path.join(CSRC, name)).read()
        if edit and name == "gmres_dev.h":
            assert text.count(edit[0]) == 1, edit[0]
            text = text.replace(*edit)
        (tmp_path / "vivlasov1d_amd" / "csrc" / name).write_text(text)
    shutil.copy(os.path.join(ROOT, "include", "vv1d.h"), tmp_path / "include")
    src = shutil.copy(os.path.join(ROOT, "tests", "native", "cycle_flags_check.cpp"), tmp_path / "tests" / "native")
    exe = str(tmp_path / "check")
    subprocess.run([_hipcc(), "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-value", str(src),
                    "-o", exe], check=True, cwd=str(tmp_path))
    out = subprocess.run([exe], capture_output=True, text=True)
    m = re.search(r"checked (\d+) launches, (\d+) failures", out.stdout)
    assert m, out.stdout
    return out, int(m.group(1)), int(m.group(2))


def test_flags(tmp_path):
    out, launches, failures = _run(tmp_path)
    assert out.returncode == 0 and failures == 0 and launches > 10000, out.stdout


PLANTED = {
    "the flag that the same launch writes": ("return g->skip[a.it & 1] != 0;", "return g->st.done != 0;"),
    "a restart that reads the reason": ("return g->over != 0;", "return !g->st.active || g->st.reason != 0;"),
    "the wrong parity": ("g->skip[(it + 1) & 1] = end;", "g->skip[it & 1] = end;"),
}


@pytest.mark.parametrize("name", sorted(PLANTED))
def test_planted_mistake_is_reported(name, tmp_path):
    out, _, failures = _run(tmp_path, PLANTED[name])
    assert out.returncode != 0 and failures > 0, out.stdout
