"""The autotuner's variants build: their values pass the kernels' compile-time checks."""
import importlib.util
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(HERE, "cpm-ibc_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _tune():
    spec = importlib.util.spec_from_file_location("tune", os.path.join(PKG, "tune.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_default_is_the_header_s():
    t = _tune()
    text = open(os.path.join(PKG, "csrc", "tuned.h")).read()
    for k, name in t.DEFINES.items():
        assert f"#define {name} {t.DEFAULT[k]}\n" in text


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_variants_pass_the_kernels_checks():
    t = _tune()
    runs = []
    for v in t.VARIANTS:
        if dict(v, xcd_run=t.DEFAULT["xcd_run"]) == t.DEFAULT:   # the XCD run is in no check
            continue
        for src in ("tpfmt.hip", "krylov.hip"):
            runs.append((v, subprocess.Popen(
                [HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-Wno-unused-function"]
                + [f"-D{t.DEFINES[k]}={v[k]}" for k in t.DEFINES] + [os.path.join(PKG, "csrc", src)],
                stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)))
            if len(runs) % 6 == 0:
                runs[-6][1].wait(timeout=300)
    for v, p in runs:
        err = p.communicate(timeout=300)[1]
        assert p.returncode == 0, f"{v}: {err[-2000:]}"
