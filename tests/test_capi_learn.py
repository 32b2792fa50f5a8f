"""include/qqt_learn.h (no GPU needed): the library exports what the header
declares, and its structs have the layout of their ctypes mirrors."""

from __future__ import annotations

import ctypes
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "qqt_learn.h")


def _text():
    return re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)


def test_the_declared_entry_points_are_exported():
    from qqtsim import _capi

    names = sorted(set(re.findall(r"^\s*[\w\s\*]+?\b(qqt_\w+)\s*\(", _text(), flags=re.M)))
    assert names == ["qqt_l1_grad_columns", "qqt_l1_grad_preferred_floats",
                     "qqt_lstm_seq_backward", "qqt_lstm_seq_forward", "qqt_ppo_step",
                     "qqt_ppo_step_workspace_bytes", "qqt_w0_pack"]
    lib = _capi.lib()
    assert all(hasattr(lib, n) for n in names)


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_struct_layouts_match_the_header(tmp_path):
    from qqtsim import _capi

    structs = {"qqt_ppo_step_args": _capi.PpoStepArgsC, "qqt_lstm_seq_args": _capi.LstmSeqArgsC}
    assert sorted(structs) == sorted(re.findall(r"typedef struct (\w+)", _text()))
    lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "qqt_hip.h"',
             '#include "qqt_learn.h"', 'int main(void) {']
    for cname, cls in structs.items():
        lines.append(f'  printf("{cname} size %zu\\n", sizeof({cname}));')
        lines += [f'  printf("{cname} {f} %zu\\n", offsetof({cname}, {f}));' for f, _ in cls._fields_]
    src, exe = tmp_path / "layout.c", tmp_path / "layout"
    src.write_text("\n".join(lines + ["  return 0;", "}"]) + "\n")
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    got = {tuple(line.split()[:2]): int(line.split()[2]) for line in out.strip().splitlines()}
    for cname, cls in structs.items():
        assert got[(cname, "size")] == ctypes.sizeof(cls), cname
        for f, _ in cls._fields_:
            assert got[(cname, f)] == getattr(cls, f).offset, (cname, f)
