"""The ctypes structures in h3_flash_amd/_ext.py against the C header: a C
program compiled from include/h3attn.h prints sizeof and offsetof of every
field that the binding declares, and both must agree (a field missing from
the header fails to compile)."""

from __future__ import annotations

import ctypes
import json
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from h3_flash_amd import _ext

ROOT = Path(__file__).resolve().parents[1]
STRUCTS = {
    "h3a_attn_args": _ext.AttnArgs,
    "h3a_qknorm_rope_args": _ext.QkNormRopeArgs,
    "h3a_pack_qkv_args": _ext.PackQkvArgs,
    "h3a_merge_heads_args": _ext.MergeHeadsArgs,
    "h3a_qknorm_rope_pack_args": _ext.QkNormRopePackArgs,
    "h3a_rmsnorm_modulate_args": _ext.RmsnormModulateArgs,
    "h3a_residual_gate_rmsnorm_modulate_args": _ext.ResidualGateRmsnormModulateArgs,
    "h3a_swiglu_args": _ext.SwigluArgs,
    "h3a_attn_merge_args": _ext.AttnMergeArgs,
    "h3a_proj_section": _ext.ProjSection,
    "h3a_proj_args": _ext.ProjArgs,
}


@pytest.fixture(scope="module")
def c_layout(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    lines = ["#include <stddef.h>", "#include <stdio.h>", '#include "h3attn.h"', "int main(void) {", 'printf("{");']
    first = True
    for cname, cls in STRUCTS.items():
        sep = "" if first else ","
        first = False
        lines.append(f'printf("{sep}\\"{cname}\\": {{\\"size\\": %zu", sizeof({cname}));')
        for field, _ in cls._fields_:
            lines.append(f'printf(", \\"{field}\\": %zu", offsetof({cname}, {field}));')
        lines.append('printf("}");')
    lines += ['printf("}\\n");', "return 0;", "}"]
    d = tmp_path_factory.mktemp("abi")
    src, exe = d / "layout.c", d / "layout"
    src.write_text("\n".join(lines) + "\n")
    subprocess.run([cc, "-std=c11", "-I", str(ROOT / "include"), str(src), "-o", str(exe)], check=True)
    return json.loads(subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout)


@pytest.mark.parametrize("cname", sorted(STRUCTS))
def test_ctypes_structure_matches_the_header(c_layout, cname):
    cls = STRUCTS[cname]
    want = c_layout[cname]
    assert ctypes.sizeof(cls) == want["size"], (cname, ctypes.sizeof(cls), want["size"])
    for field, _ in cls._fields_:
        assert getattr(cls, field).offset == want[field], (cname, field)


# The packed form of every entry point's arguments: each member at its ctypes
# offset, and values beyond a member's range as C would convert them.
@pytest.mark.parametrize(
    "launch, ctype",
    [(_ext.attn_fwd, _ext.AttnArgs), (_ext.qknorm_rope, _ext.QkNormRopeArgs), (_ext.pack_qkv, _ext.PackQkvArgs),
     (_ext.merge_heads, _ext.MergeHeadsArgs), (_ext.qknorm_rope_pack, _ext.QkNormRopePackArgs),
     (_ext.rmsnorm_modulate, _ext.RmsnormModulateArgs),
     (_ext.residual_gate_rmsnorm_modulate, _ext.ResidualGateRmsnormModulateArgs), (_ext.swiglu, _ext.SwigluArgs),
     (_ext.attn_merge, _ext.AttnMergeArgs), (_ext.proj_gemm, _ext.ProjArgs)],
)
def test_packed_arguments_match_the_structure(launch, ctype):
    def members(obj):
        for name, t in obj._fields_:
            v = getattr(obj, name)
            if hasattr(t, "_fields_"):
                yield from members(v)
            elif hasattr(t, "_length_"):
                for x in v:
                    if hasattr(x, "_fields_"):
                        yield from members(x)
                    else:
                        yield x or 0
            else:
                yield v or 0

    raw = bytes((37 * i + 11) % 120 + 1 for i in range(ctypes.sizeof(ctype)))
    args = ctype.from_buffer_copy(raw)
    packed = launch._pack(*members(args))
    assert len(packed) == ctypes.sizeof(ctype)
    assert list(members(ctype.from_buffer_copy(packed))) == list(members(args))


def test_host_tensors_never_reach_a_launch(monkeypatch):
    """An entry point called with tensors that are not on a GPU raises before
    the library is called (the kernel would read host addresses)."""
    from h3_flash_amd.projection import Section, proj_gemm

    called = []
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0, raising=False)
    monkeypatch.setattr(_ext.proj_gemm, "_proto", lambda bound: lambda *args: called.append(args) or 0)
    monkeypatch.setattr(_ext.proj_gemm, "_bound", (None, None))
    monkeypatch.setattr(_ext, "load_library", lambda path=None: called)
    x, w = torch.zeros(4, 128, dtype=torch.bfloat16), torch.zeros(128, 128, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="ROCm device"):
        proj_gemm(x, [Section(w, torch.empty(4, 128, dtype=torch.bfloat16))])
    assert called == []
