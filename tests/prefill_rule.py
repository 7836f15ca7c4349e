"""csrc/prefill_rule.h compiled by the host compiler: which kernels a prefill of 32-token chunks
runs, for tests that aim at one of them."""

from __future__ import annotations

import ctypes
import functools
import shutil
import subprocess
import tempfile
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "lightdelta_amd" / "csrc"

SHIM = r"""
#include "prefill_rule.h"
extern "C" int plan(int64_t tokens, int64_t sequences, int heads, int64_t gate_row) {
  const ld::Plan32 p = ld::plan_chunks32(tokens, sequences, heads, gate_row);
  return (p.own ? 1 : 0) | (p.heads ? 2 : 0) | (p.rows ? 4 : 0);
}
extern "C" int reads_qkv(int64_t tokens, int64_t sequences, int heads, int64_t gate_row,
                         int64_t qkv_row, int64_t qkv_width) {
  return ld::reads_qkv32(ld::plan_chunks32(tokens, sequences, heads, gate_row), qkv_row, qkv_width);
}
extern "C" int whole_heads(int64_t tokens, int64_t sequences, int heads, int64_t gate_row,
                           int64_t chunks, int64_t longest) {
  return ld::plan_chunks32(tokens, sequences, heads, gate_row).rule.whole_heads(chunks, longest);
}
"""


@functools.lru_cache(maxsize=1)
def _library():
    cxx = shutil.which("g++") or shutil.which("c++")
    with tempfile.TemporaryDirectory() as tmp:
        source, built = Path(tmp) / "rule.cpp", Path(tmp) / "rule.so"
        source.write_text(SHIM)
        subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(source),
                        "-o", str(built)], check=True, timeout=60)
        lib = ctypes.CDLL(str(built))
    i64 = ctypes.c_int64
    lib.plan.argtypes = [i64, i64, ctypes.c_int, i64]
    lib.reads_qkv.argtypes = [i64, i64, ctypes.c_int, i64, i64, i64]
    lib.whole_heads.argtypes = [i64, i64, ctypes.c_int, i64, i64, i64]
    return lib


def plan(lengths, num_v_heads, gate_row=None):
    """(own, heads, rows): the workgroups prepare their chunks themselves; which sides are
    launched."""
    row = 128 * num_v_heads if gate_row is None else gate_row
    bits = _library().plan(sum(lengths), len(lengths), num_v_heads, row)
    return bool(bits & 1), bool(bits & 2), bool(bits & 4)


def reads_qkv(lengths, num_v_heads, qkv_row, qkv_width):
    """False: the 64-token form runs instead."""
    return bool(_library().reads_qkv(sum(lengths), len(lengths), num_v_heads, 128 * num_v_heads,
                                     qkv_row, qkv_width))


def side(lengths, num_v_heads, gate_row=None):
    """The kernels whose results stand: "own" or "records" (whole heads, by who prepares the
    chunks) or "rows" (row blocks)."""
    row = 128 * num_v_heads if gate_row is None else gate_row
    own, heads, rows = plan(lengths, num_v_heads, row)
    if heads and rows:
        chunks = [(n + 31) // 32 for n in lengths]
        heads = bool(_library().whole_heads(sum(lengths), len(lengths), num_v_heads, row,
                                            sum(chunks), max(chunks)))
    if not heads:
        return "rows"
    return "own" if own else "records"
