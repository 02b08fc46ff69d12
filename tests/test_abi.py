"""The C ABI library loads and exports every symbol include/mmff_hip.h declares (no
compute calls: this runs without a GPU)."""
from __future__ import annotations

import ctypes
import re
from pathlib import Path

from mlxmolkit_archive_amd import _lib
from mlxmolkit_archive_amd._build import lib_path

HEADER = Path(__file__).resolve().parents[1] / "include" / "mmff_hip.h"


def declared_symbols():
    txt = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(mmffhip_[a-z_0-9]+)\s*\(", txt)))


def test_library_exports_every_declared_symbol():
    L = ctypes.CDLL(str(lib_path("libmmff_hip.so")))
    syms = declared_symbols()
    assert len(syms) >= 9
    for s in syms:
        assert hasattr(L, s), s
    assert set(syms) == set(_lib.SIGNATURES)  # the ctypes binding covers the whole ABI


def test_abi_version_and_struct_sizes():
    L = _lib.load()
    assert L.mmffhip_abi_version() == _lib.ABI_VERSION
    assert ctypes.sizeof(_lib.Batch) == 16 * 8 + 3 * 4 + 4  # 16 pointers + 3 int32 (+ padding)
    assert ctypes.sizeof(_lib.NkOpts) == 8 * 4 + 8 + 8 + 8  # ... precond, table_lds_bytes (+ pad), xcd_offsets


def test_oracle_is_not_linked_by_the_product():
    """The product library must not depend on the oracle in any form."""
    data = lib_path("libmmff_hip.so").read_bytes()
    assert b"oracle" not in data


def test_training_workspace_grows_with_the_batch():
    """A workspace allocated for the largest batch serves the smaller ones: the size never falls as
    atoms are added, also where the tiles spread over fewer workgroups (16,384 -> 16,385 atoms)."""
    L = _lib.load()
    sizes = []
    for n in [*range(0, 70), *range(63, 40000, 64), *range(64, 40000, 64), *range(65, 40000, 64), 2**31 - 1]:
        b = ctypes.c_size_t()
        assert L.mmffhip_mlp_workspace(n, ctypes.byref(b)) == 0
        sizes.append((n, b.value))
    sizes.sort()
    assert all(a[1] <= b[1] for a, b in zip(sizes, sizes[1:]))
    at = dict(sizes)
    assert at[1] > at[0] and at[16384] == at[16385] and at[32768] == at[32769]
