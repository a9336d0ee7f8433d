"""The build's check of device assembly, on the CPU: scalar instructions named
for a store, an atomic or the scalar data cache are listed by whatever prefix
and suffix they carry, vector memory instructions and scalar loads are not."""
import importlib.util
import pathlib

import pytest

PATH = pathlib.Path(__file__).parents[1] / "fastgeodis_amd" / "_asm_guard.py"
SPEC = importlib.util.spec_from_file_location("fg_asm_guard", PATH)
GUARD = importlib.util.module_from_spec(SPEC)
SPEC.loader.exec_module(GUARD)


@pytest.mark.parametrize("family", ["store", "atomic", "dcache"])
@pytest.mark.parametrize("before,after", [("", "_some_form"), ("other_", "_some_form_x4"), ("other_", "")])
def test_scalar_cache_writes_are_listed(family, before, after):
    name = f"s_{before}{family}{after}"
    assert GUARD.scalar_cache_writes(f"\tv_mov_b32 v0, 0\n\t{name} s4, s[0:1], 0x0\n") == [name]


@pytest.mark.parametrize("line", ["global_store_dword v[0:1], v2, off", "buffer_store_dwordx2 v[0:1], v2, s[0:3], 0 offen",
                                  "global_atomic_add_u32 v0, v1, s[0:1]", "ds_write_b32 v0, v1", "s_load_dwordx4 s[0:3], s[4:5], 0x0",
                                  "s_waitcnt vmcnt(0)", "; s_or_b32 and a store in a comment"])
def test_others_are_not(line):
    assert GUARD.scalar_cache_writes(f"\t{line}\n") == []
