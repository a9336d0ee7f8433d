"""Build-time guard: lists the instructions of the scalar data cache other than
loads (any scalar instruction named for a store, an atomic or that cache itself)
found in device assembly.  The library writes only through vector memory
instructions; the build fails if the compiler ever emits one of these.
Host-side only."""
import re

_PATTERN = re.compile(r"^\s*(s_(?:\w+_)?(?:store|atomic|dcache)\w*)", re.M)


def scalar_cache_writes(asm_text: str):
    return sorted(set(_PATTERN.findall(asm_text)))
