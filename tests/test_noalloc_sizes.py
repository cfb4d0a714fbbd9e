"""CPU check of the workspace of olx_asm_c64_noalloc: the mixed-radix passes pad the intermediate's columns, and
every field whose unpadded intermediate fits the 64 MiB that the entry point admits fits the 72 MiB it holds."""
from openol_amd import _lib


def test_padded_columns_fit():
    columns = getattr(_lib.load(), "_ZN3olx10mr_columnsEi")
    sides = [n for n in range(2, 8193) if _lib.load()._ZN3olx12mr_supportedEl(2 * n) & 1]
    assert len(sides) > 600
    for nx in sides:
        c = columns(nx)
        assert 2 * nx <= c <= 2 * (nx + 48) and c % 8 == 0
        # the tallest field of this width
        ny = max((n for n in sides if 8 * n * ((2 * nx + 7) & ~7) <= 64 << 20), default=0)
        assert 8 * ny * c <= 72 << 20
    assert columns(17) == 0
