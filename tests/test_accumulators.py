"""What the build asks of kernels whose accumulators are registers by name: that the compiler has left those alone."""
import pytest

from xgserve import _build

KERNEL = """
0000000000001000 <_ZN3xgm18tile_linear_kernelILi4ELi4EEEv>:
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[12:15], 0      // 000000001000: D3B58000 02021908
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[12:15], a[0:3] // 000000001008: D3B58000 04021908
\tv_accvgpr_read_b32 v70, a0                                 // 000000001010: D3D84046 18000100
\ts_waitcnt vmcnt(0)                                         // 000000001018: BF8C0F70
"""


def test_products_onto_themselves_and_reads_pass():
    assert _build.check_accumulators(KERNEL) == 1
    other = "0000000000002000 <_ZN3xgm11some_kernelEv>:\n\tv_accvgpr_write_b32 a0, v1\n\tscratch_store_dword off, v1, s0\n"
    assert _build.check_accumulators(KERNEL + other) == 1


@pytest.mark.parametrize("op", [
    "v_accvgpr_write_b32 a3, v1", "v_accvgpr_mov_b32 a1, a0", "v_accvgpr_read_b32 a4, a0",
    "v_mfma_f32_16x16x32_bf16 a[4:7], v[8:11], v[12:15], a[0:3]", "v_mfma_f32_16x16x32_bf16 v[4:7], v[8:11], v[12:15], a[0:3]",
    "v_mfma_f32_16x16x32_bf16 a[0:3], a[8:11], v[12:15], a[0:3]", "ds_read_b128 a[0:3], v1", "global_load_dwordx4 a[0:3], v1, s[2:3]",
    "buffer_store_dword a0, v1, s[4:7], 0 offen", "scratch_store_dword off, v1, s0", "scratch_load_dword v1, off, s0"])
def test_the_compilers_own_use_is_refused(op):
    with pytest.raises(RuntimeError, match="tile_linear_kernel"):
        _build.check_accumulators(KERNEL + "\t" + op + "   // 000000001020: 00000000\n")


def test_the_built_library():
    library = _build.PKG / f"_mixers{_build.EXT}"
    if not library.exists():
        pytest.skip("not built")
    assert _build.check_library_accumulators(library) >= 50   # sixteen tiles, gated and plain, the short forms, the grouped ones
