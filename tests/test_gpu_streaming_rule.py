"""Where sweeps start to use the cache hints: where the padded fields exceed the 256 MB
cache, by the bytes of their cells, on a line of each kernel's own.  gr_set_streaming
overrides the rule."""
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu

# kernel, dtype, flags, grid, hints.  A 128-wide FP32 grid's rows are padded by half: 128 x 300 x
# 300 of kernel 5 holds 407 MB of cells in 601 MB, 128 x 300 x 128 175 MB in 259 MB.
CASES = [(5, gpu.GR_F32, 0, (128, 300, 128), False), (5, gpu.GR_F32, 0, (128, 252, 252), False),
         (5, gpu.GR_F32, 0, (128, 300, 300), True), (5, gpu.GR_F64, 0, (128, 151, 151), False),
         (5, gpu.GR_F64, 0, (172, 172, 172), True), (5, gpu.GR_F32, gpu.GR_COEF_BF16, (280, 260, 240), True),
         (4, gpu.GR_F64, 0, (120, 120, 120), False), (4, gpu.GR_F32, 0, (183, 183, 183), True),
         (3, gpu.GR_F64, 0, (181, 181, 181), False), (3, gpu.GR_F32, 0, (228, 228, 228), True),
         (2, gpu.GR_F64, 0, (187, 187, 187), False), (2, gpu.GR_F32, 0, (250, 250, 250), True),
         (1, gpu.GR_F64, 0, (384, 384, 100), False), (1, gpu.GR_F32, 0, (128, 429, 429), True),
         (1, gpu.GR_F32, 0, (328, 328, 328), True),
         (0, gpu.GR_F32, 0, (128, 351, 351), False), (0, gpu.GR_F32, 0, (297, 297, 297), True),
         (0, gpu.GR_F64, 0, (128, 261, 261), False), (0, gpu.GR_F64, 0, (248, 248, 248), True)]


@pytest.mark.parametrize("kernel,dtype,flags,n,hints", CASES)
def test_hints_by_the_cells_bytes(kernel, dtype, flags, n, hints):
    streaming = gpu.lib().gr_internal_streaming
    with gpu.Stepper(kernel, *n, dtype=dtype, flags=flags) as st:
        assert bool(streaming(st._h)) == hints
        for mode in (0, 1):
            st.set_streaming(mode)
            assert streaming(st._h) == mode
