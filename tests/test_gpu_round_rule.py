"""The z chunk of an untuned fused pass, also where its tiles outnumber the compute units: a
last round of workgroups that is nearly empty costs as much as a full one."""
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,dtype,depth,n", [(1, gpu.GR_F64, 5, (512, 512, 256)), (1, gpu.GR_F64, 4, (700, 300, 200)),
                                                  (1, gpu.GR_F32, 6, (500, 700, 100)), (5, gpu.GR_F64, 4, (520, 290, 90)),
                                                  (5, gpu.GR_F64, 4, (512, 512, 128)), (0, gpu.GR_F64, 2, (900, 400, 40))])
def test_untuned_chunks_fill_their_rounds(kernel, dtype, depth, n):
    torch = pytest.importorskip("torch")
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    nx, ny, nz = n
    with gpu.Stepper(kernel, *n, dtype=dtype, flags=gpu.GR_ROC2_SCALAR if kernel == 0 else 0, t_block=depth) as st:
        s = st.stats()
        margin = 2 * st.R * depth

    def cost(zc):  # planes that the busiest compute unit computes
        tiles = -(-nx // s["tile_x"]) * -(-ny // s["tile_y"])
        return -(-(tiles * -(-nz // zc)) // ncu) * (zc + margin)

    print(kernel, depth, n, "tile", s["tile_x"], s["tile_y"], "chunk", s["zchunk"], flush=True)
    zc = s["zchunk"] or nz
    assert cost(zc) <= 1.1 * min(cost(z) for z in range(margin, nz + 1)) and (zc == nz or zc >= margin)
