"""First-order fused steps without the memory for a third field: two fields of 0.38 of the
free memory each leave no room for another.  The calls run (passes that end with single
sweeps) and a captured sequence is replayed, not captured again at every call."""
import pytest

from girih_amd import gpu

from test_gpu_graph_captures import captures

pytestmark = pytest.mark.gpu


def test_calls_replay_without_a_third_field():
    torch = pytest.importorskip("torch")
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    n = int((0.38 * free / 4) ** (1 / 3)) - 31  # less the rows' padding
    print("grid", n, "free", free, flush=True)
    with gpu.Stepper(1, n, n, n, dtype=gpu.GR_F32, coef=[0.4, 0.1]) as st:
        held = st.stats()["device_bytes"]
        assert held // 2 > free - held, "a third field would fit"
        st.set_config(t_block=4)
        st.set_graph(True)
        for rep in range(4):
            st.step(10)  # two passes, two sweeps: ends on the buffers and parity it began with
            assert st.stats()["last_launches"] == 4
            assert captures(st) == 1, rep
        assert st.stats()["device_bytes"] == held
