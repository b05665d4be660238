"""Graph mode captures a launch sequence once and replays it: repeated first-order calls
capture at most once, and calls of one pass, whose buffers change from call to call, not
at all.  Every call equals the eager one bit for bit."""
import pytest

from girih_amd import gpu

from test_gpu_graph import _pair, _same

pytestmark = pytest.mark.gpu


def captures(st):
    return gpu.lib().gr_internal_graph_captures(st._h)


# steps a call, captures of 7 such calls.  Odd counts of several launches alternate the
# parity, and with it the sequence, from call to call: they are captured at every one.
@pytest.mark.parametrize("kernel,dtype,depth,steps,most", [
    (1, gpu.GR_F64, 4, 4, 0), (1, gpu.GR_F32, 4, 2, 0), (1, gpu.GR_F32, 3, 3, 0), (1, gpu.GR_F64, 4, 5, 0),
    (5, gpu.GR_F64, 4, 4, 0), (5, gpu.GR_F32, 6, 6, 1), (5, gpu.GR_F32, 2, 3, 0), (1, gpu.GR_F64, 4, 8, 1),
    (1, gpu.GR_F32, 3, 4, 1), (5, gpu.GR_F32, 4, 20, 1), (1, gpu.GR_F64, 4, 7, 7)])
def test_calls_capture_once_at_most(kernel, dtype, depth, steps, most):
    (eager, graph), shape = _pair(kernel, 70, 19, 13, dtype)
    try:
        for st in (eager, graph):
            st.set_config(zchunk=6, t_block=depth)
        graph.set_graph(True)
        for rep in range(7):
            print("captures", kernel, dtype, depth, steps, rep, flush=True)
            eager.step(steps)
            graph.step(steps)
            assert graph.stats()["last_launches"] == eager.stats()["last_launches"]
            _same(eager, graph, shape, "call %d" % rep)
        assert captures(graph) <= most and captures(eager) == 0
    finally:
        eager.close()
        graph.close()


def test_one_pass_calls_keep_the_captured_sequence():
    (eager, graph), shape = _pair(1, 70, 19, 13, gpu.GR_F64)
    try:
        for st in (eager, graph):
            st.set_config(zchunk=6, t_block=4)
        graph.set_graph(True)
        for rep, n in enumerate((20, 4, 4, 20, 4, 4, 20)):  # two one-pass calls restore the buffers
            eager.step(n)
            graph.step(n)
            _same(eager, graph, shape, "call %d" % rep)
        assert captures(graph) == 1
    finally:
        eager.close()
        graph.close()
