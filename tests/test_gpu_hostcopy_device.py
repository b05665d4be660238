"""Uploads and downloads of a handle while another GPU is current: they run on the handle's
GPU and leave the caller's current."""
import numpy as np
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu


def test_host_copies_keep_the_callers_device():
    torch = pytest.importorskip("torch")
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    rng = np.random.default_rng(3)
    U1, U2 = rng.random((63, 70, 520)).astype(np.float32), rng.random((63, 70, 520)).astype(np.float32)
    with torch.cuda.device(0):
        st = gpu.Stepper(1, 518, 68, 61, dtype=gpu.GR_F32, coef=[0.4, 0.1])
    with torch.cuda.device(1):
        st.upload(U1, U2)
        assert torch.cuda.current_device() == 1
        D1, D2 = st.download(U1.shape)
        assert torch.cuda.current_device() == 1
    st.close()
    np.testing.assert_array_equal(D1, U1)
    np.testing.assert_array_equal(D2, U2)
