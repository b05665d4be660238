"""The tile variant, z chunk, order and depth that gr_get_stats reports select the same
tiles on another handle (gr_set_config, gr_set_xcd_order), for tuned and chosen settings."""
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu

WORDS = ("tile_variant", "zchunk", "xcd_order", "t_block", "tile_x", "tile_y")


def _replay(st, kernel, n, dtype, flags):
    s = st.stats()
    with gpu.Stepper(kernel, *n, dtype=dtype, flags=flags) as other:
        other.set_config(s["tile_variant"], s["zchunk"], s["t_block"])
        other.set_xcd_order(s["xcd_order"])
        o = other.stats()
    assert {k: o[k] for k in WORDS} == {k: s[k] for k in WORDS}
    return s


@pytest.mark.parametrize("kernel,dtype,flags", [(1, gpu.GR_F32, 0), (1, gpu.GR_F64, 0), (5, gpu.GR_F64, 0),
                                                (5, gpu.GR_F32, 0), (5, gpu.GR_F32, gpu.GR_COEF_BF16)])
def test_reported_settings_select_the_same_tiles(kernel, dtype, flags):
    n = (200, 180, 96)
    with gpu.Stepper(kernel, *n, dtype=dtype, flags=flags) as st:
        st.init_fields(1, 3)
        for depth in (2, 4):
            st.set_config(zchunk=32, t_block=depth)  # nobody chose a tile
            _replay(st, kernel, n, dtype, flags)
            tiles, t = {}, 0
            while True:  # every pass tile with sweep variants below and above their number
                try:
                    st.set_config(13 + 64 * (t + 1), 32, depth)
                except gpu.GirihError as e:
                    assert e.code == gpu.GR_EINVAL
                    break
                s = _replay(st, kernel, n, dtype, flags)
                tiles[t] = (s["tile_x"], s["tile_y"])
                st.set_config(t_block=depth)  # the same depth again keeps the tile
                assert _replay(st, kernel, n, dtype, flags)["tile_x"] == s["tile_x"]
                st.set_config(2 + 64 * (t + 1), 32, depth)
                s = _replay(st, kernel, n, dtype, flags)
                assert (s["tile_x"], s["tile_y"]) == tiles[t]
                t += 1
            assert len(set(tiles.values())) >= (2 if len(tiles) > 1 else 1)
            for v in range(len(tiles)):  # variants below the number of tiles select them too
                st.set_config(v, 32, depth)
                s = _replay(st, kernel, n, dtype, flags)
                assert (s["tile_x"], s["tile_y"]) == tiles[v] and s["tile_variant"] == v
        for bad in (17, 13 + 64 * 20):
            with pytest.raises(gpu.GirihError) as ei:
                st.set_config(bad, 32, 4)
            assert ei.value.code == gpu.GR_EINVAL
        with pytest.raises(gpu.GirihError):
            st.set_config(2 + 64, 32, 1)  # single sweeps have no pass tile


@pytest.mark.parametrize("kernel,dtype,n", [(1, gpu.GR_F32, (512, 512, 512)), (1, gpu.GR_F64, (389, 270, 331)),
                                            (5, gpu.GR_F32, (389, 270, 331)), (0, gpu.GR_F64, (96, 90, 70))])
def test_tuned_settings_select_the_same_tiles(kernel, dtype, n):
    with gpu.Stepper(kernel, *n, dtype=dtype, flags=gpu.GR_ROC2_SCALAR if kernel == 0 else 0, roc2=0.1) as st:
        if kernel == 5:
            st.init_coef_uniform(5, 0.3, 0.5, 0.0, 0.1)
        st.init_fields(1, 3)
        st.autotune(4)
        s = _replay(st, kernel, n, dtype, gpu.GR_ROC2_SCALAR if kernel == 0 else 0)
        print("tuned", {k: s[k] for k in WORDS}, flush=True)
        before = st.stats()
        st.set_config(t_block=s["t_block"])
        assert {k: st.stats()[k] for k in WORDS} == {k: before[k] for k in WORDS}
