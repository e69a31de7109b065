"""What bench.py reports of the dedispersion kernel: the one that ran, and HBM
traffic only where the committed counters are that kernel's."""
import bench


class Plan:
    tile, own_tile = (32, 512, 0, 16), False

    def kernel(self, d_in):
        return "window", 32, 1280, 0


def test_record_names_the_kernel_that_ran():
    rec = bench.dedisp_kernel(Plan(), None, "f32")
    assert rec["name"] == "dedisperse_window_kernel" and rec["set_tile_dm_t_chanblock_readbytes"] is None
    plan = Plan()
    plan.own_tile = True
    assert bench.dedisp_kernel(plan, None, "f32")["set_tile_dm_t_chanblock_readbytes"] == [32, 512, 0, 16]


def test_traffic_is_of_the_kernel_that_ran():
    for dtype, kernel in (("f32", "dedisperse_window_kernel"), ("f32", "dedisperse_ring_kernel"),
                          ("f16", "dedisperse_window_kernel"), ("u8", "dedisperse_u8_group_kernel")):
        assert bench.traffic_from_profile(dtype, kernel) > 1e9
    assert bench.traffic_from_profile("f32", "dedisperse_kernel") is None
    assert bench.traffic_from_profile("f16", "dedisperse_ring_kernel") is None
