"""bench.py's roofline block: the kernels it names, and a profiled traffic
figure only from a profile of those kernels."""
import json
import os

import bench


def test_names_follow_the_library_choice():
    assert bench.fwd_kernel_names(16, 12, 2, 3) == [
        "k_ntt_pass<16, 1, false, 12, 3, 0>", "k_ntt_pass<16, 2, false, 12, 3, 0>"]
    assert bench.fwd_kernel_names(16, 12, 1, 3) == ["k_ntt_fused<16, false, 12, 2>"]
    assert bench.fwd_kernel_names(12, 13, 1, 3) == ["k_ntt_fused<12, false, 13, 3>"]
    assert bench.forward_tile(14, 12, 1) == 14 and bench.forward_tile(14, 12, 2) == 12
    assert bench.forward_tile(16, 12, 2) == 12 and bench.forward_tile(13, 13, 1) == 13
    assert bench.fwd_kernel_names(14, 14, 2, 3, npoly=512) == ["k_ntt_wide<14, false>"]
    assert bench.fwd_kernel_names(14, 14, 2, 3, npoly=256) == ["k_ntt_fused<14, false, 14, 3>"]
    assert bench.fwd_kernel_names(14, 14, 2, 1, npoly=512) == ["k_ntt_fused<14, false, 14, 1>"]


def test_traffic_only_of_the_named_kernels():
    def prof(tile):
        with open(os.path.join(bench.REPO, "profiles",
                               f"ntt_fwd_n65536_x512_tile{tile}.json")) as f:
            return json.load(f)
    mc = bench.modulus_class((1 << 50) - 1)
    for tile in (11, 12):
        names = bench.fwd_kernel_names(16, tile, 2, mc)
        assert prof(tile)["kernels"] == names
        traffic, busy, path = bench.traffic_from_profile(16, 512, names)
        assert abs(traffic - prof(tile)["hbm_bytes_per_launch"]) <= 1 and 0 < busy < 1
        assert path == f"profiles/ntt_fwd_n65536_x512_tile{tile}.md"
    # the passes' tiles tuned apart
    names = bench.fwd_kernel_names(16, 12, 2, mc, 0, 11)
    traffic, _, path = bench.traffic_from_profile(16, 512, names)
    assert path.count("tile11") == path.count("tile12") == 1 and traffic > 0
    # another class's kernels, or another size: no figure
    other = bench.fwd_kernel_names(16, 12, 2, 2)
    assert bench.traffic_from_profile(16, 512, other) == (None, None, None)
    assert bench.traffic_from_profile(16, 256, names) == (None, None, None)
