"""What bench.py makes of a forward's stages (host only)."""
import bench


def test_stages_are_one_kernel_only_where_one_kernel_ran():
    """Softmax + mixing and P V in one kernel are announced as two stages at once: the first takes no time and the sum belongs to the one kernel.
    Where both take time, or neither is there (the route of single stages), the stages stay what they are."""
    assert bench.join_stages({"qk_conv": 0.24, "mix_softmax_mix": 0.002, "pv": 0.19}) == {"qk_conv": 0.24, "softmax_mix_pv": 0.192}
    for stages in ({"qk_conv": 0.24, "mix_softmax_mix": 0.18, "pv": 0.14}, {"qk": 0.3, "conv_pre": 0.2, "softmax": 0.2, "mix_post": 0.2, "pv": 0.3}):
        assert bench.join_stages(dict(stages)) == stages
        for name in bench.join_stages(dict(stages)):
            assert bench.stage_model(name, 2, 16, 4096, 128)[0] > 0
