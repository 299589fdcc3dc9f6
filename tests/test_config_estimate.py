"""The v3 entry's choice of a workgroup configuration on grids that fill no
whole round of the device (CPU: without a device the CU count is an MI355X's
256)."""


def test_configuration_between_whole_rounds(fa_lib):
    """The configuration whose workgroups divide best, by the estimate of
    auto_config; where two are within 5 % the rule's stays."""
    for shape, causal, want in [((1, 20, 1024, 64), False, (128, 2)), ((1, 20, 1024, 128), False, (128, 2)),
                                ((1, 12, 2048, 128), False, (128, 2)), ((3, 5, 1531, 64), False, (128, 2)),
                                ((1, 12, 3072, 128), False, (256, 1)), ((1, 40, 1024, 128), False, (256, 1)),
                                ((1, 48, 512, 128), True, (128, 2)), ((1, 24, 1536, 128), True, (64, 2)),
                                ((1, 192, 768, 128), True, (256, 1)), ((1, 1, 1, 64), True, (64, 2))]:
        assert fa_lib.tensorcore_v3_config(shape, causal) == want, (shape, causal)
