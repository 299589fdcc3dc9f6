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


def test_causal_grids_that_keep_the_rule(fa_lib):
    """Both sides of each edge: 64-row grids of up to one and a half rounds
    (head_dim 128: nine eighths), one or two slabs per XCD, short head_dim-64 rows in one
    round, whole rounds."""
    for shape, want in [((1, 8, 2500, 64), (64, 4)), ((1, 8, 3072, 64), (64, 4)), ((1, 8, 3840, 64), (128, 4)),
                        ((1, 16, 1152, 128), (64, 2)), ((1, 9, 2048, 128), (64, 2)), ((1, 16, 1536, 128), (128, 2)),
                        ((1, 8, 7360, 64), (128, 2)), ((1, 8, 5000, 64), (64, 2)), ((1, 9, 7360, 64), (64, 2)),
                        ((1, 16, 3600, 64), (128, 2)), ((1, 8, 9000, 64), (64, 2)),
                        ((1, 16, 2059, 128), (128, 2)), ((1, 12, 3001, 128), (128, 2)), ((2, 6, 3001, 128), (128, 2)),
                        ((1, 17, 2300, 128), (64, 2)), ((1, 21, 2496, 128), (64, 2)),
                        ((1, 28, 1000, 64), (64, 2)), ((1, 16, 2048, 128), (128, 2)), ((1, 199, 1024, 128), (128, 2))]:
        assert fa_lib.tensorcore_v3_config(shape, True) == want, (shape, fa_lib.tensorcore_v3_config(shape, True))
