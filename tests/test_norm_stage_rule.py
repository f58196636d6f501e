"""Whether the norm and the exact staging of a call run as one launch: where that was the faster form in
the usual step. Either gives the same bits."""

# (matrices, padded rows, padded columns, kept scales), whether one launch is as fast
JOIN = [((1, 128, 512, 0), 1), ((12, 512, 2048, 0), 1), ((8, 1024, 2048, 0), 1),
        ((8, 1024, 4096, 0), 1), ((8, 4096, 1024, 0), 1), ((64, 1024, 1024, 0), 1),
        ((32, 512, 8192, 0), 0), ((64, 1536, 2048, 0), 0), ((64, 2048, 1536, 0), 0),
        ((32, 1024, 4096, 0), 0), ((1, 1024, 4224, 0), 0),
        ((1, 128, 512, 1), 1), ((200, 512, 512, 1), 1), ((64, 1024, 1024, 1), 1),
        ((4, 1024, 4096, 1), 1), ((64, 1536, 2048, 1), 1), ((64, 2048, 1536, 1), 1),
        ((32, 1024, 4096, 1), 1), ((1, 1024, 16384, 1), 0)]


def test_the_faster_form(cpp_harness):
    args = [v for case, _ in JOIN for v in case]
    assert cpp_harness("norm_stage", *args) == "".join(str(want) for _, want in JOIN)
