"""Where the middle Q update of a Gram segment runs: in the idle CUs of three triangle launches, or
in a launch of its own. The choice changes no bit, only the time."""
from dmuon_amd import _C

# (rows, matrices): whether the update in the triangle launches was the faster one, measured on
# several cards
FILL = [((192, 1), 1), ((1024, 1), 1), ((1216, 1), 1), ((2048, 1), 1), ((2112, 1), 1),
        ((3072, 1), 1), ((4096, 1), 1), ((512, 3), 1), ((640, 3), 1), ((768, 2), 1), ((384, 10), 1),
        ((768, 10), 1), ((1024, 8), 1), ((1152, 8), 1), ((640, 32), 1), ((1408, 8), 1),
        ((1280, 12), 1), ((576, 8), 1), ((1408, 24), 1), ((4096, 4), 1),
        ((1280, 1), 0), ((1344, 1), 0), ((1408, 1), 0), ((1856, 1), 0), ((1920, 1), 0),
        ((1984, 1), 0), ((2560, 1), 0), ((2816, 1), 0), ((3840, 1), 0), ((256, 16), 0),
        ((384, 8), 0), ((512, 4), 0), ((512, 7), 0), ((768, 3), 0), ((896, 8), 0), ((1024, 6), 0),
        ((1280, 4), 0), ((1152, 16), 0), ((1408, 2), 0), ((1536, 6), 0), ((2048, 6), 0)]


def test_the_faster_place_of_the_q_update(cpp_harness):
    args = []
    for (m, batch), _ in FILL:
        args += [m, batch, _C.plan(m, m, batch, 0, 256, _C.NS_GRAM)[0]]
    assert cpp_harness("nt_fill", *args) == "".join(str(want) for _, want in FILL)
