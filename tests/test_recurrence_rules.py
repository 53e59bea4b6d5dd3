"""The rule that sends a step's portions through a recurrent layer in stages or has them walked: host code, held against both routes'
measured times."""

import pytest

from bitwise_amd.parts.recurrent import in_stages

# (gates, heads, key channels, value channels), portions, single tokens beside them, microseconds walked, in stages
MEASURED = [
    ((False, 16, 64, 128), (64,), 0, 12.6, 11.6), ((False, 16, 64, 128), (64,), 15, 19.3, 34.6), ((False, 16, 64, 128), (64,), 64, 52.3, 114.0),
    ((False, 16, 64, 128), (96,), 255, 164.7, 423.0), ((False, 16, 64, 128), (128,), 1, 20.5, 15.0), ((False, 16, 64, 128), (256,), 7, 37.5, 32.8),
    ((False, 16, 64, 128), (512,), 128, 142.5, 240.2), ((False, 16, 64, 128), (2048,), 31, 269.7, 180.2), ((False, 16, 64, 128), (2048,), 255, 400.3, 531.5),
    ((False, 4, 64, 64), (64,), 7, 12.2, 11.0), ((False, 4, 64, 64), (64,), 128, 21.5, 36.9), ((False, 4, 64, 64), (2048,), 128, 267.3, 149.7),
    ((False, 16, 128, 128), (64,), 64, 90.3, 256.1), ((False, 16, 128, 128), (256,), 1, 41.1, 34.3), ((False, 16, 128, 128), (2048,), 15, 286.0, 249.1),
    ((False, 8, 128, 64), (96,), 4, 16.9, 19.6), ((False, 8, 128, 64), (64,), 255, 96.1, 253.3), ((False, 8, 128, 64), (512,), 4, 72.4, 55.9),
    ((True, 8, 128, 256), (128,), 4, 40.1, 36.9), ((True, 8, 128, 256), (96,), 64, 93.4, 155.2), ((True, 8, 128, 256), (512,), 31, 159.2, 130.1),
    ((True, 8, 128, 256), (256,), 255, 358.7, 569.8), ((True, 16, 64, 128), (128,), 128, 98.2, 262.4), ((True, 4, 128, 64), (128,), 128, 53.6, 69.3),
    ((True, 4, 128, 64), (256,), 64, 75.4, 63.1), ((True, 16, 128, 256), (512, 512), 0, 160.7, 143.5),
]


@pytest.mark.parametrize("layer,portions,ones,walked,staged", MEASURED)
def test_the_route_that_is_taken_is_the_faster_one(layer, portions, ones, walked, staged):
    gates, heads, dim, vdim = layer
    taken = in_stages(max(portions), sum(portions) + ones, len(portions) + ones, heads * vdim, dim, gates)
    assert (staged if taken else walked) <= 1.08 * min(walked, staged)


def test_single_tokens_beside_a_portion_end_the_stages_and_other_heads_never_take_them():
    for gates in (False, True):
        for dim in (64, 128):
            for longest in (64, 80, 200, 600, 2048):
                taken = [in_stages(longest, longest + n, 1 + n, 2048, dim, gates) for n in range(300)]
                assert taken == sorted(taken, reverse=True) and (longest < 200 or taken[0]) and not (longest < 600 and taken[64])
        assert not any(in_stages(512, 512, 1, 512, dim, gates) for dim in (16, 32, 96, 256))
