"""How many waves a workgroup of 32-bit decode attention gets: host code, held against both forms' measured times."""

import pytest

from bitwise_amd.csrc import ops

# head size, workgroups, keys (and the most of them), microseconds in four waves, in eight
MEASURED = [(16, 64, 2400, 44.1, 33.1), (16, 256, 200, 10.3, 8.7), (16, 400, 200, 11.5, 15.1), (16, 2400, 2400, 229.8, 338.6),
            (32, 400, 20, 12.1, 10.2), (64, 2400, 60, 60.4, 52.7), (128, 2400, 4, 66.1, 51.2),
            (160, 400, 60, 10.6, 14.2), (160, 64, 800, 35.4, 25.4), (192, 1200, 20, 20.9, 30.5), (224, 64, 4, 7.0, 7.5), (224, 600, 200, 43.6, 47.4),
            (256, 256, 4, 6.9, 7.8), (256, 256, 200, 19.4, 17.6), (256, 600, 20, 13.7, 19.6), (256, 2400, 800, 616.0, 656.2)]


@pytest.mark.parametrize("head_dim,workgroups,keys,four,eight", MEASURED)
def test_the_form_that_is_taken_is_the_faster_one(head_dim, workgroups, keys, four, eight):
    waves = ops.attention_f32_waves(head_dim, workgroups, keys)
    assert {4: four, 8: eight}[waves] == min(four, eight)


def test_heads_without_a_kernel_of_four_waves_get_eight():
    for head_dim in (32, 48, 64, 80, 96, 112, 128):
        assert {ops.attention_f32_waves(head_dim, n, c) for n in (1, 256, 257, 60000) for c in (1, 64, 65, 30000)} == {8}
