"""Which kernel chains a row's fingerprint: host code, held against both kernels' measured times."""

import pytest

from bitwise_amd.csrc import ops

# rows, logits, microseconds word by word, bit by bit
MEASURED = [(8, 49152, 318, 43), (8, 3072, 21, 26), (200, 4096, 29.9, 28.4), (256, 20000, 145.7, 34.0), (300, 5645, 40.3, 33.1), (500, 7000, 49.1, 33.7),
            (787, 5000, 41.0, 46.0), (787, 5645, 42.0, 46.5), (787, 7000, 52.7, 46.6), (1024, 5000, 43.2, 46.8), (1024, 5645, 45.0, 47.2),
            (1024, 7000, 59.1, 47.4), (1100, 10000, 140.3, 60.4), (2048, 7000, 102.3, 84.3), (3000, 14000, 293.4, 122.1), (6000, 10000, 396.1, 220.3)]


@pytest.mark.parametrize("rows,vocab,words,bits", MEASURED)
def test_the_faster_kernel_is_taken(rows, vocab, words, bits):
    assert (ops.fingerprint_waves(rows, vocab) > 0) == (bits < words)
