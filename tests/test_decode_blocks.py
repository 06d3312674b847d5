"""The block sizes of a decode call that leaves them to the library (split_tokens
0), as far as the host alone shows them: through the workspace sizes.  No GPU is
needed.  The results are compared in test_gqa_gpu.py and test_zz_no_alloc.py."""
import ctypes
import random

import pytest

from pluto_amd import capi

STATIC_BYTES = 16 << 20


@pytest.fixture(scope="module")
def library():
    return capi.lib()


def size(library, qh, kh, d, rows, split, round_to_bfloat16=True):
    p = capi.attention_params(qh, kh, d, 16, capacity=1 << 20, round_to_bfloat16=round_to_bfloat16)
    positions = (ctypes.c_int * len(rows))(*[r - 1 for r in rows])
    return library.pluto_hip_gqa_decode_workspace_bytes(ctypes.byref(p), len(rows), positions, split)


def default_of(d):
    return 1024 if d == 256 else 512


@pytest.mark.parametrize("qh,kh,d,rounding", [(32, 1, 256, True), (12, 1, 128, True), (6, 1, 96, True),
                                              (24, 4, 256, False), (3, 1, 128, True)])
def test_any_shape_kernels_need_no_more_than_the_default_size(library, qh, kh, d, rounding):
    # groups, widths and roundings the fused kernel does not take: blocks are not read
    for rows in ([1], [777], [848, 5000], [4096] * 32):
        assert size(library, qh, kh, d, rows, 0, rounding) == size(library, qh, kh, d, rows, default_of(d), rounding)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_a_sequence_is_counted_alone(library, d):
    rng = random.Random(d)
    for _ in range(50):
        rows = [rng.choice([rng.randint(1, 2000), rng.randint(1, 40000)]) for _ in range(rng.randint(2, 40))]
        # regions are rounded up to 256 bytes each
        alone = sum(size(library, 24, 4, d, [r], 0) for r in rows)
        together = size(library, 24, 4, d, rows, 0)
        assert together <= alone <= together + 5 * 256 * len(rows)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_a_workspace_serves_smaller_positions(library, d):
    last = 0
    for rows in list(range(1, 4200)) + list(range(4200, 40000, 97)):
        now = size(library, 8, 1, d, [rows], 0)
        assert now >= last, rows
        assert now >= size(library, 8, 1, d, [rows], default_of(d)), rows
        last = now


@pytest.mark.parametrize("d", [64, 128, 256])
def test_what_fits_the_fixed_scratch_in_default_blocks_fits_the_array(library, d):
    """The array holds 52 / 16 of the limit that a call is measured against; a
    sequence's bytes in blocks of its own are at most (5 x 258 + 256) / (258 + 256) of
    those in default blocks, with the counters and the rounding of the regions beside."""
    rng = random.Random(d + 1)
    worst = 0.0
    for r in list(range(1, 3000)) + [rng.randint(3000, 60000) for _ in range(300)]:
        default = size(library, 24, 4, d, [r] * 64, default_of(d))
        # the reported size bounds smaller positions too: what one length needs is less
        worst = max(worst, size(library, 24, 4, d, [r] * 64, 0) / default)
    assert worst <= 3.05 < 52 / 16
