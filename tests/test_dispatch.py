"""Which kernel a call takes, where that was chosen by measurement (CPU; the rules count the CUs of the
current device, 256 where there is none).

The shapes are points of sweeps that timed both sides with each form forced; those on the wrong side of
a line were up to 2.4 times slower. The results do not depend on the choice (the GPU tests compare the
forms' bits)."""
import pytest

from ancha_amd import _native

# groups, tokens (8 heads), rotated on load, aligned rows, queries per workgroup
ATTENTION = [
    (600, 65, False, True, 128), (200, 128, True, False, 128),
    # Aligned rows, nothing rotated: one round of 512-query passes, past it, past five 4-wave workgroups.
    (1, 801, False, True, 128), (16, 512, False, True, 128), (25, 450, False, True, 512),
    (15, 801, False, True, 512), (10, 1301, False, True, 512), (8, 1722, False, True, 512),
    (20, 801, False, True, 128), (10, 1722, False, True, 128), (200, 384, False, True, 128),
    (60, 801, False, True, 512), (90, 1722, False, True, 512),
    # Rotary rows.
    (5, 801, True, True, 128), (6, 801, True, True, 512), (17, 129, True, True, 512),
    (50, 129, True, True, 512), (80, 200, True, True, 128), (200, 200, True, True, 128),
    (120, 801, True, True, 512),
    # Unaligned rows.
    (3, 1025, False, False, 128), (4, 1025, False, False, 512), (10, 1301, False, False, 512),
    (15, 801, False, False, 512), (200, 384, False, False, 512), (80, 256, False, False, 128),
    (50, 256, False, False, 512), (5, 801, True, False, 512), (200, 256, True, False, 512),
]


@pytest.mark.parametrize("groups,tokens,rotated,aligned,queries", ATTENTION)
def test_attention_passes(groups, tokens, rotated, aligned, queries):
    assert _native.lib().ancha_amd_attention_queries(groups, tokens, 8, rotated, aligned) == queries


# n, k, m, whether the weight is laid out first (scratch of k m halves)
LINEAR = [
    (32, 384, 1664, True), (300, 1536, 384, True), (96120, 384, 1664, True), (18060, 1536, 384, True),
    (9000, 384, 512, True), (33000, 640, 1664, True), (40000, 1024, 256, True), (40000, 1536, 128, True),
    # 128 x 128 tiles that linear.hip runs two to a CU.
    (65000, 256, 256, False), (32000, 512, 256, False), (24576, 1024, 256, False),
    (10500, 640, 640, False), (20000, 640, 1664, False), (96120, 128, 128, False),
    # Few rows on a very wide weight.
    (200, 256, 16384, False), (500, 512, 16384, False), (128, 256, 8192, True), (700, 512, 16384, True),
    # Shapes that only linear.hip takes, and calls that are refused.
    (1000, 384, 200, False), (1000, 64, 128, False), (0, 384, 384, False), (1 << 31, 384, 384, False),
    (4, 128, 1 << 22, False), (4, 1 << 23, 128, False),
]


@pytest.mark.parametrize("n,k,m,laid_out", LINEAR)
def test_linear_scratch(n, k, m, laid_out):
    assert _native.lib().ancha_amd_linear_workspace(n, k, m) == (2 * k * m if laid_out else 0)
