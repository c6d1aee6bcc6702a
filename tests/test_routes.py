"""Which kernel a call of given sizes runs (viper_hip_qlinear_route), at 256 CUs: sizes whose measured best kernel the
rules must keep.  Needs no GPU; on one the same holds for the MI355X's 256 CUs."""
import pytest

import viper_amd as va

Q4, Q5, Q6, W8 = 4, 5, 6, 8
BF16, INT8, FRAG = 0, 1, 2
M1, ROWS, RC_BF16, STREAM_BF16, RC_SPLIT, RC, STREAM, PAIRS = range(8)


def route(qtype, rows, N, K, M, matrices=1):
    return va.lib().viper_hip_qlinear_route(qtype, rows, N, K, M, matrices)


@pytest.mark.parametrize("qtype,rows,N,K,M,matrices,want", [
    (Q4, BF16, 10240, 2560, 1, 1, M1), (W8, INT8, 10240, 2560, 1, 2, M1), (Q4, BF16, 2560, 2560, 2, 1, ROWS),
    (Q4, BF16, 10240, 2560, 8, 1, RC_BF16), (Q4, BF16, 10240, 2560, 16, 1, RC), (Q4, BF16, 2560, 10240, 16, 1, RC_SPLIT),
    (Q4, FRAG, 2560, 10240, 16, 1, RC_SPLIT), (Q4, FRAG, 1024, 10240, 16, 2, RC), (Q5, BF16, 2560, 3520, 8, 1, STREAM_BF16),
    (Q4, FRAG, 10240, 4096, 16, 1, STREAM), (W8, INT8, 10240, 3072, 16, 1, STREAM)])
def test_route_basics(qtype, rows, N, K, M, matrices, want):
    assert route(qtype, rows, N, K, M, matrices) == want


@pytest.mark.parametrize("args", [(7, BF16, 64, 64, 2, 1), (Q4, 3, 64, 64, 2, 1), (Q4, BF16, 0, 64, 2, 1),
                                  (Q4, BF16, 64, 96, 2, 1), (Q4, BF16, 64, 64, 17, 1), (Q4, BF16, 64, 64, 2, 3),
                                  (Q4, FRAG, 64, 256, 1, 1), (Q4, FRAG, 64, 192, 2, 1), (Q4, BF16, 64, 0, 2, 1)])
def test_route_invalid(args):
    assert va.lib().viper_hip_qlinear_route(*args) == -1


# Q4, long K: the K split unless one launch serves a K of one phase (7 and 8 rows of K = 6144 are past its LDS).
@pytest.mark.parametrize("N,K,M,want", [(3072, 5376, 8, RC_SPLIT), (3072, 6144, 7, RC_SPLIT), (3072, 6144, 8, RC_SPLIT),
                                        (3072, 6144, 6, RC_BF16), (3072, 5376, 7, RC_BF16), (3072, 6144, 16, RC_SPLIT)])
def test_route_k_split(N, K, M, want):
    assert route(Q4, BF16, N, K, M) == want


# Q4, K of two phases: few rows quantized by every workgroup of the row-contiguous kernel while its rounds are few, then
# the streaming kernel's two launches; the dots up to 40 rows per CU.  A pair's two rows up to two rounds.
@pytest.mark.parametrize("qtype,N,K,M,matrices,want", [
    (Q4, 10240, 7168, 3, 1, RC_BF16), (Q4, 8192, 7168, 4, 1, RC_BF16), (Q4, 10240, 7168, 5, 1, STREAM),
    (Q4, 16384, 7168, 4, 1, STREAM), (Q4, 4352, 9216, 3, 1, ROWS), (Q5, 24576, 2048, 2, 2, RC)])
def test_route_two_phases(qtype, N, K, M, matrices, want):
    assert route(qtype, BF16, N, K, M, matrices) == want


# Two to four rows on the dots or on the matrix cores: exact tilings, two rows at 33..40 per CU, W8's short rows and its
# few long ones, several phases; int8 rows of a nibble format 3 and 4 on the matrix cores in one round.
@pytest.mark.parametrize("qtype,rows,N,K,M,want", [
    (Q4, BF16, 4096, 5120, 2, ROWS), (Q4, BF16, 10240, 5120, 2, ROWS), (Q4, BF16, 2560, 9600, 2, ROWS),
    (Q4, BF16, 10240, 2112, 2, ROWS), (Q6, BF16, 10240, 2112, 2, ROWS), (W8, BF16, 10240, 1760, 2, ROWS),
    (Q6, BF16, 8192, 2112, 2, STREAM_BF16), (Q4, BF16, 11005, 4032, 2, STREAM_BF16), (W8, BF16, 16384, 672, 2, ROWS),
    (W8, BF16, 2560, 3520, 2, ROWS), (W8, BF16, 4256, 4128, 2, ROWS), (W8, BF16, 6144, 3520, 2, STREAM_BF16),
    (Q4, INT8, 4096, 5120, 4, RC), (Q4, INT8, 28160, 2560, 3, ROWS), (W8, INT8, 2560, 2560, 4, ROWS)])
def test_route_dots(qtype, rows, N, K, M, want):
    assert route(qtype, rows, N, K, M) == want


# Past one round of the row-contiguous kernel: the streaming kernel, but for equal padding with part of a step of four
# groups idle, and two bf16 rows also before it where it pads fewer rows.
@pytest.mark.parametrize("qtype,rows,N,K,M,matrices,want", [
    (Q4, BF16, 14336, 3328, 4, 1, RC_BF16), (Q4, BF16, 14336, 4096, 4, 1, STREAM_BF16), (Q4, INT8, 16384, 4608, 16, 1, RC),
    (Q4, FRAG, 14336, 3328, 16, 1, STREAM), (Q4, INT8, 13312, 3584, 7, 2, STREAM), (Q6, BF16, 10000, 3328, 4, 1, STREAM_BF16),
    (Q5, BF16, 14000, 2048, 2, 1, STREAM_BF16), (Q4, BF16, 14000, 2048, 3, 1, RC_BF16)])
def test_route_padding(qtype, rows, N, K, M, matrices, want):
    assert route(qtype, rows, N, K, M, matrices) == want


# K of an even number of groups, not a multiple of four: gathered pairs for short rows, few rows per CU and many rows of
# the formats that decode cheapest; the streaming kernel else.
@pytest.mark.parametrize("qtype,rows,N,K,M,want", [
    (Q4, BF16, 2048, 384, 16, PAIRS), (Q4, INT8, 2048, 384, 16, PAIRS), (Q4, INT8, 256, 384, 16, STREAM),
    (Q4, BF16, 2048, 4224, 16, PAIRS), (Q6, BF16, 6144, 4224, 8, PAIRS), (Q4, BF16, 24000, 3712, 16, PAIRS),
    (W8, BF16, 24000, 2112, 16, PAIRS), (W8, BF16, 10240, 2112, 16, STREAM), (Q4, BF16, 2048, 8320, 16, PAIRS),
    (Q5, BF16, 2048, 6784, 16, STREAM), (Q4, INT8, 2048, 8320, 16, PAIRS), (Q4, INT8, 2048, 8320, 8, STREAM),
    (W8, BF16, 256, 13248, 12, STREAM), (Q4, BF16, 24576, 384, 8, PAIRS), (Q4, BF16, 2560, 3456, 8, STREAM_BF16)])
def test_route_pairs(qtype, rows, N, K, M, want):
    assert route(qtype, rows, N, K, M) == want


# Two bf16 rows over several rounds of the row-contiguous kernel: the kernel that pads fewest; a long K of a pair stays in
# one launch.
@pytest.mark.parametrize("qtype,N,K,matrices,want", [
    (Q4, 17366, 1536, 1, ROWS), (Q4, 20480, 2048, 1, ROWS), (Q4, 24320, 2048, 1, RC_BF16), (Q4, 12800, 1792, 1, ROWS),
    (Q5, 14000, 2048, 1, STREAM_BF16), (Q4, 20000, 2048, 2, RC_BF16), (Q5, 20000, 2048, 2, RC), (Q6, 25600, 1536, 1, ROWS), (W8, 26645, 5504, 2, RC_BF16), (Q4, 20736, 256, 1, RC_BF16)])
def test_route_two_rows_padding(qtype, N, K, matrices, want):
    assert route(qtype, BF16, N, K, 2, matrices) == want
