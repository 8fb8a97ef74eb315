"""Gate and up of prompt batches whose last row tile is short: which of them go to the tiled GEMM, by sizes alone."""
import pytest


# (tails of one row, of 64 and of 65; whole tiles alone; rounds that the short tiles lengthen; narrower and wider layers than were measured)
@pytest.mark.parametrize("n,k,rows,takes", [
    (28672, 4096, 1595, True), (28672, 4096, 1600, True), (28672, 4096, 1601, False), (28672, 4096, 1536, False), (28672, 4096, 1537, True),
    (28672, 4096, 1056, True), (28672, 4096, 800, False), (28672, 4096, 1300, False), (28672, 4096, 1833, False), (28672, 4096, 300, False),
    (16384, 3072, 800, True), (16384, 3072, 1595, True), (16384, 2048, 2100, True), (16384, 2048, 1300, False), (16384, 1984, 800, False),
    (28672, 5184, 1595, False), (37904, 2048, 800, False), (28672, 4096, 59, False), (0, 4096, 800, False), (28672, 4096, 0, False)])
def test_short_tails(monkeypatch, n, k, rows, takes):
    from semi_pd_amd import ops
    monkeypatch.setitem(ops._DENSE_GEMM, "cus", 0)
    assert ops.tiled_gemm_short_tail(n, k, rows) == takes
    monkeypatch.setitem(ops._DENSE_GEMM, "cus", 128)
    assert not ops.tiled_gemm_short_tail(n, k, rows)


# (sizes that the rule was not made from, on both sides of each line: a free CU for each short tile, two in turn on few and on many free CUs, a
# round of their own, four rounds; weights of many rows and of more than 256 MB)
@pytest.mark.parametrize("n,k,rows,takes", [
    (12288, 2048, 1088, True), (9728, 2560, 1344, True), (18432, 2304, 1344, False), (14336, 3584, 1832, True), (14336, 3584, 1600, False),
    (9728, 2560, 1576, False), (8704, 3072, 1856, False), (5632, 2048, 2880, False), (14336, 3584, 1064, True), (22016, 4096, 1281, True),
    (24576, 3072, 1320, True), (29568, 4096, 1041, False), (24576, 3072, 1025, False), (28672, 4096, 1856, False), (24576, 3072, 2049, True),
    (32768, 4096, 808, False), (32768, 4096, 1064, False), (35840, 5120, 1320, False), (30720, 5120, 1088, False), (27648, 5120, 1064, True),
    (37888, 3584, 1576, True), (37888, 3584, 832, False), (37889, 2048, 1576, False)])
def test_short_tails_of_other_layers(monkeypatch, n, k, rows, takes):
    test_short_tails(monkeypatch, n, k, rows, takes)
