"""The plans that gemm() picks, from its plan trace, for problems too large to
allocate in a test. Run in a process that sees no GPU: the call plans, its
launches fail, and the operands (null) are never read."""
import os
import re
import subprocess
import sys

import pytest

import bmb

PKG = bmb.PKG_DIR
NARROW = 9  # the part that runs on the element-by-element kernel

CALL = """
import sys
sys.path.insert(0, %r)
import bmb
ta, tb, M, N, K = (int(v) for v in sys.argv[1:])
bmb.gemm(bool(ta), bool(tb), M, N, K, 1.0, 0, 0, 0.0, 0)
""" % PKG


def _plan(ta, tb, M, N, K):
    """The first plan traced: (m1, [(tile, splits, k per range), ...])."""
    env = dict(os.environ, BMB_GEMM_PLAN_TRACE="1", HIP_VISIBLE_DEVICES="-1",
               ROCR_VISIBLE_DEVICES="-1", CUDA_VISIBLE_DEVICES="-1")
    r = subprocess.run([sys.executable, "-c", CALL] + [str(int(v)) for v in (ta, tb, M, N, K)],
                       capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0, r.stderr
    m = re.search(r"bf16x3 gemm plan %dx%dx%d: m1 (\d+) .* parts (.*) model" % (M, N, K), r.stderr)
    assert m, r.stderr
    parts = [tuple(int(v) for v in q.split(",")) for q in re.findall(r"\(([^)]*)\)", m.group(2))]
    return int(m.group(1)), parts


# The staging loads' 32-bit byte offsets: 33 stored rows of an operand whose m
# or n is contiguous, a tile's rows of one whose k is, have to stay below 2^32
# bytes, by the stored stride of the whole problem also in a band of it.
@pytest.mark.parametrize("ta,tb,M,N,K", [(1, 0, 40_000_000, 64, 800), (1, 1, 36_000_000, 256, 1024),
                                         (0, 0, 64, 36_000_000, 800), (0, 1, 64, 64, 40_000_000)])
def test_offsets_that_do_not_fit_take_the_element_kernel(ta, tb, M, N, K):
    m1, parts = _plan(ta, tb, M, N, K)
    assert m1 == M and parts[0][0] == NARROW, (m1, parts)


def test_element_kernel_splits_a_long_k():
    _, parts = _plan(0, 1, 64, 64, 40_000_000)
    assert parts[0][0] == NARROW and parts[0][1] > 1, parts


# A dimension that does not enter the offsets may be as long as it likes.
@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 0, 34_000_000, 64, 32), (0, 0, 40_000_000, 16, 16),
                                         (0, 1, 16, 40_000_000, 16), (1, 0, 64, 64, 40_000_000),
                                         (0, 1, 100_000_000, 8, 8)])
def test_offsets_that_fit_take_the_tiles(ta, tb, M, N, K):
    m1, parts = _plan(ta, tb, M, N, K)
    assert parts[0][0] != NARROW and (m1 == M or parts[1][0] != NARROW), (m1, parts)
    if K > 1 << 20:
        assert parts[0][1] > 1, parts


# Short dimensions: only an operand of fewer than four elements (or an empty
# product) needs the element kernel. An M (or N) below 4 is any tile's edge
# unless it is the stored row length.
@pytest.mark.parametrize("ta,tb,M,N,K,tiles", [
    (0, 1, 1, 768, 768, range(NARROW)), (0, 0, 3, 50257, 768, range(NARROW)),
    (1, 1, 2304, 2, 768, range(NARROW)), (1, 0, 768, 768, 2, range(NARROW)),
    (0, 0, 8192, 1, 768, (1, 2, 5, 7)), (1, 0, 3, 768, 8192, (1, 2, 5, 7)),
    (0, 1, 768, 768, 3, (1, 2, 5, 7)), (1, 1, 1, 768, 4096, (1, 2, 5, 7)),
    (0, 0, 1, 768, 3, (NARROW,)), (0, 1, 3, 1, 2, (NARROW,)), (0, 0, 64, 64, 0, (NARROW,))])
def test_short_dimensions(ta, tb, M, N, K, tiles):
    m1, parts = _plan(ta, tb, M, N, K)
    assert parts[0][0] in tiles, parts
