"""How far the AXPY kernel's 16-byte loads of A reach (no GPU needed).

With M not a multiple of 4 the load that crosses row M reads on into the next
column, so in the last column it would leave A; what it reads is not stored, so
no result shows it.  Here the lanes' offsets are restated, with the number of
full steps and the stride rule taken from the kernel's source."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hiperml_amd", "csrc")


def source(name):
    return open(os.path.join(CSRC, name)).read()


def constant(name):
    return int(re.search(r"constexpr int %s = (\d+);" % name, source("hml_internal.h")).group(1))


def full_steps(K, kb, ke, ragged):
    e, = re.search(r"const int64_t nfull = ke > kb \? (\(ke - kb.*?\) / kAxpyKStep) : 0;",
                   source("hml_k_skinny.hip")).groups()
    e, n = re.subn(r"\(ragged && ke == p\.K \? 1 : 0\)", "(1 if ragged and ke == K else 0)", e)
    assert n == 1, e
    step = constant("kAxpyKStep")
    return eval(e.replace("/", "//").replace("kAxpyKStep", str(step)), dict(ragged=ragged, ke=ke, kb=kb, K=K))


def reach(M, K, lda, chunks):
    """The furthest float that the full steps of any chunk touch."""
    step = constant("kAxpyKStep")
    kchunk = -(-K // chunks)
    kchunk = -(-kchunk // step) * step
    row = (M - 1) // 4 * 4  # the last lane below row M
    far = -1
    for kb in range(0, K, kchunk):
        n = full_steps(K, kb, min(K, kb + kchunk), M % 4 != 0)
        if n:
            far = max(far, (kb + n * step - 1) * lda + row + 3)
    return far


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 63, 64, 65, 127, 130, 5003])
def test_full_steps_stay_in_a(M):
    smallest, = re.search(r"p\.M % 4 != 0 && p\.sAk < (\d+) \? 0 :", source("hml_k_skinny.hip")).groups()
    for K in (16, 17, 31, 32, 33, 160, 161, 9001):
        for lda in {max(M, int(smallest)), max(M, int(smallest)) + 1, M + 61}:
            for chunks in (1, 2, 3, 8):
                assert reach(M, K, lda, chunks) <= (K - 1) * lda + M - 1, (K, lda, chunks)
