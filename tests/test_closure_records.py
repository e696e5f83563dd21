"""The record tiles of the closure's backward kernels (vpfc.hip k_bwd_out,
k_bwd_in): all threads clear the tile, then each thread below 256 writes the
five records of its position, most of them into entries that another wave has
cleared.  A barrier has to stand between the two, in the source as the kernels
have it.  Host only: what a missing one does depends on the order of the waves."""

import os
import re

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = open(os.path.join(HERE, "..", "vlapy_amd", "csrc", "vpfc.hip")).read()
NV, TAPS, WAVE = 256, 5, 64


def _body(kernel):
    m = re.search(r"^__global__[^;{]*\b%s\(.*?^}" % kernel, SRC, re.S | re.M)
    return m.group(0)


@pytest.mark.parametrize("kernel,offset", [("k_bwd_out", lambda t, k: t - 2 + k), ("k_bwd_in", lambda t, k: t + 2 - k)])
def test_barrier_between_clearing_and_writing_the_records(kernel, offset):
    body = _body(kernel)
    threads = int(re.search(r"constexpr int kBT = (\d+);", SRC).group(1))
    clear = re.search(r"for \(int i = t; i < kNV \* 16; i \+= kBT\) R\[i\]", body)
    rows = body.index("for (int row = blockIdx.x")
    record = re.search(r"R\[q \* 16 \+ k\] =", body)
    assert clear.end() < rows < record.start()
    # the entry that thread t writes for tap k, and the thread that cleared it
    crossing = sum((16 * q + k) % threads // WAVE != t // WAVE
                   for t in range(NV) for k in range(TAPS) for q in [offset(t, k)] if 0 <= q < NV)
    assert crossing > 0
    # outside the row loop and not inside another block of the kernel
    between = re.sub(r"//.*", "", body[clear.end():rows])
    assert re.search(r"^  __syncthreads\(\);", between, re.M), kernel
