"""String keys read by 8-byte words: every length around the words, strings that differ in one byte at
every place, buffers of fewer bytes than a word, and later blocks that meet the strings in the arena,
against Python's own grouping of the bytes."""
import numpy as np
import pytest

import qikkdb_amd as qk
from qikkdb_amd.strings import DeviceStrings, GPUGroupByString

pytestmark = pytest.mark.gpu


def check(blocks, capacity=4096):
    gb = GPUGroupByString([qk.AGG_SUM, qk.AGG_COUNT], qk.LONG, capacity)
    want = {}
    at = 0
    for keys in blocks:
        vals = np.arange(at, at + len(keys), dtype=np.int64)
        at += len(keys)
        for k, v in zip(keys, vals):
            s, c = want.get(k, (0, 0))
            want[k] = (s + int(v), c + 1)
        gb.ProcessBlock(DeviceStrings.from_list(keys), qk.DeviceBuffer.from_numpy(vals), len(keys))
    r = gb.results_host()
    gb.close()
    got = {k: (int(r["values"][0][i]), int(r["values"][1][i])) for i, k in enumerate(r["keys"])}
    assert r["count"] == len(want) and got == want


@pytest.mark.parametrize("first", [b"", b"a", b"abcdefg", b"abcdefgh"])
def test_buffer_start(first):
    check([[first], [first, b"", b"xy"], [b"xy", first]], 16)


@pytest.mark.parametrize("seed", [1, 2])
def test_every_length_and_place(seed):
    rng = np.random.default_rng(seed)
    base = bytes(rng.integers(0, 256, 70).astype(np.uint8))
    keys = [base[:n] for n in range(71)] + [b"\x00" * n for n in range(1, 20)]
    for n in (1, 7, 8, 9, 16, 23, 40):
        for i in range(n):
            keys.append(base[:i] + bytes([base[i] ^ 1]) + base[i + 1:n])
    blocks = []
    for _ in range(3):
        order = rng.integers(0, len(keys), 3000)
        blocks.append([keys[i] for i in order])
    check(blocks)
