"""The device kernels at the edges of their tiles and of the rules that choose between them, bit-exact against xxhash
and the oracle (MI355X)."""
import ctypes as C

import numpy as np
import pytest
import xxhash

pytestmark = pytest.mark.gpu


# Units per workgroup 1, 2, 4, 8, 16, then a quad per unit; a chunk is 512 stripes (16 KiB) over a workgroup's units.
@pytest.mark.parametrize("n", [1, 512, 513, 1025, 2049, 4097, 12288, 12289])
def test_digest_unit_counts(gpu, n):
    rng = np.random.default_rng(n)
    data = rng.integers(0, 256, 1 << 20, dtype=np.uint8)
    buf = gpu.DeviceBuffer(data.nbytes)
    buf.upload(data)
    shapes = [[0], [5], [31], [32], [63], [512], [1024 - 32], [1024], [1024 + 33], [2048 + 7], [4096], [16384 - 1], [16384],
              [3 * 16384 + 40], [32, 0], [32 * 7, 8], [96, 64, 32, 33], [1024, 1024, 1024, 1024], [16384 * 2 + 32, 4096, 17]]
    if n == 1:
        shapes = [[5 * 16384 + 32 * 511, 32 * 513, 16384, 16384 * 3 + 31]]
    units, want = [], []
    for i in range(n):
        sizes = shapes[i % len(shapes)] if i < 4 * len(shapes) else shapes[int(rng.integers(len(shapes)))]
        at = [int(rng.integers((data.nbytes - s) // 8)) * 8 for s in sizes]  # extents anywhere, 8-byte aligned
        units.append(gpu.make_unit([(buf.ptr + a, s) for a, s in zip(at, sizes)]))
        want.append(xxhash.xxh64_intdigest(b"".join(data[a:a + s].tobytes() for a, s in zip(at, sizes))))
    assert gpu.device_digests(units) == want


# Kind 2 is made in groups of nine words (four Q4 blocks), 256 groups to a workgroup; kinds 0 and 1 two words to a lane.
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("words,offset", [(1, 0), (2, 1), (8, 8), (9, 9), (511, 3), (2304, 0), (2304, 5), (2305, 2300),
                                          (3 * 2304 + 7, 9 * 77777 + 4)])
def test_synth_edges(gpu, kind, words, offset):
    from oracle import synth
    n, at = 8 * words, 8 * offset
    for lead in (8, 16):  # the destination 8-byte or 16-byte aligned, the words around it left alone
        buf = gpu.DeviceBuffer(lead + n + 16)
        buf.upload(np.full(lead + n + 16, 0xA5, dtype=np.uint8))
        gpu.check(gpu.lib().tsa_synth(C.c_void_p(buf.ptr + lead), n, 99, 5, at, kind, C.c_float(0.02), None))
        gpu.check(gpu.lib().tsa_stream_sync(None))
        got = buf.download()
        assert np.all(got[:lead] == 0xA5) and np.all(got[lead + n:] == 0xA5)
        got = got[lead:lead + n]
        if kind == 1:
            # Against 64 bits: bf16 rounding and a few 32-bit roundings (2^-8 of the value); a 24-bit u1 moves
            # r^2 = -2 ln u1 by up to 2^-24, so r by 2^-25 / r, and near r = 0 by at most its root; the angle's own
            # 32-bit roundings move a value next to a zero of cos or sin by 2^-22 r.
            w = synth.words(99, 5, 2 * offset, 2 * words)
            u = [((w >> np.uint64(32)).astype(float) + 0.5) / 2 ** 32, ((w & np.uint64(0xFFFFFFFF)).astype(float) + 0.5) / 2 ** 32]
            r = np.sqrt(-2 * np.log(u[0]))
            want = 0.02 * np.stack([r * np.cos(2 * np.pi * u[1]), r * np.sin(2 * np.pi * u[1])], axis=1).reshape(-1)
            slack = 0.02 * np.repeat(2.0 ** -24 / np.maximum(r, 2.0 ** -12) + 2.0 ** -22 * r, 2)
            have = (got.view(np.uint16).astype(np.uint32) << 16).view(np.float32)
            assert np.all(np.abs(have - want) <= np.abs(want) * 2.0 ** -8 + slack)
        else:
            assert np.array_equal(got, synth.uniform_bytes(99, 5, at, n) if kind == 0 else synth.q4_blocks(99, 5, at, n))
