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
