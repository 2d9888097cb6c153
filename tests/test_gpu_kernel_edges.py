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


# Workgroups whose units all have at most 32 stripes hash them straight from memory; one with a stripe more is fed.
@pytest.mark.parametrize("n", [2, 513, 1025, 2049, 4097, 12288])
@pytest.mark.parametrize("longest", [1024 + 31, 1024 + 32])
def test_digest_small_units(gpu, n, longest):
    rng = np.random.default_rng(n)
    data = rng.integers(0, 256, 1 << 16, dtype=np.uint8)
    buf = gpu.DeviceBuffer(data.nbytes)
    buf.upload(data)
    shapes = [[0], [7], [32], [1023], [32, 0], [512, 512], [96, 64, 32, 33], [longest], [512, 32, longest - 544]]
    units, want = [], []
    for i in range(n):
        sizes = shapes[(i + i // 9) % len(shapes)] if i % 64 < 48 else [64]  # (long ones in some workgroups only)
        at = [int(rng.integers((data.nbytes - s) // 8)) * 8 for s in sizes]
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


# The checks by segment size and by size. Streamed: 2 KiB segments; on whole cache lines also 1 KiB ones above 80 MB and, in
# the copy, any whole pair of 256-byte chunks up to 4 KiB and 80 MB, above 1 KiB. Two chunk buffers a wave, four above 80 MB
# in the copy and off the cache lines, all chunks in flight up to 96 segments of 2 KiB. The chain loop: other segments; up to
# 80 MB also arenas with a part that is 8-byte aligned; above, and in batches and the copy, the waves that hold one. Units in
# rows of workgroups or packed; parts that end inside a segment, inside a stripe, or are none.
SHAPES = [
    (1, [2048], 2048), (1, [32], 2048), (2, [8], 2048), (1, [2080, 40], 2048), (5, [65568, 4096, 1000], 2048),
    (64, [30 * 2048 + 32, 96], 2048), (3, [2048 * 17, 2048 * 15 + 64, 32, 2048], 2048), (3, [(8 << 20) + 32, 1 << 20], 2048),
    (3, [28 << 20, (3 << 20) + 48], 2048), (3, [45 << 20, 4096 + 24], 2048), (2, [65536, 2048 + 1008], 512), (3, [65536 + 96, 1024 * 16], 1024),
    (2, [9 << 20, 1024 * 3 + 8], 1024), (3, [1536 * 40 + 32, 1536 * 16 - 8], 1536), (2, [1 << 20, 4096 * 3 + 56], 4096), (2, [1 << 20, 4096 * 3 + 128], 4096),
    (1, [65536, 40], 4096), (2, [65536 + 64, 128], 1536), (64, [530016, 40], 2048), (70, [530016, 48], 2048),
    (3, [28 << 20, 4096 + 16], 4096), (3, [28 << 20, (3 << 20) + 1000], 1024),
    (1, [84 << 20, (3 << 20) + 48], 2048),
    (3, [32 * 2048, 64 * 2048], 2048), (3, [32 * 2048, 64 * 2048 + 64], 2048), (3, [44 << 20, (3 << 20) + 48], 1024), (2, [44 << 20, (3 << 20) + 128], 1024), (2, [1 << 20, 8192 + 32], 8192), (2, [1 << 18, 4000], 2080),
]


def _bad_at(parts, n):
    """A byte to spoil in each unit but the last: the first, the last, and ones next to the parts' and segments' ends."""
    ub = sum(parts)
    at = [0, ub - 1, parts[0] - 1, min(parts[0], ub - 1), min(2047, ub - 1), min(2048, ub - 1), max(0, parts[0] - 32), ub // 2]
    return [at[i % len(at)] for i in range(n - 1)]


@pytest.mark.parametrize("n,parts,seg", SHAPES)
@pytest.mark.parametrize("staged", [False, True])
def test_arena_checks_by_shape(gpu, n, parts, seg, staged):
    rng = np.random.default_rng(n + sum(parts) + seg)
    ub, slots_n = sum(parts), n + 2
    data = rng.integers(0, 256, (n, ub), dtype=np.uint8)
    cuts = np.cumsum([0] + parts)
    arrays = lambda u: [u[a:b] for a, b in zip(cuts, cuts[1:])]
    marks = [gpu.host_checkpoints(arrays(data[i]), seg) for i in range(n)]
    keys, slots = rng.permutation(n), rng.permutation(slots_n)[:n]
    states, digests = np.zeros((n, len(marks[0][0])), dtype=np.uint64), np.zeros(n, dtype=np.uint64)
    for k, (st, dg) in zip(keys, marks):
        states[k], digests[k] = st, dg
    bufs = [gpu.DeviceBuffer(slots_n * p) for p in parts]
    st_dev, dg_dev, fail = gpu.DeviceBuffer(states.nbytes), gpu.DeviceBuffer(digests.nbytes), gpu.DeviceBuffer(4 * n)
    st_dev.upload(states)
    dg_dev.upload(digests)
    src = gpu.DeviceBuffer(n * ub)
    a = gpu.TsaArenaVerify()
    for p, (buf, pb) in enumerate(zip(bufs, parts)):
        buf.upload(np.zeros(slots_n * pb, dtype=np.uint8))
        a.arena[p], a.part_bytes[p] = buf.ptr, pb
    a.n_parts, a.seg_bytes, a.states_dev, a.digests_dev = len(parts), seg, st_dev.ptr, dg_dev.ptr
    for bad in ([], _bad_at(parts, n)):
        for i, at in enumerate(bad):
            data[i, at] ^= 0x10
        fail.upload(np.zeros(n, dtype=np.uint32))
        args = [C.byref(a), (C.c_uint32 * n)(*map(int, keys)), (C.c_int32 * n)(*map(int, slots)), n]
        if staged:
            src.upload(data.reshape(-1))
            gpu.check(gpu.lib().tsa_xxh64_scatter_verify_slots(*args, C.c_void_p(src.ptr), C.c_void_p(fail.ptr), None))
        else:
            for i in range(n):
                for buf, x in zip(bufs, arrays(data[i])):
                    buf.upload(x, int(slots[i]) * x.nbytes)
            gpu.check(gpu.lib().tsa_xxh64_verify_slots(*args, C.c_void_p(fail.ptr), None))
        gpu.check(gpu.lib().tsa_stream_sync(None))
        assert list(fail.download(4 * n).view(np.uint32)) == [1 if i < len(bad) else 0 for i in range(n)]
        if staged:  # every unit in its slot, and nothing anywhere else
            for p, buf in enumerate(bufs):
                got = buf.download().reshape(slots_n, parts[p])
                for s in range(slots_n):
                    i = np.flatnonzero(slots == s)
                    assert np.array_equal(got[s], arrays(data[i[0]])[p] if len(i) else np.zeros(parts[p], dtype=np.uint8))


@pytest.mark.parametrize("align", [8, 16])
@pytest.mark.parametrize("n,parts,seg", SHAPES + [(200, [30000 + 16, 11], 2048), (70, [32, 0], 2048), (3, [0], 2048)])
def test_batch_checks_by_shape(gpu, n, parts, seg, align):
    rng = np.random.default_rng(n + sum(parts) + seg + align)
    sizes = [parts[:-1] + [parts[-1] + i % 5] for i in range(n)]
    at, pos = 0, []
    for unit in sizes:
        row = []
        for b in unit:
            at = -(-at // align) * align + align * int(rng.integers(2))
            row.append(at)
            at += b
        pos.append(row)
    host = rng.integers(0, 256, at + 32, dtype=np.uint8)
    buf = gpu.DeviceBuffer(host.nbytes)
    marks = [gpu.host_checkpoints([host[p:p + b] for p, b in zip(row, unit)], seg) for row, unit in zip(pos, sizes)]
    st_dev = gpu.DeviceBuffer(sum(st.nbytes for st, _ in marks))
    st_dev.upload(np.concatenate([st for st, _ in marks]))
    units, first = [], 0
    for row, unit, (st, dg) in zip(pos, sizes, marks):
        v = gpu.TsaVerifyUnit()
        for e, (p, b) in enumerate(zip(row, unit)):
            v.ext[e].ptr, v.ext[e].bytes = buf.ptr + p, b
        v.n_ext, v.seg_first, v.states, v.digest, v.total = len(unit), first, st_dev.ptr + 32 * first, dg, sum(unit)
        first += len(st) // 4
        units.append(v)
    table, fail = gpu.upload_struct_array(units), gpu.DeviceBuffer(4 * n)
    for spoil in (False, True):
        want = [0] * n
        if spoil:
            for i, o in enumerate(_bad_at(parts, n)):  # (a byte of the unit: counted through its extents)
                for p, b in zip(pos[i], sizes[i]):
                    if 0 <= o < b:
                        host[p + o] ^= 0x04
                        want[i] = 1
                        break
                    o -= b
        buf.upload(host)
        fail.upload(np.zeros(n, dtype=np.uint32))
        gpu.check(gpu.lib().tsa_xxh64_verify(C.c_void_p(table.ptr), n, first, seg, C.c_void_p(fail.ptr), None))
        gpu.check(gpu.lib().tsa_stream_sync(None))
        assert list(fail.download(4 * n).view(np.uint32)) == want


# A checkpoint is four 64-bit words: it may lie 8-byte aligned, and the kernels read it in 16-byte pieces.
@pytest.mark.parametrize("how", ["check", "staged", "batch"])
@pytest.mark.parametrize("parts,seg", [([65536 + 96, 4000], 2048), ([65536, 1024 * 3 + 8], 1024), ([32768 + 32, 40], 4096)])
def test_checkpoints_at_8_bytes(gpu, how, parts, seg):
    rng = np.random.default_rng(seg)
    n, ub = 3, sum(parts)
    data = rng.integers(0, 256, (n, ub), dtype=np.uint8)
    cuts = np.cumsum([0] + parts)
    marks = [gpu.host_checkpoints([u[a:b] for a, b in zip(cuts, cuts[1:])], seg) for u in data]
    words = len(marks[0][0])
    st_dev, fail = gpu.DeviceBuffer(8 + 8 * words * n), gpu.DeviceBuffer(4 * n)
    st_dev.upload(np.concatenate([np.zeros(1, dtype=np.uint64)] + [st for st, _ in marks]))
    states = st_dev.ptr + 8
    assert states % 16 == 8
    src = gpu.DeviceBuffer(n * ub)
    for bad in (None, 1):
        if bad is not None:
            data[bad, parts[0] - 1] ^= 1
        src.upload(data.reshape(-1))
        fail.upload(np.zeros(n, dtype=np.uint32))
        if how == "batch":
            units = []
            for i in range(n):
                v = gpu.TsaVerifyUnit()
                for e, (at, b) in enumerate(zip(cuts, parts)):
                    v.ext[e].ptr, v.ext[e].bytes = src.ptr + i * ub + int(at), b
                v.n_ext, v.seg_first, v.digest, v.total = len(parts), i * words // 4, marks[i][1], ub
                v.states = states + 8 * words * i
                units.append(v)
            table = gpu.upload_struct_array(units)
            gpu.check(gpu.lib().tsa_xxh64_verify(C.c_void_p(table.ptr), n, n * words // 4, seg, C.c_void_p(fail.ptr), None))
        else:
            dg_dev = gpu.DeviceBuffer(8 * n)
            dg_dev.upload(np.array([dg for _, dg in marks], dtype=np.uint64))
            bufs = [gpu.DeviceBuffer(n * p) for p in parts]
            a = gpu.TsaArenaVerify()
            for p, (buf, pb) in enumerate(zip(bufs, parts)):
                buf.upload(np.ascontiguousarray(data[:, cuts[p]:cuts[p + 1]]).reshape(-1))
                a.arena[p], a.part_bytes[p] = buf.ptr, pb
            a.n_parts, a.seg_bytes, a.states_dev, a.digests_dev = len(parts), seg, states, dg_dev.ptr
            args = [C.byref(a), (C.c_uint32 * n)(*range(n)), (C.c_int32 * n)(*range(n)), n]
            if how == "staged":
                gpu.check(gpu.lib().tsa_xxh64_scatter_verify_slots(*args, C.c_void_p(src.ptr), C.c_void_p(fail.ptr), None))
            else:
                gpu.check(gpu.lib().tsa_xxh64_verify_slots(*args, C.c_void_p(fail.ptr), None))
        gpu.check(gpu.lib().tsa_stream_sync(None))
        assert list(fail.download(4 * n).view(np.uint32)) == [int(i == bad) for i in range(n)]


# 16 KiB blocks part by part; more jobs than a wave's 64 probes.
@pytest.mark.parametrize("n,parts", [(1, [16]), (1, [16384]), (2, [16400, 32, 0, 16368]), (65, [16384 * 3, 48]),
                                     (200, [1024, 16]), (3, [13 << 20, (1 << 20) + 16])])
def test_scatter_jobs(gpu, n, parts):
    rng = np.random.default_rng(n + sum(parts))
    ub = sum(parts)
    host = rng.integers(0, 256, (n, ub), dtype=np.uint8)
    src, bufs = gpu.DeviceBuffer(host.nbytes), [gpu.DeviceBuffer((n + 1) * max(p, 16)) for p in parts]
    src.upload(host.reshape(-1))
    for buf, p in zip(bufs, parts):
        buf.upload(np.zeros((n + 1) * max(p, 16), dtype=np.uint8))
    per = int(gpu.lib().tsa_scatter_blocks((C.c_uint64 * len(parts))(*parts), len(parts)))
    slots, jobs = rng.permutation(n + 1)[:n], []
    for i in range(n):
        j = gpu.TsaScatterJob()
        j.src, j.n_parts, j.block_first = src.ptr + i * ub, len(parts), i * per
        for p, (buf, pb) in enumerate(zip(bufs, parts)):
            j.dst[p], j.bytes[p] = buf.ptr + int(slots[i]) * pb, pb
        jobs.append(j)
    table = gpu.upload_struct_array(jobs)
    gpu.check(gpu.lib().tsa_scatter(C.c_void_p(table.ptr), n, n * per, None))
    gpu.check(gpu.lib().tsa_stream_sync(None))
    cuts = np.cumsum([0] + parts)
    for p, buf in enumerate(bufs):
        want = np.zeros((n + 1, parts[p]), dtype=np.uint8)
        want[slots] = host[:, cuts[p]:cuts[p + 1]]
        assert np.array_equal(buf.download()[:want.size].reshape(want.shape), want)
