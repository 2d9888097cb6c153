"""Device-gated decode on the MI355X where the reference core is not built: every token's slot table and cache counters
against this library's own cache core on the CPU (the schedule tests/test_dgcore_parity.py pins to the reference's), and
every routed unit the engine read against its file bytes. Staged and direct units, copies on the HSA runtime's engines
and on HIP streams, the token as a graph and launched. (A corrupted unit that fails closed:
tests/test_gpu_dg_parity.py::test_device_check_gates_a_corrupted_unit.)"""
import numpy as np
import pytest

import test_gpu_dg_parity as base
from test_dgcore_parity import OurCore
from tierstream_amd import ss

pytestmark = pytest.mark.gpu
KiB = 1024


@pytest.mark.parametrize("parts,hip_copies,graph", [([64 * KiB] * 3, False, True), ([64 * KiB, 8 * KiB, 4096 + 256], False, False),
                                                    ([192 * KiB], False, True), ([192 * KiB], True, False)],
                         ids=["staged-graph", "staged-odd-launched", "hsa-graph", "hip-launched"])
def test_decode_matches_the_core(tmp_path, gpu, parts, hip_copies, graph):
    layers, units, n_ids, tokens = 4, 8, 2, 24
    m, bkw, okw = base._setup(tmp_path, layers, units, parts, 12, 1, 6, n_ids)
    routes = base._routes(layers, units, n_ids, tokens, seed=5, zipf=True)
    d = ss.Desc(m.desc_json())
    plan = ss.Plan(d, ss.budget(**bkw))
    tiers = plan.tiers()
    residents = [L * units + u for L in range(layers) for u in range(units) if tiers[L][u] == 0]
    P = sum(1 for r in tiers for t in r if t == 1)
    Q = plan.json()["spare_blocks"][0]["blocks"]
    D = sum(min(1, sum(1 for t in r if t != 0)) for r in tiers)
    core = OurCore([units] * layers, len(residents) + D, n_ids, P + Q, D, parts, residents + list(range(layers * units)),
                   wb_defer=1, inclusive=0)
    ctx = base._open(d, bkw, plan, okw, hip_copies)
    eng = ss.DgEngine(ctx, n_ids, use_graph=graph)
    try:
        assert ctx.hsa_copies() == (len(parts) == 1 and not hip_copies)
        for t in range(tokens):
            cks, _ = eng.token(routes[t])
            table, want = core.token(routes[t])
            got = ctx.dg_stats()
            assert np.array_equal(ctx.dg_table(), table), t
            assert {k: got[k] for k in base.COUNTERS} == {k: want[k] for k in base.COUNTERS}, t
            for L in range(layers):
                for i, u in enumerate(routes[t, L]):
                    assert int(cks[L, i]) == m.checksum(L, int(u)), (t, L, i)
        assert got["fetched"] > 0 and got["evicted"] > 0 and ctx.verify_failures() == 0
    finally:
        eng.close()
        ctx.close()
        core.close()
