"""The destination order's list is counted and written in blocks of 1024 physical pages (4096 of a pool past 2^22): pools
that end one page before, on and one page after a block's end, and tables spread over several blocks, place every byte as
the oracle does."""
import numpy as np
import pytest

import sc_synthetic as synth

pytestmark = pytest.mark.gpu

GEO = dict(n_layers=8, qsa_interval=4, n_head_kv=2, head_dim=256, page_size=4, ssm_state_size=32, ssm_k_heads=4,
           ssm_v_heads=8, ssm_d_conv=4, ssm_conv_channels=520)


@pytest.mark.parametrize("n_pages,T", [(1023, 3001), (1024, 4096), (1025, 4097), (2048, 5555), (2049, 6000)])
def test_order_at_the_blocks_edges(sc, oracle, cuda, n_pages, T):
    # (a table of too few pages for its pool is not ordered, so each covers at least half of them)
    print(f"case order blocks pages={n_pages} T={T}", flush=True)
    geo = sc.geometry(**GEO)
    H, D, ps = geo.n_head_kv, geo.head_dim, geo.page_size
    logical = (T + ps - 1) // ps
    rng = np.random.default_rng(n_pages + T)
    tables = []
    for _ in range(geo.n_qsa):
        t = rng.permutation(n_pages)[:logical].astype(np.int32)
        if n_pages - 1 not in t:
            t[logical // 2] = n_pages - 1   # the pool's last page is always one of them
        tables.append(t)
    case = synth.SyntheticCase(geo, tokens=T, seed=n_pages)
    previous = sc.set_order_min_pages(1)
    try:
        slot = sc.new_slot(geo, logical * ps, n_pages=n_pages, tables=sc.device_tables(tables), fill=0xEE)
        sc.device_sync()
        plan = sc.plan_carve(geo, case.prefill, slot, with_gdn=False)
        assert plan.order_groups == geo.n_qsa
    finally:
        sc.set_order_min_pages(previous)
    for _ in range(2):   # the second launch finds the inverse table cleared
        plan.launch()
    sc.device_sync()
    inputs, got = case.host_inputs(), slot.host_state()
    for j in range(geo.n_qsa):
        for kv in ("k", "v"):
            want = np.full(n_pages * H * ps * D, 0xEEEE, dtype=np.uint16)
            oracle.kv_append(inputs[kv][j], T, 0, tables[j], n_pages, H, D, ps, want)
            assert np.array_equal(got[f"{kv}{j}"].reshape(-1), want), f"{kv}{j} differs"
    plan.destroy()


@pytest.mark.parametrize("n_pages", [(1 << 22) - 1, 1 << 22, (1 << 22) + 1, (1 << 22) + 4096, (1 << 22) + 4097])
def test_order_of_a_large_pool(sc, cuda, n_pages):
    """Pools past 2^22 pages are counted and written in blocks of 4096 pages."""
    T = n_pages // 8 + 1
    print(f"case order of a large pool, pages={n_pages} T={T}", flush=True)
    geo = sc.geometry(**{**GEO, "n_layers": 4, "n_head_kv": 1, "head_dim": 8, "page_size": 1})
    table = np.random.default_rng(n_pages).permutation(n_pages)[:T].astype(np.int32)
    table[T // 2] = n_pages - 1 if n_pages - 1 not in table else table[T // 2]
    case = synth.SyntheticCase(geo, tokens=T, seed=n_pages)
    slot = sc.new_slot(geo, T, n_pages=n_pages, tables=sc.device_tables([table]), fill=0xEE)
    sc.device_sync()
    plan = sc.plan_carve(geo, case.prefill, slot, with_gdn=False)
    assert plan.order_groups == 1
    for _ in range(2):
        plan.launch()
    sc.device_sync()
    inputs, got = case.host_inputs(), slot.host_state()
    for kv in ("k", "v"):
        want = np.full((n_pages, 8), 0xEEEE, dtype=np.uint16)
        want[table] = inputs[kv][0].reshape(T, 8)
        assert np.array_equal(got[f"{kv}0"].reshape(n_pages, 8), want), f"{kv} differs"
    plan.destroy()
