"""The fused gather + hash over maps of many extents: each workgroup finds its first extent by sampling one end per share of
the table and then looking inside that share, 64 ends at a time.  Table sizes around one share per lane, one look and two
looks per share; extents of ragged lengths, some longer than a workgroup's 64 KiB, with gaps the map leaves as they are.
Bytes and hash against numpy and the oracle's byte loop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 2, 31, 32, 33, 63, 64, 65, 2048, 2080, 2200])
def test_many_extents(sc, oracle, cuda, copies):
    rng = np.random.default_rng(copies)
    sizes = rng.integers(1, 60, copies) * 16
    if copies < 100:
        sizes[rng.integers(0, copies)] += 3 * 65536 + 16      # one extent over several workgroups
    gaps = np.where(rng.random(copies) < 0.9, rng.integers(1, 5, copies) * 16, 0)
    if copies > 2:
        gaps[0] = 0
    starts = np.cumsum(gaps) + np.concatenate([[0], np.cumsum(sizes)[:-1]])
    n = int(starts[-1] + sizes[-1]) + int(rng.integers(0, 40)) * 16
    print(f"case hash map of {copies} copies, {n} bytes", flush=True)
    data = rng.integers(0, 256, int(sizes.sum()), dtype=np.uint8)
    before = rng.integers(0, 256, n, dtype=np.uint8)
    src, payload = sc.DeviceBuffer(data.size, "uint8"), sc.DeviceBuffer(n, "uint8")
    src.upload(data)
    payload.upload(before)
    offs = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    plan = sc.plan_copies([(payload.ptr + int(d), src.ptr + int(o), int(b)) for d, o, b in zip(starts, offs, sizes)])
    want = before.copy()
    for d, o, b in zip(starts, offs, sizes):
        want[d:d + b] = data[o:o + b]
    hp, hm = sc.HashPlan(n), sc.HashMap([plan], payload.ptr, n)
    for _ in range(2):
        hm.launch(hp)
        sc.device_sync()
        assert hp.result() == oracle.fnv1a64(want.tobytes())
        assert np.array_equal(payload.numpy(), want)
    hm.destroy()
    plan.destroy()
    hp.free()
    for b in (src, payload):
        b.free()
