"""The fused gather + hash over maps of many extents: each workgroup finds its first extent by sampling one end per share of
the table and sampling again inside the share found.  Table sizes around one extent per share, one more sampling and two;
extents of ragged lengths, some longer than a workgroup's 64 KiB, with gaps the map leaves as they are.  Bytes and hash against
numpy and the oracle's byte loop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 2, 31, 32, 33, 63, 64, 65, 2048, 2080, 2200, 5000, 40000])
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


@pytest.mark.parametrize("n", [16, 240, 256, 272, 65536, 65536 + 16, 65536 + 240, 65536 + 256, 2 * 65536 + 128])
def test_tail_at_the_edges_of_a_workgroup(sc, oracle, cuda, n):
    """The last partial 256 bytes, hashed by the closing kernel, alone in their workgroup's 64 KiB, after it, or none."""
    print(f"case hash tail {n}", flush=True)
    data = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    src, payload = sc.DeviceBuffer(n, "uint8"), sc.DeviceBuffer(n, "uint8")
    src.upload(data)
    payload.fill(0)
    plan = sc.plan_copies([(payload.ptr, src.ptr, n)])
    want = oracle.fnv1a64(data.tobytes())
    hp, hm = sc.HashPlan(n), sc.HashMap([plan], payload.ptr, n)
    hm.launch(hp)
    sc.device_sync()
    assert hp.result() == want and np.array_equal(payload.numpy(), data)
    seg = 65536
    parts = [sc.DeviceBuffer(seg, "uint8") for _ in range(-(-n // seg))]
    for k, b in enumerate(parts):
        b.fill(0)
        b.upload(data[k * seg:(k + 1) * seg])
    rm = sc.HashMap.read([b.ptr for b in parts], seg, n)
    rm.check(hp, want)
    sc.device_sync()
    assert hp.result() == want and int(hp.verdict.numpy()[0]) == 1
    for m in (hm, rm, plan):
        m.destroy()
    hp.free()
    for b in (src, payload, *parts):
        b.free()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 63, 64, 65, 253, 254, 255, 257, 511, 65535, 65537, 65536 + 255, 200003])
def test_odd_lengths_aligned_and_not(sc, oracle, cuda, n):
    print(f"case hash length {n}", flush=True)
    data = np.random.default_rng(n).integers(0, 256, n + 16, dtype=np.uint8)
    buf, carry = sc.DeviceBuffer(n + 16, "uint8"), sc.DeviceBuffer(16, "uint8")
    buf.upload(data)
    hp = sc.HashPlan(n)
    for shift in (0, 5):
        want = oracle.fnv1a64(data[shift:shift + n].tobytes())
        hp.launch_carry(buf.ptr + shift, n, carry.ptr)
        sc.device_sync()
        assert hp.result() == want
        hp.check_carried(buf.ptr + shift, n, want, carry.ptr)
        sc.device_sync()
        assert int(hp.verdict.numpy()[0]) == 1 and hp.fault_word() == 0
        hp.start()
        hp.chain(buf.ptr + shift, n // 2)
        hp.chain(buf.ptr + shift + n // 2, n - n // 2)
        sc.device_sync()
        assert hp.result() == want
    hp.free()
    for b in (buf, carry):
        b.free()
