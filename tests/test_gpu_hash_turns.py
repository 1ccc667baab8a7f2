"""The device FNV-1a at its launches' edges: a check given carries hands each workgroup up to four 64 KiB pieces in turn
(one below 2560 pieces, two below 5120, four from there, piece k, k + grid, ...), in grids that leave the last turn short, and
the sums of every piece are brought to the input's end.  Hashes against the oracle's byte loop; a changed byte or carry in
any turn is refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GROUP = 64 << 10


SIZES = [(0, 1), (1, 0), (1, 16), (2, GROUP - 1), (257, 255), (2559, 5), (2560, 0), (2561, 4097), (3840, 256),
         (5121, 777), (7683, 16)]


def _byte_loop(oracle, buf, start, n):
    h, step = oracle.fnv1a64(b""), 256 << 20
    for at in range(0, n, step):
        h = oracle.fnv1a64(buf.numpy(min(step, n - at), start=start + at), h)
    return h


@pytest.mark.parametrize("groups,extra,shift", [(g, x, s) for g, x in SIZES for s in (0, 3)])
def test_carried_check_in_turns(sc, oracle, cuda, groups, extra, shift):
    n = groups * GROUP + extra
    print(f"case hash turns {groups} x 64 KiB + {extra} at offset {shift}", flush=True)
    buf = sc.DeviceBuffer(n + 64, "uint8")
    sc.check(sc.lib.sc_fill_uniform_f16(buf.ptr, (n + 64) // 2, -4.0, 4.0, 77 + groups, extra, None), "fill")
    sc.device_sync()
    h = _byte_loop(oracle, buf, shift, n)
    carry = sc.DeviceBuffer(max(sc.carry_bytes(n), 16), "uint8")
    hp = sc.HashPlan(n)
    hp.launch_carry(buf.ptr + shift, n, carry.ptr)
    sc.device_sync()
    assert hp.result() == h
    # the same bytes as three chained pieces
    hp.start()
    cuts = [0, n // 3, n // 3 * 2 + 1 if n > 2 else n, n]
    for a, b in zip(cuts, cuts[1:]):
        hp.chain(buf.ptr + shift + a, b - a)
    sc.device_sync()
    assert hp.result() == h

    def check():
        hp.check_carried(buf.ptr + shift, n, h, carry.ptr)
        sc.device_sync()
        return int(hp.verdict.numpy()[0]), hp.fault_word()

    def flip(b, at):
        b.upload(b.numpy(1, start=at) ^ 1, start=at)

    assert check() == (1, 0) and int(hp.out.numpy()[0]) == h
    # a byte of each turn's first, middle and last piece, in a whole segment.  The low byte's machine is one to one from
    # any state, so the piece ends with another low byte than the carry after it, if there is one
    pieces = -(-n // GROUP)
    turns = 1 if pieces < 2560 else 2 if pieces < 5120 else 4
    grid = -(-pieces // turns)
    each = [k for t in range(turns) for k in {t * grid, (t * grid + min((t + 1) * grid, pieces)) // 2, min((t + 1) * grid, pieces) - 1}
            if k < pieces]
    whole = n // 256 * 256   # what follows is the closing kernel's (of an aligned input)
    for k in each:
        size = min((k + 1) * GROUP, whole) - k * GROUP
        if size <= 0:
            continue
        at = shift + k * GROUP + (k * 7919 + 12345) % size
        flip(buf, at)
        verdict, fault = check()
        assert verdict == 0 and fault == (sc.FNV_FAULT_CARRY if k < sc.carry_bytes(n) else 0), f"byte of piece {k}"
        flip(buf, at)
    # one carry of each turn: the workgroup before it ends elsewhere
    for k in each:
        if k < sc.carry_bytes(n):
            flip(carry, k)
            assert check() == (0, sc.FNV_FAULT_CARRY), f"carry {k}"
            flip(carry, k)
    # the last byte (the closing kernel hashes it when an aligned input ends in a partial segment)
    flip(buf, shift + n - 1)
    assert check() == (0, 0)
    flip(buf, shift + n - 1)
    assert check() == (1, 0)
    for b in (buf, carry):
        b.free()
    hp.free()


def test_input_past_65536_pieces(sc, oracle, cuda):
    """More than 4 GiB: a piece's distance from the end takes a third byte.  Plain, with carries, chained, gathered, and read
    from segments."""
    n = (65536 + 300) * GROUP + 48
    print(f"case hash {n} bytes", flush=True)
    buf = sc.DeviceBuffer(n, "uint8")
    sc.check(sc.lib.sc_fill_uniform_f16(buf.ptr, n // 2, -4.0, 4.0, 5, 6, None), "fill")
    sc.device_sync()
    h = _byte_loop(oracle, buf, 0, n)
    carry = sc.DeviceBuffer(sc.carry_bytes(n), "uint8")
    hp = sc.HashPlan(n)
    hp.launch_carry(buf.ptr, n, carry.ptr)
    assert hp.result() == h
    hp.check_carried(buf.ptr, n, h, carry.ptr)
    sc.device_sync()
    assert int(hp.verdict.numpy()[0]) == 1 and hp.fault_word() == 0
    seg = 1 << 30
    parts = [buf.ptr + at for at in range(0, n, seg)]
    rm = sc.HashMap.read(parts, seg, n)
    rm.check(hp, h)
    sc.device_sync()
    assert int(hp.verdict.numpy()[0]) == 1 and hp.fault_word() == 0
    payload = sc.DeviceBuffer(n, "uint8")
    plan = sc.plan_copies([(payload.ptr, buf.ptr, n)])
    hm = sc.HashMap([plan], payload.ptr, n)
    hm.launch(hp)
    assert hp.result() == h
    for at in (0, n // 2, n - (1 << 20)):
        assert np.array_equal(payload.numpy(1 << 20, start=at), buf.numpy(1 << 20, start=at))
    for m in (rm, hm, plan):
        m.destroy()
    for b in (buf, carry, payload):
        b.free()
    hp.free()
