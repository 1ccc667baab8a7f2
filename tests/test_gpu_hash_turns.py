"""The device FNV-1a at its launches' edges: a check given carries hands each workgroup up to four 64 KiB pieces, in grids
that leave the last turn short, and the sums of every piece are brought to the input's end.  The plain hash (one piece per
workgroup, compared with the byte loop elsewhere) and the chained one give the values to match."""
import pytest

pytestmark = pytest.mark.gpu

GROUP = 64 << 10


SIZES = [(0, 1), (1, 0), (1, 16), (2, GROUP - 1), (257, 255), (2559, 5), (2560, 0), (2561, 4097), (3840, 256),
         (5121, 777), (7683, 16)]


# an unaligned input takes the same launch and a byte at a time: its smaller sizes are enough
@pytest.mark.parametrize("groups,extra,shift", [(g, x, s) for g, x in SIZES for s in (0, 3) if not s or g <= 300])
def test_carried_check_equals_the_plain_hash(sc, cuda, groups, extra, shift):
    n = groups * GROUP + extra
    print(f"case hash turns {groups} x 64 KiB + {extra} at offset {shift}", flush=True)
    buf = sc.DeviceBuffer(n + 64, "uint8")
    sc.check(sc.lib.sc_fill_uniform_f16(buf.ptr, (n + 64) // 2, -4.0, 4.0, 77 + groups, extra, None), "fill")
    carry = sc.DeviceBuffer(max(sc.carry_bytes(n), 16), "uint8")
    hp = sc.HashPlan(n)
    hp.launch_carry(buf.ptr + shift, n, carry.ptr)
    sc.device_sync()
    h = hp.result()
    # the same bytes as three chained pieces
    hp.start()
    cuts = [0, n // 3, n // 3 * 2 + 1 if n > 2 else n, n]
    for a, b in zip(cuts, cuts[1:]):
        hp.chain(buf.ptr + shift + a, b - a)
    sc.device_sync()
    assert hp.result() == h
    hp.check_carried(buf.ptr + shift, n, h, carry.ptr)
    sc.device_sync()
    assert hp.fault_word() == 0 and int(hp.verdict.numpy()[0]) == 1 and int(hp.out.numpy()[0]) == h
    # a flipped byte in the last piece of the last turn is caught
    at = n - 1
    old = buf.numpy(1, start=shift + at)
    buf.upload(old ^ 1, start=shift + at)
    hp.check_carried(buf.ptr + shift, n, h, carry.ptr)
    sc.device_sync()
    assert int(hp.verdict.numpy()[0]) == 0
    for b in (buf, carry):
        b.free()
    hp.free()
