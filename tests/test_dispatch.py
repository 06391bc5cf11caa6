"""Dispatch of the int4 linear without a GPU (see zt_plan): the launches a call
is given, over the shapes a rule has to hold for."""
import re

from zt_plan import plans

LDS = 160 * 1024  # bytes per workgroup on gfx950


# the stream kernel's x, slabs, scales and zero points fit its LDS at every
# row and chunk count, group size and zero-point type, with few and many tiles
def test_stream_launches_fit_lds():
    calls = [dict(M=M, K=128 * C, N=N, gs=gs, zp=zp, gate_up=gu)
             for M in range(1, 17) for C in range(1, 65)
             for N, gu in ((4096, False), (12800, False), (25600, True))
             for gs in (32, 64, 128) for zp in (None, "int8")]
    seen = 0
    for call, (status, lines) in zip(calls, plans(calls)):
        for line in lines:
            m = re.search(r"lds=(\d+)", line)
            if " stream " in line:
                seen += 1
                assert int(m.group(1)) <= LDS, (call, line)
    assert seen > len(calls) // 2
