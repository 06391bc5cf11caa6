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


# a forced layout of other than eight waves is the general mode's: 8-bit zero
# points and groups of 64 leave the stream kernel's modes for it and still run
def test_forced_stream_layout_of_other_waves():
    calls = [dict(M=8, K=1024, N=64, zp="int8"), dict(M=8, K=1024, N=64, zp="uint8", gs=256),
             dict(M=8, K=1024, N=64, gs=64), dict(M=8, K=1024, N=64, gs=64, gate_up=True)]
    for status, lines in plans(calls, ZT_WOQ_STREAM="4,2,1"):
        assert "invalid argument" not in status, (status, lines)
        assert lines


# 17..64 rows with fp32 scales, or zero points that the wide kernel does not
# take: blocks of 16 rows on small matrices and few rows, the large-tile
# kernel where it reads the weights once for more
def test_general_modes_17_to_64_rows():
    cases = [(dict(M=M, K=K, N=N, **kind), prefill)
             for kind in (dict(s_dtype="float32"), dict(zp="bfloat16"), dict(zp="int32"))
             for M, K, N, prefill in [
                 (17, 4096, 4096, False), (32, 2048, 2048, False), (24, 4096, 512, False),
                 (32, 512, 512, False), (24, 2048, 1001, False), (33, 4096, 4096, False),
                 (64, 4096, 4096, True), (48, 4096, 14336, True), (24, 3584, 18944, True),
                 (32, 14336, 4096, True), (24, 8192, 8192, True), (64, 1024, 512, True)]]
    cases += [(dict(M=M, K=14336, N=4096, s_dtype="float32"), M > 21) for M in (17, 20, 26)]
    for (call, prefill), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert lines and lines[0].startswith("woq prefill") == prefill, (call, lines)


# merged gate_up on the large tiles: in one launch where its tiles fill the GPU
# or the workspace holds no K split of the plain linear, else in two steps
def test_gate_up_large_tiles_or_two_steps():
    general = (dict(s_dtype="float32"), dict(zp="bfloat16"))
    cases = [(dict(M=M, K=K, N=N, gate_up=True, **kind), merged)
             for kind in (dict(), dict(gs=32), dict(zp="int8")) + general
             for M, K, N, merged in [
                 (128, 4096, 28672, True), (512, 4096, 7168, True), (2048, 14336, 8192, True),
                 (300, 512, 512, True), (128, 4096, 3584, False), (128, 14336, 1024, False),
                 (200, 8192, 7168, False), (1024, 14336, 1024, False)]]
    cases += [(dict(M=M, K=K, N=N, gate_up=True, **kind), False)
              for kind in general for M, K, N in [(17, 4096, 3584), (32, 14336, 1024),
                                                  (64, 2048, 2048), (24, 512, 512)]]
    cases += [(dict(M=128, K=4096, N=3584, gate_up=True, workspace=4 * 128 * 3584), True),
              (dict(M=64, K=4096, N=28672, gate_up=True, zp="bfloat16"), False),
              (dict(M=64, K=3584, N=37888, gate_up=True, zp="bfloat16"), True)]
    for (call, merged), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert any(l.endswith(", gate_up") for l in lines) == merged, (call, lines)


# short K at up to 64 rows: the synchronous kernel (it prints no launch line) up to
# a limit that grows with the rows, fp32 scales, columns that are not whole quads and
# long post-ops; the large tiles past it
def test_short_k_kernel():
    limits = [(dict(gs=32), 256, 320, 384), (dict(gs=64), 256, 320, 384), (dict(gs=64), 261, 512, 704),
              (dict(gs=32, zp="int8"), 256, 256, 256), (dict(gs=32, zp="uint8"), 261, 320, 512),
              (dict(gs=64, s_dtype="float32"), 256, 704, 704),
              (dict(gs=64, s_dtype="float32", zp="int8"), 1001, 704, 704),
              (dict(gs=64, post=["mul"]), 256, 320, 384), (dict(gs=64, post=["mul", "add"]), 256, 512, 704),
              (dict(gs=64, post=["gelu_erf"]), 256, 512, 704),
              (dict(gs=32, post=["silu", "mul"]), 261, 640, 704),
              (dict(gs=64, zp="int8", post=["tanh"]), 256, 256, 576)]
    cases = [(dict(M=M, K=K, N=N, **kind), K > (few if M <= 32 else many))
             for kind, N, few, many in limits
             for M in (1, 16, 17, 32, 33, 64) for K in (64, 192, 320, 448, 576, 704, 832)]
    cases += [(dict(M=65, K=64, N=256, gs=64), True), (dict(M=65, K=704, N=261, gs=64), True)]
    for (call, prefill), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert any(l.startswith("woq prefill") for l in lines) == prefill, (call, lines)
        assert prefill or not lines, (call, lines)


# many columns of a short K past 32 rows: not the stream kernel, which reads x again
# for every 16 of them; fewer columns, or a longer K, stay
def test_short_k_many_columns():
    cases = [(dict(M=M, K=K, N=N, **kind), stream)
             for kind in (dict(gs=64), dict(gs=128, zp="int8"))
             for M, K, N, stream in [(48, 640, 28672, False), (64, 384, 28672, False),
                                     (48, 640, 12288, True), (24, 640, 28672, True),
                                     (48, 1408, 28672, True)]]
    for (call, stream), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert any(l.startswith("woq stream") for l in lines) == stream, (call, lines)


# K of three phases with post-ops at 64 rows: zero points and small groups leave the
# wide kernel for the large tiles
def test_short_k_wide_kernel():
    cases = [(dict(M=M, K=K, N=8192, post=post, **kind), wide)
             for kind in (dict(gs=32), dict(gs=128, zp="int8"))
             for M, K, post, wide in [(64, 768, ["mul", "add"], False), (64, 768, ["relu"], False),
                                      (64, 768, [], True),
                                      (64, 1024, ["add"], True)]]
    cases += [(dict(M=64, K=768, N=8192, post=["add"]), True)]
    for (call, wide), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert lines and lines[0].startswith("woq wide" if wide else "woq prefill"), (call, lines)


# merged gate_up without its workspace: taken by the decode kernels' one launch
# for signed weights in groups of 128 and up, refused for all others
def test_gate_up_short_workspace():
    cases = [(dict(M=M, K=4096, N=28672, gate_up=True, workspace=ws, **kind), ok)
             for kind, ok in ((dict(), True), (dict(zp="int8"), False), (dict(gs=64), False),
                              (dict(gs=32, zp="uint8"), False))
             for M in (1, 12, 24) for ws in (0, 4 * M * 28672 - 256)]
    cases += [(dict(M=M, K=4096, N=28672, gate_up=True, workspace=4 * M * 28672, zp="int8"), True)
              for M in (1, 12, 24)]
    cases += [(dict(M=200, K=4096, N=28672, gate_up=True, workspace=0), False)]
    for (call, ok), (status, lines) in zip(cases, plans([c for c, _ in cases])):
        assert ("workspace of" not in status) == ok, (call, status, lines)


# bf16 scales that start in the middle of a dword keep zero points and small
# groups off the kernels that move them by 4-byte DMA
def test_misaligned_scales():
    calls = [dict(M=M, K=4096, N=28672, gate_up=gu, scales=(1 << 20) + at, **kind)
             for kind in (dict(zp="int8"), dict(gs=64), dict(gs=32, zp="uint8"))
             for M in (4, 24, 64) for gu in (False, True) for at in (0, 2)]
    for call, (status, lines) in zip(calls, plans(calls)):
        staged = any(l.startswith(("woq wide", "woq gate_up stream")) for l in lines) or \
            any(l.startswith("woq stream") for l in lines) and "zp" not in call
        assert lines and (call["scales"] % 4 == 0 or not staged), (call, lines)


# 8-bit zero points and groups of 32 and 64 at up to 16 rows take the stream
# kernel at every whole number of 128-column chunks, short K included
def test_group_modes_take_the_stream_kernel():
    calls = [dict(M=M, K=128 * C, N=N, gate_up=gu, **kind)
             for M in (1, 5, 16) for C in (1, 2, 5, 8, 9, 16, 17, 32) for N, gu in ((96, False),
                                                                                  (9216, True))
             for kind in (dict(gs=64), dict(gs=32), dict(gs=128, zp="int8"), dict(gs=0, zp="uint8"))]
    for call, (status, lines) in zip(calls, plans(calls)):
        assert len(lines) == 1 and " stream " in lines[0], (call, lines)
