"""Which kernels a C-ABI call would launch, found without a GPU: the calls run
in a process that sees no device (every launch ends in an error there) on
pointers that nothing reads, and ZT_WOQ_DEBUG prints each launch shape as it
is chosen."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def plans(calls, **knobs):
    """calls: dicts of M, K, N and optionally gs (scale group, default 128; 0:
    per channel), zp and s_dtype ("int8", "float32", ..), gate_up, post (names of
    post-ops), and workspace (bytes; default what the size function asks for).  Returns one (status,
    [launch lines]) per call; knobs are ZT_ tuning knobs."""
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ZT_WOQ_DEBUG="1", **knobs)
    p = subprocess.run([sys.executable, os.path.abspath(__file__)], input=json.dumps(calls),
                       env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                       timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    out = []
    for line in p.stderr.splitlines():
        if line.startswith("[call]"):
            out.append(([], []))
        elif line.startswith("[end] "):
            out[-1][0].append(line[6:])
        elif line.startswith("[zt] ") and out:
            out[-1][1].append(line[5:])
    assert len(out) == len(calls)
    return [(status[0], lines) for status, lines in out]


def _main():
    import ctypes
    import torch
    sys.path.insert(0, HERE)
    import zt_capi as C
    assert torch.cuda.device_count() == 0
    L = C.lib()
    ptr = ctypes.c_void_p(1 << 20)
    for c in json.load(sys.stdin):
        M, K, N, gs = c["M"], c["K"], c["N"], c.get("gs", 128)
        G = K // gs if gs else 1
        dt = lambda name: C.DT[getattr(torch, name)]
        s_dt, zp = dt(c.get("s_dtype", "bfloat16")), c.get("zp")
        gu = c.get("gate_up", False)
        size = L.zt_woq_linear_gate_up_workspace_size if gu else L.zt_woq_linear_workspace_size
        ws = c.get("workspace", size(M, K, N, G))
        head = (ptr, 1, M, K, K, ptr, N, ctypes.c_void_p(c.get("scales", 1 << 20)), s_dt, G,
                ptr if zp else None, dt(zp) if zp else -1, None, -1)
        post = C.PostOps(count=len(c.get("post", ())))
        for i, name in enumerate(c.get("post", ())):
            post.ids[i] = C.PO[name]
            # (binary operands: bf16 [M, N], in the order of their ops)
            post.bufs[i], post.buf_dtypes[i], post.buf_ld[i] = ptr.value, 1, N
        print("[call]", file=sys.stderr, flush=True)
        if gu:
            rc = L.zt_woq_linear_gate_up(*head, ptr, 1, N // 2, ptr if ws else None, ws, None)
        else:
            rc = L.zt_woq_linear(*head, ctypes.byref(post), ptr, 1, N, ptr if ws else None, ws, None)
        print("[end]", L.zt_last_error_string().decode() if rc else "ok", file=sys.stderr, flush=True)


if __name__ == "__main__":
    _main()
