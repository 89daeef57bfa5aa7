"""What a call runs (rq_w4a4_product_plan), for tests that mean one kernel."""
import ctypes

import ruquant_amd as rq

DECODE, GEMV, SKINNY, FP6, INT8 = 1, 2, 3, 4, 5   # RQ_KERNEL_*


def plan(type_, K, Ns, M, multipliers=0, once=True, slabs=True, workspace=None, n_rot=None):
    """-> dict of the plan's numbers. Ns: one row count or several; multipliers: bit i for weight i; slabs: a workspace with room
    for K slices (of the size that rq.mul_mat_fused takes); workspace: its bytes instead."""
    L = rq.load_library()
    Ns = [Ns] if isinstance(Ns, int) else list(Ns)
    rows = Ns[0] if len(Ns) == 1 else sum((n + 63) // 64 * 64 for n in Ns)
    nbytes = L.rq_w4a4_workspace_bytes(type_, K, rows, M) if workspace is None else workspace
    if not slabs:
        nbytes -= 256
    out = (ctypes.c_int64 * 6)()
    rc = L.rq_w4a4_product_plan(type_, len(Ns), K, (ctypes.c_int64 * len(Ns))(*Ns), M, n_rot or K, multipliers, int(once), nbytes, out)
    assert rc == 0, rc
    return dict(zip(("kernel", "launches", "whole", "cut", "slices", "units"), out))
