"""Helpers shared by the GPU parity tests: device buffers via torch, launches via the C ABI."""
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def to_dev(x):
    """numpy array (float16 / uint16 bf16 bits / float32 / int32) -> device tensor with the same bytes."""
    x = np.ascontiguousarray(x)
    if x.dtype == np.uint16:
        return torch.from_numpy(x.view(np.int16)).cuda()
    return torch.from_numpy(x).cuda()


def tuning(tile_dim=128, segment_dim_k=64, bar_steps_a=0, bar_steps_b=0, bar_step_rows_a=None, bar_step_rows_b=None,
           tile_group_m=4, num_stages=2, num_producer_warps=2, num_consumer_warps=4, num_sms=256):
    return dict(tile_dim=tile_dim, segment_dim_k=segment_dim_k, bar_steps_a=bar_steps_a, bar_steps_b=bar_steps_b,
                bar_step_rows_a=tile_dim if bar_step_rows_a is None else bar_step_rows_a,
                bar_step_rows_b=tile_dim if bar_step_rows_b is None else bar_step_rows_b,
                tile_group_m=tile_group_m, num_stages=num_stages, num_producer_warps=num_producer_warps,
                num_consumer_warps=num_consumer_warps, num_sms=num_sms)


def wave_mode_rows(ck, t):
    wtr = ck.get_warp_tile_rows(t["tile_dim"], t["num_consumer_warps"])
    wtc = ck.get_num_acc(t["tile_dim"], t["num_consumer_warps"]) // wtr
    return wtr * 16, wtc * 16


def run_gemm(ck, dtype, a, bt, c=None, alpha=1.0, beta=0.0, t=None, poison=True):
    """Launches the port_2 entry point on device copies of the numpy inputs; returns D as numpy (M,N)."""
    t = t or tuning()
    M, K = a.shape
    N = bt.shape[0]
    da, db = to_dev(a), to_dev(bt)
    dc = None if c is None else to_dev(np.asarray(c, dtype=np.float32))
    dd = torch.full((M, N), float("nan") if poison else 0.0, dtype=torch.float32, device="cuda")
    ck.gemm_shmem_tc_async_opt_port(dtype, da, db, dc, dd, alpha, beta, M, N, K, t["tile_dim"], t["segment_dim_k"],
                                    t["bar_steps_a"], t["bar_steps_b"], t["bar_step_rows_a"], t["bar_step_rows_b"],
                                    t["tile_group_m"], t["num_stages"], t["num_producer_warps"],
                                    t["num_consumer_warps"], t["num_sms"])
    status = ck.device_status()
    assert status == 0, "device status %d (a bounded flag wait gave up)" % status
    return dd.cpu().numpy()


def bf16_bits_to_f32(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def f32_to_bf16_bits(x):
    """round-to-nearest-even float32 -> bf16 bit patterns (finite inputs)"""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def as_f64(dtype_is_bf16, x):
    return (bf16_bits_to_f32(x) if dtype_is_bf16 else x.astype(np.float32)).astype(np.float64)


def captured_kernels(launch):
    """Records launch(stream) into a HIP graph that is never run: (kernel, grid, block, LDS bytes) of its kernel nodes in order, and the
    number of its other nodes."""
    import ctypes

    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "/libamdhip64.so" in line))

    class Dim3(ctypes.Structure):
        _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]

    class KernelNodeParams(ctypes.Structure):
        _fields_ = [("blockDim", Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("gridDim", Dim3), ("kernelParams", ctypes.c_void_p), ("sharedMemBytes", ctypes.c_uint)]

    stream = torch.cuda.Stream()
    s, graph = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p()
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(s, 2) == 0   # relaxed: other work of the process is no part of it
    try:
        launch(stream)
    finally:
        assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    kernels, others = [], 0
    for node in nodes:
        kind, p = ctypes.c_int(), KernelNodeParams()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value != 0:
            others += 1
            continue
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        kernels.append((p.func, (p.gridDim.x, p.gridDim.y, p.gridDim.z), (p.blockDim.x, p.blockDim.y, p.blockDim.z), p.sharedMemBytes))
    assert hip.hipGraphDestroy(graph) == 0
    return kernels, others
