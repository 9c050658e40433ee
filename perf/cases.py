"""The work this library's performance is judged on, as cases that a timing program can prepare and run.

Each case is one call of a public launcher on operands that are already on the GPU, as a user's program makes it:
matrix-core products through the port_2 launcher on the tuple the library suggests for the size, the same launcher on a
producer/consumer tuple of the user's own choice, and products without matrix cores through matmul_shmem. Sizes and value
distributions are those of bench.py's workloads and shape grid and of the tests; draw() spreads more cases over the ranges
between and around them.
"""
import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TUPLE = ("tile_dim", "segment_dim_k", "bar_steps_a", "bar_steps_b", "bar_step_rows_a", "bar_step_rows_b", "tile_group_m", "num_stages",
         "num_producer_warps", "num_consumer_warps", "num_sms")


def package():
    """The package's directory name holds a hyphen, so it is loaded by path."""
    name = "ckopt_amd"
    if name not in sys.modules:
        where = os.path.join(ROOT, "cuda-kernel-opt_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(where, "__init__.py"), submodule_search_locations=[where])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def gemm(name, dtype, M, N, K, out="f32", beta=0.0, values="uniform"):
    """D = A Bt^T + beta C on the suggested tuple; out "f32", or "same": C and D in the operands' 16-bit type."""
    return {"name": name, "kind": "gemm", "dtype": dtype, "M": M, "N": N, "K": K, "out": out, "beta": beta, "values": values}


def staged(name, dtype, M, N, K, tile, segk, stages, producers, consumers, steps_a, steps_b):
    """The port_2 launcher with dedicated producer waves; steps_a, steps_b > 0: shift synchronisation per wave tile."""
    return {"name": name, "kind": "staged", "dtype": dtype, "M": M, "N": N, "K": K, "out": "f32", "beta": 0.0, "values": "uniform", "tile": tile,
            "segk": segk, "stages": stages, "producers": producers, "consumers": consumers, "steps_a": steps_a, "steps_b": steps_b}


def simt(name, dtype, M, N, K, transposed, tile, block_rows):
    """matmul_shmem: no matrix cores; B is N x K (transposed) or K x N."""
    return {"name": name, "kind": "simt", "dtype": dtype, "M": M, "N": N, "K": K, "transposed": transposed, "tile": tile, "block_rows": block_rows}


def listed():
    return [
        # a small product in a chain of launches: the call, the launch and one tile's latency are all there is
        gemm("small_f16_512", "f16", 512, 512, 512),
        # the smallest ragged call: rows of an odd number of bf16 values, so no row but the first starts on 16 bytes
        gemm("small_ragged_bf16", "bf16", 200, 136, 1001),
        # an ordinary mid-size product, too small to fill the device with the largest tiles
        gemm("square_f16_2048", "f16", 2048, 2048, 2048),
        # few rows against a wide weight matrix, 16-bit result: a layer applied to a small batch
        gemm("skinny_bf16", "bf16", 256, 16384, 4096, out="same"),
        # the headline size
        gemm("square_f16_8192", "f16", 8192, 8192, 8192),
        # a long reduction into few tiles, as a weight gradient over many samples has it
        gemm("long_k_f16", "f16", 2048, 2048, 32768, values="normal"),
        # a large product whose sizes fit nothing: no multiple of a tile, K odd
        gemm("ragged_bf16_6143", "bf16", 6143, 4097, 3071),
        # the largest: the size the reference's driver times, with alpha = beta = 1, so that C is read as well
        gemm("square_f16_16384_c", "f16", 16384, 16384, 16384, beta=1.0),
        # the reference's own design as its user calls it: producer waves, shift synchronisation per wave tile
        staged("staged_f16_4096", "f16", 4096, 4096, 4096, 256, 64, 2, 2, 8, 4, 2),
        # single precision without matrix cores, B transposed
        simt("simt_f32_4096", "f32", 4096, 4096, 4096, True, 128, 4),
        # half precision in and out without matrix cores, B as the reference's kernel takes it
        simt("simt_f16_2048", "f16", 2048, 2048, 2048, False, 128, 4),
        # exact integers, small values
        simt("simt_i32_1024", "i32", 1024, 1024, 1024, False, 64, 4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _round(x, unit):
    return max(unit, (x + unit // 2) // unit * unit)


def draw(rng):
    pick = rng.random()
    if pick < 0.6:
        # any matrix-core product no larger than the largest listed one; half of the extents are odd sizes
        while True:
            M, N, K = _log(rng, 64, 16384), _log(rng, 64, 16384), _log(rng, 64, 65536)
            M, N = (_round(x, 64) if rng.random() < 0.5 else x for x in (M, N))
            K = _round(K, rng.choice((64, 64, 64, 8, 1)))
            if M * N * K <= 16384 ** 3:
                break
        c = gemm("", rng.choice(("f16", "bf16")), M, N, K, rng.choice(("f32", "f32", "same")), rng.choice((0.0, 0.0, 1.0)), rng.choice(("uniform", "normal")))
    elif pick < 0.75:
        while True:
            M, N, K = _log(rng, 256, 8192), _log(rng, 256, 8192), _round(_log(rng, 256, 16384), 64)
            M, N = (_round(x, 256) if rng.random() < 0.7 else x for x in (M, N))
            if M * N * K <= 8192 ** 3:
                break
        tile, stages = rng.choice(((256, 2), (128, 3), (128, 4)))
        steps = rng.choice(((0, 0), (2, 1), (4, 2)))
        c = staged("", rng.choice(("f16", "bf16")), M, N, K, tile, 64, stages, rng.choice((2, 4)), 8, *steps)
    else:
        tile, block_rows = rng.choice(((64, 4), (128, 4), (128, 8)))
        M, N = _round(_log(rng, 128, 4096), tile), _round(_log(rng, 128, 4096), tile)
        c = simt("", rng.choice(("f32", "f16", "i32")), M, N, _round(_log(rng, 64, 4096), 16), rng.random() < 0.5, tile, block_rows)
    del c["name"]
    return c


TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i32": torch.int32}


def _values(case, shape, dtype, gen):
    if dtype == "i32":   # the reference's own range
        return torch.randint(-10, 11, shape, dtype=torch.int32, device="cuda", generator=gen)
    x = torch.empty(shape, dtype=TORCH[dtype], device="cuda")
    if case.get("values") == "normal":
        return x.normal_(0.0, 0.1, generator=gen)
    return x.uniform_(-1.0, 1.0, generator=gen)


def _operands(case, seed):
    """A, B (as the launcher takes it) and C (None: not read)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
    A = _values(case, (M, K), dtype, gen)
    if case["kind"] == "simt":
        return A, _values(case, (N, K) if case["transposed"] else (K, N), dtype, gen), None
    B = _values(case, (N, K), dtype, gen)
    return A, B, _values(case, (M, N), _result(case), gen) if case["beta"] != 0.0 else None


def _result(case):
    return case["dtype"] if case["kind"] == "simt" or case["out"] == "same" else "f32"


def prepare(case, seed):
    ck = package()
    M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
    code = {"f16": ck.DT_F16, "bf16": ck.DT_BF16, "f32": ck.DT_F32, "i32": ck.DT_I32}[dtype]
    s = {"kind": case["kind"], "code": code, "sizes": (M, N, K)}
    s["A"], s["B"], s["C"] = _operands(case, seed)
    s["D"] = torch.empty((M, N), dtype=TORCH[_result(case)], device="cuda")
    if case["kind"] == "simt":
        s["tuning"] = (case["tile"], case["block_rows"], case["transposed"])
        return s
    s["beta"] = case["beta"]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if case["kind"] == "gemm":
        t = ck.suggest_gemm_tuning(M, N, K, cus)
        s["tuning"] = tuple(t[k] for k in TUPLE)
    else:
        tile, consumers = case["tile"], case["consumers"]
        rows = (tile, tile)
        if case["steps_a"] or case["steps_b"]:   # wave-tile granularity
            wave_rows = ck.get_warp_tile_rows(tile, consumers)
            rows = (wave_rows * 16, ck.get_num_acc(tile, consumers) // wave_rows * 16)
        s["tuning"] = (tile, case["segk"], case["steps_a"], case["steps_b"], rows[0], rows[1], 4, case["stages"], case["producers"], consumers, cus)
    s["launch"] = ck.gemm_shmem_tc_async_opt_port if case["out"] == "f32" else ck.gemm_shmem_tc_async_opt_port_lp
    return s


def run(s):
    M, N, K = s["sizes"]
    if s["kind"] == "simt":
        tile, block_rows, transposed = s["tuning"]
        package().matmul_shmem(s["code"], s["A"], s["B"], s["D"], M, N, K, tile, block_rows, transposed)
    else:
        s["launch"](s["code"], s["A"], s["B"], s["C"], s["D"], 1.0, s["beta"], M, N, K, *s["tuning"])
    return s["D"]


SIZE = {"f16": 2, "bf16": 2, "f32": 4, "i32": 4}


def work(case):
    M, N, K, e = case["M"], case["N"], case["K"], SIZE[case["dtype"]]
    result = 4 if case.get("out") == "f32" else e
    c = 1 if case.get("beta", 0.0) else 0
    return {"bytes": (M * K + N * K) * e + M * N * result * (1 + c), "flops": 2.0 * M * N * K}


def exact(case, seed):
    A, B, C = _operands(case, seed)
    A, B = A.double(), B.double()
    D = A @ (B if case["kind"] == "simt" and not case["transposed"] else B.t())
    if C is not None:
        D += case["beta"] * C.double()
    return D.to(torch.int32) if case["dtype"] == "i32" else D   # (sums of whole numbers far below 2^53)


def tolerance(case):
    """About four times what results differ by from the same sums taken in 64 bits and rounded once (largest of 25 shapes
    with K from 256 to 42000): fp32 results 6.7e-9 sqrt(K) through the matrix cores and 1.8e-8 sqrt(K) in one chain of
    fused multiply-adds; 16-bit results 2.1e-5 (fp16) and 7.9e-5 (bf16), which is the share of sums that round to the
    other side, one unit in the last place (2^-10, 2^-7) apart."""
    if case["dtype"] == "i32":
        return "exact"
    if case["kind"] != "simt" and case["out"] == "f32":
        return {"rel": 2.7e-8 * math.sqrt(case["K"])}
    if case["dtype"] == "f32":
        return {"rel": 7.2e-8 * math.sqrt(case["K"])}
    return {"rel": 8.5e-5, "max": 0.002} if case["dtype"] == "f16" else {"rel": 3.2e-4, "max": 0.016}
