#!/usr/bin/env python3
"""Benchmark of the Nx eager hot path on one MI355X.

A "step" is one pass of the benchmark's configuration 2 (broadcast / strided
elementwise) over synthetic input already resident in HBM:

  f32:   a[64,512,512] viewed through permute(0,2,1); b[1,512,1] expanded
         t = add a' b ; u = mul t 0.5 ; v = cast f16 u
  int32: add a' b ; mul a' b ; m = cmplt b a' ; where m a' b

`value` is the algorithmic GB/s of that step (unique input elements read once +
outputs written once: 832 MiB + the small broadcast operands). The same JSON
line carries `roofline` for the dominant kernel (the LDS-turned elementwise
kernel, timed with HIP events on the context's stream, both launched back to
back and as the first call of the step), `cpu_baseline` (the CPU oracle — a
restatement of the reference's C backend — on the same workload, rank 0, host
cores), and in `config`, as flat scalars, every operation of configurations 1-5
timed alone (GB/s or TFLOP/s and its fraction of the 8 TB/s / MFMA peak), a
parity flag per configuration (the outputs of the timed calls against the CPU
oracle on the same seeded inputs) and the oracle's own rate on a bounded sample
of each; `ops` holds the same records in full.

Calls go straight through the C ABI with pre-built descriptors and
pre-allocated outputs ("output first"), so the timed region holds kernel
launches only: no allocation, no host<->device copies.
"""

from __future__ import annotations

import argparse
import ctypes as C
import json
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

from raven_amd import _ffi  # noqa: E402
from raven_amd import dtype as dt  # noqa: E402
from raven_amd.nx_backend import Backend, logical  # noqa: E402

MIB = 1 << 20
PEAK_HBM_GBS = 8000.0
PEAK_TFLOPS = {"bf16": 2500.0, "f16": 2500.0, "f32": 157.3}
METRIC = "Nx op GB/s (elementwise/reduce) + GEMM TFLOP/s, as % of MI355X roofline"


# HBM bytes per launch of the headline step's dominant kernel (map_tiled add, f32,
# [64,512,512]), from rocprofv3 --pmc FETCH_SIZE and --pmc WRITE_SIZE runs of
# `bench.py --only-step --no-cpu --pmc-calibration`: 32 799 KiB fetched x 1.9991 (a plain
# 64 MiB copy reads 32 782 KiB on the same counter) + 65 536 KiB written x 1.0000.
DOMINANT_KERNEL_HBM_TRAFFIC = 134252296


class Op:
    """One pre-built C-ABI call: name, thunk, algorithmic bytes / flops."""

    def __init__(self, name, fn, args, nbytes=0, flops=0, keep=()):
        self.name, self.fn, self.args, self.nbytes, self.flops, self.keep = name, fn, args, nbytes, flops, keep

    def __call__(self):
        rc = self.fn(*self.args)
        if rc != 0:
            raise RuntimeError(f"{self.name}: status {rc}")


def ref(t):
    d = t._desc()
    return d, C.byref(d)


class Workloads:
    def __init__(self, hip: Backend):
        self.hip, self.lib, self.h = hip, hip._lib, hip._h
        self.keep = []

    def dev(self, arr, d, shape=None):
        t = self.hip.from_host(arr, d)
        return self.hip.reshape(t, shape if shape is not None else arr.shape)

    def mk(self, name, fn, tensors, extra=(), pre=(), nbytes=0, flops=0):
        descs = [ref(t) for t in tensors]
        self.keep.append((tensors, descs))
        args = (self.h, *pre, *[p for _, p in descs], *extra)
        return Op(name, fn, args, nbytes, flops)

    def unary(self, op, out, x, nbytes):
        return self.mk(op, self.lib.nxh_unary, [out, x], pre=(_ffi.UNARY_OPS.index(op),), nbytes=nbytes)

    def binary(self, op, out, x, y, nbytes, name=None):
        return self.mk(name or op, self.lib.nxh_binary, [out, x, y], pre=(_ffi.BINARY_OPS.index(op),), nbytes=nbytes)

    def compare(self, op, out, x, y, nbytes):
        return self.mk(op, self.lib.nxh_compare, [out, x, y], pre=(_ffi.COMPARE_OPS.index(op),), nbytes=nbytes)

    def reduce(self, op, out, x, axes, nbytes, name):
        arr = (C.c_int32 * len(axes))(*axes)
        self.keep.append(arr)
        return self.mk(name, self.lib.nxh_reduce, [out, x], pre=(_ffi.REDUCE_OPS.index(op),),
                       extra=(arr, len(axes)), nbytes=nbytes)

    # -- config 2: the headline step ------------------------------------------
    def config2(self):
        hip = self.hip
        rng = [np.random.default_rng(s) for s in (4, 5, 6, 7)]
        shp = (64, 512, 512)
        n = 64 * 512 * 512
        a = self.dev(rng[0].standard_normal(shp).astype(np.float32), dt.float32)
        b = self.dev(rng[1].standard_normal((1, 512, 1)).astype(np.float32), dt.float32)
        ai = self.dev(rng[2].integers(-1000, 1001, shp).astype(np.int32), dt.int32)
        bi = self.dev(rng[3].integers(-1000, 1001, (1, 512, 1)).astype(np.int32), dt.int32)
        ap, aip = hip.permute(a, (0, 2, 1)), hip.permute(ai, (0, 2, 1))
        bx, bix = hip.expand(b, shp), hip.expand(bi, shp)
        half = hip.expand(hip.full(dt.float32, (), 0.5), shp)
        t, u = hip.buffer(dt.float32, shp), hip.buffer(dt.float32, shp)
        v = hip.buffer(dt.float16, shp)
        ti, ui = hip.buffer(dt.int32, shp), hip.buffer(dt.int32, shp)
        m, w = hip.buffer(dt.bool_, shp), hip.buffer(dt.int32, shp)
        small = 512 * 4
        ops = [
            self.binary("add", t, ap, bx, 8 * n + small, "cfg2 f32 add(permuted a, broadcast b)"),
            self.binary("mul", u, t, half, 8 * n + 4, "cfg2 f32 mul(t, scalar 0.5)"),
            self.mk("cfg2 cast f32->f16", self.lib.nxh_cast, [v, u], nbytes=6 * n),
            self.binary("add", ti, aip, bix, 8 * n + small, "cfg2 i32 add(permuted a, broadcast b)"),
            self.binary("mul", ui, aip, bix, 8 * n + small, "cfg2 i32 mul(permuted a, broadcast b)"),
            self.compare("cmplt", m, bix, aip, 5 * n + small),
            self.mk("cfg2 i32 where(m, permuted a, broadcast b)", self.lib.nxh_where, [w, m, aip, bix],
                    nbytes=9 * n + small),
        ]
        ops[5].name = "cfg2 i32 cmplt(broadcast b, permuted a)"
        self.cfg2_out = {"v": v, "w": w, "m": m}
        self.cfg2_in = {"a": a, "ai": ai}
        return ops

    # -- config 1: the CPU-runnable chain --------------------------------------
    def config1(self):
        hip = self.hip
        n = 4096
        host = [np.random.default_rng(s).uniform(-1, 1, (n, n)).astype(np.float32) for s in (1, 2, 3)]
        a, b, c = (self.dev(h, dt.float32) for h in host)
        t1, t2, t3 = (hip.buffer(dt.float32, (n, n)) for _ in range(3))
        z = hip.buffer(dt.float32, (n,))
        e = n * n * 4
        self.cfg1 = {"host": host, "z": z}
        return [
            self.binary("mul", t1, a, b, 3 * e, "cfg1 f32 mul"),
            self.unary("sin", t2, c, 2 * e),
            self.binary("add", t3, t1, t2, 3 * e, "cfg1 f32 add"),
            self.reduce("sum", z, t3, [1], e + n * 4, "cfg1 f32 reduce_sum axis 1"),
        ]

    # -- config 3: reductions ---------------------------------------------------
    def config3(self):
        hip = self.hip
        n = 8192
        hx = np.random.default_rng(8).standard_normal((n, n)).astype(np.float32)
        hxi = np.random.default_rng(9).integers(-1000, 1001, (n, n)).astype(np.int32)
        x, xi = self.dev(hx, dt.float32), self.dev(hxi, dt.int32)
        e = n * n * 4 + n * 4
        ops = []
        self.cfg3 = {"host": (hx, hxi), "out": {}}
        for axis in (1, 0):
            of, om = hip.buffer(dt.float32, (n,)), hip.buffer(dt.float32, (n,))
            oi, oa = hip.buffer(dt.int32, (n,)), hip.buffer(dt.int32, (n,))
            self.cfg3["out"][axis] = {"sum": of, "max": om, "argmax": oa, "isum": oi}
            ops.append(self.reduce("sum", of, x, [axis], e, f"cfg3 f32 sum axis {axis}"))
            ops.append(self.reduce("max", om, x, [axis], e, f"cfg3 f32 max axis {axis}"))
            ops.append(self.mk(f"cfg3 f32 argmax axis {axis}", self.lib.nxh_argreduce, [oa, x], pre=(0,),
                               extra=(axis,), nbytes=e))
            ops.append(self.reduce("sum", oi, xi, [axis], e, f"cfg3 i32 sum axis {axis}"))
        return ops

    # -- config 4: GEMM -----------------------------------------------------------
    def config4(self):
        hip = self.hip
        ops = []
        ha = (np.random.default_rng(10).standard_normal((2048, 2048)) * 0.02).astype(np.float32)
        hb = (np.random.default_rng(11).standard_normal((2048, 2048)) * 0.02).astype(np.float32)
        a, b = self.dev(ha, dt.float32), self.dev(hb, dt.float32)
        cf = hip.buffer(dt.float32, (2048, 2048))
        ops.append(self.mk("cfg4 f32 matmul 2048^3", self.lib.nxh_matmul, [cf, a, b],
                           flops=2 * 2048 ** 3, nbytes=3 * 2048 * 2048 * 4))
        # bf16 [16,4096,4096] x 2: sixteen distinct N(0, 0.02) matrices per operand from seeds 12 / 13,
        # drawn as float32 on the host and narrowed to bf16 (round to nearest even) on the device
        nb, n = 16, 4096
        keep = {}
        full = []
        for which, seed in (("a", 12), ("b", 13)):
            rng = np.random.default_rng(seed)
            t = hip.buffer(dt.bfloat16, (nb, n, n))
            for i in range(nb):
                m = (rng.standard_normal((n, n)) * 0.02).astype(np.float32)
                piece = hip.cast(hip.reshape(hip.from_host(m, dt.float32), (1, n, n)), dt.bfloat16)
                hip.assign(hip.shrink(t, [(i, i + 1), (0, n), (0, n)]), piece)
                if i in (0, 9):
                    keep[(which, i)] = m
            full.append(t)
        cb = hip.buffer(dt.bfloat16, (nb, n, n))
        ops.append(self.mk("cfg4 bf16 matmul [16,4096,4096]^2", self.lib.nxh_matmul, [cb, full[0], full[1]],
                           flops=2 * nb * n ** 3, nbytes=3 * nb * n * n * 2))
        self.cfg4 = {"f32": (ha, hb, cf), "bf16": (keep, cb), "skinny": {}}
        hsa = (np.random.default_rng(14).standard_normal((8, 4096)) * 0.02).astype(np.float32)
        hsb = (np.random.default_rng(15).standard_normal((4096, 16384)) * 0.02).astype(np.float32)
        for d, nm in ((dt.bfloat16, "bf16"), (dt.float32, "f32")):
            sa, sb = hip.cast(self.dev(hsa, dt.float32), d), hip.cast(self.dev(hsb, dt.float32), d)
            es = d.itemsize
            out = hip.buffer(d, (8, 16384))
            self.cfg4["skinny"][nm] = (hsa, hsb, out)
            ops.append(self.mk(f"cfg4 {nm} skinny [8,4096]x[4096,16384]", self.lib.nxh_matmul,
                               [out, sa, sb], flops=2 * 8 * 4096 * 16384,
                               nbytes=(8 * 4096 + 4096 * 16384 + 8 * 16384) * es))
        self.config4_ops = ops
        return ops


def next_ops(hip, W, linalg=False):
    """The operations beside the named hot path (pad, cat, scan, threefry,
    scatter, sort, unfold, fold), timed through the Python mirror with HIP events."""
    rng = np.random.default_rng(20)
    out = []

    def timed(name, fn, nbytes, iters=20):
        for _ in range(3):
            r = fn()
            del r
        hip.synchronize()
        hip.timer_start()
        for _ in range(iters):
            r = fn()
            del r
        ms = hip.timer_stop() / iters
        out.append({"op": name, "ms": round(ms, 5), "GB/s": round(nbytes / (ms * 1e-3) / 1e9, 1),
                    "frac_hbm": round(nbytes / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4), "bound": "hbm"})

    x = W.dev(rng.standard_normal((2048, 4100)).astype(np.float32), dt.float32)
    timed("pad [2048,4100] f32 by ((3,5),(7,1))", lambda: hip.pad(x, [(3, 5), (7, 1)], -2.5),
          2048 * 4100 * 4 + 2056 * 4108 * 4)
    parts = [W.dev(rng.standard_normal((1024, 4096)).astype(np.float32), dt.float32) for _ in range(4)]
    timed("cat 4 x [1024,4096] f32 along axis 0", lambda: hip.cat(parts, 0), 2 * 4 * 1024 * 4096 * 4)
    timed("cat 4 x [1024,4096] f32 along axis 1", lambda: hip.cat(parts, 1), 2 * 4 * 1024 * 4096 * 4)
    # a result larger than the memory-side cache that nothing reads back: written past the cache
    big = [W.dev(rng.standard_normal((2048, 8192)).astype(np.float32), dt.float32) for _ in range(4)]
    timed("cat 4 x [2048,8192] f32 along axis 0 (256 MiB result, streamed by the cache policy)", lambda: hip.cat(big, 0),
          2 * 4 * 2048 * 8192 * 4, iters=10)
    del big
    y = W.dev(rng.standard_normal((4096, 8192)).astype(np.float32), dt.float32)
    timed("cumsum [4096,8192] f32 axis 1 (scan_rows)", lambda: hip.associative_scan(1, "sum", y), 2 * 4096 * 8192 * 4)
    timed("cumsum [4096,8192] f32 axis 0 (scan_cols: one pass, carries handed down between blocks)", lambda: hip.associative_scan(0, "sum", y), 2 * 4096 * 8192 * 4)
    n = 1 << 24
    ctr = W.dev(np.arange(2 * n, dtype=np.int64).astype(np.int32).reshape(n, 2), dt.int32)
    key = hip.expand(W.dev(np.array([[1234, -99]], np.int32), dt.int32), (n, 2))
    timed("threefry 2^24 vectors (one key; threefry_dense)", lambda: hip.threefry(key, ctr), 2 * n * 8)
    vocab, dim, ntok = 50257, 768, 8192
    ids = W.dev(rng.integers(0, vocab, (ntok, 1)).astype(np.int32), dt.int32)
    idx = hip.expand(ids, (ntok, dim))
    upd = W.dev(rng.standard_normal((ntok, dim)).astype(np.float32), dt.float32)
    table = hip.full(dt.float32, (vocab, dim), 0.0)
    # template copy (read + write of the table) + indices + updates + read-modify-write of the touched rows
    timed("scatter-add [8192,768] f32 rows into [50257,768] (embedding gradient)",
          lambda: hip.scatter("add", False, table, idx, upd, 0),
          2 * vocab * dim * 4 + ntok * 4 + 3 * ntok * dim * 4, iters=5)
    del table, upd, idx, ctr, key, y, parts, x
    # sort moves each element once in and once out; the network in between is
    # compare-exchange work, so the rate is quoted in keys per second too
    rows = W.dev(rng.standard_normal((16384, 1024)).astype(np.float32), dt.float32)
    timed("sort [16384,1024] f32 axis 1 (sort_registers)", lambda: hip.sort(rows, 1, False), 2 * 16384 * 1024 * 4)
    out[-1]["Mkeys/s"] = round(16384 * 1024 / out[-1]["ms"] / 1e3, 1)
    timed("argsort [16384,1024] f32 axis 1, descending (sort_registers)", lambda: hip.argsort(rows, 1, True),
          2 * 16384 * 1024 * 4)
    out[-1]["Mkeys/s"] = round(16384 * 1024 / out[-1]["ms"] / 1e3, 1)
    one = W.dev(rng.standard_normal(1 << 24).astype(np.float32), dt.float32)
    timed("sort 2^24 f32, one slice (sort_radix)", lambda: hip.sort(one, 0, False), 2 * (1 << 24) * 4, iters=5)
    out[-1]["Mkeys/s"] = round((1 << 24) / out[-1]["ms"] / 1e3, 1)
    for rec in out[-3:]:
        rec["bound"] = "lds"  # compare-exchange steps through LDS, not bytes, set the time
    del rows, one
    img = W.dev(rng.standard_normal((8, 64, 128, 128)).astype(np.float32), dt.float32)
    geo = ([3, 3], [1, 1], [1, 1], [(1, 1), (1, 1)])
    nin, ncols = 8 * 64 * 128 * 128 * 4, 9 * 8 * 64 * 128 * 128 * 4
    timed("unfold [8,64,128,128] f32, 3x3 same (im2col)", lambda: hip.unfold(img, *geo), nin + ncols)
    cols = hip.unfold(img, *geo)
    timed("fold back to [8,64,128,128] (col2im, 9 taps per output)", lambda: hip.fold(cols, [128, 128], *geo), nin + ncols)
    del img, cols
    # matmul beside config 4's shapes: float64, and the products a convolution makes of its windows
    def mm(name, a, b, flops, peak, iters=10):
        timed(name, lambda: hip.matmul(a, b), 0, iters=iters)
        tf = flops / (out[-1]["ms"] * 1e-3) / 1e12
        out[-1] = {"op": name + f" ({hip.last_path()})", "ms": out[-1]["ms"], "TFLOP/s": round(tf, 2),
                   "frac_mfma": round(tf / peak, 4), "bound": "mfma"}
    f64 = lambda shape: W.dev(rng.standard_normal(shape), dt.float64)
    mm("matmul f64 2048^3", f64((2048, 2048)), f64((2048, 2048)), 2.0 * 2048 ** 3, 78.6, iters=5)
    mm("matmul f64 512^3", f64((512, 512)), f64((512, 512)), 2.0 * 512 ** 3, 78.6)
    f32 = lambda shape: W.dev(rng.standard_normal(shape).astype(np.float32), dt.float32)
    mm("matmul f32 1024^3", f32((1024, 1024)), f32((1024, 1024)), 2.0 * 1024 ** 3, 157.3)
    mm("matmul f32 [64,576] x [32,576,3136] (3x3 windows of [32,64,56,56])",
       hip.expand(f32((1, 64, 576)), (32, 64, 576)), f32((32, 576, 3136)), 2.0 * 32 * 64 * 576 * 3136, 157.3)
    mm("matmul f32 [256,2048] x [2048,256] (weight gradient, cut along K)", f32((256, 2048)), f32((2048, 256)),
       2.0 * 256 * 2048 * 256, 157.3)
    # the dtypes without a matrix instruction: register-blocked on the vector unit (no matrix peak applies)
    def mmv(name, a, b, ops):
        timed(name, lambda: hip.matmul(a, b), 0, iters=5)
        out[-1] = {"op": name + f" ({hip.last_path()})", "ms": out[-1]["ms"],
                   "Top/s": round(ops / (out[-1]["ms"] * 1e-3) / 1e12, 2), "bound": "valu"}
    ints = lambda shape, d: W.dev(rng.integers(-100, 100, shape).astype(d.np_storage), d)
    mmv("matmul int32 2048^3", ints((2048, 2048), dt.int32), ints((2048, 2048), dt.int32), 2.0 * 2048 ** 3)
    mmv("matmul int64 2048^3", ints((2048, 2048), dt.int64), ints((2048, 2048), dt.int64), 2.0 * 2048 ** 3)
    c64 = lambda shape: W.dev((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64), dt.complex64)
    mmv("matmul complex64 2048^3 (8 flops per term)", c64((2048, 2048)), c64((2048, 2048)), 8.0 * 2048 ** 3)
    # fused attention and the row kernels at GPT-2-small's shapes (bf16, batch 8, seq 1024)
    bf = lambda shape: W.dev((rng.standard_normal(shape).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16),
                             dt.bfloat16)
    mm("matmul bf16 [256,2304] x [32,2304,196] (3x3 windows of [32,256,14,14]; rows of 196)",
       hip.expand(bf((1, 256, 2304)), (32, 256, 2304)), bf((32, 2304, 196)), 2.0 * 32 * 256 * 2304 * 196, 2500.0)
    b, h, sq, hd = 8, 12, 1024, 64
    q, k, v = (hip.permute(hip.reshape(bf((b, sq, h * hd)), (b, sq, h, hd)), (0, 2, 1, 3)) for _ in range(3))
    timed("attention [8,12,1024,64] bf16, causal, head-split views (attention_fused)",
          lambda: hip.attention(q, k, v, 0.125, causal=True, masked_value=float("-inf")), 4 * b * sq * h * hd * 2)
    useful = 4 * b * h * sq * (sq + 1) // 2 * hd  # Q K^T and probs x V over the visible half
    # bound by the per-score VALU work (two expf, an exact division, a narrowing), not by the MFMAs
    out[-1].update({"bound": "valu", "TFLOP/s": round(useful / (out[-1]["ms"] * 1e-3) / 1e12, 1)})
    scores = W.dev(rng.standard_normal((b * h * sq, sq)).astype(np.float32), dt.float32)
    timed("softmax_rows [98304,1024] f32 -> bf16 with scale (fused)",
          lambda: hip.softmax_rows(scores, 0.125, None, None, dt.bfloat16), b * h * sq * sq * 6)
    del scores
    x = bf((b * sq, 768))
    gam, bet = bf((768,)), bf((768,))
    timed("layer_norm_rows [8192,768] bf16 (fused)", lambda: hip.layer_norm_rows(x, gam, bet, 1e-5), 2 * b * sq * 768 * 2)
    y = bf((b * sq, 3072))
    timed("gelu_tanh [8192,3072] bf16 (fused)", lambda: hip.gelu_tanh(y), 2 * b * sq * 3072 * 2)
    del x, y, gam, bet, q, k, v
    # Fourier transforms: one pass reads and writes the tensor once; the butterflies run in registers
    cplx = lambda shape: W.dev((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64),
                               dt.complex64)
    z = cplx((16384, 1024))
    timed("fft [16384,1024] complex64 axis 1 (fft_lines, up to sixteen elements a lane)", lambda: hip.fft(z, [1]), 2 * 16384 * 1024 * 8)
    out[-1]["GFLOP/s"] = round(5 * 16384 * 1024 * 10 / out[-1]["ms"] / 1e6, 1)
    z2 = cplx((4096, 4096))
    timed("fft [4096,4096] complex64 axis 0 (strided lines)", lambda: hip.fft(z2, [0]), 2 * 4096 * 4096 * 8)
    z3 = cplx((8192, 1000))
    timed("fft [8192,1000] complex64 axis 1 (Bluestein in LDS, M = 2048)", lambda: hip.fft(z3, [1]), 2 * 8192 * 1000 * 8)
    r = W.dev(rng.standard_normal((16384, 2048)).astype(np.float32), dt.float32)
    timed("rfft [16384,2048] f32 -> complex64 axis 1", lambda: hip.rfft(r, dt.complex64, [1]),
          16384 * 2048 * 4 + 16384 * 1025 * 8)
    big = cplx((4, 1 << 20))
    timed("fft [4,2^20] complex64 axis 1 (four-step through a workspace)", lambda: hip.fft(big, [1]),
          2 * 4 * (1 << 20) * 8, iters=5)
    for rec in out[-5:]:
        rec["bound"] = "latency"  # of a wave's chain of exchanges through LDS
    del z, z2, z3, r, big
    if not linalg:
        return out

    # linear algebra (only with --only-next: thousands of short launches that would drown a
    # kernel-time profile of the hot path): correctness first, times only
    def la(name, fn, iters=3):
        timed(name, fn, 0, iters=iters)
        for key in ("GB/s", "frac_hbm"):
            out[-1].pop(key)
        out[-1]["bound"] = "latency"

    g = rng.standard_normal((256, 64, 64)).astype(np.float32)
    spd = W.dev(g @ g.transpose(0, 2, 1) + 64 * np.eye(64, dtype=np.float32), dt.float32)
    gen = W.dev(g, dt.float32)
    la("cholesky [256,64,64] f32", lambda: hip.cholesky(spd))
    la("qr [256,64,64] f32, reduced", lambda: hip.qr(gen))
    la("eigh [256,64,64] f32 (Jacobi)", lambda: hip.eigh(spd))
    la("svd [256,64,64] f32 (one-sided Jacobi)", lambda: hip.svd(gen))
    la("eig [256,64,64] f32 (Hessenberg + shifted QR)", lambda: hip.eig(gen))
    one = rng.standard_normal((1, 512, 512)).astype(np.float32)
    big_spd = W.dev(one @ one.transpose(0, 2, 1) + 512 * np.eye(512, dtype=np.float32), dt.float32)
    la("cholesky [1,512,512] f32", lambda: hip.cholesky(big_spd))
    la("eigh [1,512,512] f32 (Jacobi)", lambda: hip.eigh(big_spd), iters=1)
    return out


class Telemetry:
    """Board power (hwmon power1_input, microwatts) and shader clock (the current line of
    pp_dpm_sclk) sampled from sysfs every 10 ms while a loop runs. Means over the samples taken
    after the first fifth of the loop (the clock needs a moment to settle)."""

    def __init__(self):
        import glob

        self.power = (glob.glob("/sys/class/drm/card*/device/hwmon/hwmon*/power1_input") + [None])[0]
        self.sclk = (glob.glob("/sys/class/drm/card*/device/pp_dpm_sclk") + [None])[0]
        self.samples, self._stop, self._thread = [], False, None

    def _read(self):
        w = mhz = None
        try:
            if self.power:
                w = int(open(self.power).read()) / 1e6
            if self.sclk:
                for line in open(self.sclk).read().splitlines():
                    if line.rstrip().endswith("*"):
                        mhz = float(line.split(":")[1].lower().replace("mhz", "").replace("*", "").strip())
        except (OSError, ValueError, IndexError):
            pass
        return time.perf_counter(), w, mhz

    def __enter__(self):
        import threading

        def loop():
            while not self._stop:
                self.samples.append(self._read())
                time.sleep(0.01)

        self._thread = threading.Thread(target=loop, daemon=True)
        self._thread.start()
        return self

    def __exit__(self, *exc):
        self._stop = True
        self._thread.join()
        return False

    def means(self):
        s = self.samples[len(self.samples) // 5:]
        ws, fs = [w for _, w, _ in s if w is not None], [f for _, _, f in s if f is not None]
        return (round(sum(ws) / len(ws), 1) if ws else None, round(sum(fs) / len(fs)) if fs else None, len(s))


def study_row(what, data, ms, fl, tel):
    w, mhz, k = tel.means()
    return {"kernel": what, "operands": data, "ms": round(ms, 4), "TFLOP/s": round(fl / (ms * 1e-3) / 1e12, 1),
            "frac_of_2500": round(fl / (ms * 1e-3) / 1e12 / 2500.0, 4), "board_W": w, "sclk_MHz": mhz, "samples": k}


def gemm_study_vendor(seconds):
    """The rows of gemm_study that the vendor library fills (hipBLASLt behind torch.bmm)."""
    import torch

    nb, n = 16, 4096
    flops = 2.0 * nb * n ** 3
    rows = []
    for data in ("N(0, 0.02)", "zeros"):
        if data == "zeros":
            a = torch.zeros(nb, n, n, device="cuda", dtype=torch.bfloat16)
            b = torch.zeros(nb, n, n, device="cuda", dtype=torch.bfloat16)
        else:
            g = torch.Generator(device="cuda").manual_seed(12)
            a = (torch.randn(nb, n, n, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
            b = (torch.randn(nb, n, n, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        c = torch.empty(nb, n, n, device="cuda", dtype=torch.bfloat16)
        for _ in range(5):
            torch.bmm(a, b, out=c)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        iters = max(5, int(seconds / 1.8e-3))
        with Telemetry() as tel:
            e0.record()
            for _ in range(iters):
                torch.bmm(a, b, out=c)
            e1.record()
            torch.cuda.synchronize()
        rows.append(study_row("vendor: torch.bmm (hipBLASLt)", data, e0.elapsed_time(e1) / iters, flops, tel))
        del a, b, c
    return rows


def gemm_study(hip, seconds, vendor=True):
    """Config 4's batched bf16 product on all-zero and on N(0, 0.02) operands, by this library and
    by the vendor library (hipBLASLt behind torch.bmm), beside an MFMA-only loop on the same two
    kinds of data: time, TFLOP/s, board power and shader clock of each. The board holds its power
    limit by lowering the clock, so what a GEMM reaches depends on the bits that toggle."""
    nb, n = 16, 4096
    flops = 2.0 * nb * n ** 3
    rows = []

    def record(what, data, ms, fl, tel):
        rows.append(study_row(what, data, ms, fl, tel))

    W = Workloads(hip)
    W.config4()
    keep, cb = W.cfg4["bf16"]
    desc = [d for ts, ds in W.keep for t, d in zip(ts, ds) if t is cb or (tuple(t.shape) == (nb, n, n) and t.dtype is dt.bfloat16)]
    normal = [op for op in W.config4_ops if "16,4096" in op.name][0]
    zero = [hip.full(dt.bfloat16, (nb, n, n), 0.0) for _ in range(2)]
    zc = hip.buffer(dt.bfloat16, (nb, n, n))
    zeros = W.mk("cfg4 bf16 matmul, zeros", W.lib.nxh_matmul, [zc, zero[0], zero[1]], flops=flops)
    for data, op in (("N(0, 0.02)", normal), ("zeros", zeros)):
        ms1 = time_ops(hip, [op], 5, 3)
        iters = max(5, int(seconds / (ms1 * 1e-3)))
        with Telemetry() as tel:
            ms = time_ops(hip, [op], iters, 0)
        record(f"libnxhip nxh_matmul ({hip.last_path()})", data, ms, flops, tel)
    del zero, zc, zeros, normal, desc
    W.keep.clear()
    W.cfg4 = None
    hip.trim()

    # the vendor library runs in a process of its own: torch carries its own HIP runtime, and two of
    # them in one process do not both find the device
    import subprocess

    if vendor:
        r = subprocess.run([sys.executable, str(Path(__file__).resolve()), "--gemm-study-vendor", "--study-seconds", str(seconds)],
                           capture_output=True, text=True, timeout=600)
        if r.returncode == 0:
            rows.extend(json.loads(r.stdout.strip().splitlines()[-1]))
        else:
            rows.append({"kernel": "vendor: torch.bmm (hipBLASLt)", "error": r.stderr.strip()[-200:]})

    probe = ROOT / "bench_mfma_probe.so"
    if probe.exists():
        lib = C.CDLL(str(probe))
        lib.mfma_probe_run.restype = C.c_double
        lib.mfma_probe_run.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_float)]
        blocks = 4 * hip.device_info()["compute_units"]
        out = hip.buffer(dt.float32, (blocks * 512,))
        rng = np.random.default_rng(13)
        for data in ("N(0, 0.02)", "zeros"):
            host = np.zeros(16384, np.uint16) if data == "zeros" else bf16_bits((rng.standard_normal(16384) * 0.02).astype(np.float32))
            words = hip.from_host(host.view(np.int32), dt.int32)
            hip.synchronize()
            ms = C.c_float()
            iters = 2000
            fl = lib.mfma_probe_run(words.buffer.ptr, out.buffer.ptr, blocks, iters, 2, C.byref(ms))
            reps = max(2, int(seconds / max(ms.value * 1e-3, 1e-6)))
            with Telemetry() as tel:
                fl = lib.mfma_probe_run(words.buffer.ptr, out.buffer.ptr, blocks, iters, reps, C.byref(ms))
            if fl:
                rows.append(study_row("MFMA-only loop (v_mfma_f32_16x16x32_bf16, operands in registers)", data, ms.value, fl, tel))
    return rows


def time_ops(hip, ops, iters, warmup):
    """Average milliseconds per pass of `ops`, HIP events on the context stream."""
    for _ in range(warmup):
        for op in ops:
            op()
    hip.synchronize()
    hip.timer_start()
    for _ in range(iters):
        for op in ops:
            op()
    return hip.timer_stop() / iters


def op_record(op, ms):
    rec = {"op": op.name, "ms": round(ms, 5)}
    gbs = op.nbytes / (ms * 1e-3) / 1e9
    if op.flops and "skinny" not in op.name:
        dtype = "bf16" if "bf16" in op.name else "f32"
        tf = op.flops / (ms * 1e-3) / 1e12
        rec.update({"TFLOP/s": round(tf, 2), "frac_mfma": round(tf / PEAK_TFLOPS[dtype], 4), "bound": "mfma"})
    else:
        rec.update({"GB/s": round(gbs, 1), "frac_hbm": round(gbs / PEAK_HBM_GBS, 4), "bound": "hbm"})
        if op.flops:
            rec["TFLOP/s"] = round(op.flops / (ms * 1e-3) / 1e12, 3)
    return rec


def cpu_baseline(seconds_budget=20.0):
    """The oracle (CPU restatement of the reference C backend) on config 2, with
    the reference's own thread policy, on this host's cores."""
    from oracle.nx_oracle import OracleBackend, lib

    B = OracleBackend()
    rng = [np.random.default_rng(s) for s in (4, 5, 6, 7)]
    shp = (64, 512, 512)
    n = 64 * 512 * 512
    mk = lambda arr, d: B.reshape(B.from_host(arr, d), arr.shape)  # noqa: E731
    a = mk(rng[0].standard_normal(shp).astype(np.float32), dt.float32)
    b = mk(rng[1].standard_normal((1, 512, 1)).astype(np.float32), dt.float32)
    ai = mk(rng[2].integers(-1000, 1001, shp).astype(np.int32), dt.int32)
    bi = mk(rng[3].integers(-1000, 1001, (1, 512, 1)).astype(np.int32), dt.int32)
    ap, aip = B.permute(a, (0, 2, 1)), B.permute(ai, (0, 2, 1))
    bx, bix = B.expand(b, shp), B.expand(bi, shp)
    half = B.expand(B.full(dt.float32, (), np.array([0.5], np.float32)), shp)
    threads = set()

    def step():
        t = B.binary("add", ap, bx)
        threads.add(lib().nxo_last_threads())
        u = B.binary("mul", t, half)
        v = B.cast(u, dt.float16)
        B.binary("add", aip, bix)
        B.binary("mul", aip, bix)
        m = B.compare("cmplt", bix, aip)
        w = B.where(m, aip, bix)
        return v, w

    step()  # warm: first touch of fresh pages is not the steady state
    t0 = time.perf_counter()
    reps = 0
    while reps < 3 or (time.perf_counter() - t0 < seconds_budget and reps < 40):
        out = step()
        reps += 1
    dtm = (time.perf_counter() - t0) / reps
    total_bytes = 832 * MIB + 5 * 2048 + 4
    return {
        "value": round(total_bytes / dtm / 1e9, 3), "unit": "GB/s", "cores": max(threads),
        "kind": "port",
        "sample": f"{reps} full passes of config 2 ([64,512,512] f32 + int32 chain, 832 MiB algorithmic), "
                  f"{dtm * 1e3:.1f} ms per pass; host has {lib().nxo_ncores()} cores online; threads per op "
                  "follow the reference policy (bytes/32 MiB, capped by cores)",
    }, out


class CountingBackend:
    """Forwards to the backend and counts the calls that launch work."""

    LAUNCHING = ("unary", "binary", "compare", "where", "cast", "copy", "contiguous", "gather", "reduce",
                 "matmul", "full", "from_host", "softmax_rows", "layer_norm_rows", "gelu_tanh", "attention", "linear")

    def __init__(self, inner):
        self._inner, self.calls = inner, {}

    def __getattr__(self, name):
        attr = getattr(self._inner, name)
        if name not in self.LAUNCHING:
            return attr

        def counted(*a, **k):
            self.calls[name] = self.calls.get(name, 0) + 1
            return attr(*a, **k)

        return counted


def cpu_configs():
    """The CPU oracle on bounded samples of the other configurations, on this
    host's cores with the reference's thread policy: the CPU path beside each
    GPU figure. Every sample is named in its record."""
    from oracle.nx_oracle import OracleBackend, lib

    B = OracleBackend()
    out = []
    mk = lambda arr, d: B.reshape(B.from_host(arr, d), arr.shape)  # noqa: E731

    def timed(name, fn, nbytes=0, flops=0, budget=4.0):
        fn()
        t0, reps = time.perf_counter(), 0
        while reps < 2 or (time.perf_counter() - t0 < budget and reps < 20):
            fn()
            reps += 1
        sec = (time.perf_counter() - t0) / reps
        rec = {"op": name, "ms": round(sec * 1e3, 3), "threads": lib().nxo_last_threads()}
        if nbytes:
            rec["GB/s"] = round(nbytes / sec / 1e9, 2)
        if flops:
            rec["GFLOP/s"] = round(flops / sec / 1e9, 1)
        out.append(rec)

    n = 4096
    a, b, c = (mk(np.random.default_rng(s).uniform(-1, 1, (n, n)).astype(np.float32), dt.float32) for s in (1, 2, 3))
    e = n * n * 4
    timed("cfg1 f32 mul [4096,4096]", lambda: B.binary("mul", a, b), 3 * e)
    timed("cfg1 f32 sin [4096,4096]", lambda: B.unary("sin", c), 2 * e)
    timed("cfg1 f32 reduce_sum axis 1 [4096,4096]", lambda: B.reduce("sum", [1], a), e)
    del a, b, c
    n = 8192
    x = mk(np.random.default_rng(8).standard_normal((n, n)).astype(np.float32), dt.float32)
    e = n * n * 4
    for axis in (1, 0):
        timed(f"cfg3 f32 sum axis {axis} [8192,8192]", lambda: B.reduce("sum", [axis], x), e)
        timed(f"cfg3 f32 argmax axis {axis} [8192,8192]", lambda: B.argmax(x, axis), e)
    del x
    m = 2048
    fa, fb = (mk((np.random.default_rng(s).standard_normal((m, m)) * 0.02).astype(np.float32), dt.float32) for s in (10, 11))
    timed("cfg4 f32 matmul 2048^3", lambda: B.matmul(fa, fb), flops=2 * m ** 3, budget=8.0)
    ba, bb = B.cast(B.reshape(fa, (1, m, m)), dt.bfloat16), B.cast(B.reshape(fb, (1, m, m)), dt.bfloat16)
    timed("cfg4 bf16 matmul, sample [1,2048,2048]^2 of [16,4096,4096]^2", lambda: B.matmul(ba, bb), flops=2 * m ** 3,
          budget=8.0)
    sa = mk((np.random.default_rng(14).standard_normal((8, 4096)) * 0.02).astype(np.float32), dt.float32)
    sb = mk((np.random.default_rng(15).standard_normal((4096, 16384)) * 0.02).astype(np.float32), dt.float32)
    timed("cfg4 f32 skinny [8,4096]x[4096,16384]", lambda: B.matmul(sa, sb), nbytes=(8 * 4096 + 4096 * 16384 + 8 * 16384) * 4,
          flops=2 * 8 * 4096 * 16384)
    del fa, fb, ba, bb, sa, sb
    # config 5: the eager GPT-2-small forward at batch 1 x seq 128 (1/64 of the tokens of the GPU run)
    from raven_amd.kaun_gpt2 import Config, Gpt2, host_params, upload
    from raven_amd.nx_frontend import Nx

    cfg = Config.small()
    enc = lambda v, d: ((np.ascontiguousarray(v, np.float32).view(np.uint32) + 0x7FFF  # noqa: E731
                         + ((np.ascontiguousarray(v, np.float32).view(np.uint32) >> 16) & 1)) >> 16).astype(np.uint16)
    nx = Nx(B)
    params = upload(nx, host_params(cfg, seed=16), dt.bfloat16, enc)
    ids = nx.create(dt.int32, (1, 128), np.random.default_rng(17).integers(0, cfg.vocab_size, (1, 128)).astype(np.int32))
    model = Gpt2(nx, cfg)
    t0 = time.perf_counter()
    model.logits(params, ids)
    sec = time.perf_counter() - t0
    out.append({"op": "cfg5 GPT-2 small forward, bf16, sample batch 1 x seq 128 (one pass)", "ms": round(sec * 1e3, 1),
                "tokens/s": round(128 / sec, 1)})
    return {"host_cores": lib().nxo_ncores(), "ops": out}


def bf16_bits(a):
    """f32 -> bf16 storage, round to nearest even (finite inputs)."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def bf16_values(u16):
    return (np.ascontiguousarray(u16).astype(np.uint32) << 16).view(np.float32)


class Gpt2Workload:
    """Config 5's inputs, drawn once: GPT-2 small, weights N(0, 0.02) from seed 16, ids from seed 17."""

    def __init__(self):
        from raven_amd.kaun_gpt2 import Config, host_params

        self.cfg = Config.small()
        self.batch, self.seq = 8, 1024
        self.hp = host_params(self.cfg, seed=16)
        self.ids = np.random.default_rng(17).integers(0, self.cfg.vocab_size, (self.batch, self.seq)).astype(np.int32)


def compiled_host_config5(iters=3):
    """Config 5 issued by the compiled host (raven_amd/host_c/kaun_gpt2_host.c): the same call sequence
    through the C ABI with no interpreter between the calls, in a process of its own. Wall time per
    forward, eagerly and with the library's deferred mode (no graph), and the replayed graph's GPU time."""
    import subprocess

    from raven_amd import _ffi, build

    if not build.GPT2_HOST_BIN.exists():
        return {"cfg5_c_host": "not built"}
    r = subprocess.run([str(build.GPT2_HOST_BIN), str(_ffi.LIB_PATH), "--iters", str(iters)], capture_output=True, text=True,
                       timeout=300)
    if r.returncode != 0:
        return {"cfg5_c_host": ("failed: " + r.stderr.strip())[:100]}
    t = json.loads(r.stdout.strip().splitlines()[-1])
    tokens = t["batch"] * t["seq"]
    return {"cfg5_c_host_eager_ms": t["eager_wall_ms"], "cfg5_c_host_deferred_ms": t["deferred_wall_ms"],
            "cfg5_c_host_deferred_late_free_ms": t["late_free_wall_ms"], "cfg5_c_host_replay_gpu_ms": t["replay_gpu_ms"],
            "cfg5_c_host_deferred_tokens_per_s": round(tokens / (t["deferred_wall_ms"] * 1e-3), 1),
            "cfg5_c_host_deferred_wall_over_replay_gpu": t["deferred_wall_over_replay_gpu"]}


def config5(hip, work, iters=3, warmup=1, window=False, graph=False, keep_positions=64):
    """GPT-2-small-shaped forward (12 layers, d 768, 12 heads, FFN 3072, vocab
    50257, batch 8 x seq 1024, bf16 random-init weights): tokens/s. Eager: one
    backend call per primitive. With ``window``: the same calls with the library's
    deferred mode on (nxh_set_deferred): it records the primitives and replaces the
    attention, softmax, layer-norm, GELU and linear sequences by fused kernels. With
    ``graph`` too: that forward is recorded once and each timed step is one replay.
    Returns the record and logits[0, :keep_positions, :] of the last timed step."""
    from raven_amd.kaun_gpt2 import Gpt2, upload
    from raven_amd.nx_frontend import Nx

    cfg, batch, seq = work.cfg, work.batch, work.seq
    counter = CountingBackend(hip)
    front = counter
    nx = Nx(front)
    hip.set_deferred(bool(window))
    try:
        return _config5_timed(hip, work, counter, front, nx, iters, warmup, window, graph, keep_positions)
    finally:
        hip.set_deferred(False)


def _config5_timed(hip, work, counter, front, nx, iters, warmup, window, graph, keep_positions):
    from raven_amd.kaun_gpt2 import Gpt2, upload

    cfg, batch, seq = work.cfg, work.batch, work.seq
    params = upload(nx, work.hp, dt.bfloat16, lambda a, d: bf16_bits(a))
    ids = nx.create(dt.int32, (batch, seq), work.ids)
    model = Gpt2(nx, cfg)
    for _ in range(warmup):
        out = model.logits(params, ids)
        del out
    front.synchronize()
    recorded = None
    if graph:
        front.capture_begin()
        try:
            out = model.logits(params, ids)
        finally:
            recorded = front.capture_end()
    counter.calls.clear()
    stats0 = hip.deferred_stats()
    t0 = time.perf_counter()
    front.timer_start()
    for i in range(iters):
        if recorded is not None:
            recorded.launch()
        else:
            if i:
                del out
            out = model.logits(params, ids)
    ev_ms = front.timer_stop() / iters
    front.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / iters
    calls = {k: v // iters for k, v in counter.calls.items()}
    stats1 = hip.deferred_stats()
    fused = {k: (stats1[k] - stats0[k]) // iters for k in stats1 if stats1[k] != stats0[k]}
    final = out
    head = logical(hip.contiguous(hip.shrink(final, [(0, 1), (0, keep_positions), (0, cfg.vocab_size)])))
    del out, final
    if recorded is not None:
        recorded.destroy()
    flops = 284812800 * batch * seq  # matmul FLOPs per forward
    how = ("the windowed forward recorded once, each step one graph replay" if graph else
           "the library's deferred mode: attention, layer norm, GELU and linear sequences as fused kernels" if window
           else "eager, one backend call per primitive")
    rec = {"op": f"cfg5 GPT-2 small forward, bf16, batch 8 x seq 1024 ({how})",
           "ms": round(ms, 3), "tokens/s": round(batch * seq / (ms * 1e-3), 1), "hip_event_ms": round(ev_ms, 3),
           "matmul_TFLOP/s": round(flops / (ms * 1e-3) / 1e12, 1), "backend_calls": sum(calls.values()),
           "calls_by_kind": calls}
    if window and recorded is None:
        rec["library_counters_per_forward"] = fused  # primitives recorded, issued as recorded, runs fused
    del params, ids, model, nx, front
    hip.trim()
    return rec, head


# ── parity of what was timed, and the CPU oracle's time on the same work ─────────────────────────
# Each function runs right after its configuration was timed (the outputs still hold the results
# of the timed calls), compares them with the CPU oracle on the same seeded inputs, and returns
# (parity flag, {name: CPU figure}). The oracle is the checker and the CPU baseline, never the
# product path.

def _oracle():
    from oracle.nx_oracle import OracleBackend, lib
    from oracle.nx_oracle import logical as ological

    return OracleBackend(), lib(), ological


def _cpu_time(fn, budget=1.5, max_reps=5):
    r = fn()  # warm (first touch of fresh pages)
    t0, reps = time.perf_counter(), 0
    while reps < 1 or (time.perf_counter() - t0 < budget and reps < max_reps):
        r = fn()
        reps += 1
    return (time.perf_counter() - t0) / reps, r


def check_config1(W):
    B, L, olog = _oracle()
    a, b, c = (B.reshape(B.from_host(h, dt.float32), h.shape) for h in W.cfg1["host"])
    sec, zo = _cpu_time(lambda: B.reduce("sum", [1], B.binary("add", B.binary("mul", a, b), B.unary("sin", c))))
    z, zo = logical(W.cfg1["z"]).astype(np.float64), olog(zo).astype(np.float64)
    ok = bool(np.all(np.abs(z - zo) <= 4096 * 1e-5 * (1.0 + np.abs(zo))))  # k * a_rel, backend_contract.ml:908-913
    return ok, {"cfg1_chain_cpu_GBs": round(603996160 / sec / 1e9, 2), "cfg1_cpu_threads": int(L.nxo_last_threads())}


def check_config3(W):
    B, L, olog = _oracle()
    hx, hxi = W.cfg3["host"]
    x, xi = B.reshape(B.from_host(hx, dt.float32), hx.shape), B.reshape(B.from_host(hxi, dt.int32), hxi.shape)
    ok, cpu = True, {}
    e = hx.nbytes
    for axis in (1, 0):
        out = W.cfg3["out"][axis]
        sec, r = _cpu_time(lambda: B.reduce("sum", [axis], x), 1.0, 3)
        cpu[f"cfg3_sum_axis{axis}_cpu_GBs"] = round(e / sec / 1e9, 2)
        want = olog(r).astype(np.float64)
        ok &= bool(np.all(np.abs(logical(out["sum"]).astype(np.float64) - want) <= 8192 * 1e-5 * (1.0 + np.abs(want))))
        ok &= bool(np.array_equal(logical(out["max"]).view(np.uint32), olog(B.reduce("max", [axis], x)).view(np.uint32)))
        sec, r = _cpu_time(lambda: B.argmax(x, axis), 1.0, 3)
        cpu[f"cfg3_argmax_axis{axis}_cpu_GBs"] = round(e / sec / 1e9, 2)
        ok &= bool(np.array_equal(logical(out["argmax"]), olog(r)))
        ok &= bool(np.array_equal(logical(out["isum"]), olog(B.reduce("sum", [axis], xi))))
    return ok, cpu


def check_config4(W):
    B, L, olog = _oracle()
    ok, cpu = True, {}
    ha, hb, cf = W.cfg4["f32"]
    oa, ob = B.reshape(B.from_host(ha, dt.float32), ha.shape), B.reshape(B.from_host(hb, dt.float32), hb.shape)
    sec, r = _cpu_time(lambda: B.matmul(oa, ob), 2.0, 3)
    cpu["cfg4_f32_2048_cpu_TFLOPs"] = round(2 * 2048 ** 3 / sec / 1e12, 3)
    want = olog(r).astype(np.float64)
    scale = 0.02 * 0.02 * np.sqrt(2048)
    ok &= bool(np.all(np.abs(logical(cf).astype(np.float64) - want) <= 1e-3 * (np.abs(want) + scale)))  # matmul_test.ml:831-974
    # bf16 batched: sampled outputs of two batches against the float64 product of the quantised inputs
    keep, cb = W.cfg4["bf16"]
    n = 4096
    rng = np.random.default_rng(99)
    rows, cols = rng.integers(0, n, 32), rng.integers(0, n, 32)
    for i in (0, 9):
        qa = bf16_values(bf16_bits(keep[("a", i)][rows])).astype(np.float64)
        qb = bf16_values(bf16_bits(np.ascontiguousarray(keep[("b", i)][:, cols]))).astype(np.float64)
        want = qa @ qb
        ci = W.hip.contiguous(W.hip.shrink(cb, [(i, i + 1), (0, n), (0, n)]))
        got = bf16_values(logical(ci)[0][np.ix_(rows, cols)]).astype(np.float64)
        ok &= bool(np.all(np.abs(got - want) <= 6e-2 * (np.abs(want) + 0.02 * 0.02 * np.sqrt(n))))
        del ci
    m = 2048  # CPU sample: one [2048]^3 bf16 product of the oracle (1/1024 of the batched call's work)
    sa = B.cast(B.reshape(B.from_host(keep[("a", 0)][:m, :m].copy(), dt.float32), (m, m)), dt.bfloat16)
    sb = B.cast(B.reshape(B.from_host(keep[("b", 0)][:m, :m].copy(), dt.float32), (m, m)), dt.bfloat16)
    sec, _ = _cpu_time(lambda: B.matmul(sa, sb), 1.0, 2)
    cpu["cfg4_bf16_cpu_TFLOPs"] = round(2 * m ** 3 / sec / 1e12, 4)
    for nm, d, tol in (("bf16", dt.bfloat16, 6e-2), ("f32", dt.float32, 1e-3)):
        hsa, hsb, out = W.cfg4["skinny"][nm]
        oa = B.cast(B.reshape(B.from_host(hsa, dt.float32), hsa.shape), d)
        ob = B.cast(B.reshape(B.from_host(hsb, dt.float32), hsb.shape), d)
        sec, r = _cpu_time(lambda: B.matmul(oa, ob), 1.0, 3)
        cpu[f"cfg4_skinny_{nm}_cpu_GBs"] = round((8 * 4096 + 4096 * 16384 + 8 * 16384) * d.itemsize / sec / 1e9, 2)
        got, want = logical(out), olog(r)
        if d is dt.bfloat16:
            got, want = bf16_values(got), bf16_values(want)
        got, want = got.astype(np.float64), want.astype(np.float64)
        ok &= bool(np.all(np.abs(got - want) <= tol * (np.abs(want) + 0.02 * 0.02 * 64)))
    return ok, cpu


def check_config5(work, heads):
    """The oracle runs batch row 0's first positions as a forward of its own (the model is
    causal) and is compared with logits[0, :k, :] of each timed GPU route: the contract's bf16
    tolerance (rel = abs = 6e-2, backend_contract.ml:179-188) and the top-1 agreement."""
    from raven_amd.kaun_gpt2 import Gpt2, upload
    from raven_amd.nx_frontend import Nx

    B, L, olog = _oracle()
    k = next(iter(heads.values())).shape[1]
    nx = Nx(B)
    params = upload(nx, work.hp, dt.bfloat16, lambda a, d: bf16_bits(a))
    ids = nx.create(dt.int32, (1, k), work.ids[:1, :k])
    t0 = time.perf_counter()
    want = bf16_values(olog(Gpt2(nx, work.cfg).logits(params, ids)))
    sec = time.perf_counter() - t0
    ok, out = True, {"cfg5_cpu_tokens_per_s": round(k / sec, 1), "cfg5_cpu_sample": f"batch 1 x seq {k}, one pass"}
    for name, head in heads.items():
        got = bf16_values(head)
        ok &= bool(np.all(np.abs(got - want) <= 6e-2 + 6e-2 * np.abs(want)))
        out[f"cfg5_{name}_top1_vs_oracle"] = round(float(np.mean(got.argmax(-1) == want.argmax(-1))), 4)
    return ok, out


def host_buffer_step(hip, steps, warmup):
    """The headline step as a caller with host buffers sees it: per step the two 64 MiB operands go up
    (nxh_memcpy_h2d from pageable numpy arrays, staged through the library's pinned slots), the seven
    calls run, and the f16, bool and int32 results come back (nxh_memcpy_d2h). GB/s over the same
    algorithmic bytes as the headline, so the two figures compare directly."""
    W = Workloads(hip)
    ops = W.config2()
    step_bytes = sum(o.nbytes for o in ops)
    lib, h = hip._lib, hip._h
    ups = [(t.buffer.ptr, np.ascontiguousarray(hip.to_host(t))) for t in W.cfg2_in.values()]
    downs = [(t.buffer.ptr, np.empty(t.buffer.nbytes, np.uint8)) for t in W.cfg2_out.values()]
    moved = sum(x.nbytes for _, x in ups) + sum(x.nbytes for _, x in downs)

    def step():
        for ptr, host in ups:
            hip._check(lib.nxh_memcpy_h2d(h, ptr, host.ctypes.data, host.nbytes))
        for op in ops:
            op()
        for ptr, host in downs:
            hip._check(lib.nxh_memcpy_d2h(h, host.ctypes.data, ptr, host.nbytes))

    for _ in range(warmup):
        step()
    hip.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    hip.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    return {"ms_per_step": round(ms, 3), "GBs_over_algorithmic_bytes": round(step_bytes / ms / 1e6, 1),
            "bytes_over_pcie_per_step": moved, "pcie_GBs": round(moved / ms / 1e6, 1),
            "algorithmic_bytes_per_step": step_bytes, "steps": steps}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the cpu_baseline leg")
    ap.add_argument("--only-step", action="store_true", help="time the headline step only")
    ap.add_argument("--pmc-calibration", action="store_true",
                    help="also launch 20 plain 64 MiB copies (scale for rocprofv3 FETCH_SIZE / WRITE_SIZE readings)")
    ap.add_argument("--only-config", type=int, choices=(1, 2, 3, 4), default=0,
                    help="time the operations of one configuration only and print their records")
    ap.add_argument("--only-next", action="store_true",
                    help="time the operations beside the hot path only (pad ... fft), the linear-algebra family included")
    ap.add_argument("--only-gpt2", action="store_true", help="run the GPT-2 forward leg only and print its record")
    ap.add_argument("--gemm-study", action="store_true",
                    help="config 4's bf16 product on zeros and on N(0, 0.02) data, this library / the vendor library / an "
                         "MFMA-only loop: time, board power and shader clock of each")
    ap.add_argument("--gemm-study-vendor", action="store_true",
                    help="the vendor rows of --gemm-study alone (torch.bmm, in this process)")
    ap.add_argument("--study-skip-vendor", action="store_true",
                    help="--gemm-study without the vendor rows (for counter runs: run --gemm-study-vendor as a command of its own)")
    ap.add_argument("--study-seconds", type=float, default=1.5, help="length of each timed loop of --gemm-study")
    ap.add_argument("--host-buffers", action="store_true",
                    help="the headline step with its two large operands uploaded from host memory and its three "
                         "results read back inside the timed region (the PCIe-inclusive rate; never the headline)")
    ap.add_argument("--cpu-configs", action="store_true",
                    help="time the CPU oracle on bounded samples of configurations 1, 3, 4, 5 and print the records")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this backend has no multi-GPU path (run with --gpus 1)", file=sys.stderr)
        sys.exit(2)

    if args.cpu_configs:
        print(json.dumps({"cpu_configs": cpu_configs()}))
        return
    if args.gemm_study_vendor:
        print(json.dumps(gemm_study_vendor(args.study_seconds)))
        return
    hip = Backend()
    info = hip.device_info()
    if args.only_gpt2:
        work = Gpt2Workload()
        print(json.dumps(config5(hip, work)[0]))
        print(json.dumps(config5(hip, work, window=True)[0]))
        print(json.dumps(config5(hip, work, window=True, graph=True, iters=10)[0]))
        return
    if args.only_next:
        print(json.dumps({"ops": next_ops(hip, Workloads(hip), linalg=True)}))
        return
    if args.gemm_study:
        print(json.dumps({"gemm_study": gemm_study(hip, args.study_seconds, vendor=not args.study_skip_vendor)}))
        return
    if args.host_buffers:
        print(json.dumps({"host_buffers": host_buffer_step(hip, args.steps, args.warmup)}))
        return
    if args.only_config:
        # one configuration's operations, each timed alone (for profiling runs)
        W = Workloads(hip)
        group = {1: W.config1, 2: W.config2, 3: W.config3, 4: W.config4}[args.only_config]
        recs = [op_record(op, time_ops(hip, [op], 10 if "16,4096" in op.name else 50, 3)) for op in group()]
        print(json.dumps({"config": args.only_config, "ops": recs}))
        return
    W = Workloads(hip)
    step_ops = W.config2()
    step_bytes = sum(o.nbytes for o in step_ops)

    # headline: W warm-up steps, then exactly K timed steps, synchronised on both sides
    for _ in range(args.warmup):
        for op in step_ops:
            op()
    hip.synchronize()
    policy0 = hip.cache_policy_stats()
    t0 = time.perf_counter()
    hip.timer_start()
    for _ in range(args.steps):
        for op in step_ops:
            op()
    ev_ms = hip.timer_stop()
    hip.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3
    ms_per_step = wall_ms / args.steps
    value = step_bytes / (ms_per_step * 1e-3) / 1e9
    # how many of the timed calls streamed past the memory-side cache (the library's own per-call decision)
    policy_stats = {"mode": "default (3: streaming loads and stores by block history)",
                    **{k + "_calls_in_timed_steps": v - policy0[k] for k, v in hip.cache_policy_stats().items()}}

    # the same step recorded once and replayed: what the launch gaps between the seven calls cost
    hip.capture_begin()
    try:
        for op in step_ops:
            op()
    finally:
        recorded = hip.capture_end()
    for _ in range(args.warmup):
        recorded.launch()
    hip.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        recorded.launch()
    hip.synchronize()
    replay_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    recorded.destroy()

    # parity of what was just timed, against the oracle on the same seeded inputs
    cpu, parity = None, {}
    if not args.no_cpu:
        cpu, (ov, ow) = cpu_baseline()
        from oracle.nx_oracle import logical as ological

        parity[2] = bool(np.array_equal(logical(W.cfg2_out["v"]).view(np.uint16), ological(ov).view(np.uint16))
                         and np.array_equal(logical(W.cfg2_out["w"]), ological(ow)))

    # The dominant kernel (the LDS-turned add) for the roofline object, twice: launched back to
    # back (its 64 MiB input then stays in the 256 MB memory-side cache between launches), and as
    # the first call of the step (its input was evicted by the 870 MB the step moves, and the
    # cache is full of the previous step's dirty outputs).
    dom = step_ops[0]
    dom_ms = time_ops(hip, [dom], 200, 10)
    dom_path = hip.last_path()
    in_step = []
    for _ in range(5 + 30):
        hip.timer_start()
        dom()
        in_step.append(hip.timer_stop())
        for op in step_ops[1:]:
            op()
    dom_step_ms = float(np.mean(in_step[5:]))
    roofline = {
        "kernel": f"{dom_path}_kernel<BinaryF<OpAdd, f32>, 64, 32> ({dom.name})",
        "bound": "hbm", "achieved": round(dom.nbytes / (dom_ms * 1e-3) / 1e9, 1), "peak": PEAK_HBM_GBS,
        "unit": "GB/s", "frac": round(dom.nbytes / (dom_ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4),
        "bytes_per_launch": dom.nbytes, "avg_launch_ms": round(dom_ms, 5), "traffic": DOMINANT_KERNEL_HBM_TRAFFIC,
        "achieved_in_step": round(dom.nbytes / (dom_step_ms * 1e-3) / 1e9, 1),
        "frac_in_step": round(dom.nbytes / (dom_step_ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4),
        "in_step_launch_ms": round(dom_step_ms, 5),
        "note": "achieved / frac: launched back to back, input warm in the memory-side cache; *_in_step: as the "
                "first call of the step, input from HBM (streamed past the cache by the library's cache policy)",
    }

    ops_out, flat = [], {}
    if args.pmc_calibration:
        # a plain contiguous copy of known size (64 MiB read, 64 MiB written) in the same process:
        # hardware-counter readings of the step's kernels are scaled by what the counters show here
        src, dst = hip.full(dt.float32, (64, 512, 512), 1.0), hip.buffer(dt.float32, (64, 512, 512))
        cal = W.mk("calibration copy 64 MiB", W.lib.nxh_copy, [dst, src], nbytes=2 * 64 * 512 * 512 * 4)
        for _ in range(20):
            cal()
        hip.synchronize()

    def note(key, rec):
        """One operation's figure as flat scalars of the line's `config` object."""
        if "TFLOP/s" in rec and rec.get("bound") == "mfma":
            flat[key + "_TFLOPs"], flat[key + "_frac"] = rec["TFLOP/s"], rec["frac_mfma"]
        else:
            flat[key + "_GBs"], flat[key + "_frac"] = rec["GB/s"], rec["frac_hbm"]

    if not args.only_step:
        keys2 = ["cfg2_f32_add", "cfg2_f32_mul_scalar", "cfg2_cast_f16", "cfg2_i32_add", "cfg2_i32_mul", "cfg2_i32_cmplt",
                 "cfg2_i32_where"]
        for key, op in zip(keys2, step_ops):
            ops_out.append(op_record(op, time_ops(hip, [op], 100, 5)))
            note(key, ops_out[-1])
        keys = {W.config1: ["cfg1_mul", "cfg1_sin", "cfg1_add", "cfg1_sum_axis1"],
                W.config3: [f"cfg3_{o}_axis{a}" for a in (1, 0) for o in ("sum", "max", "argmax", "isum")],
                W.config4: ["cfg4_f32_2048", "cfg4_bf16_batched", "cfg4_skinny_bf16", "cfg4_skinny_f32"]}
        checks = {W.config1: (1, check_config1), W.config3: (3, check_config3), W.config4: (4, check_config4)}
        for group in (W.config1, W.config3, W.config4):
            ops = group()
            for key, op in zip(keys[group], ops):
                iters = 10 if "16,4096" in op.name else 50
                ops_out.append(op_record(op, time_ops(hip, [op], iters, 3)))
                note(key, ops_out[-1])
            if group == W.config1:
                ms = time_ops(hip, ops, 50, 3)
                ops_out.append({"op": "cfg1 chain (4 ops, 576 MiB)", "ms": round(ms, 5),
                                "GB/s": round(603996160 / (ms * 1e-3) / 1e9, 1),
                                "frac_hbm": round(603996160 / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4), "bound": "hbm"})
                note("cfg1_chain", ops_out[-1])
            if not args.no_cpu:
                n, fn = checks[group]
                parity[n], cpu_figs = fn(W)
                flat.update(cpu_figs)
            del ops
            W.keep.clear()
            W.cfg1 = W.cfg3 = W.cfg4 = None
            hip.trim()
        work = Gpt2Workload()
        heads = {}
        for name, kw in (("eager", {}), ("window", {"window": True}), ("replay", {"window": True, "graph": True, "iters": 10})):
            rec, heads[name] = config5(hip, work, **kw)
            ops_out.append(rec)
            flat[f"cfg5_{name}_tokens_per_s"], flat[f"cfg5_{name}_ms"] = rec["tokens/s"], rec["ms"]
        flat["cfg5_replay_matmul_TFLOPs"] = ops_out[-1]["matmul_TFLOP/s"]
        if not args.no_cpu:
            parity[5], cpu_figs = check_config5(work, heads)
            flat.update(cpu_figs)
        del work, heads
        flat.update(compiled_host_config5())
        ops_out.extend(next_ops(hip, W))

    # What a reader who keeps only the first keys of `config` must see comes first: one figure per
    # configuration (the GEMM and reduction fractions the metric names), the parity flags, the CPU
    # oracle beside them; the per-operation detail of config 2 and everything else follows.
    config = {"workload": "config 2: [64,512,512] f32 add(permuted, broadcast) / mul scalar / cast f16 + int32 add / mul / "
                          "cmplt / where",
              "frac_of_hbm_peak": round(value / PEAK_HBM_GBS, 4)}
    cfg3 = {k: v for k, v in flat.items() if k.startswith("cfg3_") and k.endswith("_frac")}
    first = ["cfg4_bf16_batched_TFLOPs", "cfg4_bf16_batched_frac", "cfg4_f32_2048_TFLOPs", "cfg4_f32_2048_frac",
             "cfg4_skinny_bf16_GBs", "cfg4_skinny_bf16_frac"]
    for k in first:
        if k in flat:
            config[k] = flat[k]
    if cfg3:
        worst = min(cfg3, key=cfg3.get)
        config["cfg3_worst_op"], config["cfg3_worst_frac"] = worst[:-len("_frac")], cfg3[worst]
    for k in ("cfg1_chain_GBs", "cfg1_chain_frac", "cfg5_replay_tokens_per_s", "cfg5_c_host_deferred_tokens_per_s"):
        if k in flat:
            config[k] = flat[k]
    config["cfg2_parity_vs_oracle"] = parity.get(2)
    for n in (1, 3, 4, 5):
        if n in parity:
            config[f"cfg{n}_parity_vs_oracle"] = parity[n]
    if cpu is not None:
        config["cfg2_step_cpu_GBs"] = cpu["value"]
    for k in ("cfg4_bf16_cpu_TFLOPs", "cfg4_f32_2048_cpu_TFLOPs", "cfg4_skinny_bf16_cpu_GBs", "cfg3_sum_axis0_cpu_GBs",
              "cfg1_chain_cpu_GBs", "cfg5_cpu_tokens_per_s"):
        if k in flat:
            config[k] = flat[k]
    config.update({"calls_per_step": len(step_ops), "algorithmic_bytes_per_step": step_bytes,
                   "device": info["name"].strip(), "compute_units": info["compute_units"],
                   "hip_event_ms_per_step": round(ev_ms / args.steps, 5), "parity_vs_oracle": parity.get(2),
                   "graph_replay_ms_per_step": round(replay_ms, 5),
                   "graph_replay_GBs": round(step_bytes / (replay_ms * 1e-3) / 1e9, 1),
                   "cache_policy": policy_stats})
    for k, v in flat.items():
        config.setdefault(k, v)
    # the same figures grouped per configuration (readers that keep nested objects)
    config["per_config"] = {f"config{n}": {k: v for k, v in config.items() if k.startswith(f"cfg{n}_")} for n in (1, 2, 3, 4, 5)}
    line = {
        "metric": METRIC, "value": round(value, 1), "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_per_step, 5), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32+i32", "data": "synthetic",
        "config": config, "roofline": roofline, "cpu_baseline": cpu, "ops": ops_out,
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
