"""Timing cases of the block Gram-Schmidt library: what a user's program calls
and at which sizes.

A case is one call of a public entry point on inputs made from a seed:

  entry "device"   bcgs_hip.bcgs_device on device pointers (Q in place, R)
        "noalloc"  bcgs_hip.bcgs_device_noalloc (library-fixed scratch)
        "mixed"    bcgs_hip.bcgs_mixed_device, FP32 storage with FP64 products
        "batched"  bcgs_hip.bcgs_batched_device over `count` uneven instances
        "host"     the C symbol of include/orth.h on host memory

The in-place forms overwrite X, so a program that factors a basis it also
keeps (the residual needs X) copies it first; run() does the same.
"""
import importlib
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "one-synchronization-bcgs_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)
B = importlib.import_module("bcgs_hip")


def listed():
    return [
        # The reference driver's own test matrix (rand() entries): the
        # smallest call, all launches and latency.
        {"name": "driver_550x35_s5", "entry": "device", "variant": "bcgsi2P1s", "m": 550, "n": 35,
         "s": 5, "kappa": 0.0},
        # One s-step cycle of a small problem in a serving loop that may not
        # allocate (the smoke test's shape).
        {"name": "small_4096x64_s16", "entry": "noalloc", "variant": "bcgsi2P1s", "m": 4096,
         "n": 64, "s": 16, "kappa": 1e4},
        # The reference's CPU benchmark shape, the one-synchronization variant.
        {"name": "cpu_1e5x200_s10", "entry": "device", "variant": "bcgsi2P1s", "m": 100000,
         "n": 200, "s": 10, "kappa": 1e4},
        # The same shape by the robust variant with the most synchronizations
        # (what a program falls back to when the Pythagorean form breaks down).
        {"name": "cpu_1e5x200_s10_i2", "entry": "device", "variant": "bcgsi2", "m": 100000,
         "n": 200, "s": 10, "kappa": 1e4},
        # The drop-in replacement as the reference's caller uses it: host
        # memory, the C symbol, same shape.
        {"name": "host_1e5x200_s10", "entry": "host", "variant": "bcgsi2P1s", "m": 100000,
         "n": 200, "s": 10, "kappa": 1e4},
        # A medium slab with an odd row count, a ragged last block and narrow
        # blocks (s = 4), two synchronizations per block.
        {"name": "odd_1000003x61_s4_pipi", "entry": "device", "variant": "bcgspipi2",
         "m": 1000003, "n": 61, "s": 4, "kappa": 1e3},
        # A medium slab with s = 8 blocks.
        {"name": "mid_1048576x128_s8", "entry": "device", "variant": "bcgsi2P1s", "m": 1 << 20,
         "n": 128, "s": 8, "kappa": 1e5},
        # The benchmark's width on a mid-sized slab, by the variant whose block
        # updates run in sequence.
        {"name": "mid_1048576x256_s16_a1s", "entry": "device", "variant": "bcgsi21s",
         "m": 1 << 20, "n": 256, "s": 16, "kappa": 1e4},
        # The wide slab of the near-dependent-blocks stress (n = 512, s = 32).
        {"name": "wide_4194304x512_s32", "entry": "device", "variant": "bcgsi2P1s", "m": 1 << 22,
         "n": 512, "s": 32, "kappa": 1e4},
        # FP32 storage of the basis, FP64 arithmetic.
        {"name": "mixed_4194304x256_s16", "entry": "mixed", "variant": "bcgsi2P1s", "m": 1 << 22,
         "n": 256, "s": 16, "kappa": 1e4},
        # Many small independent problems of uneven shapes in one call.
        {"name": "batched_48_uneven", "entry": "batched", "variant": "bcgsi2P1s", "count": 48,
         "mix": 7, "kappa": 1e4},
        # The headline benchmark: the largest slab.
        {"name": "headline_16777216x256_s16", "entry": "device", "variant": "bcgsi2P1s",
         "m": 1 << 24, "n": 256, "s": 16, "kappa": 1e4},
    ]


def draw(rng):
    entry = rng.choice(["device"] * 6 + ["noalloc", "mixed", "batched", "host"])
    variant = rng.choice(["bcgsi2P1s", "bcgsi2P1s", "bcgsi2P1s", "bcgsi21s", "bcgspipi2", "bcgsi2",
                          "bcgsi2P2s"])
    kappa = 10.0 ** rng.randint(2, 5)
    if entry == "batched":
        return {"entry": entry, "variant": variant, "count": rng.randint(6, 48),
                "mix": rng.randint(100, 10 ** 6), "kappa": kappa}
    s = rng.choice([3, 4, 5, 8, 10, 16, 16, 16, 32])
    nmax = {3: 96, 4: 128, 5: 128, 8: 192, 10: 256, 16: 256, 32: 512}[s]
    n = rng.randint(2 * s, nmax)
    if rng.random() < 0.5:
        n -= n % s
    if entry == "mixed":
        variant, s, n = "bcgsi2P1s", 16, 16 * rng.randint(2, 16)
    # Bytes of the slab, spread over the logarithm of the range; the variants
    # with many passes and the host form stay smaller.
    top = {"host": 2.0 ** 24, "noalloc": 2.0 ** 28}.get(entry, 2.0 ** 30)
    if variant in ("bcgsi2", "bcgsi2P2s"):
        top /= 4
    m = int(2.0 ** rng.uniform(math.log2(4 * n + 64), math.log2(top / n)))
    if rng.random() < 0.5:
        m -= m % 32
    return {"entry": entry, "variant": variant, "m": max(m, n), "n": n, "s": s, "kappa": kappa}


def _instances(case):
    """(m, n, s) of every instance of a case."""
    if case["entry"] != "batched":
        return [(case["m"], case["n"], case["s"])]
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["count"]):
        m = int(2.0 ** r.uniform(12, 18))
        out.append((m, r.choice([32, 64, 128]), r.choice([4, 8, 16])))
    return out


def _input(m, n, kappa, g, dtype=torch.float64):
    """X^T (n x m row-major: the m x n column-major slab with ld m): uniform
    [0, 1) entries for kappa = 0, else a Gaussian slab times V diag(sigma)
    with sigma log-spaced from 1 to 1 / kappa."""
    if kappa == 0.0:
        return torch.rand((n, m), generator=g, dtype=torch.float64, device="cuda").to(dtype)
    G = torch.randn((n, m), generator=g, dtype=torch.float64, device="cuda")
    V, _ = torch.linalg.qr(torch.randn((n, n), generator=g, dtype=torch.float64,
                                       device="cuda").cpu())
    sig = torch.logspace(0, -math.log10(kappa), n, dtype=torch.float64)
    X = (V * sig).cuda() @ G
    del G
    return X.to(dtype)


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dt = torch.float32 if case["entry"] == "mixed" else torch.float64
    return [_input(m, n, case["kappa"], g, dt) for m, n, _ in _instances(case)]


def prepare(case, seed):
    shapes = _instances(case)
    Xs = _inputs(case, seed)
    st = {"case": case, "shapes": shapes}
    if case["entry"] == "host":
        m, n, _ = shapes[0]
        st["X0"] = Xs[0].cpu().numpy()
        st["X"] = st["X0"].copy()
        st["R"] = np.zeros((n, n))
        return st
    if case["entry"] == "batched":
        # One allocation for the batch, the instances back to back (each
        # 256-byte aligned).
        off, tot = [], 0
        for m, n, _ in shapes:
            off.append(tot)
            tot += (m * n + 31) // 32 * 32
        st["X0"] = torch.zeros(tot, dtype=torch.float64, device="cuda")
        for o, x in zip(off, Xs):
            st["X0"][o:o + x.numel()] = x.reshape(-1)
        st["X"] = torch.empty_like(st["X0"])
        st["Q"] = [st["X"][o:o + m * n].view(n, m) for o, (m, n, _) in zip(off, shapes)]
        st["R"] = [torch.zeros((n, n), dtype=torch.float64, device="cuda") for _, n, _ in shapes]
        return st
    m, n, _ = shapes[0]
    st["X0"] = Xs.pop()
    st["X"] = torch.empty((n, m), dtype=torch.float64, device="cuda")
    st["R"] = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    st["info"] = torch.zeros(2, dtype=torch.int32, device="cuda")
    return st


def run(st):
    case = st["case"]
    entry, variant = case["entry"], case["variant"]
    m, n, s = st["shapes"][0]
    if entry == "host":
        np.copyto(st["X"], st["X0"])
        rc = getattr(B.lib(), variant)(m, n, s, st["X"].ctypes.data, m, st["R"].ctypes.data, n,
                                       None, 0)
        if rc != 0:
            raise RuntimeError("%s returned %d" % (variant, rc))
        return {"Q": st["X"], "R": st["R"]}
    stream = torch.cuda.current_stream().cuda_stream
    if entry == "mixed":
        B.bcgs_mixed_device(variant, "fp64", m, n, s, st["X0"].data_ptr(), m, st["X"].data_ptr(),
                            m, st["R"].data_ptr(), n, stream)
        return {"Q": st["X"], "R": st["R"]}
    st["X"].copy_(st["X0"])
    if entry == "batched":
        ms, ns, ss = zip(*st["shapes"])
        info, _ = B.bcgs_batched_device(variant, ms, ns, ss, [q.data_ptr() for q in st["Q"]], ms,
                                        [r.data_ptr() for r in st["R"]], ns, stream=stream)
        # Flat, since a batch has more matrices than separate outputs allow.
        return {"Q": st["X"], "R": torch.cat([r.reshape(-1) for r in st["R"]]),
                "info": np.array(info, dtype=np.int64)}
    if entry == "noalloc":
        rc = B.bcgs_device_noalloc(variant, m, n, s, st["X"].data_ptr(), m, st["R"].data_ptr(), n,
                                   st["info"].data_ptr(), stream)
        if rc != 0:
            raise RuntimeError("orth_bcgs_device_noalloc returned %d" % rc)
        return {"Q": st["X"], "R": st["R"], "info": st["info"]}
    B.bcgs_device(variant, m, n, s, st["X"].data_ptr(), m, st["R"].data_ptr(), n, stream)
    return {"Q": st["X"], "R": st["R"]}


def work(case):
    """Reorthogonalized block Gram-Schmidt: X read and Q and R written once;
    4 m n^2 flops (two passes of projection and update)."""
    b = f = 0.0
    for m, n, _ in _instances(case):
        b += (4.0 if case["entry"] == "mixed" else 8.0) * m * n + 8.0 * m * n + 8.0 * n * n
        f += 4.0 * m * n * n
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """Q and R by LAPACK's Householder QR with a positive diagonal of R (the
    factorization every variant computes)."""
    shapes = _instances(case)
    if sum(float(m) * n * n for m, n, _ in shapes) > 2.2e10:
        return None
    qs, rs = [], []
    for X in _inputs(case, seed):
        q, r = torch.linalg.qr(X.double().cpu().T)
        d = torch.sign(torch.diagonal(r))
        qs.append((q * d).T.contiguous())
        rs.append((r.T * d).contiguous())
    if case["entry"] == "batched":
        flat = []
        for (m, n, _), q in zip(shapes, qs):
            f = torch.zeros((m * n + 31) // 32 * 32, dtype=torch.float64)
            f[:m * n] = q.reshape(-1)
            flat.append(f)
        return {"Q": torch.cat(flat), "R": torch.cat([r.reshape(-1) for r in rs]), "info": None}
    if case["entry"] == "host":
        return {"Q": qs[0].numpy(), "R": rs[0].numpy()}
    out = {"Q": qs[0], "R": rs[0]}
    if case["entry"] == "noalloc":
        out["info"] = None
    return out
