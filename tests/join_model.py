"""The fp16 joined-core tiles (csrc/trk_join_kernel.h) restated in torch, for the tests: the rule that
says which cores they are routed to (join_spread_kernel in csrc/trk_pack.hip), both kernels'
roundings, and cores that are even and uneven in every way the rule looks at."""
from __future__ import annotations

import math

import torch

INS, OUTS = (8, 12, 20), (12, 10, 24)  # 1920 -> 2880


def even(cores) -> bool:
    """Whether every slice (one index of one mode) of every core has values of the size of the core's
    largest: nonzero magnitudes that average 1/16 of it, at most a quarter of them below 1/64."""
    for g in (c.float().cpu().abs() for c in cores):
        peak = g.max()
        if not torch.isfinite(peak):
            return False
        for mode in range(4):
            s = g.transpose(0, mode).flatten(1)
            nonzero, small = (s > 0).sum(1), ((s > 0) & (s * 64 < peak)).sum(1)
            if ((nonzero > 0) & ((s.sum(1) * 16 < peak * nonzero) | (4 * small > nonzero))).any():
                return False
    return True


def _half(t):
    return t.half().float()


def joined(x, cores):
    """x [T, in] through joined fp16 cores: H and W rounded to fp16, one power of two per core."""
    e = [math.frexp(c.abs().max().item())[1] for c in cores]
    g1, g2, g3 = (_half(c.float() * 2.0 ** -k) for c, k in zip(cores, e))
    h = _half(torch.einsum("bqjc,crka->qrjkab", g2, g3))
    w = _half(torch.einsum("qrjkab,apib->ijkpqr", h, g1))
    return (x.float() @ w.reshape(x.shape[1], -1)) * 2.0 ** sum(e)


def chain(x, cores):
    """x through G3, G2, G1 one after another, U and V rounded to fp16."""
    g1, g2, g3 = (c.float() for c in cores)
    u = _half(torch.einsum("tijk,crka->tijrca", x.float().reshape(-1, *INS), g3))
    v = _half(torch.einsum("tijrca,bqjc->tiqrba", u, g2))
    return torch.einsum("tiqrba,apib->tpqr", v, g1).reshape(x.shape[0], -1)


def exact(x, cores):
    g1, g2, g3 = (c.double() for c in cores)
    w = torch.einsum("apiqjc,crka->ijkpqr", torch.einsum("apib,bqjc->apiqjc", g1, g2), g3)
    return x.double() @ w.reshape(x.shape[1], -1)


# name: (kind, size); the last four of each kind's sizes are far past the rule's bounds
CASES = {"plain": ("plain", 1), "laplace": ("laplace", 1),
         **{f"{kind}_{size}": (kind, size) for kind in ("input", "input_zero", "output", "gauge", "entry")
            for size in (2, 3, 10, 100)}}


def make(name: str, rank: int, tokens: int, seed: int = 3):
    """(x, cores) in fp16 on the CPU. input: one input digit of each core `size` times the others,
    x smaller by it there (or zero); output: one output digit; gauge: one ring index larger in one core
    and smaller in the next, which leaves the operator as it is; entry: one value of each core."""
    kind, size = CASES[name]
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(tokens, *INS, generator=gen)
    cores = [torch.randn(rank, o, i, rank, generator=gen) / math.sqrt(rank * i)
             for i, o in zip(INS, OUTS)]
    if kind == "laplace":
        cores = [c.sign() * torch.empty_like(c).exponential_(generator=gen) / math.sqrt(rank * i)
                 for c, i in zip(cores, INS)]
    digits = (3, 5, 7)
    if kind in ("input", "input_zero"):
        for m, d in enumerate(digits):
            cores[m][:, :, d] *= size
            x.select(m + 1, d).mul_(1.0 / size if kind == "input" else 0.0)
    if kind == "output":
        for c, d in zip(cores, digits):
            c[:, d] *= size
    if kind == "gauge":
        for m, d in enumerate(digits):
            cores[m][..., d] *= size
            cores[(m + 1) % 3][d] /= size
    if kind == "entry":
        for c in cores:
            c[1, 2, 3, 4] = size
    return x.reshape(tokens, -1).half(), [c.half() for c in cores]
