"""The work this library is measured on: calls of its public API over the sizes that density-fitting
programs and plain Level-3 users bring, from one small product to the full pair energy.

Families ("op") and what stands behind each:
* gemm: 2-D products in fp32 / bf16 / fp16, any transposes, with and without C. Sizes from a small
  molecule's orbital blocks (tens of rows) up, odd ones included, since basis, virtual and auxiliary
  counts are whatever the molecule gives.
* half: the first half-transform of a DF-MP2 calculation, C_occ^T on the (nbasis, nbasis naux) view
  of the three-center tensor: few rows, very many columns.
* syrk / batched: the symmetric update and the batched products (per-occupied-orbital second
  half-transform, metric contraction with one shared right operand).
* pair: the fused DF-MP2 pair energy; mp2: the energy of an amplitude block that is already there.
* fp64: the fp64-class product by Ozaki splitting.
* metric / trsm: the fp64 metric stage of the same calculations.
* chain: a whole df_mp2_energy call at a small molecule's size.
"""

import math

import torch

import trnblas_amd as tb
from trnblas_amd import df_mp2

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "f64": torch.float64}
BYTES = {"f32": 4, "bf16": 2, "f16": 2, "f64": 8}


def listed():
    return [
        # the smallest call: one orbital-block product of a small molecule, A^T B + 0.5 C
        dict(name="gemm_f32_96", op="gemm", dtype="f32", m=80, n=72, k=96, ta=True, tb=False, beta=0.5),
        # an ordinary product whose sizes are multiples of nothing
        dict(name="gemm_f32_1535", op="gemm", dtype="f32", m=1535, n=1535, k=1535, ta=False, tb=False, beta=0.0),
        # the headline product: 2048^3, A^T B + 0.5 C
        dict(name="gemm_f32_2048_tn", op="gemm", dtype="f32", m=2048, n=2048, k=2048, ta=True, tb=False, beta=0.5),
        # a 16-bit product of the size the library serves itself
        dict(name="gemm_bf16_2048_nt", op="gemm", dtype="bf16", m=2048, n=2048, k=2048, ta=False, tb=True, beta=0.0),
        # first half-transform of a medium molecule
        dict(name="half_384_48_1152", op="half", nbasis=384, nocc=48, naux=1152),
        # the headline Level-3 mix: SYRK with C in the lower triangle, and the batched product
        dict(name="syrk_f32_4096x8192", op="syrk", dtype="f32", n=4096, k=8192, trans=False, uplo="lower", beta=0.5),
        dict(name="batched_64x512x2048x512", op="batched", dtype="f32", b=64, m=512, n=512, k=2048, ta=False,
             shared=False),  # fmt: skip
        # the headline pair energy (largest case)
        dict(name="pair_96_672_2304", op="pair", nocc=96, nvir=672, naux=2304),
        # energy of one i-chunk of the example's medium shape (64 / 448)
        dict(name="mp2_16_64_448", op="mp2", ic=16, nocc=64, nvir=448),
        # fp64-class product at the size of the published figure, default slices and mode
        dict(name="fp64_4096_k8", op="fp64", m=4096, n=4096, k=4096, slices=8, mode="fast"),
        # metric factor at the example's large auxiliary count
        dict(name="metric_2304", op="metric", dtype="f64", n=2304),
        # a whole calculation at the example's small shape (128 / 16 / 384)
        dict(name="chain_128_16_384", op="chain", nbasis=128, nocc=16, naux=384),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm, odd or even as it falls."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """As _log, but a third of the time a multiple of 32, as padded programs have it."""
    n = _log(rng, lo, hi)
    return max(32, n // 32 * 32) if rng.random() < 1 / 3 else n


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "half", "syrk", "batched", "pair", "mp2", "fp64", "metric", "trsm", "chain"])
    beta = rng.choice([0.0, 0.0, 0.5])
    if op == "gemm":
        return dict(op=op, dtype=rng.choice(["f32", "f32", "f32", "bf16", "f16"]), m=_size(rng, 16, 4096),
                    n=_size(rng, 16, 4096), k=_size(rng, 16, 4096), ta=rng.random() < 0.5, tb=rng.random() < 0.5,
                    beta=beta)  # fmt: skip
    if op == "half":
        nbasis = _size(rng, 96, 384)
        nocc = max(4, nbasis // rng.choice([5, 6, 8, 10]))
        return dict(op=op, nbasis=nbasis, nocc=nocc, naux=3 * nbasis - rng.choice([0, 1, 2, 8]))
    if op == "syrk":
        return dict(op=op, dtype=rng.choice(["f32", "f32", "bf16"]), n=_size(rng, 64, 4096), k=_size(rng, 64, 8192),
                    trans=rng.random() < 0.5, uplo=rng.choice(["lower", "upper"]), beta=beta)  # fmt: skip
    if op == "batched":
        return dict(op=op, dtype=rng.choice(["f32", "f32", "bf16"]), b=_log(rng, 4, 64), m=_size(rng, 64, 640),
                    n=_size(rng, 64, 1536), k=_size(rng, 64, 1536), ta=rng.random() < 0.5,
                    shared=rng.random() < 0.5)  # fmt: skip
    if op == "pair":
        return dict(op=op, nocc=_log(rng, 4, 72), nvir=_size(rng, 40, 500), naux=_size(rng, 128, 1800))
    if op == "mp2":
        return dict(op=op, ic=_log(rng, 1, 12), nocc=_log(rng, 8, 64), nvir=_size(rng, 60, 448))
    if op == "fp64":
        return dict(op=op, m=_size(rng, 100, 4096), n=_size(rng, 100, 4096), k=_size(rng, 100, 4096),
                    slices=rng.choice([6, 7, 8, 8, 8, 9, 10]), mode=rng.choice(["fast", "fast", "crt", "exact"]))  # fmt: skip
    if op == "metric":
        return dict(op=op, dtype=rng.choice(["f64", "f64", "f32"]), n=_size(rng, 96, 2304))
    if op == "trsm":
        return dict(op=op, dtype=rng.choice(["f64", "f32"]), n=_size(rng, 96, 2304), m=_size(rng, 96, 2304),
                    left=rng.random() < 0.7, uplo=rng.choice(["lower", "upper"]), trans=rng.random() < 0.5)  # fmt: skip
    nbasis = _size(rng, 48, 160)
    return dict(op=op, nbasis=nbasis, nocc=max(4, nbasis // 8), naux=3 * nbasis)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _eps(g, nocc, nvir):
    eo = -1.5 + 1.2 * torch.rand(nocc, generator=g, device="cuda")
    ev = 0.1 + 2.9 * torch.rand(nvir, generator=g, device="cuda")
    return eo, ev


def _metric(g, n):
    """A symmetric positive definite metric: a Wishart matrix and a little of the identity."""
    x = _randn(g, n, n, dtype=torch.float64)
    return x @ x.mT / n + 0.1 * torch.eye(n, dtype=torch.float64, device="cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]
    s = dict(case)
    if op == "gemm":
        dt, m, n, k = DTYPES[case["dtype"]], case["m"], case["n"], case["k"]
        s["A"] = _randn(g, *((k, m) if case["ta"] else (m, k))).to(dt)
        s["B"] = _randn(g, *((n, k) if case["tb"] else (k, n))).to(dt)
        s["C"] = _randn(g, m, n).to(dt) if case["beta"] else None
    elif op == "half":
        nb = case["nbasis"]
        q, _ = torch.linalg.qr(_randn(g, nb, nb))
        s["A"] = q[:, : case["nocc"]].contiguous()
        s["B"] = 0.02 * _randn(g, nb, nb * case["naux"])
    elif op == "syrk":
        dt, n, k = DTYPES[case["dtype"]], case["n"], case["k"]
        s["A"] = _randn(g, *((k, n) if case["trans"] else (n, k))).to(dt)
        s["C"] = None
        if case["beta"]:
            x = _randn(g, n, n)
            s["C"] = (torch.tril(x) + torch.tril(x, -1).mT).to(dt)
    elif op == "batched":
        dt, b, m, n, k = DTYPES[case["dtype"]], case["b"], case["m"], case["n"], case["k"]
        s["A"] = _randn(g, b, *((k, m) if case["ta"] else (m, k))).to(dt)
        s["B"] = _randn(g, k, n).to(dt).unsqueeze(0).expand(b, k, n) if case["shared"] else _randn(g, b, k, n).to(dt)
    elif op == "pair":
        s["B"] = 0.05 * _randn(g, case["nocc"], case["nvir"], case["naux"])
        s["eo"], s["ev"] = _eps(g, case["nocc"], case["nvir"])
    elif op == "mp2":
        ic, nocc, nvir = case["ic"], case["nocc"], case["nvir"]
        s["T"] = 0.05 * _randn(g, ic * nvir, nocc * nvir)
        s["eo"], s["ev"] = _eps(g, nocc, nvir)
    elif op == "fp64":
        for name, shape in (("A", (case["m"], case["k"])), ("B", (case["k"], case["n"]))):
            s[name] = _randn(g, *shape, dtype=torch.float64)
    elif op == "metric":
        s["J"] = _metric(g, case["n"]).to(DTYPES[case["dtype"]])
    elif op == "trsm":
        dt, n, m = DTYPES[case["dtype"]], case["n"], case["m"]
        t = torch.linalg.cholesky(_metric(g, n))
        s["T"] = (t if case["uplo"] == "lower" else t.mT.contiguous()).to(dt)
        s["B"] = _randn(g, *((n, m) if case["left"] else (m, n)), dtype=torch.float64).to(dt)
    elif op == "chain":
        nb, nocc, naux = case["nbasis"], case["nocc"], case["naux"]
        s["C_occ"], s["C_vir"] = 0.1 * _randn(g, nb, nocc), 0.1 * _randn(g, nb, nb - nocc)
        s["eri"] = 0.01 * _randn(g, nb, nb, naux)
        j = 0.01 * _randn(g, naux, naux)
        s["J"] = j @ j.mT + torch.eye(naux, device="cuda")
        s["eo"], s["ev"] = _eps(g, nocc, nb - nocc)
    return s


def run(s):
    op = s["op"]
    if op == "gemm":
        return tb.gemm(1.0, s["A"], s["B"], s["beta"], s["C"], transA=s["ta"], transB=s["tb"])
    if op == "half":
        return tb.gemm(1.0, s["A"], s["B"], transA=True)
    if op == "syrk":
        return tb.syrk(1.0, s["A"], s["beta"], s["C"], trans=s["trans"], uplo=s["uplo"])
    if op == "batched":
        return tb.batched_gemm(1.0, s["A"], s["B"], transA=s["ta"])
    if op == "pair":
        return tb.hip.nki_batched_pair_energy(s["B"], s["eo"], s["ev"])
    if op == "mp2":
        return tb.hip.nki_mp2_energy(s["T"], s["eo"][: s["ic"]], s["eo"], s["ev"])
    if op == "fp64":
        return tb.gemm_fp64(s["A"], s["B"], slices=s["slices"], mode=s["mode"])
    if op == "metric":
        return tb.metric_inv_half(s["J"])
    if op == "trsm":
        return tb.trsm(1.0, s["T"], s["B"], side="left" if s["left"] else "right", uplo=s["uplo"], trans=s["trans"])
    return df_mp2.df_mp2_energy(s["C_occ"], s["C_vir"], s["eri"], s["J"], s["eo"], s["ev"], use_batched_pair=True)


def work(case):
    op = case["op"]
    e = BYTES[case.get("dtype", "f32")]
    if op in ("gemm", "fp64"):
        m, n, k = case["m"], case["n"], case["k"]
        e = 8 if op == "fp64" else e
        return {"bytes": e * (m * k + k * n + m * n * (2 if case.get("beta") else 1)), "flops": 2.0 * m * n * k}
    if op == "half":
        nb, o, p = case["nbasis"], case["nocc"], case["naux"]
        return {"bytes": 4 * (nb * o + nb * nb * p + o * nb * p), "flops": 2.0 * o * nb * nb * p}
    if op == "syrk":
        n, k = case["n"], case["k"]
        c = n * (n + 1) // 2 if case["beta"] else 0
        return {"bytes": e * (n * k + c + n * n), "flops": 1.0 * n * (n + 1) * k}
    if op == "batched":
        b, m, n, k = case["b"], case["m"], case["n"], case["k"]
        return {"bytes": e * (b * m * k + k * n * (1 if case["shared"] else b) + b * m * n), "flops": 2.0 * b * m * n * k}
    if op == "pair":
        o, v, p = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": 4 * (o * v * p + o + v), "flops": o * (o + 1) / 2 * (2.0 * v * v * p + 8.0 * v * v)}
    if op == "mp2":
        t = case["ic"] * case["nocc"] * case["nvir"] ** 2
        return {"bytes": 4 * (t + case["nocc"] + case["nvir"]), "flops": 8.0 * t}
    if op == "metric":
        n = case["n"]
        return {"bytes": e * 2 * n * n, "flops": 2.0 * n**3 / 3.0}
    if op == "trsm":
        n, m = case["n"], case["m"]
        return {"bytes": e * (n * (n + 1) // 2 + 2 * n * m), "flops": 1.0 * n * n * m}
    nb, o, p = case["nbasis"], case["nocc"], case["naux"]
    v = nb - o
    flops = 2.0 * p**3 / 3.0 + 2.0 * nb * nb * o * p + 2.0 * o * v * nb * p + 2.0 * o * v * p * p + o * (o + 1) * v * v * p
    return {"bytes": 4 * (nb * nb + nb * nb * p + p * p + nb), "flops": flops}


def tolerance(case):
    """About four times the largest error against `exact` over 130 drawn cases."""
    op = case["op"]
    if op in ("gemm", "half", "syrk", "batched"):
        if case.get("dtype", "f32") == "f32":
            return {"rel": 1e-6, "max": 6e-6}  # fp32 products and sums
        # fp32 sums, one rounding to the output type
        return {"rel": 8e-3, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 2e-3}
    if op == "fp64":
        # what `slices` digits of 7 bits keep of each operand, and fp64 rounding
        return {"rel": 1.3e-11 * 2.0 ** (-7 * (case["slices"] - 6)) + 2e-15}
    if op == "metric":
        return {"rel": 6e-15 if case["dtype"] == "f64" else 1.2e-7}  # fp64 inside, one rounding to fp32
    if op == "trsm":
        return {"rel": 4e-15 if case["dtype"] == "f64" else 1e-6}
    return {"rel": 3e-7}  # energies: sums of fp32 products, returned in fp32


def _exact_product(A, B):
    """A @ B for fp64 operands to about one rounding: each operand in two parts of at most 22 bits
    (per row of A / column of B) and a rest, the leading products exact in fp64."""

    def parts(x, dim):
        top = torch.exp2(torch.ceil(torch.log2(x.abs().amax(dim, keepdim=True).clamp_min(1e-300))))
        out, rest = [], x
        for bits in (20, 40):
            q = top * 2.0**-bits
            p = torch.round(rest / q) * q
            out.append(p)
            rest = rest - p
        return out + [rest]

    a, b = parts(A, 1), parts(B, 0)
    low = a[2] @ B + (a[0] + a[1]) @ b[2]
    low = low + a[1] @ b[1]
    return a[0] @ b[0] + (a[0] @ b[1] + a[1] @ b[0] + low)


def _exact_pair(B, eo, ev):
    nocc, nvir, naux = B.shape
    B, eo, ev = B.double(), eo.double(), ev.double()
    vv = ev[:, None] + ev[None, :]
    e = torch.zeros((), dtype=torch.float64, device=B.device)
    for i in range(nocc):
        T = (B[i] @ B[i:].reshape(-1, naux).mT).reshape(nvir, nocc - i, nvir).permute(1, 0, 2)
        d = eo[i] + eo[i:, None, None] - vv
        ei = (T * (2.0 * T - T.mT) / d).sum((1, 2))
        e = e + 2.0 * ei.sum() - ei[0]
    return e


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op in ("gemm", "half", "batched"):
        A, B = s["A"].double(), s["B"].double()
        A = A.mT if (op == "half" or case["ta"]) else A
        B = B.mT if case.get("tb") else B
        D = torch.matmul(A.contiguous(), B.contiguous())
        return D + case["beta"] * s["C"].double() if case.get("beta") else D
    if op == "syrk":
        A = s["A"].double()
        A = A.mT.contiguous() if case["trans"] else A
        D = A @ A.mT
        return D + case["beta"] * s["C"].double() if case["beta"] else D
    if op == "pair":
        return _exact_pair(s["B"], s["eo"], s["ev"])
    if op == "mp2":
        ic, nocc, nvir = case["ic"], case["nocc"], case["nvir"]
        T4 = s["T"].reshape(ic, nvir, nocc, nvir)
        eo, ev = s["eo"].double(), s["ev"].double()
        vv = ev[:, None] + ev[None, :]
        e = torch.zeros((), dtype=torch.float64, device="cuda")
        for i in range(ic):
            T = T4[i].double().permute(1, 0, 2)
            e = e + (T * (2.0 * T - T.mT) / (eo[i] + eo[:, None, None] - vv)).sum()
        return e
    if op == "fp64":
        return _exact_product(s["A"], s["B"])
    if op == "metric":
        L = torch.linalg.cholesky(s["J"].double())
        eye = torch.eye(case["n"], dtype=torch.float64, device="cuda")
        return torch.linalg.solve_triangular(L.mT, eye, upper=True)
    if op == "trsm":
        T, B = s["T"].double(), s["B"].double()
        T, upper = (T.mT, case["uplo"] == "lower") if case["trans"] else (T, case["uplo"] == "upper")
        return torch.linalg.solve_triangular(T, B, upper=upper, left=case["left"])
    eri, J, C_occ, C_vir = (s[x].double() for x in ("eri", "J", "C_occ", "C_vir"))
    nb, nocc, naux = case["nbasis"], case["nocc"], case["naux"]
    eye = torch.eye(naux, dtype=torch.float64, device="cuda")
    X = torch.linalg.solve_triangular(torch.linalg.cholesky(J).mT, eye, upper=True)
    iv = (C_occ.mT @ eri.reshape(nb, nb * naux)).reshape(nocc, nb, naux)
    ia = torch.stack([C_vir.mT @ iv[i] for i in range(nocc)])
    return float(_exact_pair((ia.reshape(-1, naux) @ X).reshape(nocc, nb - nocc, naux), s["eo"], s["ev"]))
