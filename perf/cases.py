"""Performance cases of dmrg_amd: the calls a DMRG program makes on the GPU, through the public entry points.

Kinds of case (each a dict of plain values):
  matvec  y_i = H_eff x_i, the call an eigensolver makes in its inner loop. entry "operator": a device-resident
          MatVecMPOS (MultAx_device), nvec vectors per call, dtype f64/c128, or f32/c64 for the FP32 matvecs of the
          mixed-precision solver; entry "stateless": tools::common::contraction::matrix_vector_product.
  group   matvecs of many small operators of uneven shapes in one call (a request loop's resident problems).
  env     EnvBase::build_block, the environment update after a site was solved; D = 25 is the block of an MPO^2.
  solve   one step of a DMRG sweep: the local ground state of H_eff and the environment update with it. H_eff is the
          critical Ising chain's, with blocks in a random orthonormal basis, as a sweep meets it.
  sweep   a whole fDMRG ground-state search of ising_tf_rf from a product state.

Tensors are torch tensors on the GPU whose contiguous layout is the column-major layout of the C ABI with the
indices reversed: theta (b, a, s), env (w, a', a), mpo (s', s, w', w).
"""
import ctypes as C
import math

import numpy as np
import torch

import dmrg_amd
from dmrg_amd import _lib

DTYPE = {"f64": torch.float64, "c128": torch.complex128, "f32": torch.float32, "c64": torch.complex64}
CODE = {"f64": _lib.DMRG_FP64, "c128": _lib.DMRG_CX64, "f32": _lib.DMRG_FP32, "c64": _lib.DMRG_CX32}
SIZE = {"f64": 8, "c128": 16, "f32": 4, "c64": 8}
WIDE = {"f64": "f64", "c128": "c128", "f32": "f64", "c64": "c128"}
NUMPY = {"f64": np.float64, "c128": np.complex128}
MAX_MACS = 4.0 * 1024**3 * 8 * 2 * 1.01  # the two-site matvec at chi = 1024, the largest listed case
TOL = 1e-12  # the library's default eigensolver tolerance


def listed():
    def mv(name, dtype, d, chiL, chiR, D, entry="operator", nvec=1):
        return {"name": name, "kind": "matvec", "entry": entry, "dtype": dtype, "d": d, "chiL": chiL, "chiR": chiR, "D": D, "nvec": nvec}

    return [
        # Smallest calls: a site near the edge of a real chain (ising MPO, D = 3); latency and launches.
        mv("matvec_chi24_f64", "f64", 2, 24, 24, 3),
        # An ordinary complex site away from the tuned sizes: chi_L < chi_R, odd bonds.
        mv("matvec_173x211_c128", "c128", 2, 173, 211, 5),
        # The headline workload: single-site complex double at chi = 512, D = 5.
        mv("matvec_chi512_c128", "c128", 2, 512, 512, 5),
        # The same matvec as the mixed-precision solver's inner loop calls it: FP32 matrix cores.
        mv("matvec_chi512_c64", "c64", 2, 512, 512, 5),
        # Block eigensolver (blockSize 8) on a mid-size ragged site in real double, larger MPO.
        mv("matvec_block8_120x88_f64", "f64", 2, 120, 88, 8, nvec=8),
        # Largest: two-site update (d = 4) at chi = 1024 with D = 8.
        mv("matvec_two_site_chi1024_c128", "c128", 4, 1024, 1024, 8, entry="stateless"),
        # A request loop's resident problems: 32 operators of chi 16..64.
        {"name": "group32_chi16_64_f64", "kind": "group", "dtype": "f64", "d": 2, "lo": 16, "hi": 64, "D": 5, "count": 32},
        # Environment update in the rightward half-sweep at the headline size.
        {"name": "env_L_chi512_c128", "kind": "env", "side": "L", "dtype": "c128", "d": 2, "chiL": 512, "chiR": 512, "D": 5},
        # Variance environment (MPO^2, D = 25) in the leftward half-sweep, ragged bonds, real.
        {"name": "env_R_201x164_D25_f64", "kind": "env", "side": "R", "dtype": "f64", "d": 2, "chiL": 201, "chiR": 164, "D": 25},
        # A local solve of an ordinary sweep in real double, and its environment update.
        {"name": "solve_chi64_f64", "kind": "solve", "dtype": "f64", "chiL": 64, "chiR": 64, "mixed": False},
        # A large complex local solve in mixed precision (FP32 matrix-core phase, FP64 refinement).
        {"name": "solve_240x256_c128_mixed", "kind": "solve", "dtype": "c128", "chiL": 240, "chiR": 256, "mixed": True},
        # A whole program: the ground state of a random-field chain, bonds grown by subspace expansion.
        {"name": "sweep_L16_chi32_f64", "kind": "sweep", "L": 16, "chi": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec"] * 6 + ["group", "env", "env", "solve", "sweep"])
    if kind in ("matvec", "env"):
        while True:
            d = rng.choice([2, 2, 2, 4])
            chiL = _log_int(rng, 12, 1024)
            chiR = max(8, min(1024, int(chiL * rng.uniform(0.5, 2.0))))
            D = rng.choice([3, 5, 5, 8, 25])
            dtype = rng.choice(["f64", "c128", "c128", "f32", "c64"] if kind == "matvec" else ["f64", "c128"])
            nvec = rng.choice([1, 1, 1, 2, 4, 8]) if kind == "matvec" and chiL * chiR < 200 * 200 else 1
            if _macs(d, chiL, chiR, D) * nvec <= 0.5 * MAX_MACS and chiL * chiL * D <= 8 << 20 and chiR * chiR * D <= 8 << 20:
                break
        if kind == "env":
            return {"kind": "env", "side": rng.choice("LR"), "dtype": dtype, "d": d, "chiL": chiL, "chiR": chiR, "D": D}
        entry = "operator" if nvec > 1 or rng.random() < 0.7 else "stateless"
        return {"kind": "matvec", "entry": entry, "dtype": dtype, "d": d, "chiL": chiL, "chiR": chiR, "D": D, "nvec": nvec}
    if kind == "group":
        lo = _log_int(rng, 8, 40)
        return {"kind": "group", "dtype": rng.choice(["f64", "c128"]), "d": 2, "lo": lo, "hi": lo * rng.choice([2, 3, 4]),
                "D": rng.choice([3, 5, 8]), "count": rng.randint(8, 48)}
    if kind == "solve":
        chiL = _log_int(rng, 24, 256)
        chiR = max(16, min(256, int(chiL * rng.uniform(0.6, 1.6))))
        return {"kind": "solve", "dtype": rng.choice(["f64", "c128"]), "chiL": chiL, "chiR": chiR, "mixed": rng.random() < 0.5}
    return {"kind": "sweep", "L": rng.randint(8, 16), "chi": rng.randint(12, 32)}


# ------------------------------------------------------------------------------------------------ inputs


class _Buf:
    """A torch tensor's memory as the package's device-array arguments take it."""

    def __init__(self, t):
        self.t = t
        self.ptr = C.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(shape, dtype, g):
    return torch.randn(shape, dtype=DTYPE[dtype], device="cuda", generator=g)


def _theta(d, chiL, chiR, dtype, g):
    t = _normal((chiR, chiL, d), dtype, g)
    return t / torch.linalg.vector_norm(t)


def _env(chi, D, dtype, g):
    """Hermitian slices (A + A^H) / 2 with A ~ N(0, 1), as the bond blocks of a Hermitian MPO are."""
    a = _normal((D, chi, chi), dtype, g)
    return ((a + a.mH) / 2).contiguous()


def _mpo(DL, DR, d, dtype, g):
    """Real symmetric N(0, 1) blocks."""
    a = torch.randn((d, d, DR, DL), dtype=torch.float64, device="cuda", generator=g)
    return ((a + a.permute(1, 0, 2, 3)) / 2).to(DTYPE[dtype]).contiguous()


def _host(t):
    """A (reversed) torch tensor as the column-major host array that the operator's constructor takes."""
    return t.to(torch.complex128).cpu().numpy().transpose()


def _tensors(case, g, dtype):
    """theta (nvec of them), mpo, envL, envR of a matvec case."""
    d, D = case["d"], case["D"]
    th = torch.stack([_theta(d, case["chiL"], case["chiR"], dtype, g) for _ in range(case.get("nvec", 1))])
    return th, _mpo(D, D, d, dtype, g), _env(case["chiL"], D, dtype, g), _env(case["chiR"], D, dtype, g)


def _matvec_tensors(case, seed):
    """The values the call works on. The FP32 matvecs of an operator round its FP64 blocks, so those cases draw in
    FP64 what the operator holds and in FP32 the vectors."""
    th, W, L, R = _tensors(case, _gen(seed), WIDE[case["dtype"]])
    if case["dtype"] in ("f32", "c64"):
        th, W, L, R = (t.to(DTYPE[case["dtype"]]) for t in (th, W, L, R))
    return th, W, L, R


def _group_shapes(case):
    """Bonds spread evenly over [lo, hi], right bonds running against the left ones."""
    k, lo, hi = case["count"], case["lo"], case["hi"]
    chis = [lo + (hi - lo) * i // max(1, k - 1) for i in range(k)]
    return [(a, chis[(7 * i + 3) % k]) for i, a in enumerate(chis)]


def _group_tensors(case, seed):
    g = _gen(seed)
    return [tuple(t[0] if i == 0 else t for i, t in enumerate(_tensors({"d": case["d"], "D": case["D"], "chiL": a, "chiR": b}, g, case["dtype"])))
            for a, b in _group_shapes(case)]


def _env_tensors(case, seed):
    g = _gen(seed)
    th = _theta(case["d"], case["chiL"], case["chiR"], case["dtype"], g)
    W = _mpo(case["D"], case["D"], case["d"], case["dtype"], g)
    return th, W, _env(case["chiL"] if case["side"] == "L" else case["chiR"], case["D"], case["dtype"], g)


def _ising_mpo(dtype):
    """Site MPO of -sum sz sz - sum sx: row 2 starts a term, column 0 ends it."""
    W = np.zeros((3, 3, 2, 2))
    z, x = np.array([[1.0, 0.0], [0.0, -1.0]]), np.array([[0.0, 1.0], [1.0, 0.0]])
    W[0, 0] = W[2, 2] = np.eye(2)
    W[1, 0], W[2, 1], W[2, 0] = z, -z, -x
    return torch.from_numpy(np.ascontiguousarray(W.transpose())).to("cuda", DTYPE[dtype])


def _chain_block(chi, side, W, dtype, g):
    """Environment of a piece of the critical Ising chain in a random orthonormal basis of chi states: sites are
    added one by one from the chain's end, the basis doubling until chi."""
    E = torch.zeros((3, 1, 1), dtype=DTYPE[dtype], device="cuda")
    E[2 if side == "L" else 0] = 1.0
    m = 1
    while m < chi:
        r = min(2 * m, chi)
        q = torch.linalg.qr(_normal((2 * m, r), dtype, g))[0].reshape(m, 2, r)
        th = (q.permute(2, 0, 1) if side == "L" else q.permute(0, 2, 1)).contiguous()
        E = _exact_env(side, th, W, E)
        m = r
    E = E.contiguous()
    return ((E + E.mH) / 2).contiguous()


def _solve_tensors(case, seed):
    g = _gen(seed)
    W = _ising_mpo(case["dtype"])
    L = _chain_block(case["chiL"], "L", W, case["dtype"], g)
    R = _chain_block(case["chiR"], "R", W, case["dtype"], g)
    return _theta(2, case["chiL"], case["chiR"], case["dtype"], g), W, L, R


def _fields(case, seed):
    return np.random.default_rng(int(seed)).uniform(-0.5, 0.5, case["L"])


def _dims(*n):
    return (C.c_int64 * len(n))(*n)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sweep":
        return {"case": case, "h": _fields(case, seed)}
    if kind == "group":
        ops, xs, ys = [], [], []
        for th, W, L, R in _group_tensors(case, seed):
            ops.append(dmrg_amd.MatVecMPOS([_host(W)], _host(L), _host(R), dtype=NUMPY[case["dtype"]]))
            xs.append(_Buf(th))
            ys.append(_Buf(torch.zeros_like(th)))
        torch.cuda.synchronize()
        return {"case": case, "group": dmrg_amd.MatvecGroup(ops, xs, ys), "ys": ys}
    if kind == "matvec":
        th, W, L, R = _matvec_tensors(case, seed)
        s = {"case": case, "x": _Buf(th), "y": _Buf(torch.zeros_like(th))}
        if case["entry"] == "operator":
            s["op"] = dmrg_amd.MatVecMPOS([_host(W)], _host(L), _host(R), dtype=NUMPY[WIDE[case["dtype"]]])
        else:
            d, cL, cR, D = case["d"], case["chiL"], case["chiR"], case["D"]
            s.update(W=_Buf(W), L=_Buf(L), R=_Buf(R), dims=(_dims(d, cL, cR), _dims(D, D, d, d), _dims(cL, cL, D), _dims(cR, cR, D)))
        return s
    if kind == "env":
        th, W, E = _env_tensors(case, seed)
        d, cL, cR, D = case["d"], case["chiL"], case["chiR"], case["D"]
        out = torch.zeros((D, cR, cR) if case["side"] == "L" else (D, cL, cL), dtype=th.dtype, device="cuda")
        return {"case": case, "x": _Buf(th), "W": _Buf(W), "E": _Buf(E), "y": _Buf(out),
                "dims": (_dims(d, cL, cR), _dims(D, D, d, d), _dims(*reversed(E.shape)))}
    th, W, L, R = _solve_tensors(case, seed)
    cfg = _lib.EigsConfig()
    _lib.load().dmrg_eigs_default_config(C.byref(cfg))
    cfg.tol, cfg.mixed = TOL, int(case["mixed"])
    cL, cR = case["chiL"], case["chiR"]
    return {"case": case, "op": dmrg_amd.MatVecMPOS([_host(W)], _host(L), _host(R), dtype=NUMPY[case["dtype"]]), "cfg": cfg,
            "x": _Buf(th), "v": _Buf(torch.zeros_like(th)), "W": _Buf(W), "L": _Buf(L),
            "y": _Buf(torch.zeros((3, cR, cR), dtype=th.dtype, device="cuda")),
            "dims": (_dims(2, cL, cR), _dims(3, 3, 2, 2), _dims(cL, cL, 3))}


# ------------------------------------------------------------------------------------------------ one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "matvec":
        if case["entry"] == "operator":
            s["op"].MultAx_device(s["x"], s["y"], nvec=case["nvec"], fp32=case["dtype"] in ("f32", "c64"))
        else:
            m, w, l, r = s["dims"]
            _lib.call("dmrg_matrix_vector_product", CODE[case["dtype"]], s["y"].ptr, s["x"].ptr, m, s["W"].ptr, w, s["L"].ptr, l, s["R"].ptr, r, None)
        return s["y"].t
    if kind == "group":
        s["group"].run()
        return [y.t for y in s["ys"]]
    if kind == "env":
        m, w, o = s["dims"]
        _lib.call("dmrg_env_build_block", CODE[case["dtype"]], case["side"].encode(), s["y"].ptr, s["E"].ptr, o, s["x"].ptr, m, s["W"].ptr, w, None)
        return s["y"].t
    if kind == "solve":
        res = _lib.EigsResult()
        m, w, o = s["dims"]
        _lib.call("dmrg_eigs", s["op"].h, C.byref(s["cfg"]), s["x"].ptr, s["v"].ptr, C.byref(res), None)
        _lib.call("dmrg_env_build_block", CODE[case["dtype"]], b"L", s["y"].ptr, s["L"].ptr, o, s["v"].ptr, m, s["W"].ptr, w, None)
        return {"energy": res.eigval[0], "env": s["y"].t}
    r = dmrg_amd.fdmrg_ising_tf_rf(case["L"], s["h"], chi_max=case["chi"])
    return {"energy": r["energy"], "entropies": r["entropies"]}


# ------------------------------------------------------------------------------------------------ what a pass needs


def _macs(d, chiL, chiR, D):
    return float(d) * chiL * chiR * D * (chiL + chiR + D * d)


def work(case):
    kind = case["kind"]
    if kind == "sweep":  # one matvec and one environment update per site, at the bonds the chain can have
        b, f = 0.0, 0.0
        for i in range(case["L"]):
            cL, cR = (min(case["chi"], 2 ** min(k, case["L"] - k)) for k in (i, i + 1))
            b += 8.0 * (4 * cL * cR + 6 * (cL * cL + cR * cR))
            f += 4.0 * _macs(2, cL, cR, 3)
        return {"bytes": b, "flops": f}
    size, cplx = SIZE[case["dtype"]], 4.0 if case["dtype"] in ("c128", "c64") else 1.0

    def matvec(d, cL, cR, D, nvec=1):
        return (float(size) * (2 * nvec * d * cL * cR + D * (cL * cL + cR * cR) + D * D * d * d), 2 * cplx * nvec * _macs(d, cL, cR, D))

    if kind == "group":
        each = [matvec(case["d"], a, b, case["D"]) for a, b in _group_shapes(case)]
        return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}
    if kind == "matvec":
        b, f = matvec(case["d"], case["chiL"], case["chiR"], case["D"], case["nvec"])
    elif kind == "env":
        cL, cR, d, D = case["chiL"], case["chiR"], case["d"], case["D"]
        a, c = (cL, cR) if case["side"] == "L" else (cR, cL)  # the old block's bond and the new one's
        b = float(size) * (d * cL * cR + D * (cL * cL + cR * cR) + D * D * d * d)
        f = 2 * cplx * float(d) * a * c * D * (a + D * d + c)
    else:  # at least one matvec and the environment update
        cL, cR = case["chiL"], case["chiR"]
        b, f = matvec(2, cL, cR, 3)
        b += float(size) * 3 * cR * cR
        f *= 2
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------------------------------------ 64-bit values


def _wide(*ts):
    return [t.to(torch.complex128 if t.is_complex() else torch.float64) for t in ts]


def _exact_matvec(th, W, L, R):
    t = torch.tensordot(L, th, dims=([2], [1]))  # (w, a', b, s)
    t = torch.tensordot(t, W, dims=([0, 3], [3, 1]))  # (a', b, s', w')
    return torch.tensordot(t, R, dims=([1, 3], [2, 0])).permute(2, 0, 1)  # (a', s', b') -> (b', a', s')


def _exact_env(side, th, W, E):
    if side == "L":
        t = torch.tensordot(E, th, dims=([2], [1]))  # (w, a', b, s)
        t = torch.tensordot(t, W, dims=([0, 3], [3, 1]))  # (a', b, s', w')
        return torch.tensordot(t, th.conj(), dims=([0, 2], [1, 2])).permute(1, 2, 0)  # (b, w', b') -> (w', b', b)
    t = torch.tensordot(E, th, dims=([2], [0]))  # (w', b', a, s)
    t = torch.tensordot(t, W, dims=([0, 3], [2, 1]))  # (b', a, s', w)
    return torch.tensordot(t, th.conj(), dims=([0, 2], [0, 2])).permute(1, 2, 0)  # (a, w, a') -> (w, a', a)


def _exact_ground_state(th, W, L, R, steps=220):
    """Lanczos with full reorthogonalisation; the spectrum is wide against its gap by a factor of some tens."""
    V = torch.empty((steps, th.numel()), dtype=th.dtype, device=th.device)
    V[0] = th.reshape(-1) / torch.linalg.vector_norm(th)
    alpha, beta = [], []
    for j in range(steps):
        w = _exact_matvec(V[j].reshape(th.shape), W, L, R).reshape(-1)
        alpha.append(float(torch.vdot(V[j], w).real))
        for _ in range(2):
            w = w - (V[: j + 1].conj() @ w) @ V[: j + 1]
        b = float(torch.linalg.vector_norm(w))
        if j + 1 == steps or b < 1e-10:
            break
        beta.append(b)
        V[j + 1] = w / b
    T = np.diag(alpha) + np.diag(beta[: len(alpha) - 1], 1) + np.diag(beta[: len(alpha) - 1], -1)
    vals, vecs = np.linalg.eigh(T)
    y = torch.from_numpy(np.ascontiguousarray(vecs[:, 0])).to(V.device, V.dtype)
    return float(vals[0]), (y @ V[: len(alpha)]).reshape(th.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        th, W, L, R = _wide(*_matvec_tensors(case, seed))
        return torch.stack([_exact_matvec(t, W, L, R) for t in th])
    if kind == "group":
        return [_exact_matvec(*_wide(*t)) for t in _group_tensors(case, seed)]
    if kind == "env":
        th, W, E = _env_tensors(case, seed)
        return _exact_env(case["side"], *_wide(th, W, E))
    if kind == "solve":
        th, W, L, R = _solve_tensors(case, seed)
        e, v = _exact_ground_state(th, W, L, R)
        return {"energy": e, "env": _exact_env("L", v, W, L)}
    # The free-fermion closed form: H is quadratic in Majorana operators with the bidiagonal coupling matrix M.
    L, g = case["L"], 1.0 + _fields(case, seed)
    U, S, Vt = np.linalg.svd(np.diag(g) + np.diag(np.ones(L - 1), 1))
    G = U @ Vt
    ent = np.zeros(L + 1)
    for l in range(1, L):
        if 2 ** min(l, L - l) > case["chi"]:
            return {"energy": float(-S.sum()), "entropies": None}  # the bond dimension cuts the state: no closed form
        p = np.clip((1 + np.linalg.svd(G[:l, :l], compute_uv=False)) / 2, 1e-300, 1 - 1e-16)
        ent[l] = float(-np.sum(p * np.log(p) + (1 - p) * np.log1p(-p)))
    return {"energy": float(-S.sum()), "entropies": ent}
