"""The work a program has this library do, as timed cases.

Every case is one call path of a DMRG program on the U(1) block-sparse
library: a one-shot contraction, Krylov steps on an effective Hamiltonian, the
eigensolve of one bond, the truncated SVD of one bond, the SVD that
canonicalises a site, a run of environment updates, and a whole DMRG run.
Sectors are Gaussian in Sz (ttgpu.workloads): a wide distribution is the
synthetic one of the matvec benchmark (many small sectors), a narrow one is
what truncation leaves of a ground state (few large sectors).  Operands are
N(0,1), MPO tensors are the exact AutoMPO ones of the benchmark's lattices,
and two-site states have the decaying singular spectrum of a ground state.

Results stay on the device in a DMRG run; here each pass ends with one
download of its result into pinned host memory that the state keeps.  The
FP32 and split-BF16 forms carry 32-bit results, which is how they are
returned.
"""
import ctypes as C
import functools
import itertools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tensor-tools_amd", "python"))

from ttgpu import host as P  # noqa: E402
from ttgpu import lib as T  # noqa: E402
from ttgpu import workloads as W  # noqa: E402
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, legal_blocks, make_index  # noqa: E402

LATTICE = {"chain": "j1j2_chain_N100_m512", "cyl6": "heisenberg_cyl6x12_m2048", "cyl8": "j1j2_cyl8x16_m8192"}
PREC = {"fp64": T.FP64, "fp32": T.FP32, "bf16x3": T.BF16X3}


def listed():
    return [
        # operator* once on small ragged blocks, as observables and set-up code call it
        dict(name="contract_m48", kind="contract", lattice="chain", m=48, sigma=2.0, prec="fp64"),
        # Krylov steps y = H x on one operator: a chain at modest m ...
        dict(name="heff_chain_m512", kind="heff", lattice="chain", m=512, sigma=6.0, prec="fp64", steps=4),
        # ... the benchmark's cylinder in the reference's arithmetic and in the fast form ...
        dict(name="heff_cyl6_m2048", kind="heff", lattice="cyl6", m=2048, sigma=9.0, prec="fp64", steps=4),
        dict(name="heff_cyl6_m2048_bf16x3", kind="heff", lattice="cyl6", m=2048, sigma=9.0, prec="bf16x3", steps=4),
        # ... and the largest system
        dict(name="heff_cyl8_m8192", kind="heff", lattice="cyl8", m=8192, sigma=12.0, prec="fp64", steps=2),
        # the eigensolve of one bond: a new operator, planned, and the Davidson iteration DMRG runs on it
        dict(name="davidson_cyl6_m1024", kind="davidson", lattice="cyl6", m=1024, sigma=3.0, prec="fp64"),
        # the truncated SVD of one bond: bulk of a large run moving right, a ragged middle size moving left,
        # and a small one whose sectors are all narrow
        dict(name="svd_m1500", kind="svd", m=1500, sigma=3.0, dir=0),
        dict(name="svd_m333_back", kind="svd", m=333, sigma=1.7, dir=1),
        dict(name="svd_m100", kind="svd", m=100, sigma=2.0, dir=0),
        # right-canonicalisation of a random site (no cutoff): how every run starts
        dict(name="canon_m701", kind="canon", m=701, sigma=3.0, dir=1),
        # environments grown over three bulk sites, as buildEnv and the sweep do
        dict(name="env_cyl6_m1200", kind="env", lattice="cyl6", m=1200, sigma=4.0, prec="fp64", dir=0, sites=3),
        # a whole DMRG run on a short chain: every step, latency first
        dict(name="dmrg_N20_m48", kind="dmrg", n=20, m=48, sigma=2.0, sweeps=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = {"contract": 2e11, "heff": 2e11, "davidson": 6e10, "svd": 2e10, "canon": 1e10, "env": 2e11, "dmrg": 1e12}
    kind = rng.choice(["contract", "heff", "heff", "heff", "davidson", "svd", "svd", "canon", "env", "env", "dmrg"])
    while True:
        if kind == "dmrg":
            c = dict(kind=kind, n=2 * rng.randint(5, 10), m=_log(rng, 12, 48), sigma=round(rng.uniform(1.5, 3.0), 2),
                     sweeps=rng.randint(1, 2))
        else:
            hi = {"contract": 2048, "heff": 8192, "davidson": 2048, "svd": 1500, "canon": 701, "env": 2048}[kind]
            c = dict(kind=kind, m=_log(rng, 40, hi), sigma=round(rng.uniform(1.5, 12.0 if kind == "heff" else 6.0), 2))
            if c["m"] < 16 * c["sigma"]:
                c["sigma"] = round(max(1.2, c["m"] / 32), 2)
            if kind in ("svd", "canon"):
                c["dir"] = rng.randint(0, 1)
            else:
                c["lattice"] = rng.choice(["chain", "cyl6", "cyl8"])
                c["prec"] = rng.choice(["fp64", "fp64", "fp32", "bf16x3"]) if kind != "davidson" else "fp64"
            if kind == "heff":
                c["steps"] = 4 if c["m"] < 4096 else 2
            if kind == "env":
                c["dir"], c["sites"] = rng.randint(0, 1), 3
        if work(c)["flops"] <= most[kind]:
            return c


# ------------------------------------------------------------------ structures
@functools.lru_cache(maxsize=None)
def _mpo(lattice, n):
    """n consecutive MPO tensors at the lattice's middle bond, and the first site"""
    lat, nx, ny, yper, j2, site, *_ = W.WORKLOADS[LATTICE[lattice]]
    T.init(0)
    h = P.mpo_autompo(nx * ny, W.lattice_terms(P, lat, nx, ny, yper, j2))
    return [h.tensor(site + i).to_flat() for i in range(n)], site


def _link(arrow, name, level, m, sigma, odd=0):
    """a link of total dimension m: Sz sectors Gaussian of width sigma (charges odd at every other link)"""
    smax = max(1, min(int(round(3.4 * sigma)), (m - 2) // 4))
    return make_index(arrow, name, LINK, level, [((q + odd, 0), d) for q, d in W.sector_dims(m, smax, sigma)])


def _struct(idx):
    idx = [ix.copy() for ix in idx]
    return FlatTensor(idx, legal_blocks(idx), np.zeros(0))


def _bond_structs(c):
    """L (l', w, l), W1, W2, R (r', w, r) and x (l, s1, s2, r) of a two-site bond"""
    (w1, w2), site = _mpo(c["lattice"], 2)
    link = functools.partial(_link, m=c["m"], sigma=c["sigma"])
    l, r = link(INWARD, "ID1Link%d" % site, 0), link(OUTWARD, "ID1Link%d" % (site + 2), 0)
    lp, rp = link(INWARD, l.name, 1), link(OUTWARD, r.name, 1)
    s1, s2 = W.site_index(INWARD, "Site%d" % site, 0), W.site_index(INWARD, "Site%d" % (site + 1), 0)
    return (_struct([lp, w1.idx[0].dag(), l.dag()]), w1, w2, _struct([rp, w2.idx[3].dag(), r.dag()]),
            _struct([l, s1, s2, r]))


def _env_structs(c):
    """the first environment, then per updated site its psi (l, s, r) and its W, in the order of the updates"""
    ws, site = _mpo(c["lattice"], c["sites"])
    n = c["sites"]
    link = functools.partial(_link, m=c["m"], sigma=c["sigma"])
    psis = [_struct([link(INWARD, "ID1Link%d" % (site + i), 0, odd=i % 2), W.site_index(INWARD, "Site%d" % (site + i), 0),
                     link(OUTWARD, "ID1Link%d" % (site + i + 1), 0, odd=(i + 1) % 2)]) for i in range(n)]
    if c["dir"] == 0:
        l = psis[0].idx[0]
        env = _struct([link(INWARD, l.name, 1), ws[0].idx[0].dag(), l.dag()])
    else:
        psis, ws = psis[::-1], ws[::-1]
        r = psis[0].idx[2]
        env = _struct([link(OUTWARD, r.name, 1, odd=n % 2), ws[0].idx[3].dag(), r.dag()])
    return env, psis, ws


def _theta_struct(c):
    """the tensor an SVD case splits, and how many of its indices form the rows"""
    link = functools.partial(_link, m=c["m"], sigma=c["sigma"])
    l, s1, s2 = link(INWARD, "ID1Link4", 0), W.site_index(INWARD, "Site4", 0), W.site_index(INWARD, "Site5", 0)
    if c["kind"] == "svd":
        return _struct([l, s1, s2, link(OUTWARD, "ID1Link6", 0)]), 2
    site = _struct([l, s1, link(OUTWARD, "ID1Link5", 0, odd=1)])
    return site, (1 if c["dir"] else 2)   # moving left splits off the right part, moving right the left part


# the index pairs of operator* for these layouts (position in A, position in B, in B's order)
HEFF_PAIRS = [[(2, 0)], [(1, 0), (2, 1), (3, 3)], [(4, 1), (1, 2)]]
ENV_PAIRS = {0: [[(0, 0)], [(2, 0), (0, 2)], [(1, 0), (2, 1)]], 1: [[(2, 0)], [(1, 2), (2, 3)], [(3, 1), (1, 2)]]}


def _fill(t, seed, k, scale=1.0):
    """t with N(0,1) values times scale"""
    g = torch.Generator("cuda").manual_seed(97 * seed + k)
    data = torch.randn(int(t.block_sizes().sum()), dtype=torch.float64, device="cuda", generator=g)
    return FlatTensor(t.idx, t.block_qi, data.mul_(scale).cpu().numpy())


def _sectors(t, nleft):
    """per mid charge (ascending): {left tuple: row offset}, rows, {right tuple: column offset}, columns"""
    found = {}
    for b in t.block_qi.tolist():
        q = sum((1 if t.idx[j].arrow == INWARD else -1) * t.idx[j].qn[b[j]][0] for j in range(nleft))
        s = found.setdefault(q, (set(), set()))
        s[0].add(tuple(b[:nleft]))
        s[1].add(tuple(b[nleft:]))
    out = []
    for q in sorted(found):
        sides = []
        for side, first in zip(found[q], (0, nleft)):
            off, n = {}, 0
            for key in sorted(side):
                off[key] = n
                n += math.prod(t.idx[first + j].qdim[p] for j, p in enumerate(key))
            sides += [off, n]
        out.append((q, *sides))
    return out


def _theta(c, seed):
    """the tensor of an SVD case.  A site to canonicalise is random; a two-site
    state's sectors have random singular vectors and singular values that fall
    by 13 decades, and the charges away from the middle weigh less"""
    t, nleft = _theta_struct(c)
    if c["kind"] == "canon":
        return _fill(t, seed, 0, 1.0 / math.sqrt(2 * max(t.idx[0].qdim))), nleft
    g = torch.Generator("cuda").manual_seed(97 * seed)
    off, blocks = t.block_offsets(), {tuple(b): i for i, b in enumerate(t.block_qi.tolist())}
    data = torch.zeros(int(off[-1]), dtype=torch.float64, device="cuda")
    for q, left, rows, right, cols in _sectors(t, nleft):
        k = min(rows, cols)
        s = torch.logspace(0, -13, k, dtype=torch.float64, device="cuda") * math.exp(-((q / 2 - 0.3) ** 2) / (4 * c["sigma"] ** 2))
        u, v = (torch.linalg.qr(torch.randn(n, k, dtype=torch.float64, device="cuda", generator=g))[0] for n in (rows, cols))
        mat = (u * s) @ v.t()
        for a, b in itertools.product(left, right):
            i = blocks.get(a + b)
            if i is not None:
                d = t.block_dims(i)
                ls, rs = math.prod(d[:nleft]), math.prod(d[nleft:])
                data[off[i]:off[i + 1]] = mat[left[a]:left[a] + ls, right[b]:right[b] + rs].t().reshape(-1)
    return FlatTensor(t.idx, t.block_qi, (data / data.norm()).cpu().numpy()), nleft


def _heff_inputs(c, seed):
    L, w1, w2, R, x = _bond_structs(c)
    return _fill(L, seed, 1), w1, w2, _fill(R, seed, 2), _fill(x, seed, 3)


def _env_inputs(c, seed):
    env, psis, ws = _env_structs(c)
    return _fill(env, seed, 1), [_fill(p, seed, 2 + i, 1.0 / math.sqrt(2 * max(p.idx[0].qdim))) for i, p in enumerate(psis)], ws


# ------------------------------------------------------------------ the passes
def prepare(case, seed):
    c, kind = case, case["kind"]
    T.init(0)
    st = {"c": c, "out": {}}
    if kind in ("contract", "heff"):
        L, w1, w2, R, x = _heff_inputs(c, seed)
        st["L"], st["x"] = T.DTensor.from_flat(L), T.DTensor.from_flat(x)
        if kind == "heff":
            st["R"] = T.DTensor.from_flat(R)
            st["W"] = T.contract(T.DTensor.from_flat(w1), T.DTensor.from_flat(w2), [(3, 0)])
            st["H"] = T.Heff(st["L"], st["W"], st["R"], st["x"], HEFF_PAIRS, PREC[c["prec"]])
            st["v"] = [st["H"].new_output(), st["H"].new_output()]
    elif kind == "davidson":
        st["ops"] = [P.PTensor.from_flat(t) for t in _heff_inputs(c, seed)]
    elif kind in ("svd", "canon"):
        theta, st["nleft"] = _theta(c, seed)
        st["theta"] = T.DTensor.from_flat(theta)
    elif kind == "env":
        env, psis, ws = _env_inputs(c, seed)
        st["env"], st["psis"], st["ws"] = T.DTensor.from_flat(env), [T.DTensor.from_flat(p) for p in psis], [
            T.DTensor.from_flat(w) for w in ws]
    else:
        st["H"] = P.mpo_heisenberg_nn(c["n"])
        st["sites"] = [P.PTensor.from_flat(t) for t in W.random_mps(c["n"], c["m"], c["sigma"], 1000 * seed)]
    T.sync()
    return st


def _download(st, name, h, f32=False):
    """the tensor with handle h in the state's pinned buffer `name`"""
    rank, nb, n = C.c_int(0), C.c_int(0), C.c_size_t(0)
    T.check(T.lib().ttg_tensor_info(h, C.byref(rank), C.byref(nb), C.byref(n)))
    buf = st["out"].get(name)
    if buf is None or buf.numel() != n.value:
        buf = st["out"][name] = torch.empty(n.value, dtype=torch.float64, pin_memory=True)
    T.check(T.lib().ttg_tensor_download(h, buf.numpy(), n.value))
    return buf.float() if f32 else buf


def run(state):
    st = state
    c = st["c"]
    f32 = c.get("prec", "fp64") != "fp64"
    if c["kind"] == "contract":
        t1 = T.contract(st["L"], st["x"], HEFF_PAIRS[0], PREC[c["prec"]])
        return _download(st, "c", t1.h, f32)
    if c["kind"] == "heff":
        src, norms = st["x"], []
        for i in range(c["steps"]):
            dst = st["v"][i % 2]
            st["H"].apply(src, dst)
            norms.append(dst.norm())
            dst.scale(1.0 / norms[-1])
            src = dst
        return {"y": _download(st, "y", src.h, f32), "norms": np.array(norms, np.float32 if f32 else np.float64)}
    if c["kind"] == "davidson":
        L, w1, w2, R, x0 = st["ops"]
        P.set_precision(PREC[c["prec"]])
        x = x0.copy()
        E, _ = P.PBig(L, w1, w2, R).davidson(x, 2, 1e-12)
        return {"E": E, "x": x.to_flat().data}
    if c["kind"] in ("svd", "canon"):
        K, cutoff = (c["m"], 1e-9) if c["kind"] == "svd" else (0, 0.0)
        u, s, v, uv = (C.c_void_p() for _ in range(4))
        tr, kept = C.c_double(0), C.c_int64(0)
        T.check(T.lib().ttg_svd(st["theta"].h, st["nleft"], c["dir"], cutoff, K, C.byref(u), C.byref(s), C.byref(v),
                                C.byref(tr), C.byref(kept)))
        own = [T.DTensor(h, []) for h in (u, s, v)]
        # vectors are free up to signs: the factors come back as the state they make up, beside S.  The kept
        # weight is the sum the cutoff is applied to
        T.check(T.lib().ttg_contract(u, v, 1, np.array([st["nleft"]], np.int32), np.zeros(1, np.int32), T.FP64, C.byref(uv)))
        own.append(T.DTensor(uv, []))
        return {"uv": _download(st, "uv", uv), "s": _download(st, "s", s), "kept": kept.value, "weight": 1.0 - tr.value}
    if c["kind"] == "env":
        env = st["env"]
        for psi, w in zip(st["psis"], st["ws"]):
            env = T.env_update(psi, env, w, c["dir"], PREC[c["prec"]])
        return _download(st, "env", env.h, f32)
    P.set_precision(T.FP64)
    psi = P.mps_product([i % 2 for i in range(c["n"])])
    for i, t in enumerate(st["sites"]):
        psi.set_tensor(i, t)
    psi.set_center(-1)
    r = P.dmrg(psi, st["H"], c["sweeps"], [c["m"]], [1e-10], [2], 1e-12)
    return {"E": r["E"], "halfsweep_E": r["halfsweep_E"], "bond_E": r["bond_E"]}


# ------------------------------------------------------------------ operations and bytes
def _flux(t, tup, pos, sign):
    return sum(sign * (1 if t.idx[j].arrow == INWARD else -1) * t.idx[j].qn[tup[j]][0] for j in pos)


def _plan(A, B, pairs):
    """operator* on block structures: the result's indices and block tuples in creation order (charge, right, left)
    and, per result block, the (A block, B block) pairs that add up to it"""
    pa, pb = [p for p, _ in pairs], [p for _, p in pairs]
    fa, fb = [j for j in range(A.rank) if j not in pa], [j for j in range(B.rank) if j not in pb]
    qs, amap, bmap = {}, {}, {}
    for i, t in enumerate(A.block_qi.tolist()):
        left = tuple(t[j] for j in fa)
        qs.setdefault(_flux(A, t, fa, 1), (set(), set()))[0].add(left)
        amap.setdefault(left, {})[tuple(t[j] for j in pa)] = i
    for i, t in enumerate(B.block_qi.tolist()):
        right, q = tuple(t[j] for j in fb), _flux(B, t, fb, -1)
        if q in qs:
            qs[q][1].add(right)
        bmap.setdefault(right, {})[tuple(t[j] for j in pb)] = i
    tuples, terms = [], []
    for q in sorted(qs):
        for right in sorted(qs[q][1]):
            for left in sorted(qs[q][0]):
                tuples.append(left + right)
                terms.append([(i, bmap[right][mid]) for mid, i in sorted(amap[left].items()) if mid in bmap[right]])
    idx = [A.idx[j] for j in fa] + [B.idx[j] for j in fb]
    return FlatTensor(idx, np.array(tuples, np.int32).reshape(-1, len(idx)), np.zeros(0)), terms, fa, fb, pa, pb


def _mul_flops(A, B, pairs):
    Cs, terms, _, _, pa, _ = _plan(A, B, pairs)
    size = Cs.block_sizes()
    return Cs, sum(2.0 * size[c] * math.prod(A.idx[j].qdim[A.block_qi[i, j]] for j in pa) for c, tt in enumerate(terms) for i, _ in tt)


def _bond_work(L, w1, w2, R, x):
    w12, _ = _mul_flops(w1, w2, [(3, 0)])
    t1, f1 = _mul_flops(L, x, HEFF_PAIRS[0])
    t2, f2 = _mul_flops(t1, w12, HEFF_PAIRS[1])
    _, f3 = _mul_flops(t2, R, HEFF_PAIRS[2])
    n = sum(int(t.block_sizes().sum()) for t in (L, w12, R, x)) + int(x.block_sizes().sum())
    return n, f1 + f2 + f3


def _n(t):
    return int(t.block_sizes().sum())


def work(case):
    c, kind = case, case["kind"]
    es = 8 if c.get("prec", "fp64") == "fp64" else 4
    if kind == "contract":
        L, _, _, _, x = _bond_structs(c)
        t1, f = _mul_flops(L, x, HEFF_PAIRS[0])
        return {"bytes": 8 * (_n(L) + _n(x) + _n(t1)), "flops": f}
    if kind in ("heff", "davidson"):
        n, f = _bond_work(*_bond_structs(c))
        steps = c["steps"] if kind == "heff" else 3
        return {"bytes": es * n * steps, "flops": f * steps}
    if kind in ("svd", "canon"):
        t, nleft = _theta_struct(c)
        f = sum(4.0 * r * k * min(r, k) + 8.0 * min(r, k) ** 3 for _, _, r, _, k in _sectors(t, nleft))
        return {"bytes": 8 * 3 * _n(t), "flops": f}
    if kind == "env":
        env, psis, ws = _env_structs(c)
        n = f = 0.0
        for psi, w in zip(psis, ws):
            t, bra = env, FlatTensor([ix.dag() for ix in psi.idx], psi.block_qi, psi.data)
            n += _n(env) + _n(psi) + _n(w)
            t, f1 = _mul_flops(bra, env, ENV_PAIRS[c["dir"]][0])
            t, f2 = _mul_flops(t, w, ENV_PAIRS[c["dir"]][1])
            env, f3 = _mul_flops(t, psi, ENV_PAIRS[c["dir"]][2])
            n, f = n + _n(env), f + f1 + f2 + f3
        return {"bytes": es * n, "flops": f}
    # dmrg: three products of each bond's operator (nearest-neighbour MPO, w = 5) and the bond's SVD, on the start's
    # link dimensions; the state is read and written once per half-sweep
    n = f = 0.0
    d = [sum(k for _, k in W.mps_link_sectors(c["n"], b, c["m"], c["sigma"])) for b in range(c["n"] + 1)]
    for b in range(c["n"] - 1):
        l, r = d[b], d[b + 2]
        f += 3 * 2.0 * 4 * (5 * l * l * r + 5 * l * r * r) / 4 + 12.0 * (l + r) ** 3 / 4
        n += 2 * 8.0 * 4 * l * r / 2
    return {"bytes": 2 * c["sweeps"] * n, "flops": 2 * c["sweeps"] * f}


# ------------------------------------------------------------------ the same in plain torch, 64 bits
def _blocks(t):
    """the blocks of a flat tensor (column-major, packed) as device tensors"""
    data, off, out = torch.from_numpy(np.ascontiguousarray(t.data)).cuda(), t.block_offsets(), []
    for b in range(t.nblocks):
        d = t.block_dims(b)
        out.append(data[int(off[b]):int(off[b + 1])].view(*d[::-1]).permute(*range(len(d) - 1, -1, -1)))
    return out


def _pack(blocks):
    return torch.cat([b.permute(*range(b.dim() - 1, -1, -1)).reshape(-1) for b in blocks]).cpu()


def _mul(A, a, B, b, pairs):
    """block product of (structure A, blocks a) and (structure B, blocks b)"""
    Cs, terms, fa, fb, pa, pb = _plan(A, B, pairs)
    mats = {}

    def mat(which, i):   # A block as (free, paired), B block as (paired, free)
        if (which, i) not in mats:
            t, first, then = (a[i], fa, pa) if which == 0 else (b[i], pb, fb)
            mats[which, i] = t.permute(*first, *then).reshape(math.prod(t.shape[j] for j in first), -1)
        return mats[which, i]

    out = []
    for k, tt in enumerate(terms):
        d = Cs.block_dims(k)
        acc = torch.zeros(math.prod(d[:len(fa)]), math.prod(d[len(fa):]), dtype=torch.float64, device="cuda")
        for i, j in tt:
            acc.addmm_(mat(0, i), mat(1, j))
        out.append(acc.view(*d))
    return Cs, out


def _operator(L, w1, w2, R, x):
    """H as a function on x's packed blocks (a device vector)"""
    bl, br = _blocks(L), _blocks(R)
    w12, bw = _mul(w1, _blocks(w1), w2, _blocks(w2), [(3, 0)])
    off, at = x.block_offsets(), {tuple(b): i for i, b in enumerate(x.block_qi.tolist())}

    def apply(v):
        vb = [v[int(off[i]):int(off[i + 1])].view(*x.block_dims(i)[::-1]).permute(3, 2, 1, 0) for i in range(x.nblocks)]
        s, t = _mul(L, bl, x, vb, HEFF_PAIRS[0])
        s, t = _mul(s, t, w12, bw, HEFF_PAIRS[1])
        s, t = _mul(s, t, R, br, HEFF_PAIRS[2])
        y = torch.zeros_like(v)
        for tup, blk in zip(s.block_qi.tolist(), t):
            i = at[tuple(tup)]
            y[int(off[i]):int(off[i + 1])] = blk.permute(3, 2, 1, 0).reshape(-1)
        return y

    return apply, torch.from_numpy(np.ascontiguousarray(x.data)).cuda()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "contract":
        L, _, _, _, x = _heff_inputs(c, seed)
        return _pack(_mul(L, _blocks(L), x, _blocks(x), HEFF_PAIRS[0])[1])
    if kind == "heff":
        H, v = _operator(*_heff_inputs(c, seed))
        norms = []
        for _ in range(c["steps"]):
            v = H(v)
            norms.append(float(v.norm()))
            v = v / norms[-1]
        return {"y": v.cpu(), "norms": np.array(norms)}
    if kind == "davidson":
        # the lowest Ritz pair of the three-dimensional Krylov space, the products' lower triangle symmetrised
        H, v = _operator(*_heff_inputs(c, seed))
        vs = [v / v.norm()]
        vas = [H(vs[0])]
        M = torch.zeros(3, 3, dtype=torch.float64)
        M[0, 0] = vas[0] @ vs[0]
        for n in range(1, 4):
            e, z = torch.linalg.eigh(M[:n, :n])
            z = z[:, 0] * (-1.0 if z[0, 0] < 0 else 1.0)
            x = sum(float(z[k]) * vs[k] for k in range(n))
            if n == 3:
                return {"E": float(e[0]), "x": (x / x.norm()).cpu()}
            q = sum(float(z[k]) * vas[k] for k in range(n)) - float(e[0]) * x
            q = q - sum((q @ w) * w for w in vs)
            vs.append(q / q.norm())
            vas.append(H(vs[n]))
            for k in range(n + 1):
                M[n, k] = M[k, n] = vas[n] @ vs[k]
    if kind in ("svd", "canon"):
        t, nleft = _theta(c, seed)
        bl, at = _blocks(t), {tuple(b): i for i, b in enumerate(t.block_qi.tolist())}
        K, cutoff = (c["m"], 1e-9) if kind == "svd" else (0, 0.0)
        secs, facs = _sectors(t, nleft), []
        for _, left, rows, right, cols in secs:
            m = torch.zeros(rows, cols, dtype=torch.float64, device="cuda")
            for a, b in itertools.product(left, right):
                if a + b in at:
                    blk = bl[at[a + b]]
                    # rows and columns run column-major inside a tuple
                    x = blk.permute(*range(nleft - 1, -1, -1), *range(blk.dim() - 1, nleft - 1, -1))
                    x = x.reshape(math.prod(blk.shape[:nleft]), -1)
                    m[left[a]:left[a] + x.shape[0], right[b]:right[b] + x.shape[1]] = x
            facs.append(torch.linalg.svd(m.cpu(), full_matrices=False))
        every = sorted(((float(s), i) for i, (_, sv, _) in enumerate(facs) for s in sv), key=lambda p: -p[0])
        total, run_, dims, kept = sum(s * s for s, _ in every), 0.0, [0] * len(secs), 0
        for s, i in every:
            run_ += s * s / total
            if s == 0.0 and cutoff:
                break
            dims[i] += 1
            kept += 1
            if (cutoff and 1 - run_ < cutoff) or (K and kept >= K):
                break
        uv = []
        for (_, left, _, right, _), (u, s, vh), k in zip(secs, facs, dims):
            if k:
                m = (u[:, :k] * s[:k]) @ vh[:k]
                for b in sorted(right):
                    for a in sorted(left):
                        d = [t.idx[j].qdim[p] for j, p in enumerate(a + b)]
                        ls, rs = math.prod(d[:nleft]), math.prod(d[nleft:])
                        uv.append(m[left[a]:left[a] + ls, right[b]:right[b] + rs].t().reshape(-1))
        return {"uv": torch.cat(uv), "s": torch.cat([s[:k] for (_, s, _), k in zip(facs, dims)]), "kept": kept, "weight": min(run_, 1.0)}
    if kind == "env":
        env, psis, ws = _env_inputs(c, seed)
        e, be = env, _blocks(env)
        for psi, w in zip(psis, ws):
            bra, bp = FlatTensor([ix.dag() for ix in psi.idx], psi.block_qi, psi.data), _blocks(psi)
            s, t = _mul(bra, bp, e, be, ENV_PAIRS[c["dir"]][0])
            s, t = _mul(s, t, w, _blocks(w), ENV_PAIRS[c["dir"]][1])
            e, be = _mul(s, t, psi, bp, ENV_PAIRS[c["dir"]][2])
        return _pack(be)
    return None
