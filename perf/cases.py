"""What a user of this framework has it do, as cases that can be timed.

Every case goes through the package's public calls on device data with a default
(blocking) context, as a host program does.  Kinds of work, and the ranges `draw` covers:

  tree      one WT() tree of n symbols of 1, 2, 4 or 8 bytes with its WTnode records
            and, where asked, the rank directory over its bits
  wtint     sdsl::wt_int<> construction: tree, rank, select1, select0
  wtquery   batches of rank, access, select, inverse_select, lex_count and
            range_search_2d counts on a wt_int that the program keeps
  bits      rank + select1 + select0 of one bit vector, then a batch of each query
  huff      wt_huff<> over a byte text
  fmbuild   FMIndex(): suffix array, BWT and wt_huff of a DNA text
  fmcount   backward-search counts and ranks on an FM-index that the program keeps
  batch     one run of a kept plan over many uneven byte sequences
  lsel      learned select: models of some vectors, and one batch of answers
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()


def _package():
    name = "wavelet_suffix_fm_index_amd"
    if name not in sys.modules:
        d = os.path.join(ROOT, "wavelet-suffix-fm-index_amd")
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        m = importlib.util.module_from_spec(spec)
        sys.modules[name] = m
        spec.loader.exec_module(m)
    return sys.modules[name]


_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(_package().Context(0))
    return _CTX[0]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one protein-sized sequence: the call's own latency
        {"name": "tree_small", "kind": "tree", "n": 5003, "bytes": 1, "sigma": 20, "dist": "zipf", "rank": False},
        # the byte tree of the levelWT driver: 2^24 Zipf bytes, 8 levels, rank directory
        {"name": "tree_bytes", "kind": "tree", "n": 1 << 24, "bytes": 1, "sigma": 256, "dist": "zipf", "rank": True},
        # a column of 16-bit codes, skewed, at an odd length
        {"name": "wtint_u16", "kind": "wtint", "n": 3000017, "bytes": 2, "levels": 12, "dist": "geometric"},
        # the headline integer tree: 2^28 uint32 symbols below 2^20
        {"name": "wtint_u32", "kind": "wtint", "n": 1 << 28, "bytes": 4, "levels": 20, "dist": "uniform"},
        # values wider than 24 bits (ids, timestamps) in 64-bit words
        {"name": "wtint_u64", "kind": "wtint", "n": 6000011, "bytes": 8, "levels": 40, "dist": "uniform"},
        # a program that keeps a 20-level tree and asks it for a million of each answer
        {"name": "wtint_query", "kind": "wtquery", "n": (1 << 24) + 5, "levels": 20, "nq": 1000000},
        # rank/select over one long bit vector and ten million queries of each kind
        {"name": "bits_2e30", "kind": "bits", "nbits": (1 << 30) + 77, "density": 0.5, "nq": 10000000},
        # wt_huff over text with a natural-language-like spread of byte values
        {"name": "huff_text", "kind": "huff", "n": (1 << 26) + 11, "dist": "zipf", "sigma": 256},
        # the whole FM-index construction over a genome-like text
        {"name": "fm_build", "kind": "fmbuild", "n": (1 << 25) + 3},
        # a million 20-byte reads counted, and as many symbol ranks
        {"name": "fm_count", "kind": "fmcount", "n": 1 << 25, "m": 20, "nq": 1000000},
        # the batched builder: 1024 sequences of 2^10 to 2^22 bytes, alphabets 4, 20, 256
        {"name": "batch_1024", "kind": "batch", "nseq": 1024, "log2_max": 22},
        # learned select: 16 vectors of 2^25 bits built and asked ten million times
        {"name": "learned_select", "kind": "lsel", "nvec": 16, "nbits": 1 << 25, "nq": 10000000},
    ]


def _size(rng, lo, hi):
    """Log-uniform, mostly odd sizes, a power of two now and then."""
    x = int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))
    x = max(lo, min(hi, x))
    return 1 << (x.bit_length() - 1) if rng.random() < 0.15 and (1 << (x.bit_length() - 1)) >= lo else x


def draw(rng):
    kind = rng.choice(["tree", "tree", "wtint", "wtint", "wtquery", "bits", "huff", "fmbuild", "fmcount", "batch", "lsel"])
    if kind == "tree":
        w = rng.choice([1, 1, 2, 4, 8])
        levels = rng.randint(1, 8 if w == 1 else 14 if w == 2 else 20)
        sigma = rng.choice([4, 20, 256]) if w == 1 else (1 << levels) - rng.randint(0, (1 << levels) // 3)
        return {"kind": kind, "n": _size(rng, 1 << 10, 1 << 24), "bytes": w, "sigma": max(2, sigma),
                "dist": rng.choice(["zipf", "uniform"]) if w == 1 else rng.choice(["uniform", "geometric"]),
                "rank": rng.random() < 0.5}
    if kind == "wtint":
        w = rng.choice([1, 2, 4, 4, 8])
        levels = {1: lambda: rng.randint(2, 8), 2: lambda: rng.randint(6, 16), 4: lambda: rng.randint(8, 32),
                  8: lambda: rng.randint(16, 64)}[w]()
        return {"kind": kind, "n": _size(rng, 1 << 12, (1 << 26) if levels <= 24 else 6000011), "bytes": w, "levels": levels,
                "dist": rng.choice(["uniform", "geometric"])}
    if kind == "wtquery":
        return {"kind": kind, "n": _size(rng, 1 << 14, 1 << 25), "levels": rng.randint(4, 24), "nq": _size(rng, 1000, 1000000)}
    if kind == "bits":
        return {"kind": kind, "nbits": _size(rng, 1 << 16, 1 << 30), "density": round(math.exp(rng.uniform(math.log(0.01), math.log(0.9))), 4),
                "nq": _size(rng, 1000, 10000000)}
    if kind == "huff":
        return {"kind": kind, "n": _size(rng, 1 << 14, 1 << 26), "dist": rng.choice(["zipf", "zipf", "uniform", "dna"]),
                "sigma": rng.choice([20, 64, 96, 256])}
    if kind == "fmbuild":
        return {"kind": kind, "n": _size(rng, 1 << 16, 1 << 25)}
    if kind == "fmcount":
        return {"kind": kind, "n": _size(rng, 1 << 18, 1 << 25), "m": rng.randint(8, 32), "nq": _size(rng, 1000, 1000000)}
    if kind == "batch":
        return {"kind": kind, "nseq": _size(rng, 64, 1024), "log2_max": rng.choice([16, 18, 20, 22])}
    return {"kind": kind, "nvec": rng.randint(1, 16), "nbits": _size(rng, 1 << 20, 1 << 25), "nq": _size(rng, 10000, 10000000)}


# ------------------------------------------------------------- device buffers
class _Array:
    """A torch tensor as the package's calls take device arrays."""

    def __init__(self, t, dtype):
        self.t, self.dtype = t, np.dtype(dtype)
        self.ptr = ctypes.c_void_p(t.data_ptr())
        self.size, self.nbytes = t.numel(), t.numel() * t.element_size()


_NP = {torch.uint8: np.uint8, torch.int16: np.uint16, torch.int32: np.uint32, torch.int64: np.uint64}
_TYPESTR = {torch.uint8: "|u1", torch.int32: "<i4", torch.int64: "<i8", torch.float32: "<f4"}


def _array(t):
    return _Array(t, _NP[t.dtype])


def _buf(n, dtype=torch.int64):
    return _array(torch.empty(int(n), dtype=dtype, device="cuda"))


class _Owner:
    """A handle of the library that is given back with its last user."""

    def __init__(self, handle):
        self.h = handle

    def __del__(self):
        try:
            self.h.free()
        except Exception:
            pass


class _Mem:
    """Device memory inside a handle, for torch to look at without a copy."""

    def __init__(self, owner, ptr, n, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": _TYPESTR[dtype], "data": (int(ptr), False),
                                         "version": 2, "strides": None}


def _view(owner, ptr, n, dtype=torch.int64):
    ptr = getattr(ptr, "value", ptr)
    if not n or not ptr:
        return torch.empty(0, dtype=dtype, device="cuda")
    return torch.as_tensor(_Mem(owner, ptr, n, dtype), device="cuda")


def _select_views(owner, s):
    """The samples of one select structure; the rows of its pool for sparse stretches are as many as the order of
    the input makes them, and are seen through their number and index only."""
    sb, nl = int(s.sb), int(s.n_long)
    return {"count": [int(s.arg_cnt), sb, nl],
            "superblock": _view(owner, s.superblock, sb), "mini": _view(owner, s.mini, sb * 64, torch.int32),
            "mini_width": _view(owner, s.mini_width, sb, torch.uint8), "long_index": _view(owner, s.long_index, sb),
            "long_width": _view(owner, s.long_width, sb, torch.uint8)}


# -------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


#: The seed orders the input: its values are the same multiset for every seed, so that the sizes of what is built
#: from it (bits of a Huffman-shaped tree, samples of a select structure) do not change from input to input.
VALUES = 0x5EED2026


def _values(n, nbytes, limit, dist):
    """n values in [0, limit) of one distribution, on the GPU."""
    if dist == "zipf":
        a = torch.from_numpy(_package().gen_zipf_bytes(VALUES, n, 1.1)).cuda()
        return a if limit >= 256 else a % limit
    out = torch.empty(n, dtype={1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}[nbytes], device="cuda")
    g, step = _gen(VALUES), 1 << 26
    for at in range(0, n, step):
        m = min(step, n - at)
        if dist == "geometric":  # most symbols small, a long tail
            mean = max(1.0, min(1e4, limit / 16.0))
            x = torch.rand(m, generator=g, device="cuda").clamp_min_(1e-7).log_().mul_(-mean).to(torch.int64).clamp_(max=limit - 1)
        elif limit > 1 << 62:
            x = torch.randint(-(1 << 63), (1 << 63) - 1, (m,), generator=g, device="cuda")
            x = x & ((1 << 63) - 1) if limit == 1 << 63 else x
        else:
            x = torch.randint(0, limit, (m,), generator=g, device="cuda")
        out[at:at + m] = x.to(out.dtype)
    return out


def _symbols(n, nbytes, limit, dist, seed):
    """n symbols in [0, limit) in an order of the seed's."""
    if dist == "dna":
        return _dna(n, seed)
    return _values(n, nbytes, limit, dist)[torch.randperm(n, generator=_gen(seed), device="cuda")]


def _dna(n, seed):
    """Genome-like text ending in its one 0 byte: segments of 4096 bytes in an order of the seed's."""
    t = torch.from_numpy(_package().gen_dna(VALUES, n)).cuda()
    k = (n - 1) // 4096
    if k > 1:
        t[:k * 4096] = t[:k * 4096].view(k, 4096)[torch.randperm(k, generator=_gen(seed), device="cuda")].reshape(-1)
    return t


def _bits(nbits, density, seed):
    """ceil(nbits/64) words of independent bits, their order the seed's, and a zero padding word."""
    g = _gen(VALUES)
    nw = (nbits + 63) // 64
    w = torch.zeros(nw + 1, dtype=torch.int64, device="cuda")
    step = 1 << 21
    for at in range(0, nw, step):
        m = min(step, nw - at)
        if density == 0.5:
            w[at:at + m] = torch.randint(-(1 << 63), (1 << 63) - 1, (m,), generator=g, device="cuda")
        else:
            b = (torch.rand(m, 64, generator=g, device="cuda") < density).to(torch.int64)
            w[at:at + m] = (b << torch.arange(64, device="cuda")).sum(1)
    if nbits % 64:
        w[nw - 1] &= (1 << (nbits % 64)) - 1
    full = nbits // 64
    w[:full] = w[:full][torch.randperm(full, generator=_gen(seed), device="cuda")]
    return w


def _uniform(lo, hi, n, g):
    """int64 tensor, uniform in [lo, hi]."""
    return torch.randint(int(lo), int(hi) + 1, (n,), generator=g, device="cuda")


def _fm_index(text):
    """(wt_huff of the BWT, BWT, suffix array) of a device text."""
    p, ctx, n = _package(), _ctx(), text.size
    sa = _buf(n)
    bwt = _buf(n, torch.uint8)
    p._check(p.lib().wtg_suffix_array_gpu(ctx.h, text.ptr, n, sa.ptr))
    p._check(p.lib().wtg_bwt_from_sa_gpu(ctx.h, text.ptr, sa.ptr, n, bwt.ptr))
    return ctx.huff_build(bwt, n), bwt, sa


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    p, ctx = _package(), _ctx()
    st = {"case": case}
    if kind == "tree":
        L = p.levels_of_sigma(case["sigma"])
        n = case["n"]
        st["L"] = L
        st["sym"] = _array(_symbols(n, case["bytes"], case["sigma"], case["dist"], seed))
        st["words"] = _buf(p.lib().wtg_levels_words(n, L))
        st["nodes"] = _buf((1 << L) * 5)
        if case["rank"]:
            st["dir"] = _buf(p.lib().wtg_rank9_words(n * L))
    elif kind == "wtint":
        st["sym"] = _array(_symbols(case["n"], case["bytes"], 1 << case["levels"], case["dist"], seed))
    elif kind == "wtquery":
        n, L, nq = case["n"], case["levels"], case["nq"]
        s = _symbols(n, 4, 1 << L, "geometric", seed)
        sym = _array(s)
        torch.cuda.synchronize()
        st["wt"] = _Owner(ctx.wtint_build(sym, n, L))
        g = _gen(seed + 1)
        at = _uniform(0, n - 1, nq, g)
        i, j = torch.sort(torch.stack([_uniform(0, n - 1, nq, g), at]), dim=0)[0]
        c = s[_uniform(0, n - 1, nq, g)].to(torch.int64)
        c2 = s[_uniform(0, n - 1, nq, g)].to(torch.int64)
        st["at"], st["i"], st["j"], st["c"] = (_array(x.contiguous()) for x in (at, i, j, c))
        st["lo"], st["hi"] = _array(torch.minimum(c, c2)), _array(torch.maximum(c, c2))
        counts = torch.bincount(s, minlength=1 << L)
        k = (torch.rand(nq, generator=g, device="cuda", dtype=torch.float64) * counts[c]).to(torch.int64) + 1
        st["k"] = _array(torch.minimum(k, counts[c]))
        st["out"] = {x: _buf(nq) for x in ("rank", "access", "select", "inv_rank", "inv_sym", "lex_rank", "lex_less", "lex_more", "range")}
    elif kind == "bits":
        nbits, nq = case["nbits"], case["nq"]
        st["words"] = _array(_bits(nbits, case["density"], seed))
        g = _gen(seed + 1)
        st["idx"] = _array(_uniform(0, nbits, nq, g))
        st["u"] = torch.rand(nq, generator=g, device="cuda", dtype=torch.float64)
        torch.cuda.synchronize()
        D, s1, s0 = ctx.rank9_select_build(st["words"], nbits)
        ones, zeros = s1.arg_cnt, s0.arg_cnt
        for x in (D, s1, s0):
            x.free()
        st["i1"] = _array((st["u"] * ones).to(torch.int64).clamp_(0, ones - 1) + 1)
        st["i0"] = _array((st.pop("u") * zeros).to(torch.int64).clamp_(0, zeros - 1) + 1)
        st["out"] = {x: _buf(nq) for x in ("rank", "select1", "select0")}
    elif kind == "huff":
        st["text"] = _array(_symbols(case["n"], 1, case["sigma"], case["dist"], seed))
    elif kind == "fmbuild":
        st["text"] = _array(_dna(case["n"], seed))
    elif kind == "fmcount":
        n, m, nq = case["n"], case["m"], case["nq"]
        text = _array(_dna(n, seed))
        st["pats"] = _array(torch.from_numpy(p.gen_patterns(int(seed) + 2, text.t.cpu().numpy(), m, nq).reshape(-1)).cuda())
        g = _gen(seed + 1)
        st["i"] = _array(_uniform(0, n, nq, g))
        st["c"] = _array(text.t[_uniform(0, n - 1, nq, g)].to(torch.int32))
        torch.cuda.synchronize()
        st["wt"] = _Owner(_fm_index(text)[0])
        st["out"] = {x: _buf(nq) for x in ("count", "rank")}
    elif kind == "batch":
        n, sigma, _ = p.gen_batch(VALUES, case["nseq"], 10.0, float(case["log2_max"]), symbols=False)
        each = torch.repeat_interleave(torch.from_numpy(sigma.astype(np.float32)).cuda(), torch.from_numpy(n.astype(np.int64)).cuda())
        st["sym"] = _array(each.mul_(torch.rand(each.numel(), generator=_gen(seed), device="cuda")).floor_().clamp_(max=255).to(torch.uint8))
        del each
        torch.cuda.synchronize()
        st["plan"] = _Owner(p.Batch(ctx, st["sym"], n, sigma))
    else:
        w, _ = p.gen_select_vectors(int(seed) + 1, case["nvec"], case["nbits"])
        ones = np.array([int(np.bitwise_count(r).sum()) for r in w], np.int64)
        w = np.concatenate([w, np.zeros((case["nvec"], 1), np.uint64)], axis=1)
        t = torch.from_numpy(w.view(np.int64)).cuda()
        st["vecs"] = [_array(t[k].clone()) for k in range(case["nvec"])]
        g = _gen(seed + 1)
        v = _uniform(0, case["nvec"] - 1, case["nq"], g)
        most = torch.from_numpy(ones).cuda()[v]
        j = (torch.rand(case["nq"], generator=g, device="cuda", dtype=torch.float64) * most).to(torch.int64)
        st["v"], st["j"] = _array(v.to(torch.int32)), _array(torch.minimum(j, most - 1) + 1)
        st["out"] = {"select": _buf(case["nq"])}
    torch.cuda.synchronize()  # the library's context has a stream of its own
    return st


# ----------------------------------------------------------------------- run
def run(st):
    case = st["case"]
    kind = case["kind"]
    p, ctx = _package(), _ctx()
    L = p.lib()
    if kind == "tree":
        n = case["n"]
        ctx.levels_build(st["sym"], n, st["L"], st["words"], st["nodes"], 1 << st["L"])
        out = {"words": st["words"].t, "nodes": st["nodes"].t}
        if case["rank"]:
            p._check(L.wtg_rank9_build(ctx.h, st["words"].ptr, n * st["L"], st["dir"].ptr))
            out["dir"] = st["dir"].t
        return out
    if kind == "wtint":
        st["wt"] = None
        wt = st["wt"] = _Owner(ctx.wtint_build(st["sym"], case["n"], case["levels"]))
        h = wt.h
        return {"sigma": int(h.sigma), "words": _view(wt, h.words_ptr, (h.nbits + 63) // 64),
                "dir": _view(wt, h.dir_ptr, L.wtg_rank9_words(h.nbits)),
                "select1": _select_views(wt, h.select1().st), "select0": _select_views(wt, h.select0().st)}
    if kind == "wtquery":
        h, nq, o = st["wt"].h.h, case["nq"], st["out"]
        p._check(L.wtg_wtint_rank_batch(ctx.h, h, st["at"].ptr, st["c"].ptr, nq, o["rank"].ptr))
        p._check(L.wtg_wtint_access_batch(ctx.h, h, st["at"].ptr, nq, o["access"].ptr))
        p._check(L.wtg_wtint_select_batch(ctx.h, h, st["k"].ptr, st["c"].ptr, nq, o["select"].ptr))
        p._check(L.wtg_wtint_inverse_select_batch(ctx.h, h, st["at"].ptr, nq, o["inv_rank"].ptr, o["inv_sym"].ptr))
        p._check(L.wtg_wtint_lex_count_batch(ctx.h, h, st["i"].ptr, st["j"].ptr, st["c"].ptr, nq, o["lex_rank"].ptr,
                                             o["lex_less"].ptr, o["lex_more"].ptr))
        p._check(L.wtg_wtint_range_count_batch(ctx.h, h, st["i"].ptr, st["j"].ptr, st["lo"].ptr, st["hi"].ptr, nq,
                                               o["range"].ptr))
        return {k: v.t for k, v in o.items()}
    if kind == "bits":
        nbits, nq, o = case["nbits"], case["nq"], st["out"]
        st["sup"] = None
        D, s1, s0 = ctx.rank9_select_build(st["words"], nbits)
        sup = st["sup"] = [_Owner(x) for x in (D, s1, s0)]
        ctx.rank9_batch(st["words"], D, nbits, st["idx"], o["rank"])
        ctx.select_batch(s1, st["words"], st["i1"], o["select1"])
        ctx.select_batch(s0, st["words"], st["i0"], o["select0"])
        return {"dir": _view(sup[0], D.ptr, L.wtg_rank9_words(nbits)), "s1": _select_views(sup[1], s1.st),
                "s0": _select_views(sup[2], s0.st), "answers": {k: v.t for k, v in o.items()}}
    if kind in ("huff", "fmbuild"):
        st["wt"] = None
        out = {}
        if kind == "huff":
            wt = st["wt"] = _Owner(ctx.huff_build(st["text"], case["n"]))
        else:
            h, bwt, sa = _fm_index(st["text"])
            wt = st["wt"] = _Owner(h)
            out = {"bwt": bwt.t, "sa": sa.t}
        h, s = wt.h, wt.h.shape
        return {**out, "words": _view(wt, h.words_ptr, (h.nbits + 63) // 64 + 1), "dir": _view(wt, h.dir_ptr, L.wtg_rank9_words(h.nbits)),
                "select1": _select_views(wt, h.select1().st), "select0": _select_views(wt, h.select0().st),
                "C": np.array(s.C[:], np.int64), "bv_pos": np.array(s.bv_pos[:s.n_inner], np.int64),
                "bv_pos_rank": np.array(s.bv_pos_rank[:s.n_inner], np.int64), "sym": np.array(s.sym[:s.n_nodes], np.int32),
                "path": np.array(s.path[:], np.uint64).view(np.int64), "path_len": np.array(s.path_len[:], np.int32)}
    if kind == "fmcount":
        h, nq, o = st["wt"].h.h, case["nq"], st["out"]
        p._check(L.wtg_fm_count_batch(ctx.h, h, st["pats"].ptr, case["m"], nq, o["count"].ptr))
        p._check(L.wtg_huff_rank_batch(ctx.h, h, st["i"].ptr, st["c"].ptr, nq, o["rank"].ptr))
        return {k: v.t for k, v in o.items()}
    if kind == "batch":
        plan = st["plan"].h
        plan.run()
        w, nw = ctypes.c_void_p(), ctypes.c_uint64()
        p._check(L.wtg_batch_words(plan.h, ctypes.byref(w), ctypes.byref(nw)))
        return {"words": _view(st["plan"], w, nw.value)}
    st["ls"] = None
    ls = st["ls"] = _Owner(p.LearnedSelect(ctx, st["vecs"], [case["nbits"]] * case["nvec"]))
    ls.h.query(st["v"], st["j"], st["out"]["select"])
    f = [ls.h.info(b) for b in range(case["nvec"])]
    whole = ("ones", "learned", "nknots", "eps", "eps_init", "trained", "lut_log")
    return {"select": st["out"]["select"].t, "models": np.array([[x[k] for k in whole] for x in f], np.int64),
            "loss": np.array([[x["loss_init"], x["loss_final"]] for x in f])}


# ---------------------------------------------------------------------- work
def _supports(nbits):
    """Bytes of rank directory and select samples: 16 per 512 bits, 4 per 64 arguments of either value."""
    return nbits / 512 * 16 + nbits / 64 * 4


def work(case):
    """Every input read once and every output written once; a query reads one 64-byte sector for each
    rank it cannot do without, or the whole structure once where that is less.  No floating-point work."""
    kind = case["kind"]
    if kind == "tree":
        L = max(1, (case["sigma"] - 1).bit_length())
        n = case["n"]
        b = n * case["bytes"] + n * L / 8 + (1 << L) * 40 + (n * L / 512 * 16 if case["rank"] else 0)
    elif kind == "wtint":
        nb = case["n"] * case["levels"]
        b = case["n"] * case["bytes"] + nb / 8 + _supports(nb)
    elif kind == "wtquery":
        n, L, nq = case["n"], case["levels"], case["nq"]
        tree = n * L / 8 + _supports(n * L)
        sectors = nq * 64 * L
        # rank, access, select and inverse_select follow one path, lex_count and range_count two
        b = 6 * min(tree, sectors) + 2 * min(tree, sectors) + nq * 8 * (3 + 2 + 3 + 3 + 6 + 5)
    elif kind == "bits":
        nb, nq = case["nbits"], case["nq"]
        b = nb / 8 + _supports(nb) + 3 * nq * 16 + 3 * min(nb / 8 + _supports(nb), nq * 64 * 2)
    elif kind == "huff":
        h = {"dna": 2.3}.get(case["dist"], math.log2(case["sigma"]))
        nb = case["n"] * (h if case["dist"] != "zipf" else 0.8 * h)
        b = case["n"] + nb / 8 + _supports(nb)
    elif kind == "fmbuild":
        n = case["n"]
        b = n + 8 * n + n + 2.3 * n / 8 + _supports(2.3 * n)
    elif kind == "fmcount":
        n, nq, m = case["n"], case["nq"], case["m"]
        tree = 2.3 * n / 8 * 1.25
        b = nq * (m + 8 + 20) + min(tree, nq * m * 64 * 2.3) + min(tree, nq * 64 * 2.3)
    elif kind == "batch":
        # mean length of 2^U(10, hi), widths 2, 5 and 8 equally often
        hi = case["log2_max"]
        mean = (2.0 ** hi - 2.0 ** 10) / ((hi - 10) * math.log(2))
        b = case["nseq"] * mean * (1 + 5 / 8)
    else:
        nb, nq = case["nvec"] * case["nbits"], case["nq"]
        b = nb / 8 + _supports(nb) + nq * (4 + 8 + 8) + min(nb / 8 + _supports(nb), nq * 64 * 2)
    return {"bytes": float(b), "flops": 0.0}
