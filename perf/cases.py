"""The work this library is timed on: SIP block contractions, permutes, block
operations and (T) energies, through the public entry points of
aces4_amd.sipgpu and aces4_amd.triples.

A case names one pass of a user's program: `prepare` holds what the program
has before the pass (blocks in HBM, planned batches), `run` makes the calls,
`exact` gives the same outputs in plain 64-bit torch.  Blocks are dense FP64,
column-major, with the values and distributions of aces4_amd/workloads.py and
aces4_amd/triples.py.
"""
import itertools
import math

import torch

from aces4_amd import sipgpu as sg
from aces4_amd import triples as tp

# The terms of a coupled-cluster iteration that the workloads use: (labels of
# the result, left and right operand; arrays of the operands).
TERMS = {
    "ladder": ("abij", "abcd", "cdij", "V", "T"),
    "ring": ("aibj", "kbcj", "aick", "W", "U"),
    "hole": ("abij", "abkl", "klij", "T", "H"),
}
KIND = {x: "v" for x in "abcd"} | {x: "o" for x in "ijkl"}
# Array values: normal with this deviation, or uniform in [-0.5, 0.5).
SIGMA = {"V": 0.1, "T": 1e-2, "U": 1e-2, "H": 0.1, "W": None}


def listed():
    return [
        # The smallest call of the SIP's worker: one pair of 10^4-double
        # ladder blocks (M = N = K = 100), contracted on its own.  Launch and
        # latency bound.
        dict(name="contract_small", kind="contract", term="ladder", v="10,10,10,10", o="10,10",
             accumulate=False),
        # One ring block pair (450^3), accumulated into its result block: the
        # unbatched `contract` of a pardo body; all three blocks permuted.
        dict(name="contract_ring", kind="contract", term="ring", v="30,30,30", o="15,15,15",
             accumulate=True),
        # The same contraction with uneven extents through the reference's own
        # symbol on host buffers: what a SIP linked against the library calls.
        dict(name="dropin_contract", kind="dropin", term="ring", v="31,29,30", o="14,15,13"),
        # One large block with odd extents, indices reversed: HBM bound.
        dict(name="permute_large", kind="permute", dims="113,97,109,101", perm="4,3,2,1"),
        # All blocks of an array with uneven segments, transposed as (3,4,1,2)
        # in one launch: the permutes of a whole pardo.
        dict(name="permute_blocks", kind="permute_blocks", v="31,39,37,24,40,10", o="22,17",
             perm="3,4,1,2"),
        # The ladder term of a small molecule, segments of 10: 16 result
        # blocks, 256 pairs of 100^3 in one planned batch.
        dict(name="ladder", kind="batch", term="ladder", v="10,10,10,10", o="10", moduli=0,
             accumulate=True),
        # The ring term with 30/15 blocks, 1728 pairs, 1.8e11 flop.
        dict(name="ring", kind="batch", term="ring", v="30,30,30,30,15,15", o="15,15", moduli=0,
             accumulate=True),
        # A block-sparse ladder term: uneven segments with irreps, a block
        # exists where its segments' irreps cancel.
        dict(name="ladder_sparse", kind="batch", term="ladder", v="35,14,17,18,17,35",
             o="13,14,13", v_irreps="0,0,0,0,0,2", o_irreps="0,0,0", moduli=0, accumulate=False),
        # The ring term in split precision (13 moduli: 1e-12 of the FP64 path).
        dict(name="ring_split", kind="batch", term="ring", v="30,30,30,30,15,15", o="15,15",
             moduli=13, accumulate=True),
        # The whole (T) energy of a system with segments of 20 and 10: pack the
        # blocks' panels, run every box, sum the energy.
        dict(name="triples", kind="triples", v="20,20,20", o="20,10"),
        # The same with uneven segments.
        dict(name="triples_uneven", kind="triples", v="17,18,17,14", o="13,14"),
        # An amplitude update on one large 4-index block: residual scaled into
        # the block, divided by its orbital energies, its energy and norm, and
        # a sub-block taken out and put into another block.
        dict(name="block_update", kind="update", dims="64,62,63,61", cut="30,62,31,40",
             at="17,0,20,11"),
    ]


def _spread(rng, lo, hi):
    """An integer in lo..hi, even in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _text(values):
    return ",".join(str(x) for x in values)


def _ints(text):
    return [int(x) for x in str(text).split(",")]


def draw(rng):
    """One more case of the listed ranges: segments 8..64 for single blocks,
    8..40 inside batches, any permutation."""
    kind = rng.choice(["contract", "contract", "dropin", "permute", "permute_blocks", "batch", "batch",
                       "batch", "split", "triples", "triples", "update"])
    if kind in ("contract", "dropin"):
        term = rng.choice(sorted(TERMS))
        hi = 40 if kind == "dropin" else 64
        c = dict(kind=kind, term=term, v=_text(_spread(rng, 8, hi) for _ in range(4)),
                 o=_text(_spread(rng, 8, hi) for _ in range(4)))
        if kind == "contract":
            c["accumulate"] = rng.random() < 0.5
        return c
    if kind == "permute":
        rank = rng.choice([2, 3, 4, 5, 6])
        n = math.exp(rng.uniform(math.log(2e4), math.log(1e8)))
        dims = [max(2, int(round(n ** (1.0 / rank) * math.exp(rng.uniform(-0.4, 0.4)))))
                for _ in range(rank)]
        perm = list(range(1, rank + 1))
        while perm == sorted(perm):
            rng.shuffle(perm)
        return dict(kind=kind, dims=_text(dims), perm=_text(perm))
    if kind == "permute_blocks":
        perm = [1, 2, 3, 4]
        while perm == sorted(perm):
            rng.shuffle(perm)
        return dict(kind=kind, v=_text(rng.randint(8, 40) for _ in range(rng.randint(2, 6))),
                    o=_text(rng.randint(8, 40) for _ in range(rng.randint(1, 3))), perm=_text(perm))
    if kind in ("batch", "split"):
        term = rng.choice(["ladder", "ring"])
        nv, no = rng.randint(3, 5), rng.randint(1, 3)
        hi = _spread(rng, 9, 34 if term == "ladder" else 30)
        v = [rng.randint(max(6, hi // 2), hi) for _ in range(nv)]
        o = [rng.randint(max(5, hi // 3), max(6, hi // 2)) for _ in range(no)]
        c = dict(kind="batch", term=term, v=_text(v), o=_text(o),
                 moduli=rng.choice([12, 13, 14]) if kind == "split" else 0,
                 accumulate=rng.random() < 0.5)
        if kind == "batch" and rng.random() < 0.3:
            c["v_irreps"] = _text(rng.choice([0, 0, 0, 1, 2, 3]) for _ in v)
            c["o_irreps"] = _text(0 for _ in o)
        return c
    if kind == "triples":
        return dict(kind=kind, v=_text(rng.randint(7, 21) for _ in range(rng.randint(2, 3))),
                    o=_text(rng.randint(6, 15) for _ in range(rng.randint(1, 2))))
    dims = [rng.randint(20, 66) for _ in range(4)]
    cut = [rng.randint(max(1, x // 3), x) for x in dims]
    return dict(kind=kind, dims=_text(dims), cut=_text(cut),
                at=_text(rng.randint(0, x - y) for x, y in zip(dims, cut)))


# ------------------------------------------------------------------- inputs ----

class _Blocks:
    """A blocked array in HBM: `flat` holds the kept blocks one after another,
    each column-major, first block index fastest."""

    def __init__(self, segs, irreps=None):
        self.segs = segs
        irreps = irreps or [[0] * len(s) for s in segs]
        self.offset, n = {}, 0
        for t in itertools.product(*reversed([range(len(s)) for s in segs])):
            blk = tuple(reversed(t))
            keep = 0
            for d, s in enumerate(blk):
                keep ^= irreps[d][s]
            if keep == 0:
                self.offset[blk] = n
                n += math.prod(self.dims(blk))
        self.size, self.flat, self.dev = n, None, None

    def dims(self, blk):
        return [self.segs[d][s] for d, s in enumerate(blk)]

    def fill(self, seed, tag, sigma):
        self.flat = self.dev = _random(self.size, seed, tag, sigma)
        return self

    def addr(self, blk):
        return self.flat.data_ptr() + 8 * self.offset[blk]

    def block(self, blk):
        """The block as a tensor whose indices stand in the block's order."""
        dims = self.dims(blk)
        x = self.flat[self.offset[blk]:self.offset[blk] + math.prod(dims)]
        return x.view(dims[::-1]).permute(*range(len(dims) - 1, -1, -1))

    def dense(self):
        out = torch.empty([sum(s) for s in self.segs], dtype=torch.float64, device="cuda")
        for blk in self.offset:
            at = [sum(s[:i]) for s, i in zip(self.segs, blk)]
            out[tuple(slice(a, a + n) for a, n in zip(at, self.dims(blk)))] = self.block(blk)
        return out


class _Values:
    """A device array of orbital energies, as FusedTriples takes them."""

    def __init__(self, x):
        self.x, self.ptr = x, x.data_ptr()


def _random(n, seed, tag, sigma, lo=-0.5, hi=0.5):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 64 + tag)
    if sigma is None:
        return torch.rand(n, dtype=torch.float64, device="cuda", generator=g) * (hi - lo) + lo
    return torch.randn(n, dtype=torch.float64, device="cuda", generator=g) * sigma


def _pattern(dl, ll, rl):
    code = {x: i + 1 for i, x in enumerate(dict.fromkeys(dl + ll + rl))}
    ptrn, ierr = sg.get_contraction_ptrn(len(dl), len(ll), len(rl), [code[x] for x in dl + ll + rl])
    if ierr:
        raise ValueError("contraction labels %s %s %s" % (dl, ll, rl))
    return [int(x) for x in ptrn]


def _extents(case):
    """Extents of a single contraction's labels, taken in turn."""
    dl, ll, rl = TERMS[case["term"]][:3]
    pool = {"v": iter(_ints(case["v"])), "o": iter(_ints(case["o"]))}
    return {x: next(pool[KIND[x]]) for x in dict.fromkeys(dl + ll + rl)}


def _pair_inputs(case, seed):
    dl, ll, rl, ln, rn = TERMS[case["term"]]
    ext = _extents(case)
    ld, rd, dd = ([ext[x] for x in labels] for labels in (ll, rl, dl))
    return (ld, rd, dd, _random(math.prod(ld), seed, 1, SIGMA[ln]),
            _random(math.prod(rd), seed, 2, SIGMA[rn]), _random(math.prod(dd), seed, 3, 1e-2))


def _batch_arrays(case, seed):
    dl, ll, rl, ln, rn = TERMS[case["term"]]
    segs = {"v": _ints(case["v"]), "o": _ints(case["o"])}
    irr = {k: _ints(case[k + "_irreps"]) if k + "_irreps" in case else [0] * len(segs[k])
           for k in "vo"}

    def arr(labels, tag, sigma):
        return _Blocks([segs[KIND[x]] for x in labels], [irr[KIND[x]] for x in labels]).fill(
            seed, tag, sigma)

    return arr(dl, 3, 1e-2), arr(ll, 1, SIGMA[ln]), arr(rl, 2, SIGMA[rn])


def _batch_pairs(case, D, L, R):
    """(result, left, right) block ids in the SIP's pardo order."""
    dl, ll, rl = TERMS[case["term"]][:3]
    nseg = {"v": len(_ints(case["v"])), "o": len(_ints(case["o"]))}
    summed = [x for x in dict.fromkeys(ll + rl) if x not in dl]
    for db in D.offset:
        idx = dict(zip(dl, db))
        for at in itertools.product(*[range(nseg[KIND[x]]) for x in reversed(summed)]):
            idx.update(zip(reversed(summed), at))
            lb, rb = tuple(idx[x] for x in ll), tuple(idx[x] for x in rl)
            if lb in L.offset and rb in R.offset:
                yield db, lb, rb


def _triples_arrays(case, seed):
    vs, os_ = _ints(case["v"]), _ints(case["o"])
    w = {"V1": _Blocks([vs, vs, vs, os_]).fill(seed, 11, 0.1),
         "V2": _Blocks([os_, vs, os_, os_]).fill(seed, 12, 0.1),
         "T": _Blocks([vs, vs, os_, os_]).fill(seed, 13, 1e-2),
         "v_segs": vs, "o_segs": os_}
    w["e_occ_dev"] = _Values(_random(sum(os_), seed, 21, None, -2.0, -0.3))
    w["e_vir_dev"] = _Values(_random(sum(vs), seed, 22, None, 0.1, 3.0))
    return w


def _update_inputs(case, seed):
    dims = _ints(case["dims"])
    x = _random(math.prod(dims), seed, 1, 1e-2)
    # (a, b, i, j): two virtual, then two occupied orbital energies
    eps = [_random(d, seed, 5 + n, None, *((0.1, 3.0) if n < 2 else (-2.0, -0.3)))
           for n, d in enumerate(dims)]
    return dims, x, eps, _random(x.numel(), seed, 3, 1e-2)


UPDATE_SIGNS = (-1, -1, 1, 1)


def prepare(case, seed):
    sg.init(0)
    kind = case["kind"]
    st = {"kind": kind}
    if kind in ("contract", "dropin"):
        st["ptrn"] = _pattern(*TERMS[case["term"]][:3])
        st["ld"], st["rd"], st["dd"], l, r, d = _pair_inputs(case, seed)
        st["l"], st["r"], st["d"] = (l, r, d) if kind == "contract" else (
            l.cpu().numpy(), r.cpu().numpy(), None)
        st["acc"] = case.get("accumulate", False)
    elif kind == "permute":
        st["dims"], st["perm"] = _ints(case["dims"]), [1] + _ints(case["perm"])
        st["in"] = _random(math.prod(st["dims"]), seed, 1, 1e-2)
        st["out"] = torch.empty_like(st["in"])
    elif kind == "permute_blocks":
        vs, os_ = _ints(case["v"]), _ints(case["o"])
        st["in"] = _Blocks([vs, os_, vs, os_]).fill(seed, 1, 1e-2)
        st["out"] = torch.empty_like(st["in"].flat)
        base, perm = st["out"].data_ptr(), [1] + _ints(case["perm"])
        st["batch"] = sg.PermuteBatch([
            sg.permutation(st["in"].dims(b), perm, st["in"].addr(b), base + 8 * at)
            for b, at in st["in"].offset.items()])
    elif kind == "batch":
        D, L, R = st["arrays"] = _batch_arrays(case, seed)
        ptrn, entries, seen = _pattern(*TERMS[case["term"]][:3]), [], set()
        for db, lb, rb in _batch_pairs(case, D, L, R):
            entries.append(sg.make_contraction(ptrn, L.addr(lb), L.dims(lb), R.addr(rb), R.dims(rb),
                                               D.addr(db), D.dims(db),
                                               accumulate=case["accumulate"] or db in seen))
            seen.add(db)
        torch.cuda.synchronize()
        st["batch"] = sg.Batch(entries, moduli=case["moduli"] or None)
    elif kind == "triples":
        w = st["arrays"] = _triples_arrays(case, seed)
        torch.cuda.synchronize()
        st["plan"] = tp.FusedTriples(w)
        st["e"] = torch.zeros(1, dtype=torch.float64, device="cuda")
        plan = st["plan"]
        st["keep"] = _Destroy(plan)
    else:
        st["dims"], st["x"], st["eps"], st["u"] = _update_inputs(case, seed)
        st["cut"], st["at"] = _ints(case["cut"]), _ints(case["at"])
        st["t"] = torch.empty_like(st["x"])
        st["s"] = torch.empty(math.prod(st["cut"]), dtype=torch.float64, device="cuda")
        st["e"], st["n"] = (torch.zeros(1, dtype=torch.float64, device="cuda") for _ in range(2))
        st["eptr"] = [x.data_ptr() for x in st["eps"]]
    torch.cuda.synchronize()
    return st


class _Destroy:
    """Gives a plan's memory back with the state that holds it."""

    def __init__(self, plan):
        self.plan = plan

    def __del__(self):
        self.plan.destroy()


# --------------------------------------------------------------------- pass ----

def run(st):
    kind = st["kind"]
    if kind == "contract":
        sg.contract(st["ptrn"], st["l"].data_ptr(), st["ld"], st["r"].data_ptr(), st["rd"],
                    st["d"].data_ptr(), st["dd"], accumulate=st["acc"])
        return st["d"]
    if kind == "dropin":
        out, ierr = sg.tensor_block_contract(st["ptrn"], st["l"], st["ld"], st["r"], st["rd"],
                                             st["dd"])
        if ierr:
            raise RuntimeError("ierr %d" % ierr)
        return out
    if kind == "permute":
        sg.permute(st["dims"], st["perm"], st["in"].data_ptr(), st["out"].data_ptr())
        return st["out"]
    if kind == "permute_blocks":
        st["batch"].execute()
        return st["out"]
    if kind == "batch":
        st["batch"].execute()
        return st["arrays"][0].flat
    if kind == "triples":
        sg.block_init(st["e"].data_ptr(), [1], 0.0)
        st["plan"].pack()
        st["plan"].run()
        st["plan"].energy(st["e"].data_ptr())
        return st["e"]
    dims, t, e = st["dims"], st["t"].data_ptr(), st["e"].data_ptr()
    sg.block_init(t, dims, 0.0)
    sg.block_add(t, st["x"].data_ptr(), dims, 2.0)
    sg.block_scale(t, dims, 0.25)
    sg.energy_denominator(dims, t, st["eptr"], UPDATE_SIGNS)
    sg.block_init(e, [1], 0.0)
    sg.energy_sum(dims, st["x"].data_ptr(), t, st["eptr"], UPDATE_SIGNS, 1.0, e)
    sg.block_norm2(t, dims, st["n"].data_ptr())
    sg.block_slice(t, dims, st["s"].data_ptr(), st["cut"], st["at"])
    sg.block_insert(st["u"].data_ptr(), dims, st["s"].data_ptr(), st["cut"], st["at"])
    return {"t": st["t"], "energy": st["e"], "norm2": st["n"], "slice": st["s"], "into": st["u"]}


# --------------------------------------------------------------------- work ----

def work(case):
    """Inputs read once, outputs written once (an accumulated block also read),
    and the multiplications and additions of the products."""
    kind = case["kind"]
    if kind in ("contract", "dropin"):
        dl, ll, rl = TERMS[case["term"]][:3]
        ext = _extents(case)
        size = [math.prod(ext[x] for x in labels) for labels in (ll, rl, dl)]
        d = size[2] * (2 if case.get("accumulate") else 1)
        return {"bytes": 8.0 * (size[0] + size[1] + d),
                "flops": 2.0 * math.prod(ext.values())}
    if kind == "permute":
        return {"bytes": 16.0 * math.prod(_ints(case["dims"])), "flops": 0.0}
    if kind == "permute_blocks":
        return {"bytes": 16.0 * (sum(_ints(case["v"])) * sum(_ints(case["o"]))) ** 2, "flops": 0.0}
    if kind == "batch":
        dl, ll, rl = TERMS[case["term"]][:3]
        segs = {"v": _ints(case["v"]), "o": _ints(case["o"])}
        irr = {k: _ints(case[k + "_irreps"]) if k + "_irreps" in case else [0] * len(segs[k])
               for k in "vo"}
        D, L, R = (_Blocks([segs[KIND[x]] for x in labels], [irr[KIND[x]] for x in labels])
                   for labels in (dl, ll, rl))
        summed = [n for n, x in enumerate(ll) if x not in dl]
        flops = sum(2.0 * math.prod(D.dims(db)) * math.prod(L.dims(lb)[n] for n in summed)
                    for db, lb, rb in _batch_pairs(case, D, L, R))
        return {"bytes": 8.0 * (L.size + R.size + D.size * (2 if case["accumulate"] else 1)),
                "flops": flops}
    if kind == "triples":
        v, o = sum(_ints(case["v"])), sum(_ints(case["o"]))
        return {"bytes": 8.0 * (v ** 3 * o + v * o ** 3 + v * v * o * o + v + o),
                "flops": 12.0 * v ** 3 * o ** 3 * (v + o)}
    n, cut = math.prod(_ints(case["dims"])), math.prod(_ints(case["cut"]))
    # x read, t written; t read back for the energy, the norm and the slice;
    # the slice written, read and put into the other block
    return {"bytes": 8.0 * (2 * n + 4 * cut), "flops": 20.0 * n}


# -------------------------------------------------------------------- exact ----

def _view(flat, dims):
    return flat.view(dims[::-1]).permute(*range(len(dims) - 1, -1, -1))


def _flat(x):
    """A tensor in block order as its column-major values."""
    return x.permute(*range(x.dim() - 1, -1, -1)).contiguous().view(-1)


def _product(dl, ll, rl, L, R):
    """sum over the shared labels of L and R as a tensor in dl's order."""
    lf, rf = [x for x in ll if x in dl], [x for x in rl if x in dl]
    sm = [x for x in ll if x not in dl]
    a = L.permute(*[ll.index(x) for x in lf + sm]).contiguous()
    b = R.permute(*[rl.index(x) for x in sm + rf]).contiguous()
    m, n = list(a.shape[:len(lf)]), list(b.shape[len(sm):])
    c = torch.matmul(a.view(math.prod(m), -1), b.view(-1, math.prod(n))).view(m + n)
    return c.permute(*[(lf + rf).index(x) for x in dl])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("contract", "dropin"):
        dl, ll, rl = TERMS[case["term"]][:3]
        ld, rd, dd, l, r, d = _pair_inputs(case, seed)
        c = _flat(_product(dl, ll, rl, _view(l, ld), _view(r, rd)))
        if kind == "dropin":
            return c.cpu().numpy()
        return c + d if case["accumulate"] else c
    if kind == "permute":
        dims, perm = _ints(case["dims"]), _ints(case["perm"])
        x = _view(_random(math.prod(dims), seed, 1, 1e-2), dims)
        return _flat(x.permute(*[perm.index(n + 1) for n in range(len(dims))]))
    if kind == "permute_blocks":
        vs, os_ = _ints(case["v"]), _ints(case["o"])
        A = _Blocks([vs, os_, vs, os_]).fill(seed, 1, 1e-2)
        perm = _ints(case["perm"])
        return torch.cat([_flat(A.block(b).permute(*[perm.index(n + 1) for n in range(4)]))
                          for b in A.offset])
    if kind == "batch":
        dl, ll, rl = TERMS[case["term"]][:3]
        D, L, R = _batch_arrays(case, seed)
        sums = {}
        for db, lb, rb in _batch_pairs(case, D, L, R):
            c = _product(dl, ll, rl, L.block(lb), R.block(rb))
            sums[db] = sums[db] + c if db in sums else c
        for db, c in sums.items():
            D.block(db).copy_(D.block(db) + c if case["accumulate"] else c)
        return D.flat
    if kind == "triples":
        return _exact_triples(case, seed)
    dims, x, eps, u = _update_inputs(case, seed)
    X = _view(x, dims)
    den = torch.zeros(dims, dtype=torch.float64, device="cuda")
    for n in (2, 3, 0, 1):
        shape = [1] * 4
        shape[n] = dims[n]
        den = den + UPDATE_SIGNS[n] * eps[n].view(shape)
    t = 0.5 * X / den
    box = tuple(slice(a, a + n) for a, n in zip(_ints(case["at"]), _ints(case["cut"])))
    into = _view(u, dims).clone()
    into[box] = t[box]
    return {"t": _flat(t), "energy": (X / den * t).sum().reshape(1),
            "norm2": t.square().sum().reshape(1), "slice": _flat(t[box]), "into": _flat(into)}


def _exact_triples(case, seed):
    """E = sum W^2 / D over all of W, one (i, j, k) at a time:
    W_ijk(a,b,c) = sum over the permutations of the pairs (a,i), (b,j), (c,k) of
    sum_d V1(b,c,d,k) T(a,d,i,j) + sum_l V2(l,c,j,k) T(a,b,i,l)."""
    w = _triples_arrays(case, seed)
    V1, V2, T = (w[k].dense() for k in ("V1", "V2", "T"))
    eo, ev = w["e_occ_dev"].x, w["e_vir_dev"].x
    v, o = ev.numel(), eo.numel()
    V1 = V1.permute(3, 2, 0, 1).reshape(o, v, v * v).contiguous()   # k, d, (b c)
    Td = T.permute(2, 3, 0, 1).contiguous()                         # i, j, a, d
    Tl = T.permute(2, 0, 1, 3).reshape(o, v * v, o).contiguous()    # i, (a b), l
    V2 = V2.permute(2, 3, 0, 1).contiguous()                        # j, k, l, c
    dv = ev.view(v, 1, 1) + ev.view(1, v, 1) + ev.view(1, 1, v)
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    for i in range(o):
        for j in range(i + 1):
            for k in range(j + 1):
                occ, W = (i, j, k), None
                for p in itertools.permutations(range(3)):
                    x, y, z = (occ[n] for n in p)
                    m = torch.matmul(Td[x, y], V1[z]).view(v, v, v)
                    m += torch.matmul(Tl[x], V2[y, z]).view(v, v, v)
                    # m's indices belong to the pairs p[0], p[1], p[2]
                    m = m.permute(*[p.index(n) for n in range(3)])
                    W = m.clone() if W is None else W.add_(m)
                # W of a permuted (i, j, k) is W with its virtual indices permuted
                same = len({*itertools.permutations(occ)})
                total += same * (W.square() / (eo[i] + eo[j] + eo[k] - dv)).sum()
    return total.reshape(1)
