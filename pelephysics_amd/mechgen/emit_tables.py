"""Emit the constant-memory tables of one mechanism for the table-driven kernels.

The table-driven device code (pelephysics_amd/csrc/chem_table.h) walks these
tables with a uniform (wavefront-wide) index, so every parameter is a scalar
load and the loop body is the same few hundred instructions for all
reactions, instead of one unrolled block per reaction.

Reaction order: elementary, then three-body, then falloff (Troe, then
Lindemann), each group contiguous so the kernels run one loop per group with
no per-reaction branching.  For every reaction:

* ``rxA/rxB/rxE``: k = A T^b exp(-E/T) (SI-mol units; high-pressure for falloff);
* ``rxR[3]``/``rxP[3]``: reactant/product species, repeated for coefficient 2
  or 3, -1 when unused (products only matter for reversible reactions);
* ``rxDelta``: sum(nu') - sum(nu''), the power of refC in the reverse rate;
* ``rxNet[6]``/``rxNu[6]``: net stoichiometry (species, coefficient), -1 unused;
* ``rxEff0/rxEffN`` into ``effK``/``effV``: third-body enhancement (eff - 1)
  per listed species (default efficiency 1);
* falloff: ``foA/foB/foE`` (low-pressure rate, SI-mol) and Troe parameters
  ``troe[4]`` with ``troeT2`` flag;
* ``rxIndex``: position of the reaction in the YAML file (progress-rate and
  sensitivity outputs are reported in YAML order);
* ``spPtr/spRx/spNu``: the same net stoichiometry by species (compressed rows,
  reactions in table order), for kernels that form each species' production
  rate in its own lane.

``kPack`` is a second, compact copy of what one right-hand side reads, laid out
for the group kernels (group_bdf.h), which copy it to LDS as it stands: per
species the NASA7 coefficients of both ranges, per reaction 32 bytes (rate,
species as bytes with NX for an unused place, refC power, flags), the third
bodies and falloff parameters, and the net stoichiometry by species cut into
chunks of 8 terms (``ch``: reaction in 12 bits, coefficient + 8 in 4 bits, an
unused place is reaction NR with coefficient 0; ``spCh``: first chunk of each
species), so that the lanes of a group share the long rows.  Its reaction
order is the table order with the reversible elementary reactions first
(``perm``: position in the tables above), so that a wave's lanes agree on
whether there is a reverse rate.  A mechanism beyond those records (254 species,
4095 reactions) gets no ``kPack``.  QSS mechanisms add the balances' terms in the
same chunks (``qch``, reaction + NR for a reverse rate), by matrix entry, then by
right-hand side (``qRow``: first chunk of each; ``qInit``: the entries' constant
parts), and the elimination as code (``qss_eliminate``).

QSS mechanisms (``NQ`` > 0) index their quasi-steady-state species NS..NS+NQ-1
in ``rxR``/``rxP`` and the thermo tables; ``rxNet`` and ``spPtr`` keep the
transported species only.  Their extra tables:

* ``rxFwdOff``: 1 where the QSS reduction removed the forward direction;
* ``qRx``: the reactions with a QSS species (table order), and per such
  reaction ``qTermPtr`` into the balance terms ``tSlot`` (entry of the QSS
  matrix, or -1 - q for the right-hand side of species q), ``tMul`` (signed
  coefficient), ``tDir`` (0 forward, 1 reverse rate), ``tRow``/``tCol`` (the
  term's species and its coupled species, -1 for production);
* the QSS matrix in ``NSLOT`` entries (``slotInit``: -eps on the structural
  entries, 0 on fill-in) and its elimination without pivoting in a
  fill-reducing order: ``luA/luB/luC`` (A[a] /= A[b] when c < 0, else
  A[a] -= A[b] A[c]), ``fsI/fsS/fsP`` (b[i] -= A[s] b[p]) and, per pivot in
  reverse order, ``bsRow/bsDiag/bsPtr`` with ``bsSlot/bsCol``
  (x[row] = (b[row] - sum A[slot] x[col]) / A[diag]).
"""
from __future__ import annotations

from typing import List

from .emit_hip import _f
from .model import Mechanism, Reaction

MAXR = 3
MAXNET = 6


def ordered(m: Mechanism) -> List[int]:
    el = [j for j, r in enumerate(m.reactions) if r.kind == "elementary"]
    tb = [j for j, r in enumerate(m.reactions) if r.kind == "three-body"]
    ft = [j for j, r in enumerate(m.reactions) if r.kind == "falloff" and r.troe is not None]
    fl = [j for j, r in enumerate(m.reactions) if r.kind == "falloff" and r.troe is None]
    return el + tb + ft + fl


def _expand(stoich) -> List[int]:
    out = []
    for k, nu in sorted(stoich.items()):
        n = int(round(nu))
        if abs(nu - n) > 1e-12 or n < 1:
            raise ValueError("non-integer stoichiometry")
        out += [k] * n
    if len(out) > MAXR:
        raise ValueError("more than 3 reactant/product molecules")
    return out + [-1] * (MAXR - len(out))


class _Tables:
    """Members of the one constant-memory struct of a mechanism: a single base
    address serves every table (one scalar register pair in the kernels)."""

    def __init__(self):
        self.items = []

    def __call__(self, name: str, ctype: str, vals):
        vals = list(vals)
        if not vals:
            vals = ["0" if ctype != "double" else "0.0"]
        self.items.append((name, ctype, vals))

    def emit(self, w, sname: str):
        w(f"struct {sname} {{")
        for name, ctype, vals in self.items:
            w(f"  {ctype} {name}[{len(vals)}];")
        w("};")
        w("")
        w(f"static __constant__ {sname} kTab = {{")
        for name, _, vals in self.items:
            w(f"    /* {name} */ {{{', '.join(vals)}}},")
        w("};")


def qss_elimination(m: Mechanism):
    """Slots of the QSS matrix, their initial values and the elimination
    program (no pivoting, greedy minimum-degree order on the symmetrised
    pattern)."""
    from .model import QSS_EPS
    nq = m.n_qss
    terms = m.qss_terms()
    struct = {(q, q) for q in range(nq)} | {(r, c) for r, c, _, _, _ in terms if c >= 0}
    pat = set(struct)
    left = set(range(nq))
    order = []
    while left:
        def degree(p):
            return len({i for i in left if i != p and ((i, p) in pat or (p, i) in pat)})
        p = min(sorted(left), key=degree)
        order.append(p)
        left.discard(p)
        rows = [i for i in sorted(left) if (i, p) in pat]
        cols = [j for j in sorted(left) if (p, j) in pat]
        for i in rows:
            for j in cols:
                pat.add((i, j))
    slots = sorted(pat, key=lambda e: (order.index(e[0]), order.index(e[1])))
    slot = {e: k for k, e in enumerate(slots)}
    init = [(-QSS_EPS if e in struct else 0.0) for e in slots]
    lu, fs, bs = [], [], []
    done = []
    for p in order:
        rest = [q for q in order if q not in done and q != p]
        rows = [i for i in rest if (i, p) in pat]
        cols = [j for j in rest if (p, j) in pat]
        for i in rows:
            lu.append((slot[(i, p)], slot[(p, p)], -1))
            for j in cols:
                lu.append((slot[(i, j)], slot[(i, p)], slot[(p, j)]))
            fs.append((i, slot[(i, p)], p))
        done.append(p)
    for p in reversed(order):
        later = order[order.index(p) + 1:]
        bs.append((p, slot[(p, p)], [(slot[(p, j)], j) for j in later if (p, j) in pat]))
    return terms, slot, init, lu, fs, bs


CHUNK = 8


class Unpackable(ValueError):
    """A mechanism that the packed tables cannot hold: its header has none, and
    its calls run on the one-lane-per-cell kernels."""


def qss_program(w, lu, fs, bs) -> None:
    """The elimination and the solution of the QSS balances as straight-line
    code: every lane of a group runs it on registers."""
    w("  // QSS balances A x = r, factors and solution in place (no pivoting)")
    w("  PPC_DI static void qss_eliminate(double* A, double* r) {")
    for a, b, c in lu:
        w(f"    A[{a}] /= A[{b}];" if c < 0 else f"    A[{a}] -= A[{b}] * A[{c}];")
    for i, sl, p in fs:
        w(f"    r[{i}] -= A[{sl}] * r[{p}];")
    for row, d, ents in bs:
        for sl, c in ents:
            w(f"    r[{row}] -= A[{sl}] * r[{c}];")
        w(f"    r[{row}] /= A[{d}];")
    w("  }")


def emit_pack(w, m: Mechanism, R: List[Reaction], n_el: int) -> None:
    """The Packed struct and its values (see the module's docstring); R is in
    table order, its first n_el reactions elementary."""
    ns, nx, nr = m.n_species, m.n_species + m.n_qss, len(R)
    if nx > 254 or nr > 4095:
        raise Unpackable("mechanism too large for the packed tables")

    def shape(j):
        r = R[j]
        return (0 if r.reversible else 1, sum(r.reactants.values()) > 2, sum(r.products.values()) > 2, j)

    perm = sorted(range(n_el), key=shape) + list(range(n_el, nr))
    rx, rx_eff, effk, effv = [], [], [], []
    for j in perm:
        r = R[j]
        rr = [nx if k < 0 else k for k in _expand(r.reactants)]
        pp = [nx if k < 0 else k for k in (_expand(r.products) if r.reversible else [-1] * MAXR)]
        d = int(round(r.delta_order()))
        if r.reversible and abs(d) > 100:
            raise Unpackable("reaction order out of range")
        flags = (1 if r.reversible else 0) + (2 if r.fwd_removed else 0)
        rx.append(f"{{{_f(r.rate.A)}, {_f(r.rate.b)}, {_f(r.rate.EaR)}, "
                  f"{{{', '.join(map(str, rr))}}}, {{{', '.join(map(str, pp))}}}, {d if r.reversible else 0}, {flags}}}")
    for r in R[n_el:]:
        e = [(k, v - 1.0) for k, v in sorted(r.efficiencies.items()) if v != 1.0]
        rx_eff.append(f"{{{len(effk)}, {len(e)}}}")
        effk += [str(k) for k, _ in e]
        effv += [_f(v) for _, v in e]
    fo = []
    for r in R:
        if r.kind != "falloff":
            continue
        t = list(r.troe or []) + [0.0] * 4
        fo.append("{" + ", ".join(_f(x) for x in (r.low.A, r.low.b, r.low.EaR, t[0], t[1], t[2], t[3],
                                                  1.0 if r.troe and len(r.troe) == 4 else 0.0)) + "}")
    sp = [f"{{{{{', '.join(_f(x) for x in s.low)}}}, {_f(s.tmid)}, {{{', '.join(_f(x) for x in s.high)}}}, {_f(s.imw)}}}"
          for s in m.all_species]
    pos = {j: i for i, j in enumerate(perm)}
    chunks, first = [], [0]
    for k in range(ns):
        terms = []
        for j, r in enumerate(R):
            v = r.net_stoich().get(k, 0.0)
            if v:
                if v != int(v) or not -8 <= v <= 7:
                    raise Unpackable("net coefficient out of range")
                terms.append((pos[j], int(v)))
        terms.sort()
        for i in range(0, len(terms), CHUNK):
            c = terms[i:i + CHUNK] + [(nr, 0)] * (CHUNK - len(terms[i:i + CHUNK]))
            chunks.append("{" + ", ".join(str(((v + 8) << 12) | j) for j, v in c) + "}")
        first.append(len(chunks))
    qch, qfirst, qinit = [], [], []
    if m.n_qss:
        if any(k >= ns for r in R for k in r.efficiencies):
            raise Unpackable("a QSS species as a third body is not supported")
        terms, slot, init, _, _, _ = qss_elimination(m)
        order = ordered(m)
        yaml_pos = {order[j]: i for j, i in pos.items()}
        qrows = [[] for _ in range(len(slot) + m.n_qss)]
        for q, c, j, d, cf in terms:
            row = len(slot) + q if c < 0 else slot[(q, c)]
            mul = cf if c < 0 or c == q else -cf
            if mul != int(mul) or not -8 <= mul <= 7:
                raise Unpackable("QSS balance coefficient out of range")
            qrows[row].append((yaml_pos[j] + (nr if d else 0), int(mul)))
        if 2 * nr > 4095:
            raise Unpackable("mechanism too large for the packed QSS balances")
        qfirst = [0]
        for t in qrows:
            for i in range(0, len(t), CHUNK):
                c = t[i:i + CHUNK] + [(2 * nr, 0)] * (CHUNK - len(t[i:i + CHUNK]))
                qch.append("{" + ", ".join(str(((v + 8) << 12) | j) for j, v in c) + "}")
            qfirst.append(len(qch))
        qinit = [_f(v) for v in init] + ["QSS_EPS"] * m.n_qss
    rows = [("PackSp", "sp", sp), ("PackRx", "rx", rx), ("PackFo", "fo", fo or ["{}"]),
            ("PackCh", "ch", chunks), ("double", "mw", [_f(s.mw) for s in m.species]),
            ("double", "effV", effv or ["0.0"]), ("PackEff", "eff", rx_eff or ["{0, 0}"]),
            ("unsigned short", "spCh", list(map(str, first))), ("unsigned short", "perm", list(map(str, perm))),
            ("unsigned char", "effK", effk or ["0"])]
    if m.n_qss:
        rows += [("PackCh", "qch", qch), ("double", "qInit", qinit), ("unsigned short", "qRow", list(map(str, qfirst)))]
    w("struct alignas(16) Packed {")
    for t, nm, v in rows:
        w(f"  {t} {nm}[{len(v)}];")
    w("};")
    w("")
    w("static __constant__ Packed kPack = {")
    for _, nm, v in rows:
        w(f"    /* {nm} */ {{{', '.join(v)}}},")
    w("};")
    w("")
    w(f"constexpr int kChunks = {len(chunks)};")


def emit(m: Mechanism, source: str) -> str:
    order = ordered(m)
    R = [m.reactions[j] for j in order]
    n_el = sum(r.kind == "elementary" for r in R)
    n_tb = sum(r.kind == "three-body" for r in R)
    n_troe = sum(r.kind == "falloff" and r.troe is not None for r in R)
    n_lind = sum(r.kind == "falloff" and r.troe is None for r in R)
    ns = m.n_species
    nq = m.n_qss
    L = []
    w = L.append
    w(f"// Generated by pelephysics_amd.mechgen.emit_tables from {source}. Do not edit.")
    w("#pragma once")
    w('#include "../pack.h"')
    w("")
    w("namespace ppc {")
    w("namespace tab {")
    w(f"namespace {m.name}_t {{")
    w("")
    tab = _Tables()
    # thermo
    lo = [c for s in m.all_species for c in s.low]
    hi = [c for s in m.all_species for c in s.high]
    tab("nasaLo", "double", (_f(x) for x in lo))
    tab("nasaHi", "double", (_f(x) for x in hi))
    tab("tmid", "double", (_f(s.tmid) for s in m.all_species))
    tab("mw", "double", (_f(s.mw) for s in m.species))
    tab("imw", "double", (_f(s.imw) for s in m.species))
    # reactions
    tab("rxA", "double", (_f(r.rate.A) for r in R))
    tab("rxB", "double", (_f(r.rate.b) for r in R))
    tab("rxE", "double", (_f(r.rate.EaR) for r in R))
    rr, pp, net, nu, delta, rev = [], [], [], [], [], []
    for r in R:
        rr += _expand(r.reactants)
        pp += _expand(r.products) if r.reversible else [-1] * MAXR
        ns_ = sorted((k, v) for k, v in r.net_stoich().items() if k < ns)
        if len(ns_) > MAXNET:
            raise ValueError("more than 6 species in one reaction")
        net += [k for k, _ in ns_] + [-1] * (MAXNET - len(ns_))
        nu += [_f(v) for _, v in ns_] + ["0.0"] * (MAXNET - len(ns_))
        d = r.delta_order()
        delta.append(str(int(round(d))))
        rev.append("1" if r.reversible else "0")
    tab("rxR", "int", map(str, rr))
    tab("rxP", "int", map(str, pp))
    tab("rxNet", "int", map(str, net))
    tab("rxNu", "double", nu)
    tab("rxDelta", "int", delta)
    tab("rxRev", "int", rev)
    eff0, effn, effk, effv = [], [], [], []
    for r in R:
        eff0.append(str(len(effk)))
        cnt = 0
        if r.has_third_body:
            if r.default_eff != 1.0:
                raise ValueError("default efficiency other than 1 is not supported")
            for k, e in sorted(r.efficiencies.items()):
                if e != 1.0:
                    effk.append(str(k))
                    effv.append(_f(e - 1.0))
                    cnt += 1
        effn.append(str(cnt))
    tab("rxEff0", "int", eff0)
    tab("rxEffN", "int", effn)
    tab("effK", "int", effk)
    tab("effV", "double", effv)
    fo = [r for r in R if r.kind == "falloff"]
    tab("foA", "double", (_f(r.low.A) for r in fo))
    tab("foB", "double", (_f(r.low.b) for r in fo))
    tab("foE", "double", (_f(r.low.EaR) for r in fo))
    tr = [r for r in R if r.kind == "falloff" and r.troe is not None]
    tv = []
    for r in tr:
        t = list(r.troe) + [0.0] * (4 - len(r.troe))
        tv += [_f(x) for x in t]
    tab("troe", "double", tv)
    tab("troeT2", "int", ("1" if len(r.troe) == 4 else "0" for r in tr))
    tab("rxIndex", "int", (str(j) for j in order))
    rows = [[] for _ in range(ns)]
    for jj, r in enumerate(R):
        for k, v in sorted(r.net_stoich().items()):
            if k < ns:
                rows[k].append((jj, v))
    ptr, srx, snu = [0], [], []
    for k in range(ns):
        srx += [str(jj) for jj, _ in rows[k]]
        snu += [_f(v) for _, v in rows[k]]
        ptr.append(len(srx))
    tab("spPtr", "int", map(str, ptr))
    tab("spRx", "int", srx)
    tab("spNu", "double", snu)
    qss_counts = {"NQR": 0, "NSLOT": 1, "NLU": 0, "NFS": 0}
    if nq:
        terms, slot, init, lu, fs, bs = qss_elimination(m)
        pos = {j: jj for jj, j in enumerate(order)}
        tab("rxFwdOff", "int", ("1" if r.fwd_removed else "0" for r in R))
        qrx = sorted(pos[j] for j in m.qss_reactions())
        by_rx = {jj: [] for jj in qrx}
        for q, c, j, d, cf in terms:
            if c < 0:
                sl, mul = -1 - q, cf
            elif c == q:
                sl, mul = slot[(q, q)], cf
            else:
                sl, mul = slot[(q, c)], -cf
            by_rx[pos[j]].append((sl, mul, d, q, c))
        tp, tsl, tmul, tdir, trow, tcol = [0], [], [], [], [], []
        for jj in qrx:
            for sl, mul, d, q, c in by_rx[jj]:
                tsl.append(str(sl))
                tmul.append(_f(mul))
                tdir.append(str(d))
                trow.append(str(q))
                tcol.append(str(c))
            tp.append(len(tsl))
        tab("qRx", "int", map(str, qrx))
        tab("qTermPtr", "int", map(str, tp))
        tab("tSlot", "int", tsl)
        tab("tMul", "double", tmul)
        tab("tDir", "int", tdir)
        tab("tRow", "int", trow)
        tab("tCol", "int", tcol)
        tab("slotInit", "double", (_f(v) for v in init))
        tab("luA", "int", (str(a) for a, _, _ in lu))
        tab("luB", "int", (str(b) for _, b, _ in lu))
        tab("luC", "int", (str(c) for _, _, c in lu))
        tab("fsI", "int", (str(i) for i, _, _ in fs))
        tab("fsS", "int", (str(sl) for _, sl, _ in fs))
        tab("fsP", "int", (str(p) for _, _, p in fs))
        bptr, bsl, bcol = [0], [], []
        for _, _, ents in bs:
            bsl += [str(sl) for sl, _ in ents]
            bcol += [str(c) for _, c in ents]
            bptr.append(len(bsl))
        tab("bsRow", "int", (str(p) for p, _, _ in bs))
        tab("bsDiag", "int", (str(d) for _, d, _ in bs))
        tab("bsPtr", "int", map(str, bptr))
        tab("bsSlot", "int", bsl)
        tab("bsCol", "int", bcol)
        qss_counts = {"NQR": len(qrx), "NSLOT": len(slot), "NLU": len(lu), "NFS": len(fs)}
    tab.emit(w, "Tables")
    w("")
    try:
        emit_pack(w, m, R, n_el)
        packed = True
    except Unpackable as e:
        w(f"// no packed tables: {e}")
        packed = False
    w("")
    w("}  // namespace")
    w("")
    w(f"struct {m.name} {{")
    w(f"  static constexpr int NS = {ns};")
    w(f"  static constexpr int NR = {m.n_reactions};")
    w(f"  static constexpr int NEQ = {ns + 1};")
    w(f"  static constexpr int NQ = {nq}, NX = {ns + nq};")
    w("  static constexpr int " + ", ".join(f"{k} = {v}" for k, v in qss_counts.items()) + ";")
    w(f"  static constexpr int N_EL = {n_el}, N_TB = {n_tb}, N_TROE = {n_troe}, N_LIND = {n_lind};")
    w(f"  static constexpr int MAXR = {MAXR}, MAXNET = {MAXNET};")
    if packed:
        w(f"  static constexpr int NCH = {m.name}_t::kChunks;")
        w(f"  using Packed = {m.name}_t::Packed;")
        w(f"  PPC_DI static const Packed& pack() {{ return {m.name}_t::kPack; }}")
    for nm in ("nasaLo", "nasaHi", "tmid", "mw", "imw", "rxA", "rxB", "rxE", "rxNu", "effV", "foA",
               "foB", "foE", "troe", "spNu"):
        w(f"  PPC_DI static double {nm}_(int i) {{ return {m.name}_t::kTab.{nm}[i]; }}")
    for nm in ("rxR", "rxP", "rxNet", "rxDelta", "rxRev", "rxEff0", "rxEffN", "effK", "troeT2",
               "rxIndex", "spPtr", "spRx"):
        w(f"  PPC_DI static int {nm}_(int i) {{ return {m.name}_t::kTab.{nm}[i]; }}")
    if nq:
        qss_program(w, lu, fs, bs)
        for nm in ("tMul", "slotInit"):
            w(f"  PPC_DI static double {nm}_(int i) {{ return {m.name}_t::kTab.{nm}[i]; }}")
        for nm in ("rxFwdOff", "qRx", "qTermPtr", "tSlot", "tDir", "tRow", "tCol", "luA", "luB", "luC", "fsI",
                   "fsS", "fsP", "bsRow", "bsDiag", "bsPtr", "bsSlot", "bsCol"):
            w(f"  PPC_DI static int {nm}_(int i) {{ return {m.name}_t::kTab.{nm}[i]; }}")
    w("};")
    w("")
    w("}  // namespace tab")
    w("}  // namespace ppc")
    return "\n".join(L) + "\n"
