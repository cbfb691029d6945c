"""Mechanism code generator: a finite-rate mechanism -> an unrolled HIP production function.

The reference renders its rate fold at build time with every species index and
every per-reaction choice (product or log form, which terms are zero) fixed in
the text (``peregrine/simulator/mixture/chemistry/kernels/finiterate.mako:7-236``).
This generator does the same for gfx950: species indices are literals, so the
concentrations, Gibbs terms and production rates stay in registers; the
numeric rate constants are read from a per-case table at literal offsets,
which the compiler turns into scalar loads.

The structure the code depends on is summarised in a signature string; a case
is run on a compiled mechanism only when its signature matches.
"""

import hashlib
import json

import numpy as np

# the per-reaction row of the constant table
RFIELDS = ("logA", "b", "EaR", "logprA", "prb", "prEaR", "nusum")
W = 4
ROW = len(RFIELDS) + 5 * W  # + fwdorder, reactnu, prodnu, netnu, netnuMW
SCALARS = ("logprefRu", "prefRu", "Rupref", "logcfloor", "expclamp", "troeuc", "troeuhinv", "cfloor")
HEAD = 8
LFCTERMS = 13


class Layout:
    def __init__(self, nr, ntroe, ntb, ns):
        self.nr, self.ntroe, self.ntb, self.ns = nr, ntroe, ntb, ns
        self.rec = HEAD
        self.lfc = HEAD + nr * ROW
        self.tb = self.lfc + ntroe * LFCTERMS
        self.size = self.tb + ntb * (ns + 1)

    def scalar(self, name):
        return SCALARS.index(name)

    def field(self, k, name):
        return self.rec + k * ROW + RFIELDS.index(name)

    def listed(self, k, name, j):
        base = {"fwdorder": 0, "reactnu": 1, "prodnu": 2, "netnu": 3, "netnuMW": 4}[name]
        return self.rec + k * ROW + len(RFIELDS) + base * W + j

    def lfcpoly(self, t, m):
        return self.lfc + t * LFCTERMS + m

    def tbdefeff(self, j):
        return self.tb + j * (self.ns + 1)

    def tbeffdev(self, j, e):
        return self.tb + j * (self.ns + 1) + 1 + e


def _layout(records, sets, ns):
    return Layout(len(records), sum(1 for r in records if r.troe), len(sets), ns)


def pack(records, sets, scalars, ns):
    """The constant table a generated mechanism reads, as float64."""
    L = _layout(records, sets, ns)
    t = np.zeros(L.size)
    for name in SCALARS:
        t[L.scalar(name)] = scalars[name]
    for k, r in enumerate(records):
        for name in RFIELDS:
            t[L.field(k, name)] = getattr(r, name)
        for j, (_, v) in enumerate(r.fwd):
            t[L.listed(k, "fwdorder", j)] = v
        for j, (_, v) in enumerate(r.react):
            t[L.listed(k, "reactnu", j)] = v
        for j, (_, v) in enumerate(r.prod):
            t[L.listed(k, "prodnu", j)] = v
        for j, (_, v, m) in enumerate(r.net):
            t[L.listed(k, "netnu", j)] = v
            t[L.listed(k, "netnuMW", j)] = m
        if r.troe:
            for m, c in enumerate(r.lfcpoly):
                t[L.lfcpoly(r.troeidx, m)] = c
    for j, s in enumerate(sets):
        t[L.tbdefeff(j)] = s.defeff
        for e, (_, dev) in enumerate(s.eff):
            t[L.tbeffdev(j, e)] = dev
    return t


def signature(records, sets, ns):
    """What the generated code fixes: every index, form and zero test it was rendered with."""
    rows = []
    for r in records:
        rows.append(
            dict(
                kind=r.name, rev=r.reversible, prod=r.product, tb=r.tb, troe=r.troeidx, nfc=len(r.fcent),
                fwd=[s for s, _ in r.fwd], react=[[s, int(v)] for s, v in r.react],
                products=[[s, int(v)] for s, v in r.prod], net=[s for s, _, _ in r.net],
                b=r.b != 0.0, EaR=r.EaR != 0.0, prb=r.prb != 0.0, prEaR=r.prEaR != 0.0,
                nusum=int(r.nusum) if float(r.nusum).is_integer() else r.nusum, lfc=len(r.lfcpoly),
            )
        )
    body = dict(ns=ns, reactions=rows, tb=[[s for s, _ in t.eff] for t in sets])
    text = json.dumps(body, sort_keys=True, separators=(",", ":"))
    return f"ns{ns}-nr{len(records)}-" + hashlib.sha256(text.encode()).hexdigest()[:24]


def render(name, records, sets, ns):
    """C++ for the device: the rate state and the production fold of one mechanism."""
    L = _layout(records, sets, ns)
    logform = any(not r.product for r in records)
    product = any(r.product for r in records)
    plainbodies = sorted({r.tb for r in records if r.product and r.thirdbody and not r.falloff})
    logbodies = sorted({r.tb for r in records if r.thirdbody and (r.falloff or not r.product)})
    out = []
    w = out.append
    w(f"// generated by peregrine_amd/mechgen.py: mechanism {name}, {ns} species, {len(records)} reactions")
    w("#pragma once")
    w('#include "../pga_chem.hpp"')
    w("namespace pga {")
    w(f"struct Mech_{name} {{")
    w(f"  static constexpr int NS = {ns};")
    w(f"  static constexpr int NR = {len(records)};")
    w(f"  static constexpr int TABLE = {L.size};")
    w(f'  static constexpr const char *NAME_ = "{name}";')
    w(f'  static constexpr const char *SIGNATURE = "{signature(records, sets, ns)}";')
    w(f"  static constexpr int CFLOOR = {L.scalar('cfloor')};")
    # the rate state, finiterate.mako:136-182: what one temperature and composition fix
    w("  struct Rates {")
    w("    double logT, Tinv, ctot;")
    if logform:
        w(f"    double logprefRuT, logc[{ns}];")
    if product:
        w(f"    double prefRuT, prefRuTinv, cG[{ns}];")
    w(f"    double gRT[{ns}];")
    if sets:
        w(f"    double ctb[{len(sets)}], logtb[{len(sets)}];")
    w("  };")
    w("  __device__ __forceinline__ static void ratestate(const Gas<NS> &g, Constants C, double rho,")
    w("                                                   const double (&Y)[NS], double T, Rates &s) {")
    w("#pragma clang fp contract(off)")
    w("    s.logT = tlog(T);")
    w("    s.Tinv = 1.0 / T;")
    w("    const double logT = s.logT, Tinv = s.Tinv;")
    w("    // the Gibbs polynomials in ln T cancel like the caloric ones: one rounding per operation")
    if logform:
        w(f"    s.logprefRuT = C[{L.scalar('logprefRu')}] - logT;")
    if product:
        w(f"    s.prefRuT = C[{L.scalar('prefRu')}] * Tinv;")
        w(f"    s.prefRuTinv = C[{L.scalar('Rupref')}] * T;")
    w("    double ctot = 0.0;")
    w("#pragma unroll")
    w(f"    for (int n = 0; n < {ns}; n++) {{")
    w("      const double c = rho * Y[n] * g.MWinv(n);")
    w("      ctot += c;")
    w("      s.gRT[n] = gibbs_rt(g, n, logT, Tinv);")
    if logform:
        w(f"      s.logc[n] = fmax(C[{L.scalar('logcfloor')}], tlog(c));")
    if product:
        w("      s.cG[n] = fmax(c, 0.0) * texp(s.gRT[n]);")
    w("    }")
    w("    s.ctot = ctot;")
    _ctb(w, L, sets, plainbodies, logbodies)
    w("  }")
    # the fold, finiterate.mako:185-236: omega and, with WITHD, the destruction rates D
    w("  template <bool WITHD>")
    w("  __device__ __forceinline__ static void fold(Constants C, const Rates &s, double (&omega)[NS],")
    w("                                              double (&D)[NS]) {")
    _fold_prologue(w, L, records, ns, logform, product)
    _fold_reactions(w, L, records)
    w("  }")
    # what the rates at one T share whatever the composition, for the forward-difference columns of
    # implicit chemistry (a species column changes the composition at the same T): each value is the
    # expression ratestate and fold evaluate, so tstate_part + fold_columns give fold's bits
    w(f"  static constexpr int NX = {len(records)};")
    w("  struct TCache {")
    w("    double logT, Tinv;")
    if logform:
        w("    double logprefRuT;")
    if product:
        w(f"    double prefRuT, prefRuTinv, eG[{ns}];")
    w(f"    double gRT[{ns}], kx[{len(records)}];")
    w("  };")
    off = {"logT": 0, "Tinv": 1}
    at = 2
    if logform:
        off["logprefRuT"] = at
        at += 1
    if product:
        off["prefRuT"], off["prefRuTinv"], off["eG"] = at, at + 1, at + 2
        at += 2 + ns
    off["gRT"] = at
    off["kx"] = at + ns
    if ns <= IMPLICIT_NS:
        _tstate_part(w, L, records, ns, off, logform, product)
        _fold_columns(w, L, records, sets, ns, off, logform, product)
    w("  __device__ __forceinline__ static void production(const Gas<NS> &g, Constants C,")
    w("                                                    double rho, const double (&Y)[NS], double T, double (&omega)[NS]) {")
    w("    Rates s;")
    w("    ratestate(g, C, rho, Y, T, s);")
    w("    fold<false>(C, s, omega, omega);")
    w("  }")
    w("};")
    w("}  // namespace pga")
    return "\n".join(out) + "\n"


def _fold_prologue(w, L, records, ns, logform, product):
    w("    // one rounding per written operation, as the oracle evaluates the fold")
    w("#pragma clang fp contract(off)")
    w("    const double logT = s.logT, Tinv = s.Tinv;")
    w("    (void)logT, (void)Tinv;")
    if logform:
        w("    const double logprefRuT = s.logprefRuT;")
    if product:
        w("    const double prefRuT = s.prefRuT, prefRuTinv = s.prefRuTinv;")
        w("    (void)prefRuT, (void)prefRuTinv;")
    w(f"    const double expclamp = C[{L.scalar('expclamp')}];")
    w("    (void)expclamp;")
    if any(r.troe for r in records):
        w("    const double log10e = 0.4342944819032518, ln10 = 2.302585092994046;")
    w("#pragma unroll")
    w(f"    for (int n = 0; n < {ns}; n++) omega[n] = 0.0;")
    w("    if constexpr (WITHD) {")
    w("#pragma unroll")
    w(f"      for (int n = 0; n < {ns}; n++) D[n] = 0.0;")
    w("    }")


def _ctb(w, L, sets, plainbodies, logbodies):
    for j, tb in enumerate(sets):
        if not (j in plainbodies or j in logbodies):
            continue
        w("    {")
        w(f"      double ctbc = C[{L.tbdefeff(j)}] * ctot;")
        for e, (sp, _) in enumerate(tb.eff):
            w(f"      ctbc += C[{L.tbeffdev(j, e)}] * (rho * Y[{sp}] * g.MWinv({sp}));")
        if j in plainbodies:
            w(f"      s.ctb[{j}] = ctbc;")
        if j in logbodies:
            w(f"      s.logtb[{j}] = tlog(fmax(2.2250738585072014e-308, ctbc));")
        w("    }")


def _arrhenius(w, L, k, r):
    w(f"      double lk = C[{L.field(k, 'logA')}];")
    if r.b != 0.0:
        w(f"      lk += C[{L.field(k, 'b')}] * logT;")
    if r.EaR != 0.0:
        w(f"      lk -= C[{L.field(k, 'EaR')}] * Tinv;")


class _Names:
    """What a reaction's rate is written in: the rate state s."""

    def cG(self, sp):
        return f"s.cG[{sp}]"

    def logc(self, sp):
        return f"s.logc[{sp}]"

    def gRT(self, sp):
        return f"s.gRT[{sp}]"

    def ctb(self, j):
        return f"s.ctb[{j}]"

    def logtb(self, j):
        return f"s.logtb[{j}]"


def _reaction_rate(w, L, k, r, kind, x):
    """fwd, rev and rp of reaction k; kind: its T-only value (_cached) read rather than evaluated, each
    the same expression in the same order."""
    if kind == "lk":
        w(f"      double lk = {x.kx(k)};")
    elif kind != "K":
        _arrhenius(w, L, k, r)
    if r.product:
        if r.falloff:
            _logpr(w, L, k, r, x)
            w("      const double pr = texp(fmin(logpr, expclamp));")
            w("      const double pfac = pr / (1.0 + pr);")
        if r.troe:
            _troe_lfc(w, L, r) if kind != "lfc" else w(f"      const double lfc = {x.kx(k)};")
            _troe_use(w)
        if kind == "K":
            w(f"      double K = {x.kx(k)};")
        else:
            w("      double xk = lk;")
            for j, (sp, _) in enumerate(r.react):
                w(f"      xk -= C[{L.listed(k, 'reactnu', j)}] * {x.gRT(sp)};")
            w("      double K = texp(fmin(xk, expclamp));")
        if r.thirdbody and not r.falloff:
            w(f"      K *= {x.ctb(r.tb)};")
        if r.falloff:
            w("      K *= pfac;")
        w("      double fwd = K;")
        for sp, nu in r.react:
            for _ in range(int(nu)):
                w(f"      fwd *= {x.cG(sp)};")
        if r.reversible:
            w("      double rev = K;")
            for _ in range(int(abs(r.nusum))):
                w(f"      rev *= {'prefRuTinv' if r.nusum > 0 else 'prefRuT'};")
            for sp, nu in r.prod:
                for _ in range(int(nu)):
                    w(f"      rev *= {x.cG(sp)};")
        else:
            w("      const double rev = 0.0;")
        w("      const double rp = fwd - rev;")
    else:
        if r.thirdbody and not r.falloff:
            w(f"      lk += {x.logtb(r.tb)};")
        if r.falloff:
            _logpr(w, L, k, r, x)
            w("      const double prexp = texp(-fabs(logpr));")
            w("      lk += fmin(logpr, 0.0) - dlog1p(prexp);")
        if r.troe:
            _troe_lfc(w, L, r) if kind != "lfc" else w(f"      const double lfc = {x.kx(k)};")
            _troe_use(w)
        w("      double lrp = lk;")
        for j, (sp, _) in enumerate(r.fwd):
            w(f"      lrp += C[{L.listed(k, 'fwdorder', j)}] * {x.logc(sp)};")
        if r.reversible:
            first = f"C[{L.field(k, 'nusum')}] * logprefRuT" if r.nusum != 0.0 else "0.0"
            w(f"      double diff = {first};")
            for j, (sp, _, _) in enumerate(r.net):
                w(f"      diff -= C[{L.listed(k, 'netnu', j)}] * ({x.gRT(sp)} + {x.logc(sp)});")
            w("      const double fwd = texp(fmin(lrp, expclamp)), rev = texp(fmin(lrp - diff, expclamp));")
            w("      const double rp = fwd - rev;")
        else:
            w("      const double fwd = texp(fmin(lrp, expclamp)), rev = 0.0;")
            w("      const double rp = fwd;")


def _fold_reactions(w, L, records):
    """The fold's reactions (finiterate.mako:185-236)."""
    x = _Names()
    for k, r in enumerate(records):
        w(f"    {{  // reaction {k}: {r.equation} ({r.name}{', reversible' if r.reversible else ''}, {'product' if r.product else 'log'} form)")
        _reaction_rate(w, L, k, r, None, x)
        for j, (sp, _, nuMW) in enumerate(r.net):
            w(f"      omega[{sp}] += C[{L.listed(k, 'netnuMW', j)}] * rp;")
        w("      if constexpr (WITHD) {")
        for j, (sp, _, nuMW) in enumerate(r.net):
            a = f"-C[{L.listed(k, 'netnuMW', j)}]" if nuMW < 0 else "0.0"
            b = f"C[{L.listed(k, 'netnuMW', j)}]" if nuMW > 0 else "0.0"
            w(f"        D[{sp}] += {a} * fwd + {b} * rev;")
        w("      }")
        w("      (void)rev;")
        w("    }")


class _ColumnNames(_Names):
    """Column v >= 1 of a group, its (v - 1)-th species moved (v = 0: the base): the moved species' values are
    the column's own, the others the base's."""

    def __init__(self, v, moved, off):
        self.v, self.moved, self.off = v, moved, off

    def of(self, name, sp):
        return f"{name}{sp}_{self.v}" if self.v and sp == self.moved else f"{name}{sp}_0"

    def cG(self, sp):
        return self.of("cG", sp)

    def logc(self, sp):
        return self.of("logc", sp)

    def gRT(self, sp):
        return f"X({self.off['gRT'] + sp})"

    def ctb(self, j):
        return f"ctb{j}_{self.v}"

    def logtb(self, j):
        return f"logtb{j}_{self.v}"

    def kx(self, k):
        return f"X({self.off['kx'] + k})"


# the species columns a lane takes beside the base (implicit chemistry's workgroups have a wave a group)
COLUMNS = 3
# the species whose matrices implicit chemistry takes (IM_N less T, pga_implicit.hpp): a mechanism of more has
# no columns
IMPLICIT_NS = 11


def _touches(r, sp):
    """Whether the reaction's rate changes with species sp alone at one T."""
    if r.thirdbody or r.falloff:
        return True
    if r.product:
        return any(s == sp for s, _ in r.react) or (r.reversible and any(s == sp for s, _ in r.prod))
    return any(s == sp for s, _ in r.fwd) or (r.reversible and any(s == sp for s, _, _ in r.net))


def _tstate_part(w, L, records, ns, off, logform, product):
    """One of GROUPS shares of the TCache at T, each value put (put(index, value)) where TCache's member lies."""
    groups = -(-ns // COLUMNS)
    w(f"  static constexpr int COLS = {COLUMNS}, GROUPS = {groups};")
    w("  template <int G, class PUT>")
    w("  __device__ __forceinline__ static void tstate_part(const Gas<NS> &g, Constants C, double T, const PUT &put) {")
    w("#pragma clang fp contract(off)")
    w("    const double logT = tlog(T), Tinv = 1.0 / T;")
    w(f"    double gRT[{ns}];")
    w("#pragma unroll")
    w(f"    for (int n = 0; n < {ns}; n++) gRT[n] = gibbs_rt(g, n, logT, Tinv);")
    w(f"    const double expclamp = C[{L.scalar('expclamp')}];")
    w("    (void)expclamp;")
    for G in range(groups):
        w(f"    if constexpr (G == {G}) {{")
        if G == 0:
            w(f"    put({off['logT']}, logT);")
            w(f"    put({off['Tinv']}, Tinv);")
            if logform:
                w(f"    put({off['logprefRuT']}, C[{L.scalar('logprefRu')}] - logT);")
            if product:
                w(f"    put({off['prefRuT']}, C[{L.scalar('prefRu')}] * Tinv);")
                w(f"    put({off['prefRuTinv']}, C[{L.scalar('Rupref')}] * T);")
        for n in range(G, ns, groups):
            w(f"    put({off['gRT'] + n}, gRT[{n}]);")
            if product:
                w(f"    put({off['eG'] + n}, texp(gRT[{n}]));")
        for k, r in list(enumerate(records))[G::groups]:
            kind = _cached(r)
            at = off["kx"] + k
            if kind is None:
                w(f"    put({at}, 0.0);")
                continue
            w(f"    {{  // reaction {k}: {kind}")
            if kind == "lfc":
                _troe_lfc(w, L, r)
                w(f"      put({at}, lfc);")
            else:
                _arrhenius(w, L, k, r)
                if kind == "lk":
                    w(f"      put({at}, lk);")
                else:
                    w("      double xk = lk;")
                    for j, (sp, _) in enumerate(r.react):
                        w(f"      xk -= C[{L.listed(k, 'reactnu', j)}] * gRT[{sp}];")
                    w(f"      put({at}, texp(fmin(xk, expclamp)));")
            w("    }")
        w("    }")
    w("  }")


def _fold_columns(w, L, records, sets, ns, off, logform, product):
    """The rates at one T of a base composition, omega[0], and with one species moved for each of a group's
    COLUMNS species: ratestate + fold's values of each, a reaction's rate evaluated again only for the
    columns whose species it reads."""
    w("  template <int G, class TC>")
    w("  __device__ __forceinline__ static void fold_columns(Constants K, Constants C, double rho,")
    w("                                                      const double (&Y)[NS], const double (&Yp)[COLS], const TC &X,")
    w("                                                      double (&omega)[COLS + 1][NS]) {")
    w("    // one rounding per written operation, as the oracle evaluates the fold")
    w("#pragma clang fp contract(off)")
    w(f"    const double logT = X({off['logT']}), Tinv = X({off['Tinv']});")
    w("    (void)logT, (void)Tinv;")
    if logform:
        w(f"    const double logprefRuT = X({off['logprefRuT']});")
        w("    (void)logprefRuT;")
    if product:
        w(f"    const double prefRuT = X({off['prefRuT']}), prefRuTinv = X({off['prefRuTinv']});")
        w("    (void)prefRuT, (void)prefRuTinv;")
    w(f"    const double expclamp = C[{L.scalar('expclamp')}];")
    w("    (void)expclamp;")
    if any(r.troe for r in records):
        w("    const double log10e = 0.4342944819032518, ln10 = 2.302585092994046;")
    w("#pragma unroll")
    w("    for (int v = 0; v <= COLS; v++)")
    w("#pragma unroll")
    w(f"      for (int n = 0; n < {ns}; n++) omega[v][n] = 0.0;")

    def species(n, v, y):
        w(f"    const double c{n}_{v} = rho * {y} * K[Gas<NS>::O.MWinv + {n}];")
        if product:
            w(f"    const double cG{n}_{v} = fmax(c{n}_{v}, 0.0) * X({off['eG'] + n});")
        if logform:
            w(f"    const double logc{n}_{v} = fmax(C[{L.scalar('logcfloor')}], tlog(c{n}_{v}));")

    for n in range(ns):
        species(n, 0, f"Y[{n}]")
    for G in range(-(-ns // COLUMNS)):
        moved = list(range(G * COLUMNS, min(ns, (G + 1) * COLUMNS)))
        w(f"    if constexpr (G == {G}) {{  // species {moved[0]} to {moved[-1]}")
        for v, m in enumerate(moved, 1):
            species(m, v, f"Yp[{v - 1}]")
        cols = [_ColumnNames(0, -1, off)] + [_ColumnNames(v, m, off) for v, m in enumerate(moved, 1)]
        for x in cols:
            w(f"    double ctot_{x.v} = 0.0;")
            for n in range(ns):
                w(f"    ctot_{x.v} += {x.of('c', n)};")
        summed, logged = set(), set()
        for k, r in enumerate(records):
            if r.thirdbody or r.falloff:
                # a third body's sums, made where a reaction first reads them
                for x in cols:
                    if r.tb not in summed:
                        w(f"    double ctb{r.tb}_{x.v} = C[{L.tbdefeff(r.tb)}] * ctot_{x.v};")
                        for e, (sp, _) in enumerate(sets[r.tb].eff):
                            w(f"    ctb{r.tb}_{x.v} += C[{L.tbeffdev(r.tb, e)}] * {x.of('c', sp)};")
                    if (r.falloff or not r.product) and r.tb not in logged:
                        w(f"    const double logtb{r.tb}_{x.v} = tlog(fmax(2.2250738585072014e-308, ctb{r.tb}_{x.v}));")
                summed.add(r.tb)
                if r.falloff or not r.product:
                    logged.add(r.tb)
            own = [x for x in cols[1:] if _touches(r, x.moved)]
            for x, takers in [(cols[0], [y for y in cols if y not in own])] + [(x, [x]) for x in own]:
                w(f"    {{  // reaction {k}: {r.equation}")
                _reaction_rate(w, L, k, r, _cached(r), x)
                for y in takers:
                    for j, (sp, _, _) in enumerate(r.net):
                        w(f"      omega[{y.v}][{sp}] += C[{L.listed(k, 'netnuMW', j)}] * rp;")
                w("      (void)rev;")
                w("    }")
        w("    }")
    w("  }")


def _logpr(w, L, k, r, x):
    w(f"      double logpr = {x.logtb(r.tb)} + C[{L.field(k, 'logprA')}];")
    if r.prb != 0.0:
        w(f"      logpr += C[{L.field(k, 'prb')}] * logT;")
    if r.prEaR != 0.0:
        w(f"      logpr -= C[{L.field(k, 'prEaR')}] * Tinv;")


def _troe_lfc(w, L, r, into="const double lfc"):
    """log10 Fcent of a Troe falloff: its fit in ln T (depends on T alone)."""
    if not r.fcent:
        w(f"      {into} = {np.log(np.finfo(np.float64).tiny) * 0.4342944819032518!r};")
    else:
        n = len(r.lfcpoly)
        w(f"      const double tf = (logT - C[{L.scalar('troeuc')}]) * C[{L.scalar('troeuhinv')}];")
        w(f"      double lfcp = C[{L.lfcpoly(r.troeidx, n - 1)}];")
        for m in reversed(range(n - 1)):
            w(f"      lfcp = lfcp * tf + C[{L.lfcpoly(r.troeidx, m)}];")
        w(f"      {into} = lfcp;")


def _troe_use(w):
    w("      const double Cc = -0.4 - 0.67 * lfc, Nn = 0.75 - 1.27 * lfc;")
    w("      const double Aa = logpr * log10e + Cc, Bb = Nn - 0.14 * Aa, B2 = Bb * Bb;")
    w("      lk += lfc * B2 / (B2 + Aa * Aa) * ln10;")


def _troe(w, L, r):
    _troe_lfc(w, L, r)
    _troe_use(w)


def _cached(r):
    """What a reaction's T-only cache slot holds: 'K' (a product-form rate constant with its
    equilibrium exponential), 'lk' (a log-form ln k), 'lfc' (a Troe fit's value) or None."""
    if r.troe and r.fcent:
        return "lfc"
    if r.falloff:
        return None
    return "K" if r.product else "lk"
