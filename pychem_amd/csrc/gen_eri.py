"""Generate straight-line HIP code for the integral classes (eri_classes.inc).

For every shell-quartet class (la lb | lc ld) with s..d shells -- each pair in
"primary first" orientation (the VRR runs on the shell of larger l, as the
reference's goofy handling does, Methods/integrals.py:79-85) and the bra
pair class >= the ket pair class -- it emits one kernel:

  * loop over bra and ket primitive pairs (runtime trip counts),
  * Boys F_0..F_L, then the Obara-Saika VRR of only the [e0|f0]^(m) terms the
    targets need (ket first, then bra with the cross term; the same
    recurrences as Methods/c_ints/two_electron_vrr.c:92-109, written in the
    unscaled form), as named scalars so they live in registers,
  * contraction of the m=0 targets into per-thread accumulators,
  * HRR on contracted classes (ket then bra, Methods/c_ints/two_electron_hrr.c:82),
  * per-Cartesian-component normalisation (Util/structures.py:850-856) and a
    coalesced store: out[component * nq + quartet].

It also emits one one-electron kernel per pair class (S, T, V; the reference's
Methods/integrals.py:220-370 path: overlap VRR/HRR to (a|b+2), kinetic by the
derivative formula of Methods/c_ints/one_electron_kinetic.c:60-64, nuclear
VRR/HRR per atom).

Run: python pychem_amd/csrc/gen_eri.py   (writes eri_classes.inc next to it)
"""
import math
import os
import re
from fractions import Fraction

PAIRS = [(0, 0), (1, 0), (1, 1), (2, 0), (2, 1), (2, 2)]   # pair classes (primary, secondary)
CLASSES = [(X, Y) for X in range(len(PAIRS)) for Y in range(X + 1)]


def comps(l):
    return [(lx, ly, l - lx - ly) for lx in range(l, -1, -1) for ly in range(l - lx, -1, -1)]


def lev(c):
    return c[0] + c[1] + c[2]


def axis(c):
    return 0 if c[0] else (1 if c[1] else 2)


def dec(c, i, k=1):
    c = list(c); c[i] -= k; return tuple(c)


def inc(c, i):
    c = list(c); c[i] += 1; return tuple(c)


def nm(c):
    return "%d%d%d" % c


def cnorm(c):
    return 1.0 / math.sqrt(math.gamma(c[0] + 0.5) * math.gamma(c[1] + 0.5) * math.gamma(c[2] + 0.5))


XYZ = "xyz"


class Emitter:
    def __init__(self, indent="      "):
        self.lines = []
        self.done = set()
        self.ind = indent

    def emit(self, s):
        self.lines.append(self.ind + s)


def gen_eri_class(la, lb, lc, ld, asel=None, csel=None, suffix=""):
    """Device function eri_body_<tag><suffix>: the outputs (a b | c d) with a
    in ``asel`` and c in ``csel`` (default: all), each stored at its index in
    the class's full component order.  The VRR accumulators are only the
    [e0|f0] those outputs' HRR reaches."""
    emax, fmax = la + lb, lc + ld
    L = emax + fmax
    tag = "%d%d%d%d" % (la, lb, lc, ld)
    asel = comps(la) if asel is None else asel
    csel = comps(lc) if csel is None else csel
    em = Emitter()

    flops = {"vrr": 0, "contract": 0, "hrr": 0}
    terms = {}           # summands of each recurrence

    def vrr(e, f, m):
        # flops priced as the reference's two_electron_vrr.c:92-109: 6 for the
        # base terms, +5 with the a-term, +4 with the cross term
        key = (e, f, m)
        name = "v%s_%s_%d" % (nm(e), nm(f), m)
        if key in em.done:
            return name
        if lev(e) == 0 and lev(f) == 0:
            expr = "pref * F[%d]" % m
        elif lev(e) == 0:
            i = axis(f)
            f1 = dec(f, i)
            t = ["QC%s * %s" % (XYZ[i], vrr(e, f1, m)), "WQ%s * %s" % (XYZ[i], vrr(e, f1, m + 1))]
            flops["vrr"] += 6
            if f1[i] > 0:
                f2 = dec(f1, i)
                t.append("(real)%d * oo2q * (%s - rho_q * %s)" % (f1[i], vrr(e, f2, m), vrr(e, f2, m + 1)))
                flops["vrr"] += 5
            expr = " + ".join(t)
        else:
            i = axis(e)
            e1 = dec(e, i)
            t = ["PA%s * %s" % (XYZ[i], vrr(e1, f, m)), "WP%s * %s" % (XYZ[i], vrr(e1, f, m + 1))]
            flops["vrr"] += 6
            if e1[i] > 0:
                e2 = dec(e1, i)
                t.append("(real)%d * oo2p * (%s - rho_p * %s)" % (e1[i], vrr(e2, f, m), vrr(e2, f, m + 1)))
                flops["vrr"] += 5
            if f[i] > 0:
                t.append("(real)%d * oo2pq * %s" % (f[i], vrr(e1, dec(f, i), m + 1)))
                flops["vrr"] += 4
            expr = " + ".join(t)
        em.emit("const real %s = %s;" % (name, expr))
        em.done.add(key)
        if not (lev(e) == 0 and lev(f) == 0):
            terms[name] = t
        return name

    def reach(a, b):     # the [e0| components the bra HRR of (a b| reads
        if lev(b) == 0:
            return {a}
        i = axis(b)
        return reach(inc(a, i), dec(b, i)) | reach(a, dec(b, i))
    eneed = set().union(*[reach(a, b) for a in asel for b in comps(lb)])
    fneed = set().union(*[reach(c, d) for c in csel for d in comps(ld)])
    ecomps = [c for l in range(la, emax + 1) for c in comps(l) if c in eneed]
    fcomps = [c for l in range(lc, fmax + 1) for c in comps(l) if c in fneed]
    acc_names = {}
    for e in ecomps:
        for f in fcomps:
            acc_names[(e, f)] = "c%s_%s" % (nm(e), nm(f))
    # primitive-quartet body; a target no other recurrence reads is added to
    # its accumulator term by term, each a fused multiply-add
    targets = {}
    for e in ecomps:
        for f in fcomps:
            targets[vrr(e, f, 0)] = acc_names[(e, f)]
            flops["contract"] += 3   # two_electron_contract.c:45
    read = {w for l in em.lines for w in re.findall(r"v\w+", l.split(" = ")[1])}
    body = []
    for line in em.lines:
        v = line.split(" = ")[0].split()[-1]
        if v in targets and v in terms and v not in read:
            body += ["%s%s += %s;" % (em.ind, targets[v], t) for t in terms[v]]
        else:
            body.append(line)
            if v in targets:
                body.append("%s%s += %s;" % (em.ind, targets[v], v))
    nbody = len(em.lines) + len(targets)

    # HRR (post loop)
    hr = Emitter(indent="  ")

    def ket(e, c, d):
        if lev(d) == 0:
            return acc_names[(e, c)]
        key = ("k", e, c, d)
        name = "k%s_%s_%s" % (nm(e), nm(c), nm(d))
        if key in hr.done:
            return name
        i = axis(d)
        d1 = dec(d, i)
        expr = "%s + CD%s * %s" % (ket(e, inc(c, i), d1), XYZ[i], ket(e, c, d1))
        flops["hrr"] += 2   # two_electron_hrr.c:82
        hr.emit("const real %s = %s;" % (name, expr))
        hr.done.add(key)
        return name

    def bra(a, b, c, d):
        if lev(b) == 0:
            return ket(a, c, d)
        key = ("b", a, b, c, d)
        name = "h%s_%s_%s_%s" % (nm(a), nm(b), nm(c), nm(d))
        if key in hr.done:
            return name
        i = axis(b)
        b1 = dec(b, i)
        expr = "%s + AB%s * %s" % (bra(inc(a, i), b1, c, d), XYZ[i], bra(a, b1, c, d))
        flops["hrr"] += 2
        hr.emit("const real %s = %s;" % (name, expr))
        hr.done.add(key)
        return name

    idx = 0
    for a in comps(la):
        for b in comps(lb):
            for c in comps(lc):
                for d in comps(ld):
                    if a in asel and c in csel:
                        v = bra(a, b, c, d)
                        nrm = cnorm(a) * cnorm(b) * cnorm(c) * cnorm(d)
                        hr.emit("out[(size_t)%d * nq + q] = (real)(%s * (real)%.17g);" % (idx, v, nrm))
                    idx += 1
    ncomp = idx

    lines = []
    lines.append("template <typename real, int OP = 0>")
    lines.append("__device__ __forceinline__ void eri_body_%s%s(const EriArgs<real>& args, const int t, "
                 "const double* __restrict__ btab)" % (tag, suffix))
    lines.append("{")
    lines.append("  const int nq = args.nq;")
    lines.append("  if (t >= nq) return;")
    lines.append("  const int q = args.order ? (int)min((unsigned)args.order[t], (unsigned)(nq - 1)) : t;")
    lines.append("  const int2 pr = args.quartets[q];")
    lines.append("  const PairHdr bh = args.pairs[pr.x];")
    lines.append("  const PairHdr kh = args.pairs[pr.y];")
    lines.append("  real * __restrict__ out = args.out;")
    for n in acc_names.values():
        lines.append("  real %s = 0;" % n)
    # Ket primitive pairs in the outer loop, bra pairs in the inner one: the
    # quartet lists run over the kets of one bra, so the lanes of a wave
    # mostly share the bra.  For the light classes, whose few VALU
    # operations per primitive quartet left them bound by the vector-memory
    # path, a wave whose lanes all have one bra reads its primitive pairs
    # with scalar loads (the bra index is wave-uniform there); other waves
    # take the per-lane loads.
    def loops(uniform):
        out = ["  for (int j = 0; j < kh.n; ++j) {",
               "    const PrimPair<double> Q = args.prims[kh.off + j];"]
        if uniform:
            out += ["    for (int i = 0; i < bn; ++i) {",
                    "      const PrimPair<double> P = prim_ld_u(bp + i);"]
        else:
            out += ["    for (int i = 0; i < bh.n; ++i) {",
                    "      const PrimPair<double> P = args.prims[bh.off + i];"]
        out.append("      ERI_PRIM_SETUP(%d)" % L)
        out.extend(body)
        out += ["    }", "  }"]
        return out

    if nbody <= UNIFORM_MAX_BODY:
        lines.append("  if (__all(pr.x == __builtin_amdgcn_readfirstlane(pr.x))) {")
        lines.append("    const int bn = __builtin_amdgcn_readfirstlane(bh.n);")
        lines.append("    const ERI_CONST PrimPair<double>* __restrict__ bp =")
        lines.append("        (const ERI_CONST PrimPair<double>*)args.prims + __builtin_amdgcn_readfirstlane(bh.off);")
        lines.extend(["  " + x for x in loops(True)])
        lines.append("  } else {")
        lines.extend(["  " + x for x in loops(False)])
        lines.append("  }")
    else:
        lines.extend(loops(False))
    lines.append("  const real ABx = (real)bh.ab[0], ABy = (real)bh.ab[1], ABz = (real)bh.ab[2];")
    lines.append("  const real CDx = (real)kh.ab[0], CDy = (real)kh.ab[1], CDz = (real)kh.ab[2];")
    lines.append("  (void)ABx; (void)ABy; (void)ABz; (void)CDx; (void)CDy; (void)CDz;")
    lines.extend(hr.lines)
    lines.append("}")
    gen_eri_class.flops = dict(flops, boys=L + 1)
    gen_eri_class.naccum = len(acc_names)
    return "\n".join(lines), ncomp, nbody


# Classes whose one-thread-per-quartet kernel would hold too many [e0|f0]
# accumulators (31 x 31 for (dd|dd)) and spill: their outputs are split into
# groups of primary components, (bra groups, ket groups) below, one group
# per wave (blockIdx.y), each keeping only the accumulators its own HRR
# reaches (e.g. (dd|dd): 100 instead of 961) at the price of repeating part
# of the VRR in every group.
SPLIT = {"2111": (6, 1), "2121": (1, 6), "2211": (6, 3), "2220": (1, 6), "2221": (6, 6), "2222": (6, 6)}


def split_groups(la, lc, na, nc):
    return [(comps(la)[i::na], comps(lc)[k::nc]) for i in range(na) for k in range(nc)]


# Occupancy floor per class kernel (waves per SIMD, the second argument of
# __launch_bounds__); 1 leaves the register count to the compiler.
MINW = {"2020": 2, "2220": 2, "2110": 2}   # measured on C20H42/6-31G*: 0.087 -> 0.067 ms, 0.085 -> 0.064 ms

# classes with at most this many VRR/contraction lines per primitive quartet
# get the scalar-load path for wave-uniform bras
UNIFORM_MAX_BODY = 100


def gen_eri_class_split(la, lb, lc, ld):
    """The class's device function(s): eri_body_<tag> dispatching on the
    output group (blockIdx.y) when the class is split, else the whole body.
    Returns (code, components, body lines of the largest group, groups,
    flop model of the whole class, largest accumulator count)."""
    tag = "%d%d%d%d" % (la, lb, lc, ld)
    code_full, ncomp, nbody = gen_eri_class(la, lb, lc, ld)
    flops = gen_eri_class.flops
    if tag not in SPLIT:
        return code_full, ncomp, nbody, 1, flops, gen_eri_class.naccum
    na, nc = SPLIT[tag]
    parts, worst, wbody = [], 0, 0
    groups = split_groups(la, lc, na, nc)
    for g, (asel, csel) in enumerate(groups):
        code, _, nb = gen_eri_class(la, lb, lc, ld, asel, csel, suffix="_g%d" % g)
        parts.append(code)
        worst = max(worst, gen_eri_class.naccum)
        wbody = max(wbody, nb)
    disp = ["template <typename real, int OP = 0>",
            "__device__ __forceinline__ void eri_body_%s(const EriArgs<real>& args, const int t, "
            "const double* __restrict__ btab)" % tag,
            "{",
            "  switch (blockIdx.y) {   // one output group per wave"]
    for g in range(len(groups)):
        disp.append("  case %d: eri_body_%s_g%d<real, OP>(args, t, btab); break;" % (g, tag, g))
    disp += ["  default: break;", "  }", "}"]
    return "\n".join(parts + ["\n".join(disp)]), ncomp, wbody, len(groups), flops, worst


def gen_onee(la, lb):
    """S, T, V for one pair class as a device function for the fused launch:
    G consecutive lanes (a power of two <= 64, aligned) share one shell pair;
    lane g sums the nuclear attraction over atoms g, g + G, ... of the pair's
    molecule, the lanes combine with shuffles, and lane 0 also forms S and T
    and writes the three blocks."""
    tag = "%d%d" % (la, lb)
    es = Emitter(indent="    ")

    def ovl(e):          # primitive overlap VRR, s(e) on the primary centre
        key = ("s", e)
        name = "s%s" % nm(e)
        if key in es.done:
            return name
        if lev(e) == 0:
            expr = "P.K"
        else:
            i = axis(e)
            e1 = dec(e, i)
            expr = "PA%s * %s" % (XYZ[i], ovl(e1))
            if e1[i] > 0:
                expr += " + (double)%d * P.inv2p * %s" % (e1[i], ovl(dec(e1, i)))
        es.emit("const double %s = %s;" % (name, expr))
        es.done.add(key)
        return name

    def ohrr(a, b):
        if lev(b) == 0:
            return ovl(a)
        key = ("sh", a, b)
        name = "sh%s_%s" % (nm(a), nm(b))
        if key in es.done:
            return name
        i = axis(b)
        b1 = dec(b, i)
        es.emit("const double %s = %s + AB%s * %s;" % (name, ohrr(inc(a, i), b1), XYZ[i], ohrr(a, b1)))
        es.done.add(key)
        return name

    for a in comps(la):
        for b in comps(lb):
            sab = ohrr(a, b)
            t = ["beta * (double)%d * %s" % (2 * lb + 3, sab)]
            for i in range(3):
                t.append("- 2.0 * beta * beta * %s" % ohrr(a, tuple(b[k] + (2 if k == i else 0) for k in range(3))))
                if b[i] > 1:
                    t.append("- %r * %s" % (0.5 * b[i] * (b[i] - 1), ohrr(a, dec(b, i, 2))))
            es.emit("s_%s_%s += %s;" % (nm(a), nm(b), sab))
            es.emit("t_%s_%s += %s;" % (nm(a), nm(b), " ".join(t)))
    sbody = es.lines

    ev = Emitter(indent="      ")
    Lv = la + lb

    def nuc(e, m):
        key = (e, m)
        name = "n%s_%d" % (nm(e), m)
        if key in ev.done:
            return name
        if lev(e) == 0:
            expr = "vpref * F[%d]" % m
        else:
            i = axis(e)
            e1 = dec(e, i)
            expr = "PA%s * %s - PC%s * %s" % (XYZ[i], nuc(e1, m), XYZ[i], nuc(e1, m + 1))
            if e1[i] > 0:
                e2 = dec(e1, i)
                expr += " + (double)%d * P.inv2p * (%s - %s)" % (e1[i], nuc(e2, m), nuc(e2, m + 1))
        ev.emit("const double %s = %s;" % (name, expr))
        ev.done.add(key)
        return name

    def nhrr(a, b):
        if lev(b) == 0:
            return nuc(a, 0)
        key = ("vh", a, b)
        name = "vh%s_%s" % (nm(a), nm(b))
        if key in ev.done:
            return name
        i = axis(b)
        b1 = dec(b, i)
        ev.emit("const double %s = %s + AB%s * %s;" % (name, nhrr(inc(a, i), b1), XYZ[i], nhrr(a, b1)))
        ev.done.add(key)
        return name

    for a in comps(la):
        for b in comps(lb):
            ev.emit("v_%s_%s += %s;" % (nm(a), nm(b), nhrr(a, b)))
    vbody = ev.lines

    lines = []
    lines.append("__device__ __forceinline__ void onee_body_%s(const OneeArgs& args, int t, int g, int G)" % tag)
    lines.append("{")
    lines.append("  if (t >= args.npair) return;   // uniform over the pair's lanes")
    lines.append("  const int pidx = args.pair_list[t];")
    lines.append("  const PairHdr h = args.pairs[pidx];")
    lines.append("  const MolInfo mi = args.mols[h.mol];")
    lines.append("  const double ABx = h.ab[0], ABy = h.ab[1], ABz = h.ab[2];")
    lines.append("  (void)ABx; (void)ABy; (void)ABz;")
    for a in comps(la):
        for b in comps(lb):
            lines.append("  double s_%s_%s = 0, t_%s_%s = 0, v_%s_%s = 0;" % ((nm(a), nm(b)) * 3))
    lines.append("  for (int i = 0; i < h.n; ++i) {")
    lines.append("    const PrimPair<double> P = args.prims[h.off + i];")
    lines.append("    const double PAx = P.PAx, PAy = P.PAy, PAz = P.PAz;")
    lines.append("    const double beta = P.beta;")
    lines.append("    if (g == 0) {")
    lines.extend(["  " + x for x in sbody])
    lines.append("    }")
    lines.append("    for (int c = mi.atom_lo + g; c < mi.atom_hi; c += G) {")
    lines.append("      const double PCx = P.Px - args.atoms[4 * c], PCy = P.Py - args.atoms[4 * c + 1], PCz = P.Pz - args.atoms[4 * c + 2];")
    lines.append("      const double Tn = P.p * (PCx * PCx + PCy * PCy + PCz * PCz);")
    lines.append("      double F[%d];" % (Lv + 1))
    lines.append("      boys_eval<%d>(Tn, F);" % Lv)
    lines.append("      const double vpref = -args.atoms[4 * c + 3] * 1.1283791670955126 * sqrt(P.p) * P.K;")
    lines.extend(vbody)
    lines.append("    }")
    lines.append("  }")
    lines.append("  for (int o = G >> 1; o > 0; o >>= 1) {")
    for a in comps(la):
        for b in comps(lb):
            lines.append("    v_%s_%s += __shfl_xor(v_%s_%s, o, 64);" % ((nm(a), nm(b)) * 2))
    lines.append("  }")
    lines.append("  if (g != 0) return;")
    lines.append("  const int o1 = args.cart_off[h.s1], o2 = args.cart_off[h.s2];")
    lines.append("  const int N = mi.n;")
    lines.append("  double* const Sm = args.S + mi.base;")
    lines.append("  double* const Tm = args.T + mi.base;")
    lines.append("  double* const Vm = args.V + mi.base;")
    ia = 0
    for a in comps(la):
        ib = 0
        for b in comps(lb):
            nrm = cnorm(a) * cnorm(b)
            lines.append("  { const size_t u = (size_t)(o1 + %d) * N + (o2 + %d), w = (size_t)(o2 + %d) * N + (o1 + %d);" % (ia, ib, ib, ia))
            for M, v in (("S", "s"), ("T", "t"), ("V", "v")):
                lines.append("    %sm[u] = %s_%s_%s * %.17g; %sm[w] = %s_%s_%s * %.17g;" %
                             (M, v, nm(a), nm(b), nrm, M, v, nm(a), nm(b), nrm))
            lines.append("  }")
            ib += 1
        ia += 1
    lines.append("}")
    return "\n".join(lines)


_written = set()


def _write_if_changed(path, text):
    """Keep mtimes of unchanged generated files so incremental builds skip them."""
    _written.add(os.path.basename(path))
    if os.path.exists(path):
        with open(path) as fh:
            if fh.read() == text:
                return
    with open(path, "w") as fh:
        fh.write(text)


def jk_tile(la, lb, lc, ld, budget=72):
    """Bra tile (TA, TB) of the tiled J/K kernel: the fewest tiles whose
    per-lane live state, 2 (TA + TB)(N4 + 1) + 2 TA TB doubles, fits the
    budget (ties: the smaller state).  Returns (TA, TB, number of tiles)."""
    nc = lambda l: (l + 1) * (l + 2) // 2
    n1, n2, n4 = nc(la), nc(lb), nc(ld)
    best = None
    for ta in [t for t in range(1, n1 + 1) if n1 % t == 0]:
        for tb in [t for t in range(1, n2 + 1) if n2 % t == 0]:
            cost = 2 * (ta + tb) * (n4 + 1) + 2 * ta * tb
            if cost > budget and (ta, tb) != (1, 1):
                continue
            key = ((n1 // ta) * (n2 // tb), cost)
            if best is None or key < best[0]:
                best = (key, ta, tb)
    _, ta, tb = best
    return ta, tb, (n1 // ta) * (n2 // tb)


# J/K launch groups by rows staged (TA + TB), which also orders the classes by
# the registers their digestion takes (86, 128, 207 and 230 at most)
JK_GROUPS = [(0, 4), (7, 7), (5, 6), (8, 99)]


def jk_group(la, lb, lc, ld):
    ta, tb, _ = jk_tile(la, lb, lc, ld)
    if (la, lb, lc, ld) in ((2, 2, 2, 2), (2, 0, 1, 1)):
        return 2          # few rows, but the registers of the 3 x 3 tiles
    return next(g for g, (lo, hi) in enumerate(JK_GROUPS) if lo <= ta + tb <= hi)


def boys_rows(here):
    """Grid step and rows F_0..F_{NCOL-1}(T_k) of boys_table.inc."""
    with open(os.path.join(here, "boys_table.inc")) as fh:
        text = fh.read()
    step = float(text.split("#define BOYS_STEP")[1].split()[0])
    ncol = int(text.split("#define BOYS_NCOL")[1].split()[0])
    body = text.split("{", 1)[1].split("}", 1)[0]
    vals = [float(x) for x in body.replace("\n", " ").split(",") if x.strip()]
    return step, [vals[i:i + ncol] for i in range(0, len(vals), ncol)]


# Up to this Boys order a class takes F_L and F_{L-1} from one polynomial
# (boys_eval_s); must equal BOYS_PAIR_MAX of eri_common.h.
BOYS_PAIR_MAX = 5


def economised(c, h):
    """The polynomial sum_j c[j] x^j less its top Chebyshev component on
    |x| <= h: one degree lower, off by c[n] h^n / 2^(n-1) at most."""
    n = len(c) - 1
    t0, t1 = [1], [0, 1]                        # Chebyshev T_0, T_1, ..., T_n
    for _ in range(n - 1):
        t2 = [0] + [2 * v for v in t1]
        for k, v in enumerate(t0):
            t2[k] -= v
        t0, t1 = t1, t2
    return [c[k] - c[n] * h ** (n - k) * t1[k] / 2 ** (n - 1) for k in range(n)]


def boys_lds_table(L, step, rows):
    """The LDS image a class kernel of Boys order L stages (boys_stage_copy),
    10 doubles per grid point T_k: polynomial coefficients of F_0(T_k - x)
    (L = 0: 8) or F_{L-1}(T_k - x) (to BOYS_PAIR_MAX: 9), the Taylor series
    economised by one degree; above that the 9 Taylor coefficients
    F_{L+c}(T_k) / c! and e^{-T_k} (T_k the double k * step, as the kernel
    forms it)."""
    out = []
    h = Fraction(step) / 2
    for k, r in enumerate(rows):
        if L <= BOYS_PAIR_MAX:
            n, m = (8, 0) if L == 0 else (9, L - 1)
            c = economised([Fraction(r[m + j]) / math.factorial(j) for j in range(n + 1)], h)
            out += [float(v) for v in c] + [0.0] * (10 - n)
        else:
            out += [r[L + c] * (1.0 / math.factorial(c)) for c in range(9)] + [math.exp(-(k * step))]
    name = "boys_lds_L%d" % L
    lines = ["// Boys coefficients staged in LDS by the class kernels of order %d" % L,
             "static __device__ __align__(16) const double %s[BOYS_LDS_DOUBLES] = {" % name]
    for i in range(0, len(out), 6):
        lines.append("  " + ", ".join("%.17e" % v for v in out[i:i + 6]) + ",")
    lines.append("};")
    return name, "\n".join(lines)


def main():
    here = os.path.dirname(os.path.abspath(__file__))
    gdir = os.path.join(here, "gen")
    os.makedirs(gdir, exist_ok=True)
    bstep, brows = boys_rows(here)
    table = []
    flop_table = {}
    for X, Y in CLASSES:
        la, lb = PAIRS[X]
        lc, ld = PAIRS[Y]
        tag = "%d%d%d%d" % (la, lb, lc, ld)
        Lc = la + lb + lc + ld
        code, ncomp, nbody, ngrp, flops, nacc = gen_eri_class_split(la, lb, lc, ld)
        table.append((la, lb, lc, ld, ncomp, X, Y, nbody))
        flop_table[tag] = dict(flops, jk_tile=list(jk_tile(la, lb, lc, ld)), groups=ngrp, accumulators=nacc)
        _write_if_changed(os.path.join(gdir, "body_%s.h" % tag),
                          "\n".join(["// generated by gen_eri.py -- do not edit", "#pragma once",
                                     '#include "../eri_common.h"', code]) + "\n")
        btname, btcode = boys_lds_table(Lc, bstep, brows)
        src = ["// generated by gen_eri.py -- do not edit", '#include "body_%s.h"' % tag, btcode,
               "// occupancy floor (waves per SIMD) of the class kernels: caps their registers",
               "#if defined(ERI_MINW_ALL)",
               "#define ERI_MINW ERI_MINW_ALL",
               "#else",
               "#define ERI_MINW %d" % MINW.get(tag, 1),
               "#endif",
               "template <typename real>",
               "__global__ void __launch_bounds__(ERI_BLOCK, ERI_MINW) eri_k%s(const EriArgs<real> args)" % tag,
               "{",
               "  __shared__ __align__(16) double btab[BOYS_LDS_DOUBLES];",
               "  boys_stage_copy(btab, %s, BOYS_LDS_DOUBLES);" % btname,
               "  eri_body_%s<real>(args, blockIdx.x * blockDim.x + threadIdx.x, btab);" % tag,
               "}"]
        # both lists of the class in one launch (FP64 blocks first): the FP32
        # list of a mixed-precision plan costs no launch of its own
        src.append("__global__ void __launch_bounds__(ERI_BLOCK, ERI_MINW) eri_kmix%s(const EriArgs<double> d, "
                   "const EriArgs<float> f, int nb64)" % tag)
        src.append("{")
        src.append("  __shared__ __align__(16) double btab[BOYS_LDS_DOUBLES];")
        src.append("  boys_stage_copy(btab, %s, BOYS_LDS_DOUBLES);" % btname)
        src.append("  if ((int)blockIdx.x < nb64) eri_body_%s<double>(d, blockIdx.x * blockDim.x + threadIdx.x, btab);" % tag)
        src.append("  else eri_body_%s<float>(f, (blockIdx.x - nb64) * blockDim.x + threadIdx.x, btab);" % tag)
        src.append("}")
        src.append("void eri_run_%s_mix(const EriArgs<double>& d, const EriArgs<float>& f, hipStream_t st)" % tag)
        src.append("{ const int nb64 = (d.nq + ERI_BLOCK - 1) / ERI_BLOCK, nb32 = (f.nq + ERI_BLOCK - 1) / ERI_BLOCK;")
        src.append("  if (nb64 + nb32 > 0) hipLaunchKernelGGL(eri_kmix%s, dim3(nb64 + nb32, %d), dim3(ERI_BLOCK), 0, st, d, f, nb64); }" % (tag, ngrp))
        # the electron-scattering operator (FP64 only)
        src.append("__global__ void __launch_bounds__(ERI_BLOCK, ERI_MINW) eri_ks%s(const EriArgs<double> args)" % tag)
        src.append("{ eri_body_%s<double, 1>(args, blockIdx.x * blockDim.x + threadIdx.x, nullptr); }" % tag)
        src.append("void eri_run_%s_s(const EriArgs<double>& a, hipStream_t st)" % tag)
        src.append("{ hipLaunchKernelGGL(eri_ks%s, dim3((a.nq + ERI_BLOCK - 1) / ERI_BLOCK, %d), dim3(ERI_BLOCK), 0, st, a); }" % (tag, ngrp))
        src.append("size_t eri_scratch_%s_s()" % tag)
        src.append("{ hipFuncAttributes f; return hipFuncGetAttributes(&f, (const void*)eri_ks%s) == hipSuccess ? "
                   "f.localSizeBytes : (size_t)1 << 30; }" % tag)
        src.append("size_t eri_scratch_%s_mix()" % tag)
        src.append("{ hipFuncAttributes f; return hipFuncGetAttributes(&f, (const void*)eri_kmix%s) == hipSuccess ? "
                   "f.localSizeBytes : (size_t)1 << 30; }" % tag)
        jsrc = ["// generated by gen_eri.py -- do not edit", '#include "../jk_common.h"']
        for rn, rt in (("d", "double"), ("f", "float")):
            src.append("void eri_run_%s_%s(const EriArgs<%s>& a, hipStream_t st)" % (tag, rn, rt))
            src.append("{ hipLaunchKernelGGL(eri_k%s<%s>, dim3((a.nq + ERI_BLOCK - 1) / ERI_BLOCK, %d), dim3(ERI_BLOCK), 0, st, a); }" % (tag, rt, ngrp))
            src.append("size_t eri_scratch_%s_%s()" % (tag, rn))
            src.append("{ hipFuncAttributes f; return hipFuncGetAttributes(&f, (const void*)eri_k%s<%s>) == hipSuccess ? "
                       "f.localSizeBytes : (size_t)1 << 30; }" % (tag, rt))
            jsrc.append("void jk_run_%s_%s(const JkArgs<%s>& a, hipStream_t st)" % (tag, rn, rt))
            jsrc.append("{ hipLaunchKernelGGL((jk_kernel<%d, %d, %d, %d, %s>), dim3((a.nq + 127) / 128), dim3(128), 0, st, a); }" % (la, lb, lc, ld, rt))
            jsrc.append("void scatter_run_%s_%s(const ScatterArgs<%s>& a, hipStream_t st)" % (tag, rn, rt))
            jsrc.append("{ hipLaunchKernelGGL((scatter_kernel<%d, %d, %d, %d, %s>), dim3((unsigned)((a.nq * %dLL + 255) / 256)), "
                        "dim3(256), 0, st, a); }" % (la, lb, lc, ld, rt, ncomp))
            jsrc.append("void pairscatter_run_%s_%s(const PairScatterArgs<%s>& a, hipStream_t st)" % (tag, rn, rt))
            n12 = (la + 1) * (la + 2) // 2 * ((lb + 1) * (lb + 2) // 2)
            jsrc.append("{ hipLaunchKernelGGL((pair_scatter_kernel<%d, %d, %d, %d, %s>), dim3((a.nq + 255) / 256, "
                        "%d / PairScatterSplit<%d, %d>::AB), dim3(256), 0, st, a); }"
                        % (la, lb, lc, ld, rt, n12, n12, ncomp // n12))
        _write_if_changed(os.path.join(gdir, "cls_%s.hip" % tag), "\n".join(src) + "\n")
        _write_if_changed(os.path.join(gdir, "jk_%s.hip" % tag), "\n".join(jsrc) + "\n")
    # J/K launch groups: classes whose kernels need about the same registers
    # and LDS rows in one kernel
    for g in range(len(JK_GROUPS)):
        js = ["// generated by gen_eri.py -- do not edit", '#include "../jk_common.h"',
              "__global__ void __launch_bounds__(256, 2) jk_group_kernel_%d(const JkGroupArgs g)" % g, "{",
              "  extern __shared__ double lds[];", "  const int s = jk_group_slot(g);",
              "  const JkClassArgs& a = g.c[s];", "  const int local = blockIdx.x - a.block0;",
              "  jk_clock(g, a.cls, 0);", "  switch (a.cls) {"]
        for k, t in enumerate(table):
            la, lb, lc, ld = t[:4]
            if jk_group(la, lb, lc, ld) != g:
                continue
            ta, tb, nt = jk_tile(la, lb, lc, ld)
            js.append("  case %d: jk_tile_class<%d, %d, %d, %d, %d, %d>(g, a, local, lds); break;"
                      % (k, la, lb, lc, ld, ta, tb))
        js += ["  default: break;", "  }", "  jk_clock(g, a.cls, 1);", "}",
               "void jk_group_run_%d(const JkGroupArgs& g, int blocks, int block, size_t lds, hipStream_t st)" % g,
               "{ hipLaunchKernelGGL(jk_group_kernel_%d, dim3(blocks), dim3(block), lds, st, g); }" % g]
        _write_if_changed(os.path.join(gdir, "jk_group_%d.hip" % g), "\n".join(js) + "\n")
    onee = ["// generated by gen_eri.py -- do not edit", '#include "../eri_common.h"']
    for la, lb in PAIRS:
        onee.append(gen_onee(la, lb))
    onee.append("// every pair class in one launch: block -> class by the first-block table")
    onee.append("__global__ void __launch_bounds__(128) onee_fused_k(const OneeFusedArgs a)")
    onee.append("{")
    onee.append("  const int b = blockIdx.x;")
    onee.append("  int j = 0;")
    onee.append("  while (j + 1 < 6 && b >= a.block0[j + 1]) ++j;")
    onee.append("  const int lt = (b - a.block0[j]) * 128 + threadIdx.x;")
    onee.append("  const int t = lt / a.G, g = lt - (lt / a.G) * a.G;")
    onee.append("  switch (j) {")
    for p, (la, lb) in enumerate(PAIRS):
        onee.append("  case %d: onee_body_%d%d(a.cls[%d], t, g, a.G); break;" % (p, la, lb, p))
    onee.append("  default: break;")
    onee.append("  }")
    onee.append("}")
    onee.append("void onee_fused_run(const OneeFusedArgs& a, hipStream_t st)")
    onee.append("{ if (a.block0[6] > 0) hipLaunchKernelGGL(onee_fused_k, dim3(a.block0[6]), dim3(128), 0, st, a); }")
    _write_if_changed(os.path.join(gdir, "onee.hip"), "\n".join(onee) + "\n")
    for f in os.listdir(gdir):   # of an older generator
        if f.endswith((".hip", ".h")) and f not in _written:
            os.remove(os.path.join(gdir, f))
    # dispatch header
    d = ["// generated by gen_eri.py -- do not edit", "#pragma once", '#include "jk_common.h"',
         "#define ERI_NCLASS %d" % len(CLASSES)]
    for la, lb, lc, ld, ncomp, X, Y, nbody in table:
        tag = "%d%d%d%d" % (la, lb, lc, ld)
        for rn, rt in (("d", "double"), ("f", "float")):
            d.append("void eri_run_%s_%s(const EriArgs<%s>&, hipStream_t);" % (tag, rn, rt))
            d.append("size_t eri_scratch_%s_%s();" % (tag, rn))
            d.append("void jk_run_%s_%s(const JkArgs<%s>&, hipStream_t);" % (tag, rn, rt))
            d.append("void scatter_run_%s_%s(const ScatterArgs<%s>&, hipStream_t);" % (tag, rn, rt))
            d.append("void pairscatter_run_%s_%s(const PairScatterArgs<%s>&, hipStream_t);" % (tag, rn, rt))
        d.append("void eri_run_%s_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);" % tag)
        d.append("size_t eri_scratch_%s_mix();" % tag)
        d.append("void eri_run_%s_s(const EriArgs<double>&, hipStream_t);" % tag)
        d.append("size_t eri_scratch_%s_s();" % tag)
    d.append("void onee_fused_run(const OneeFusedArgs& a, hipStream_t st);")
    d.append("// la, lb, lc, ld, components, bra pair class, ket pair class")
    d.append("static const int eri_class_table[ERI_NCLASS][7] = {")
    for la, lb, lc, ld, ncomp, X, Y, nbody in table:
        d.append("  {%d, %d, %d, %d, %d, %d, %d}," % (la, lb, lc, ld, ncomp, X, Y))
    d.append("};")
    d.append("// VRR and contraction lines per primitive quartet (of one output group)")
    d.append("static const int eri_body_lines[ERI_NCLASS] = {")
    d.append("  " + ", ".join(str(t[7]) for t in table))
    d.append("};")
    d.append("// the electron-scattering operator's class kernels (FP64)")
    d.append("static void (*const eri_table_s[ERI_NCLASS])(const EriArgs<double>&, hipStream_t) = {")
    d.append("  " + ", ".join("eri_run_%d%d%d%d_s" % (t[0], t[1], t[2], t[3]) for t in table))
    d.append("};")
    d.append("// per-lane scratch (spill) bytes of each class kernel, FP64, FP32, mixed and scattering forms")
    for rn in ("d", "f", "mix", "s"):
        d.append("static size_t (*const eri_scratch_table_%s[ERI_NCLASS])() = {" % rn)
        d.append("  " + ", ".join("eri_scratch_%d%d%d%d_%s" % (t[0], t[1], t[2], t[3], rn) for t in table))
        d.append("};")
    d.append("// tiled J/K: bra tile TA x TB, tiles per quartet, LDS doubles per basis function")
    d.append("static const int jk_tile_table[ERI_NCLASS][4] = {")
    for la, lb, lc, ld, ncomp, X, Y, nbody in table:
        ta, tb, nt = jk_tile(la, lb, lc, ld)
        d.append("  {%d, %d, %d, %d}," % (ta, tb, nt, 2 * ((ta + tb) | 1)))
    d.append("};")
    ng = len(JK_GROUPS)
    d.append("// J/K launch groups")
    d.append("#define JK_NGROUP %d" % ng)
    d.append("static const int jk_group_table[ERI_NCLASS] = {")
    d.append("  " + ", ".join(str(jk_group(*t[:4])) for t in table))
    d.append("};")
    for g in range(ng):
        d.append("void jk_group_run_%d(const JkGroupArgs&, int, int, size_t, hipStream_t);" % g)
    d.append("static void (*const jk_group_run[JK_NGROUP])(const JkGroupArgs&, int, int, size_t, hipStream_t) = {")
    d.append("  " + ", ".join("jk_group_run_%d" % g for g in range(ng)))
    d.append("};")
    d.append("// both lists of a class in one launch")
    d.append("static void (*const eri_table_mix[ERI_NCLASS])(const EriArgs<double>&, const EriArgs<float>&, hipStream_t) = {")
    d.append("  " + ", ".join("eri_run_%d%d%d%d_mix" % (t[0], t[1], t[2], t[3]) for t in table))
    d.append("};")
    for kname, targ in (("eri", "EriArgs"), ("jk", "JkArgs"), ("scatter", "ScatterArgs"),
                        ("pairscatter", "PairScatterArgs")):
        for rn, rt in (("d", "double"), ("f", "float")):
            d.append("static void (*const %s_table_%s[ERI_NCLASS])(const %s<%s>&, hipStream_t) = {" % (kname, rn, targ, rt))
            d.append("  " + ", ".join("%s_run_%d%d%d%d_%s" % (kname, t[0], t[1], t[2], t[3], rn) for t in table))
            d.append("};")
        d.append("template <typename real> static inline void %s_launch(int cls, const %s<real>& a, hipStream_t st)" % (kname, targ))
        d.append("{ if (sizeof(real) == 8) %s_table_d[cls]((const %s<double>&)a, st); else %s_table_f[cls]((const %s<float>&)a, st); }" % (kname, targ, kname, targ))
    _write_if_changed(os.path.join(here, "eri_dispatch.h"), "\n".join(d) + "\n")
    import json
    _write_if_changed(os.path.join(here, "eri_flops.json"), json.dumps(flop_table, indent=1, sort_keys=True) + "\n")
    for la, lb, lc, ld, ncomp, X, Y, nbody in table:
        tag = "%d%d%d%d" % (la, lb, lc, ld)
        print("class (%d%d|%d%d) comps=%d body_lines=%d groups=%d accumulators=%d" %
              (la, lb, lc, ld, ncomp, nbody, flop_table[tag]["groups"], flop_table[tag]["accumulators"]))
    print("wrote", gdir)


if __name__ == "__main__":
    main()
