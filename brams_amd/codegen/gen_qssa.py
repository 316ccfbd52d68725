"""Generate the QSSA kernel's wave programs (csrc/generated/<mech>_qssa.h).

A workgroup holds 64 cells, one to a lane, and shares a cell's work between
its waves: each wave computes some of the rate constants, and integrates some
of the species.  What the waves exchange (rate constants, concentrations)
goes through LDS, so no lane keeps a cell's whole state:

  1  rates that depend on T (and J) alone; one wave takes the pressure
  2  rates that depend on M or H2O; each wave gathers its species
  3  production, loss and sub-steps of the wave's species
  4  tendencies

Both distributions are greedy, longest first, on the estimated number of
FP64 instructions.
"""
import re

from gen_coop import lit

WAVES = 8
GROUP = 6                        # terms of a sum between scheduling fences
FENCE = 100                      # instructions between scheduling fences
PRE_COST = 260                   # Exner pressure, M, H2O and the gather's factor


def rate_cost(text):
    """Estimated FP64 instructions of a rate expression."""
    c = 4
    for name, cost in (("rl_arr_tn(", 40), ("rl_arr(", 36), ("rl_hno3_oh(", 140), ("rl_troe_ca(", 700),
                       ("rl_troe(", 430), ("pow(T", 150)):
        c += cost * text.count(name)
    c += 36 * len(re.findall(r"(?<!_)exp\(", text))
    return c


def spread(items, cost, start):
    """Items to waves, the costliest first, each to the wave with least."""
    load, out = list(start), [[] for _ in start]
    for x in sorted(items, key=lambda x: (-cost[x], x)):
        n = min(range(len(load)), key=lambda k: load[k])
        out[n].append(x)
        load[n] += cost[x]
    return [sorted(x) for x in out]


def emit(ns, nr, react, prod, reactions, rate_rhs, literals, mech, name):
    rhs = [rate_rhs(r) for r in range(nr)]
    used = sorted({r for terms in prod.values() for _, r in terms if r not in literals})
    slot = {r: k for k, r in enumerate(used)}
    ybase = len(used)
    m_slot = ybase + ns
    nslots = m_slot + 3                                     # M, H2O, avo * volmol

    # reactions with the same fall-off go to one wave, which computes it once
    groups = {}
    for r in used:
        t = re.search(r"rl_troe\([^)]*\)", rhs[r])
        groups.setdefault(t.group(0) if t else r, []).append(r)
    late, early, cost = [], [], {}
    for k, rs in enumerate(groups.values()):
        c = sum(rate_cost(rhs[r]) for r in rs)
        if len(rs) > 1:
            c -= 400 * (len(rs) - 1)
        cost[k] = c
        (late if any(re.search(r"\b(M|H2O)\b", rhs[r]) for r in rs) else early).append(k)
    glist = list(groups.values())
    first = spread(early, cost, [0] * (WAVES - 1) + [PRE_COST])
    second = spread(late, cost, [0] * WAVES)

    def others(r, s):
        """Reaction and species whose product is dw_r/dc_s."""
        rs = react[r]
        if s not in rs:          # negative product (CB07_TUV): dratedc never assigns dw(r,s)
            return None
        return [r] + ([rs[1] if rs[0] == s else rs[0]] if len(rs) == 2 else [])

    def terms(out, ts):
        """A sum c * rk * y..., read from LDS term by term."""
        w("    %s = 0.0;" % out)
        for n, (c, x) in enumerate(ts):
            if x is None:
                f = "0.0"
            else:
                f = " * ".join([literals.get(x[0]) or "s.get(%d)" % slot[x[0]]]
                               + ["s.get(%d)" % (ybase + y) for y in x[1:]])
            w("    %s %s= %s;" % (out, "+" if n else "", f if c == 1.0 else "%s * (%s)" % (lit(c), f)))
            if n % GROUP == GROUP - 1:
                w("    coop_fence();")

    ptab = {s: [(c, r) for c, r in prod.get(s, []) if c > 0] for s in range(ns)}
    ltab = {s: [(-c, r) for c, r in prod.get(s, []) if c < 0] for s in range(ns)}
    scost = {s: 150 + sum(3 + len(react[r]) for _, r in ptab[s] + ltab[s]) for s in range(ns)}
    mine = spread(range(ns), scost, [0] * WAVES)

    L = []
    w = L.append
    w("// Generated by brams_amd/codegen/gen_qssa.py from brams_amd/mechanism/%s.json." % mech)
    w("// %s: the QSSA step of 64 cells as %d waves' programs." % (name, WAVES))
    w("#pragma once")
    w("#define MECH_QSSA_WAVES %d" % WAVES)
    w("#define MECH_QSSA_SLOTS %d" % nslots)
    w("")
    for n in range(WAVES):
        w("__device__ __forceinline__ void qssa_program_%d(const QssaCell& q, const CoopLds& s) {" % n)
        w("  const QssaTemp T = q.temp;")
        for k, sp in enumerate(mine[n]):
            w("  const float x%d = q.load(%d);" % (sp, sp))

        def rates(gs):
            left = FENCE
            for r in [r for g in gs for r in glist[g]]:
                w("  s.put(%d, %s);" % (slot[r], re.sub(r"J\[(\d+)\]", r"q.photolysis(\1)", rhs[r])))
                left -= rate_cost(rhs[r])
                if left <= 0:
                    w("  coop_fence();")
                    left = FENCE

        lnt = any("lnT" in rhs[r] for g in first[n] + second[n] for r in glist[g])
        if lnt:
            w("  const double lnT = log(q.temp.t);")
        if n == WAVES - 1:
            w("  q.pressure(s, %d);" % m_slot)
        rates(first[n])
        w("  coop_barrier();")
        if second[n]:
            w("  const double M = s.get(%d), H2O = s.get(%d);" % (m_slot, m_slot + 1))
            w("  (void)M; (void)H2O;")
        rates(second[n])
        w("  const double av = s.get(%d);" % (m_slot + 2))
        w("  constexpr int N = %d;" % len(mine[n]))
        w("  double v[N], P[N], L[N];")
        for k, sp in enumerate(mine[n]):
            w("  v[%d] = q.gather(x%d, av, %d); s.put(%d, v[%d]);" % (k, sp, sp, ybase + sp, k))
        w("  coop_barrier();")
        for k, sp in enumerate(mine[n]):
            w("  { // species %d" % sp)
            terms("P[%d]" % k, [(c, [r] + react[r]) for c, r in ptab[sp]])
            terms("L[%d]" % k, [(c, others(r, sp)) for c, r in ltab[sp]])
            w("    qssa_here(P[%d], L[%d]);" % (k, k))
            w("  }")
        w("  if (q.advance<N>(v, P, L)) q.fatal[q.lane] = 1;")
        w("  coop_barrier();")
        w("  if (!q.store(%s)) return;" % ("true" if n == 0 else "false"))
        for k, sp in enumerate(mine[n]):
            w("  q.tendency(%d, x%d, v[%d], av);" % (sp, sp, k))
        w("}")
        w("")
    w("__device__ __forceinline__ void qssa_program(int wave, const QssaCell& q, const CoopLds& s) {")
    w("  switch (wave) {")
    for n in range(WAVES):
        w("    case %d: qssa_program_%d(q, s); break;" % (n, n))
    w("  }")
    w("}")
    return "\n".join(L) + "\n"
