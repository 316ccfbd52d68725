"""Split one block's Rosenbrock attempt over the waves of a workgroup.

A cell's working set (the factors, the rate constants and the stage vectors,
about a thousand doubles) fits the registers and the LDS of a whole CU, not
one lane's.  So a workgroup of WAVES waves integrates one 64-cell block: lane
l of every wave works on cell l, and each wave owns some species.  It holds
their rows of the matrix, evaluates their rates and carries their entries of
the stage vectors.  What another wave needs goes through LDS, one 512-byte
row ("slot") per value of the 64 cells.

This module builds the data flow of one attempt as scalar operations, places
each on the wave that owns its row, and cuts the result into phases: an
operation's phase is that of its inputs, one later where an input comes from
another wave.  A barrier separates two phases.  The code of every wave is
straight-line, with the same number of barriers.

The last `dense` pivots, nearly a dense block, are eliminated by one wave
(the dense wave), which keeps U in registers and L in LDS: a chain of
dependent pivots costs a barrier each when it is spread over waves, and a few
FMA latencies when it is not.  Their rows of the matrix are assembled, and
eliminated by the other pivots, on the other waves.

coop_rows.json says for each mechanism how many waves, how large the dense
block, and which wave owns the row of each pivot.  RELACS_TUV's rows were found
by simulated annealing on Layout.stats; the search is not part of the
repository.  Where rows is null, default_rows deals them.
"""
LDS_SLOTS = 320                  # 160 KB / (64 lanes x 8 bytes)
DENSE_PARTS = 3                  # phases of the dense wave's elimination
# Operations between scheduling fences, chunks a value read is kept, and
# chunks by which a read is issued ahead of its use.  Clocks move little with
# them as long as the registers hold (RODAS3 on 164k cells, us a block's
# attempt: 6/6/1 21.0, 6/6/2 20.8, 6/6/3 21.3, 4/8/2 21.3, 8/4/2 21.6, 3/8/4
# 22.2); chunks of 24 and more spill.
CHUNK, KEEP, AHEAD = 6, 6, 1


def lit(x):
    s = repr(float(x))
    if "e" not in s and "." not in s and "inf" not in s and "nan" not in s:
        s += ".0"
    return s


class Mech:
    """The mechanism's tables in the form the passes below use."""

    def __init__(self, ns, nr, react, prod, jt, perm, F, sidx):
        self.ns, self.nr, self.react, self.prod, self.jt, self.perm, self.F, self.sidx = (
            ns, nr, react, prod, jt, perm, F, sidx)
        self.pos = {s: k for k, s in enumerate(perm)}
        self.coef = {(sp, r): c for sp, terms in prod.items() for c, r in terms}


class Val:
    __slots__ = ("wave", "phase", "expr", "slot", "home", "uses", "into", "store", "count_only")

    def __init__(self, wave, phase, expr, home="reg"):
        self.wave, self.phase, self.expr, self.home = wave, phase, expr, home
        self.slot, self.uses, self.into, self.store, self.count_only = None, [], None, None, False


class Op:
    __slots__ = ("wave", "phase", "outs", "ins", "text", "cost", "movable", "count_only")

    def __init__(self, wave, phase, outs, ins, text, cost, movable):
        self.wave, self.phase, self.outs, self.ins, self.text, self.cost = wave, phase, outs, ins, text, cost
        self.movable, self.count_only = movable, False


class Flow:
    """Operations of one straight-line section over all waves."""

    def __init__(self):
        self.ops, self.n = [], 0
        self.movable = False             # whether level() may move the operations added now

    def at(self, v, w):
        """First phase in which wave w can use v."""
        if v.home == "free":
            return 0
        if v.home == "lds":                      # persistent slot
            return 0
        return v.phase if v.wave == w else v.phase + 1

    def op(self, w, text, ins, cost=1.0, outs=1, home="reg", count_only=False, first=0):
        ph = max([first] + [self.at(v, w) for v in ins])
        res = []
        for _ in range(outs):
            res.append(Val(w, ph, "v%d" % self.n, home))
            self.n += 1
        o = Op(w, ph, res, ins, text, cost, self.movable)
        o.count_only = count_only
        for v in res:
            v.count_only = count_only
        self.ops.append(o)
        return res[0] if outs == 1 else res

    def level(self, waves, least=16.0):
        """Moves the movable operations out of the phases that they would
        lengthen.  One may run in any phase from its inputs' to the last that
        its consumers allow; it goes to the first where its wave has time left
        beside the busiest wave, and else to where it adds the least."""
        P = self.phases()
        users = {}
        for o in self.ops:
            for v in o.ins:
                if v.home not in ("free", "lds"):
                    users.setdefault(id(v), []).append(o)
        last = {}
        load = [[0.0] * waves for _ in range(P)]
        for o in reversed(self.ops):
            if not o.movable:
                if not o.count_only:
                    load[o.phase][o.wave] += o.cost
                last[id(o)] = o.phase
                continue
            last[id(o)] = min([P - 1] + [last[id(u)] - (0 if u.wave == o.wave else 1)
                                         for v in o.outs for u in users.get(id(v), [])])
        for o in self.ops:
            if not o.movable:
                continue
            e, q = max([0] + [self.at(v, o.wave) for v in o.ins]), last[id(o)]

            def extra(p):
                return max(0.0, load[p][o.wave] + o.cost - max([least] + load[p]))
            o.phase = min(range(e, q + 1), key=lambda p: (extra(p), p))
            load[o.phase][o.wave] += o.cost
            for v in o.outs:
                v.phase = o.phase

    def settle(self):
        """Operations whose results wait in registers for a later phase move
        there, unless that keeps more values waiting; then the uses are noted."""
        users = {}
        for o in self.ops:
            for v in o.ins:
                if v.home != "free":
                    users.setdefault(id(v), []).append(o)
        for o in reversed(self.ops):
            if o.count_only or not o.outs:
                continue
            us = [u for v in o.outs for u in users.get(id(v), [])]
            if not us or any(u.wave != o.wave for u in us) or any(v.store is not None or v.home == "park" for v in o.outs):
                continue
            q = min(u.phase for u in us)
            if q <= o.phase:
                continue
            longer = 0
            for v in set(o.ins):
                if v.home in ("free", "lds") or v.wave != o.wave:
                    continue
                if not any(u is not o and u.wave == o.wave and u.phase >= q for u in users[id(v)]):
                    longer += 1
            if longer < len(o.outs) or (longer == len(o.outs) and longer == 0):
                o.phase = q
                for v in o.outs:
                    v.phase = q
        for o in self.ops:
            for v in o.ins:
                if v.home != "free":
                    v.uses.append((o.wave, o.phase))

    def phases(self):
        return 1 + max(o.phase for o in self.ops)


def free(expr):
    return Val(None, 0, expr, "free")


class Plan:
    """Which wave owns which row, and the LDS slots that hold a value throughout."""

    def __init__(self, m, waves, dense, row_wave, rk_lit=None):
        self.m, self.waves, self.dense, self.t0 = m, waves, dense, m.ns - dense
        self.row_wave, self.dw = row_wave, waves - 1         # by pivot position; the dense wave
        self.rk_lit = rk_lit or {}                           # constants that depend on nothing
        self.own = [[] for _ in range(waves)]                # species of each wave
        for I, w in enumerate(row_wave):
            self.own[w].append(m.perm[I])
        self.idx = {s: k for w in range(waves) for k, s in enumerate(self.own[w])}
        # rate constants each wave's rows need
        self.need = []
        for w in range(waves):
            self.need.append(sorted({r for s in self.own[w] for _, r in m.prod.get(s, [])}))
        users = {}
        for w in range(waves):
            for r in self.need[w]:
                users.setdefault(r, []).append(w)
        # the rate constants, those with the fewest users first
        self.rk_lds = [r for r in sorted(users, key=lambda r: (len(users[r]), r)) if r not in self.rk_lit]
        # persistent slots: the concentrations, then the rate constants
        self.yslot = {s: s for s in range(m.ns)}
        self.rkslot = {r: len(self.yslot) + k for k, r in enumerate(self.rk_lds)}
        self.nfix = len(self.yslot) + len(self.rkslot)
        self.mask_own = [dict() for _ in range(waves)]       # mask words of each wave's rows


class Builder:
    def __init__(self, plan):
        self.p, self.m = plan, plan.m
        self.f = Flow()
        self.yc = {s: Val(None, -1, None, "lds") for s in range(self.m.ns)}
        for s, v in self.yc.items():
            v.slot = plan.yslot[s]
        self.rkl = {r: Val(None, -1, None, "lds") for r in plan.rk_lds}
        for r, v in self.rkl.items():
            v.slot = plan.rkslot[r]

    def rk(self, r):
        return free(self.p.rk_lit[r]) if r in self.p.rk_lit else self.rkl[r]

    def add_rate(self, w, acc, rows, r, t, last):
        """Adds the rate t * last of reaction r to the sums of `rows`."""
        m, f = self.m, self.f
        fuse = len(rows) == 1 and abs(m.coef[(rows[0], r)]) == 1.0
        if not fuse:
            t = f.op(w, "{0} * {1}", [t, last])
        for s in rows:
            c = m.coef[(s, r)]
            if fuse:
                sg = "" if c > 0 else "-"
                if s in acc:
                    acc[s] = f.op(w, "fma(%s{0}, {1}, {2})" % sg, [t, last, acc[s]])
                else:
                    acc[s] = f.op(w, "%s({0} * {1})" % sg, [t, last])
            elif s not in acc:
                acc[s] = t if c == 1.0 else f.op(w, "%s * {0}" % lit(c), [t])
            elif abs(c) == 1.0:
                acc[s] = f.op(w, "{0} %s {1}" % ("+" if c > 0 else "-"), [acc[s], t])
            else:
                acc[s] = f.op(w, "fma(%s, {0}, {1})" % lit(c), [t, acc[s]])

    # f at the concentrations yv (species -> Val) for every wave's species
    def fun(self, yv):
        m, p, f = self.m, self.p, self.f
        out = {}
        f.movable = True
        for w in range(p.waves):
            acc = {}
            for r in p.need[w]:
                rows = [s for s in p.own[w] if (s, r) in m.coef]
                rs = m.react[r]
                t = self.rk(r)
                for s in rs[:-1]:
                    t = f.op(w, "{0} * {1}", [t, yv[s]])
                self.add_rate(w, acc, rows, r, t, yv[rs[-1]])
            for s in p.own[w]:
                out[s] = acc.get(s, free("0.0"))
        f.movable = False
        return out

    # rows of the masked 1/(gamma h) I - J, {(I, J): Val} on the rows' waves
    def matrix(self):
        m, p, f = self.m, self.p, self.f
        A = {}
        for w in range(p.waves):
            acc, prods = {}, {}

            def product(r, slot):
                """d(rate r)/d(its reactant in `slot`)"""
                rs = m.react[r]
                if len(rs) == 1:
                    return self.rk(r)
                o = rs[1 - slot]
                if (r, o) not in prods:
                    prods[(r, o)] = f.op(w, "{0} * {1}", [self.rk(r), self.yc[o]])
                return prods[(r, o)]

            for r in p.need[w]:
                for s in p.own[w]:
                    if (s, r) not in m.coef:
                        continue
                    c = m.coef[(s, r)]
                    for slot, j in enumerate(m.react[r]):
                        q = product(r, slot)
                        # off the diagonal -J is summed, on it J
                        sc = c if s == j else -c
                        e = (s, j)
                        if e not in acc:
                            acc[e] = (q if sc == 1.0 else f.op(w, "-{0}", [q]) if sc == -1.0
                                      else f.op(w, "%s * {0}" % lit(sc), [q]))
                        elif abs(sc) == 1.0:
                            acc[e] = f.op(w, "{0} %s {1}" % ("+" if sc > 0 else "-"), [acc[e], q])
                        else:
                            acc[e] = f.op(w, "fma(%s, {0}, {1})" % lit(sc), [q, acc[e]])
            for s in p.own[w]:
                d = acc.get((s, s))
                acc[(s, s)] = f.op(w, "igdt - {0}", [d]) if d is not None else free("igdt")
            # the mask: one uniform test a row, the selects only where a bit is clear
            for s in p.own[w]:
                ent = sorted(e for e in acc if e[0] == s)
                bits = [m.sidx[e] for e in ent]
                words = {}
                for b in bits:
                    words[b // 32] = words.get(b // 32, 0) | (1 << (b % 32))
                ins = [acc[e] for e in ent]
                text = ["@DECL", "  if constexpr (DYN) {", "    if (dyn) {"]
                for k, b in enumerate(bits):
                    text.append("      mw[%d] = (mw[%d] & 0x%08xu) | (coop_lane0_nonzero($%d$) << %d);"
                                % (b // 32, b // 32, 0xffffffff ^ (1 << (b % 32)), k, b % 32))
                text += ["    }", "  }"]
                text.append("  if (__builtin_expect(%s, 0)) {" % " || ".join(
                    "(mw[%d] & 0x%08xu) != 0x%08xu" % (q, v, v) for q, v in sorted(words.items())))
                for k, b in enumerate(bits):
                    text.append("    if (!((mw[%d] >> %d) & 1u)) $%d$ = 0.0;" % (b // 32, b % 32, k))
                text.append("  }")
                for q, v in words.items():
                    p.mask_own[w][q] = p.mask_own[w].get(q, 0) | v
                outs = f.op(w, text, ins, cost=1.0, outs=len(ent))
                if len(ent) == 1:
                    outs = [outs]
                for e, v in zip(ent, outs):
                    A[(m.pos[e[0]], m.pos[e[1]])] = v
        return A

    def factor(self, A):
        m, p, f = self.m, self.p, self.f
        F, t0 = m.F, p.t0
        self.L, self.U, self.R = {}, {}, {}
        pivots, checks = {}, []

        def over(w, I, K, lik, d, first=0):
            # Sparse1.3's threshold rule fails at pivot K where some
            # |L(I,K)| * 1e-3 >= |pivot|
            f.op(w, "if constexpr (COUNT) viol[%d] |= (fabs({0}) * 1.0e-3 >= fabs({1}) ? 1u : 0u) << %d;"
                 % (K // 32, K % 32), [lik, d], cost=0.0, outs=0, count_only=True, first=first)

        rows = []
        for I in range(m.ns):
            w = p.row_wave[I]
            row = {J: A[(I, J)] for J in range(m.ns) if (I, J) in A}
            rows.append(row)

            def eliminate(I, K, w):
                row, lik = rows[I], rows[I][K]
                self.L[(I, K)] = lik
                checks.append((w, I, K, lik))
                for J in range(K + 1, m.ns):
                    if F[K][J]:
                        if J in row:
                            row[J] = f.op(w, "fma(-{0}, {1}, {2})", [lik, self.U[(K, J)], row[J]])
                        else:
                            row[J] = f.op(w, "-({0} * {1})", [lik, self.U[(K, J)]])

            def pivot(I, w):
                d = rows[I][I]
                pivots[I] = d
                if not any(F[Q][I] for Q in range(I + 1, m.ns)):
                    f.op(w, "if constexpr (COUNT) viol[%d] |= ({0} == 0.0 ? 1u : 0u) << %d;" % (I // 32, I % 32),
                         [d], cost=0.0, outs=0, count_only=True)
                self.R[I] = f.op(w, "1.0 / {0}", [d], cost=12.0)
                for J in range(I + 1, m.ns):
                    if F[I][J]:
                        self.U[(I, J)] = f.op(w, "{0} * {1}", [rows[I][J], self.R[I]])

            # in the order in which the U rows arrive, after the pivots that
            # change this row's entry of column K
            left = [K for K in range(min(I, t0)) if F[I][K]]
            while left:
                ready = [K for K in left if not any(F[Q][K] for Q in left if Q < K)]
                K = min(ready, key=lambda K: (self.arrival(K, w), K))
                eliminate(I, K, w)
                left.remove(K)
            if I < t0:
                pivot(I, w)
        # The dense block crosses to its wave as a whole: the entries are
        # stored one phase after the last of them is ready, when the slots of
        # the other pivots' U rows are free again.
        w = p.dw
        self.cross = 1 + max(v.phase for I in range(t0, m.ns) for J, v in rows[I].items() if J >= t0)
        for I in range(t0, m.ns):
            for J, v in rows[I].items():
                if J >= t0 and v.home == "reg" and v.wave != w:
                    v.store = self.cross
        # The dense wave's elimination takes DENSE_PARTS phases, so that the
        # first solve's forward levels can run beside it.
        work = [sum(m.ns - 1 - K for K in range(t0, I)) + 12.0 + m.ns - I for I in range(t0, m.ns)]
        for I in range(t0, m.ns):
            part = int(DENSE_PARTS * (sum(work[:I - t0]) + 0.5 * work[I - t0]) / sum(work))
            row0 = dict(rows[I])
            for J in sorted(rows[I]):
                if J >= t0:
                    rows[I][J] = self.move(w, rows[I][J], first=self.cross + 1 + part)
            for K in range(t0, I):
                if F[I][K]:
                    eliminate(I, K, w)
                    v = self.L[(I, K)]
                    v.home = "park"
                    arrived = row0.get(K)                    # parked in the slot that brought the entry here
                    if arrived is not None and arrived.store is not None:
                        v.into = arrived
            pivot(I, w)
        # the pivots cross for the threshold check once the slots are free
        for w, I, K, lik in checks:
            if pivots[K].wave is not None and pivots[K].wave != w:
                pivots[K].store = self.cross + 2
            over(w, I, K, lik, pivots[K], first=self.cross + 3)

    def arrival(self, K, w):
        """Phase from which wave w can read row K of U."""
        return max([self.f.at(pivot, w) for pivot in [self.R[K]]]
                   + [self.f.at(v, w) for (I, J), v in self.U.items() if I == K])

    def move(self, w, v, first=0):
        """v as a value of wave w's own (read once from LDS, then in a register)."""
        if v.home == "free" or v.wave == w:
            return v
        return self.f.op(w, "{0}", [v], cost=0.0, first=first)

    # b: {I: Val}; returns {I: Val}
    def solve(self, b, first=0):
        m, p, f = self.m, self.p, self.f
        F, t0 = m.F, p.t0
        z, x = {}, {}
        for I in range(m.ns):
            w, c = p.row_wave[I], b[I]
            for K in sorted((K for K in range(min(I, t0)) if F[I][K]), key=lambda K: (f.at(z[K], w), K)):
                c = f.op(w, "fma(-{0}, {1}, {2})", [z[K], self.L[(I, K)], c], first=first)
            if I >= t0:
                w = p.dw
                for K in range(t0, I):
                    if F[I][K]:
                        c = f.op(w, "fma(-{0}, {1}, {2})", [z[K], self.L[(I, K)], c])
            z[I] = f.op(w, "{0} * {1}", [c, self.R[I]], first=first)
        for I in range(m.ns - 1, -1, -1):
            w, c = (p.dw if I >= t0 else p.row_wave[I]), z[I]
            for J in sorted((J for J in range(I + 1, m.ns) if F[I][J]), key=lambda J: (f.at(x[J], w), -J)):
                c = f.op(w, "fma(-{0}, {1}, {2})", [self.U[(I, J)], x[J], c])
            x[I] = c
        return x

    def spec(self, x):
        """Solution by species, on the species' waves."""
        return {self.m.perm[I]: self.move(self.p.row_wave[I], v) for I, v in x.items()}

    def each(self, fn):
        return {s: fn(self.p.row_wave[self.m.pos[s]], s) for s in range(self.m.ns)}

    def rows(self, v):
        return {self.m.pos[s]: x for s, x in v.items()}

    def attempt(self, solver):
        f = self.f
        # f(y0) shares the Jacobian's products, but beside all of a wave's
        # matrix entries its sums do not fit the registers
        self.factor(self.matrix())
        f0 = self.fun(self.yc)
        # the first forward elimination runs beside the dense wave's
        k1 = self.spec(self.solve(self.rows(f0), first=self.cross + 1))
        if solver == "ros2":
            yn = self.each(lambda w, s: f.op(w, "fma(kRos2GammaInv, {0}, {1})", [k1[s], self.yc[s]]))
            ft = self.fun(yn)
            b = self.each(lambda w, s: f.op(w, "fma(-2.0 * kRos2GammaInv * dti, {0}, {1})", [k1[s], ft[s]]))
            k2 = self.spec(self.solve(self.rows(b)))
            self.each(lambda w, s: f.op(
                w, "coop_end_ros2({0}, {1}, {2}, atol[%d], rtol[%d], yn[%d], e);" % (s, s, self.p.idx[s]),
                [k1[s], k2[s], self.yc[s]], cost=22.0, outs=0))
            return
        b = self.each(lambda w, s: f.op(w, "fma(4.0 * dti, {0}, {1})", [k1[s], f0[s]]))
        k2 = self.spec(self.solve(self.rows(b)))
        yk = self.each(lambda w, s: f.op(w, ["@DECL2", "  coop_stage3({0}, {1}, $0$, $1$);"],
                                         [k1[s], self.yc[s]], cost=4.0, outs=2))
        yn, k1 = {s: v[0] for s, v in yk.items()}, {s: v[1] for s, v in yk.items()}
        ft = self.fun(yn)
        d = self.each(lambda w, s: f.op(w, "{0} - {1}", [k1[s], k2[s]]))
        b = self.each(lambda w, s: f.op(w, "fma(dti, {0}, {1})", [d[s], ft[s]]))
        k3 = self.spec(self.solve(self.rows(b)))
        yk = self.each(lambda w, s: f.op(w, ["@DECL2", "  coop_stage4({0}, {1}, {2}, $0$, $1$);"],
                                         [k1[s], k3[s], self.yc[s]], cost=6.0, outs=2))
        yn, k3 = {s: v[0] for s, v in yk.items()}, {s: v[1] for s, v in yk.items()}
        ft = self.fun(yn)
        b = self.each(lambda w, s: f.op(w, "fma(dti, fma(-(8.0 / 3.0), {0}, {1}), {2})", [k3[s], d[s], ft[s]], cost=2.0))
        k4 = self.spec(self.solve(self.rows(b)))
        self.each(lambda w, s: f.op(
            w, "coop_end_rodas3({0}, {1}, {2}, {3}, atol[%d], rtol[%d], yn[%d], e);" % (s, s, self.p.idx[s]),
            [k1[s], k3[s], k4[s], self.yc[s]], cost=24.0, outs=0))


class Layout:
    """LDS slots of a section's exchanged values, and the section's code."""

    def __init__(self, flow, nfix, waves):
        flow.level(waves)
        flow.settle()
        self.f, self.waves, self.P = flow, waves, flow.phases()
        vals = []
        for o in flow.ops:
            for v in o.outs:
                later = [u for u in v.uses if u[0] != v.wave or (v.home == "park" and u[1] > v.phase)]
                if later:
                    vals.append((v, max(u[1] for u in later)))
        def born(v):
            return v.phase if v.store is None else v.store

        # first fit by birth; a slot is free again one phase after its last read
        busy = []                                           # slot -> last phase in use
        end = {id(v): last for v, last in vals}
        for v, last in vals:
            if v.into is not None and id(v.into) in end:
                end[id(v.into)] = max(end[id(v.into)], last)
        for v, last in sorted(vals, key=lambda t: born(t[0])):
            if v.into is not None and id(v.into) in end:
                continue
            last = end[id(v)]
            for k, b in enumerate(busy):
                if b < born(v):
                    break
            else:
                busy.append(-1)
                k = len(busy) - 1
            busy[k] = last
            v.slot = nfix + k
        for v, _ in vals:
            if v.into is not None and id(v.into) in end:
                v.slot = v.into.slot
        self.slots = nfix + len(busy)
        self.writes = sum(1 for v, _ in vals)

    def stats(self, sync=180.0):
        """Modelled clocks of the section: per phase the longest of the waves
        (latency of their operations and reads), the SIMDs (two waves' issue)
        and the LDS transfers, plus the barrier."""
        ops = [[0.0] * self.waves for _ in range(self.P)]
        reads = [[0] * self.waves for _ in range(self.P)]
        lds = [0] * self.P
        seen = set()
        for o in self.f.ops:
            if o.count_only:
                continue
            ops[o.phase][o.wave] += o.cost
            for v in o.ins:
                if self.remote(v, o.wave, o.phase):
                    k = (id(v), o.wave, o.phase)
                    if k not in seen:
                        seen.add(k)
                        lds[o.phase] += 1
                        reads[o.phase][o.wave] += 1
            for v in o.outs:
                if v.slot is not None:
                    lds[o.phase] += 1
                    reads[o.phase][o.wave] += 1
        rows = []
        for ph in range(self.P):
            wave = max(5.5 * a + 4.0 * r for a, r in zip(ops[ph], reads[ph]))
            simd = max(sum(4.6 * ops[ph][w] + 3.0 * reads[ph][w] for w in range(s, self.waves, 4)) for s in range(4))
            rows.append((round(wave), round(simd), round(2.8 * lds[ph])))
        return sum(max(r) for r in rows) + sync * self.P, rows, sum(lds)

    def remote(self, v, w, ph):
        """Whether wave w reads v from LDS in phase ph."""
        return v.home != "free" and not (v.wave == w and not (v.home == "park" and ph > v.phase))

    def emit(self, w, chunk=CHUNK, keep=KEEP, ahead=AHEAD):
        """Code of wave w, phases separated by coop_barrier().

        A phase runs in chunks of `chunk` operations with a scheduling fence
        between them: each chunk's LDS reads are issued with the chunk before
        it, and a value read stays in a register for the `keep` chunks after
        its use, else it is read again.  Left to itself the compiler's
        scheduler issues the reads of a whole phase first and spills."""
        out, n = [], 0
        for ph in range(self.P):
            ops = [o for o in self.f.ops if o.wave == w and o.phase == ph]
            parts = [ops[k:k + chunk] for k in range(0, len(ops), chunk)] or [[]]
            # reads of each chunk, and the name each value has there
            names, reads, alive = [], [[] for _ in parts], {}
            for c, part in enumerate(parts):
                here = {}
                for o in part:
                    if o.count_only:
                        continue
                    for v in o.ins:
                        if not self.remote(v, w, ph) or id(v) in here:
                            continue
                        if id(v) in alive and c - alive[id(v)][1] <= keep:
                            here[id(v)] = alive[id(v)][0]
                        else:
                            here[id(v)] = "r%d" % n
                            n += 1
                            reads[c].append((here[id(v)], v.slot))
                        alive[id(v)] = (here[id(v)], c)
                names.append(here)

            def issue(c):
                for name, slot in reads[c]:
                    out.append("  const double %s = S.get(%d);" % (name, slot))
            for c in range(min(ahead, len(parts))):
                issue(c)
            for c, part in enumerate(parts):
                if c + ahead < len(parts):
                    issue(c + ahead)
                for o in part:
                    if o.count_only:
                        args = [v.expr if not self.remote(v, w, ph) else names[c].get(id(v), "S.get(%d)" % v.slot)
                                for v in o.ins]
                        out.append("  " + o.text.format(*args))
                        continue
                    args = [names[c][id(v)] if self.remote(v, w, ph) else v.expr for v in o.ins]
                    if isinstance(o.text, list):
                        outs = [v.expr for v in o.outs]
                        for line in o.text:
                            if line == "@DECL":
                                out.append("  double " + ", ".join("%s = %s" % t for t in zip(outs, args)) + ";")
                            elif line == "@DECL2":
                                out.append("  double %s;" % ", ".join(outs))
                            else:
                                for k, x in enumerate(outs):
                                    line = line.replace("$%d$" % k, x)
                                for k, x in enumerate(args):
                                    line = line.replace("{%d}" % k, x)
                                out.append(line)
                    elif not o.outs:
                        out.append("  " + o.text.format(*args))
                    else:
                        out.append("  const double %s = %s;" % (o.outs[0].expr, o.text.format(*args)))
                    for v in o.outs:
                        if v.slot is not None and v.store is None:
                            only_count = all(v_users_count(self.f, v))
                            st = "S.put(%d, %s);" % (v.slot, v.expr)
                            out.append("  if constexpr (COUNT) { %s }" % st if only_count else "  " + st)
                if c + 1 < len(parts):
                    out.append("  coop_fence();")
            for o in self.f.ops:
                if o.wave == w:
                    for v in o.outs:
                        if v.store == ph:
                            only_count = all(v_users_count(self.f, v))
                            st = "S.put(%d, %s);" % (v.slot, v.expr)
                            out.append("  if constexpr (COUNT) { %s }" % st if only_count else "  " + st)
            if ph + 1 < self.P:
                out.append("  coop_barrier();")
        return out


def v_users_count(flow, v):
    """For each use of v by another wave (or after parking): whether it is a count-only use."""
    if not hasattr(flow, "_users"):
        u = {}
        for o in flow.ops:
            for x in o.ins:
                if x.home != "free":
                    u.setdefault(id(x), []).append(o)
        flow._users = u
    return [o.count_only for o in flow._users.get(id(v), [])
            if o.wave != v.wave or (v.home == "park" and o.phase > v.phase)]


def kinetic_shares(waves, cost):
    """Reactions of each wave's share of the rate laws, largest first to the
    least loaded wave."""
    load, share = [0.0] * waves, [[] for _ in range(waves)]
    for r in sorted(cost, key=lambda r: (-cost[r], r)):
        w = min(range(waves), key=lambda w: (load[w], w))
        load[w] += cost[r]
        share[w].append(r)
    return [sorted(x) for x in share]


FAMILY_COST = {"arrhenius": 45, "arrhenius_tn": 50, "m_power": 160, "exp_plus_m_exp": 90, "troe": 420,
               "troe_ca": 700, "hno3_oh": 150, "m_exp_h2o": 100}


def law_cost(law):
    c = FAMILY_COST.get(law["family"], 2)
    if law["family"] == "exp_sum":
        c = 45 * ((len(law["params"]) - 1) // 3)
    for q in law["post"]:
        c += 420 if q[0] == "mul_troe" else 2
    return c


def emit(m, plan, reactions, rate_line, name, mech_name):
    """Text of the generated header: one struct a wave."""
    W = plan.waves
    L = []
    w_ = L.append
    secs = {}
    slots = 0
    for solver in ("rodas3", "ros2"):
        b = Builder(plan)
        b.attempt(solver)
        lay = Layout(b.f, plan.nfix, W)
        secs[solver] = lay
        slots = max(slots, lay.slots)
    eslot = slots
    slots += W                       # error partials
    vslot = slots
    vwords = (m.ns + 31) // 32
    slots += (vwords + 1) // 2       # pivots failing the threshold rule, 32-bit words
    mslot = slots
    slots += 1                       # mask words on their way to memory
    if slots > LDS_SLOTS:
        raise ValueError("%s: %d LDS slots of %d" % (mech_name, slots, LDS_SLOTS))
    w_("// Generated by brams_amd/codegen/gen_coop.py from brams_amd/mechanism/%s.json." % name)
    w_("// One block's attempt spread over %d waves: RODAS3 in %d phases, ROS2 in %d;" % (
        W, secs["rodas3"].P, secs["ros2"].P))
    w_("// the last %d pivots on wave %d; %d rate constants in LDS.  Modelled clocks of an" % (
        plan.dense, plan.dw, len(plan.rk_lds)))
    w_("// attempt, barriers included: %d and %d." % (secs["rodas3"].stats()[0], secs["ros2"].stats()[0]))
    w_("#pragma once")
    w_("#define MECH_COOP_WAVES %d" % W)
    w_("#define MECH_COOP_SLOTS %d" % slots)
    w_("#define MECH_COOP_ESLOT %d" % eslot)
    w_("#define MECH_COOP_VSLOT %d" % vslot)
    w_("#define MECH_COOP_VWORDS %d" % vwords)
    w_("#define MECH_COOP_MSLOT %d" % mslot)
    w_("")
    shares = kinetic_shares(W, {r: law_cost(reactions[r]["rate"]) for r in plan.rk_lds})
    nwords = (len(m.sidx) + 31) // 32
    for w in range(W):
        own = plan.own[w]
        n = max(1, len(own))
        w_("struct CoopWave%d {" % w)
        w_("  static constexpr int kOwn = %d;" % len(own))
        w_("  // species (0-based); a species' concentration lies in the slot of its number")
        w_("  static constexpr int own[%d] = {%s};" % (n, ", ".join(map(str, own)) or "0"))
        mo = [plan.mask_own[w].get(q, 0) for q in range(nwords)]
        w_("  static constexpr unsigned mask_own[%d] = {%s};" % (nwords, ", ".join("0x%08xu" % v for v in mo)))
        w_("  // this wave's share of the rate laws (chem_spack_kinetic.f90), into LDS")
        w_("  static __device__ __forceinline__ void kinetic(double T, double P, double vapp, const double* J, const CoopLds& S) {")
        w_("    const double M = P * 7.243e16 / T;")
        w_("    const double H2O = 29.0 * M * vapp / (18.0 + 11.0 * vapp);")
        w_("    const double lnT = log(T);")
        w_("    (void)M; (void)H2O; (void)lnT; (void)J;")
        for r in shares[w]:
            w_("    S.put(%d, %s);" % (plan.rkslot[r], rate_line(r)))
        w_("  }")
        for solver in ("rodas3", "ros2"):
            w_("  template <bool DYN, bool COUNT>")
            w_("  static __device__ __forceinline__ void %s(const CoopLds& S," % solver)
            w_("      double igdt, double dti, unsigned* mw, bool dyn, const double* atol, const double* rtol,")
            w_("      double* yn, double& e, unsigned* viol) {")
            L.extend("  " + x for x in secs[solver].emit(w))
            w_("  }")
        w_("};")
        w_("")
    return "\n".join(L) + "\n"


def default_rows(m, waves, dense):
    """Rows dealt to the waves by their work where no placement is on file."""
    t0 = m.ns - dense
    cost = []
    for I in range(m.ns):
        c = sum(2 * len(m.react[r]) for _, r in m.prod.get(m.perm[I], []))
        c += sum(sum(m.F[K][J] for J in range(K + 1, m.ns)) for K in range(min(I, t0)) if m.F[I][K])
        cost.append(c + 4 * sum(m.F[I]) + 40)
    rows, load = [None] * m.ns, [0.0] * waves
    load[waves - 1] = sum(cost) / waves * 0.8
    for I in sorted(range(m.ns), key=lambda I: (-cost[I], I)):
        w = min(range(waves), key=lambda w: (load[w], w))
        rows[I] = w
        load[w] += cost[I]
    return rows


def literal_rates(reactions):
    """Rate constants that depend on neither T, p nor J: {reaction: text}."""
    out = {}
    for r, rx in enumerate(reactions):
        law = rx["rate"]
        if law["family"] in ("constant", "unset") and not law["post"]:
            out[r] = lit(law["params"][0]) if law["params"] else "0.0"
    return out
