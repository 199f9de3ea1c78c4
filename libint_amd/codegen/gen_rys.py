"""Generator of the Rys-quadrature kernels: a tile of lanes per shell quartet.

The contracted targets [e0|f0] of a class are sums over its primitive quartets
and the nodes r of the n-point Rys rule (n = L // 2 + 1) of products of
two-dimensional integrals (M. Dupuis, J. Rys, H. F. King, J. Chem. Phys. 65,
111 (1976)),

  [e0|f0] = sum_p sum_r X_pr(ex, fx) Y_pr(ey, fy) Z_pr(ez, fz),

followed by the same horizontal recurrences, solid-harmonic transforms and
store or digest as the per-lane kernels of gen_eri.py.

Mapping to the hardware.  A lane owns one or two components e of one quartet
and keeps its accumulators for every f in registers, so a quartet takes a tile
of ceil(ne / 2) (or ne) lanes instead of one lane that has to walk its targets
in groups and recompute shared recursion for each.  A block of 1, 2 or 4 waves
holds as many quartets as fit.  Per batch of NB primitive quartets:

  0. primitive stage: a lane per (primitive, quartet) evaluates prefactors and
     screening and leaves a record of 15 doubles in LDS (evaluated by every
     lane of the root stage instead, the light classes spent 40 % of their
     instructions on it: (pp|dp) 0.067 -> 0.053 ns a primitive quartet);
  1. root stage: a lane per (primitive, quartet, node) evaluates node and
     weight from the table (codegen/rys_table.py);
  2. 2D stage: a lane per (quartet, node, axis) runs the two-index recurrence
     and leaves its (na+1)(nc+1) values in LDS;
  3. product stage: a lane reads the rows of its components per axis and does
     one fused multiply-add per target and node, the products X(fx) Y(fy)
     shared by the two components of its tile (they differ on one axis only).
     The nodes of a primitive quartet are summed before they are added to the
     accumulators: on ill-conditioned deep (dd|dd) quartets adding every node
     to the accumulators left 1.9 times the Obara-Saika sum's rounding error
     (n times as many roundings at the accumulators' size), summing them
     first 0.95 times.  Where targets, their node sums and the rows do not fit
     the registers of two waves per SIMD, the targets are done in parts.

Per primitive quartet (dd|dd) takes about 500 x 16 lane operations in the
product stage where the Obara-Saika kernels evaluate 4123 recursion nodes of
two to five operations with half of the live values in accumulation registers.
Measured per class on an MI355X, K = 6 shells (77 primitive quartets a quartet
on average), when the kernels came: 34,000 (dd|dd) quartets 55.6 -> 2.0 ms,
40,000 (dp|dp) 11.0 -> 0.71 ms, 40,000 (pp|pp) 2.35 -> 0.37 ms, 2,200 (fd|fd)
3.9 -> 0.60 ms, 1,000 (ff|ff) 17 -> 2.4 ms; what bounds the heavy ones is the FP64 VALU: of the 820
instructions a wave issues per primitive quartet of (dd|dd) 60 % are the
product stage's multiplies and adds.
The contracted block then goes through LDS: a lane per bra component for the
ket recurrence, a lane per ket function for the bra recurrence, and coalesced
stores (or, in J/K builds, a lane per element of the six Fock blocks).
"""
from __future__ import annotations

import functools
import random

import gen_eri as ge
import rys_table

REC = 15


def comps(l1, l2):
    return [c for l in range(l1, l1 + l2 + 1) for c in ge.cart(l)]


@functools.lru_cache(maxsize=None)
def pair_tiles(cs):
    """Components in tiles of two that share two axes: (axis they differ on, i, j); a component left over pairs with itself."""
    n = len(cs)
    adj = [[j for j in range(n) if j != i and sum(a != b for a, b in zip(cs[i], cs[j])) == 1] for i in range(n)]
    best = None
    rng = random.Random(1)
    for _ in range(400):
        free, pairs = set(range(n)), []
        while free:
            deg = {i: sum(j in free for j in adj[i]) for i in free}
            i = min(free, key=lambda k: (deg[k] or 99, rng.random()))
            free.remove(i)
            c = [j for j in adj[i] if j in free]
            if not c:
                pairs.append((2, i, i))
                continue
            j = min(c, key=lambda k: (deg[k], rng.random()))
            free.remove(j)
            ax = next(a for a in range(3) if cs[i][a] != cs[j][a])
            pairs.append((ax, i, j))
        if best is None or len(pairs) < len(best):
            best = pairs
        if len(best) == (n + 1) // 2:
            break
    return sorted(best)


@functools.lru_cache(maxsize=None)
def split_parts(inner, n):
    """The inner components in n parts by their power on axis C: indices of each part, the largest part as
    small as can be, then the fewest X Y products."""
    cs = sorted({f[2] for f in inner})
    best = None

    def go(k, groups):
        nonlocal best
        if k == len(cs):
            if all(groups):
                parts = [[i for i, f in enumerate(inner) if f[2] in g] for g in groups]
                c = (max(map(len, parts)) // 2, sum(len({inner[i][:2] for i in x}) for x in parts), max(map(len, parts)))
                if best is None or c < best[0]:
                    best = (c, parts)
            return
        for g in range(n):
            go(k + 1, groups[:g] + [groups[g] | {cs[k]}] + groups[g + 1:])
            if not groups[g]:
                break
    if n > len(cs):
        return None
    go(0, [set() for _ in range(n)])
    return best[1]


class Plan:
    """Layout of one class: side of the lanes, tile, waves, quartets per block."""

    def __init__(self, la, lb, lc, ld, side, te, nw, nparts, rl=False, nb=None):
        self.l = (la, lb, lc, ld)
        self.side, self.te, self.nw, self.rl = side, te, nw, rl
        self.ecs, self.fcs = comps(la, lb), comps(lc, ld)
        self.ne, self.nf = len(self.ecs), len(self.fcs)
        self.na, self.nc = la + lb, lc + ld
        self.nr = (la + lb + lc + ld) // 2 + 1
        self.outer, self.inner = (self.ecs, self.fcs) if side == 'bra' else (self.fcs, self.ecs)
        self.no, self.ni = (self.na, self.nc) if side == 'bra' else (self.nc, self.na)
        self.tiles = pair_tiles(tuple(self.outer)) if te == 2 else [(2, i, i) for i in range(len(self.outer))]
        self.nl = len(self.tiles)
        self.nt = 64 * nw
        self.q = self.nt // self.nl
        self.parts = self.split(nparts)
        self.gb = ((self.no + 1) * (self.ni + 1)) | 1          # doubles of one axis block (odd: no bank conflicts)
        if self.q == 0:
            return
        self.ng = 1 if rl else self.nr   # nodes whose 2D integrals are in LDS at a time
        self.nb = nb
        self.root_rounds = -(-self.q * nb * self.nr // self.nt) / nb
        self.prim_rounds = -(-self.q * nb // self.nt) / nb
        # row stride of the contracted block in LDS (odd), and doubles per
        # quartet of a pass: with every shell a solid harmonic / Cartesian
        self.rstr = max(self.nf, ge.ncart(lc) * ge.ncart(ld)) | 1
        self.erow = self.ne * self.rstr
        self.lds_main = self.nb * self.q * (2 * self.nr + REC) + self.q * self.ng * 3 * self.gb

    def split(self, n):
        return split_parts(tuple(self.inner), n)

    def nxy(self, part):
        return len({self.inner[i][:2] for i in part})

    def rows_of(self, part):
        """Powers read on axes A, B, C for a part."""
        return [sorted({self.inner[i][a] for i in part}) for a in range(3)]

    def dims(self, pure):
        return [2 * l + 1 if pure and l >= 2 else ge.ncart(l) for l in self.l]

    def layout(self, mode, pure):
        """(quartets per pass, passes, LDS doubles of each, offset of the finished block in them).  The block goes over
        the rows it is made from where a pass has at most one column a lane (every row is read before), else behind
        them, and a lane loops over its columns; whichever takes fewer passes."""
        n = self.dims(pure)
        nv = n[0] * n[1] * n[2] * n[3]
        tail = sum(n[i] * n[j] for i in range(4) for j in range(i + 1, 4)) if mode == 'fock' else 0
        # LDS that leaves the occupancy to the registers
        cap = max(self.lds_main, (163840 // (4 * min(4, 512 // self.regs())) * self.nw - 144 * self.q) // 8)
        ncol = n[2] * n[3]
        best = None
        for over in (True, False):
            if over:  # a block that does not fit over its rows is stored directly by an ERI batch
                d = self.erow if mode == 'eri' else max(self.erow, nv + tail)
            else:
                d = self.erow + nv + tail
            if not over and ncol > self.nt and d > cap:
                continue
            qp = max(1, min(self.q, cap // d, self.nt // ncol if over else self.q))
            np_ = -(-self.q // qp)
            qp = -(-self.q // np_)
            if best is None or np_ < best[1]:
                best = (qp, np_, d, 0 if over else self.erow)
        return best

    def passes(self, mode, pure=True):
        return self.layout(mode, pure)[:2]

    def lds_doubles(self, mode):
        lay = [self.layout(mode, x) for x in (True, False)]
        return max([self.lds_main] + [x[0] * x[2] for x in lay])

    def lds_bytes(self, mode):
        return 8 * self.lds_doubles(mode) + self.q * 72 + (self.q * 128 if mode == 'fock' else 0)

    def occupancy(self):
        """Waves per SIMD that registers and LDS allow."""
        return max(1, min(4, 512 // max(1, self.regs()), int(163840 / (self.lds_bytes('fock') / self.nw) / 4)))

    def cost(self):
        """Lane operations per primitive quartet (product, 2D, root and primitive stages), over the share of the VALU that so many
        waves per SIMD were seen to fill, or the LDS clocks where those are more."""
        main = self.nr * (self.te * len(self.inner) + sum(self.nxy(x) for x in self.parts)) + self.te * len(self.inner)
        reads = self.nr * sum(len(a) + len(b) + self.te * len(c) for a, b, c in map(self.rows_of, self.parts))
        rounds = self.nr // self.ng * -(-self.q * self.ng * 3 // self.nt)
        two = rounds * (3.5 * (self.na + 1) * (self.nc + 1) + 40)
        root = self.prim_rounds * 150 + self.root_rounds * 85 + 60 / self.nb
        valu = main + reads // 2 + two + root + 30
        lds = (reads + rounds * (self.gb + 12)) * 4.0  # quarter clocks of the CU's LDS for four SIMDs
        return max(valu / {1: 0.35, 2: 0.6, 3: 0.75, 4: 0.85}[self.occupancy()], lds / 0.8) * self.nt / self.q * \
            (1.05 if self.nw > 1 else 1.0)

    def regs(self):
        rows = max(len(a) + len(b) + self.te * len(c) for a, b, c in map(self.rows_of, self.parts))
        return 2 * (self.te * (len(self.inner) + max(map(len, self.parts))) + rows) + 34


# Layouts that measured faster than the model's choice: (side, tile, waves, node by node, parts, batch), with the
# nanoseconds per primitive quartet of the model's choice and of this one on one MI355X (ERI batches of
# 25,000 to 150,000 quartets, 80 primitive quartets each on average).
TUNED = {
    '0021': ('ket', 1, 1, False, 1, 12),  # 0.064 -> 0.054
    '0022': ('ket', 2, 1, False, 1, 12),  # 0.081 -> 0.076
    '0030': ('bra', 1, 1, True, 1, 1),  # 0.059 -> 0.049
    '0031': ('ket', 2, 1, False, 1, 12),  # 0.087 -> 0.074
    '0033': ('ket', 2, 2, False, 1, 16),  # 0.276 -> 0.235
    '1010': ('ket', 1, 1, True, 1, 3),  # 0.047 -> 0.043
    '1020': ('bra', 1, 1, True, 1, 3),  # 0.052 -> 0.051
    '1021': ('bra', 1, 1, True, 1, 2),  # 0.091 -> 0.088
    '1022': ('bra', 1, 1, True, 1, 3),  # 0.144 -> 0.115
    '1030': ('bra', 1, 1, True, 1, 2),  # 0.085 -> 0.082
    '1031': ('bra', 1, 1, True, 1, 2),  # 0.103 -> 0.103, the loop of few quartets is shorter
    '1033': ('ket', 2, 2, False, 1, 16),  # 0.428 -> 0.350
    '1120': ('ket', 1, 1, False, 1, 4),  # 0.113 -> 0.097
    '1132': ('bra', 1, 1, False, 1, 3),  # 0.496 -> 0.403
    '2011': ('bra', 1, 1, False, 1, 4),  # 0.112 -> 0.098
    '2020': ('bra', 1, 1, False, 1, 4),  # 0.099 -> 0.095
    '2021': ('bra', 1, 1, True, 1, 4),  # 0.167 -> 0.135
    '2022': ('ket', 2, 1, False, 1, 8),  # 0.202 -> 0.196
    '2031': ('bra', 1, 1, False, 1, 4),  # 0.223 -> 0.197
    '2032': ('bra', 1, 2, True, 1, 6),  # 0.304 -> 0.294
    '2033': ('ket', 2, 2, False, 1, 16),  # 0.622 -> 0.568
    '2121': ('ket', 1, 1, False, 1, 8),  # 0.212 -> 0.206
    '2133': ('bra', 1, 1, False, 3, 16),  # 1.195 -> 1.021
    '2232': ('bra', 1, 1, False, 1, 16),  # 1.312 -> 0.803
    '3030': ('ket', 1, 1, False, 1, 8),  # 0.288 -> 0.274
    '3032': ('bra', 1, 1, False, 1, 1),  # 0.666 -> 0.504
    '3033': ('ket', 2, 2, False, 1, 16),  # 0.925 -> 0.895
    '3132': ('bra', 1, 1, False, 1, 16),  # 1.115 -> 0.798
    '3133': ('ket', 1, 4, False, 1, 16),  # 2.074 -> 1.593
}


@functools.lru_cache(maxsize=None)
def plan(la, lb, lc, ld):
    best = None
    if f"{la}{lb}{lc}{ld}" in TUNED:
        side, te, nw, rl, nparts, nb = TUNED[f"{la}{lb}{lc}{ld}"]
        return Plan(la, lb, lc, ld, side, te, nw, nparts, rl, nb)
    for side in ('bra', 'ket'):
        for te in (1, 2):
            for nw in (1, 2, 4):
                for rl, nparts in ((True, 1), (False, 1), (False, 2), (False, 3)):
                    for nb in (1, 2, 3, 4, 6, 8, 12, 16):
                        p = Plan(la, lb, lc, ld, side, te, nw, nparts, rl, nb)
                        if p.parts is None or p.q == 0 or p.regs() > 270 or p.lds_bytes('fock') > 150 * 1024:
                            continue
                        if nb > 1 and p.q * nb > p.nt:
                            continue
                        c = p.cost()
                        if best is None or c < best[0]:
                            best = (c, p)
    return best[1]


def emit(p, mode):
    la, lb, lc, ld = p.l
    E = ge.Emitter()
    ge._R = 'double'
    ge._FUSED = True
    name = f"l2g_rys_{mode}_{la}{lb}{lc}{ld}"
    NT, Q, NL, NR, NB, NW = p.nt, p.q, p.nl, p.nr, p.nb, p.nw
    lay = {x: p.layout(mode, x) for x in (True, False)}
    qps, regs_, vofs = ({x: lay[x][k] for x in lay} for k in (0, 2, 3))
    QP = max(qps.values())
    ni1, no1 = p.ni + 1, p.no + 1
    swz = [(0, 1, 2), (0, 2, 1), (1, 2, 0)]  # axes (A, B, C) by C axis z, y, x
    order = {2: swz[0], 1: swz[1], 0: swz[2]}
    E(f"// class ({la}{lb}|{lc}{ld}): {p.ne} x {p.nf} targets, {NR} nodes; lanes on the {p.side}, tiles of {p.te}, "
      f"{NL} lanes a quartet, {Q} quartets a block of {NT}")
    # per tile: LDS offsets of rows A, B, C0, C1 within a node's three axis blocks, C axis, components
    rows = []
    for ax, i, j in p.tiles:
        a, b, c = order[ax]
        ci, cj = p.outer[i], p.outer[j]
        off = [a * p.gb + ci[a] * ni1, b * p.gb + ci[b] * ni1, c * p.gb + ci[c] * ni1, c * p.gb + cj[c] * ni1]
        assert max(off) < 256 and max(i, j) < 128
        rows.append((off[0] | off[1] << 8 | off[2] << 16 | off[3] << 24, i | j << 8 | ax << 16))
    E(f"static __device__ const unsigned {name}_tab[{2 * NL}] = {{" +
      ', '.join(f"{x}u" for r in rows for x in r) + "};")
    lb2 = p.occupancy()
    E(f"__global__ void __launch_bounds__({NT}, {lb2}) {name}(const L2gEriArgs A) {{")
    E.ind += 1
    E(f"__shared__ double sm[{p.lds_doubles(mode)}];")
    E(f"__shared__ RysItem items[{Q}];")
    if mode == 'fock':
        E(f"__shared__ RysDigest dig[{QP}];")
    uw, rec = 0, NB * Q * NR * 2
    g0 = rec + NB * Q * REC
    E("const int tid = threadIdx.x;")
    if mode == 'fock':  # deep items are cut into ranges before the launch
        E(f"constexpr int S = 1, NI = {Q};")
        E(f"const struct {{ int first, end; }} tier = {{(int)blockIdx.x * {Q}, A.n}};")
    else:
        E("// S slots of the block share a work item (tiers of deep items first, see RysTier), each a part of its")
        E("// primitive quartets")
        E(f"const RysTier<{Q}> tier(A, blockIdx.x);")
        E("const int S = tier.S, NI = tier.NI;")
    E.block(f"if (tid < {Q})")
    E("RysItem I;")
    E("const int qi = tier.first + tid / S;")
    E("I.qi = tid < NI * S && qi < tier.end ? qi : -1;")
    E("I.nsurv = 0;")
    E("I.pb0 = I.pk0 = I.npk = I.pbeg = I.pend = I.bp = I.kp = I.meta = 0;")
    E("I.lnprec = A.ln_precision, I.qprec = A.precision, I.npbk = I.rnpk = 0.0;")
    E.block("if (I.qi >= 0)")
    E("I.bp = A.bra_pair[qi], I.kp = A.ket_pair[qi], I.meta = A.meta[qi];")
    E("I.pb0 = A.pair_first[I.bp], I.pk0 = A.pair_first[I.kp];")
    E("const int npb = A.pair_np[I.bp];")
    E("I.npk = A.pair_np[I.kp];")
    E("I.npbk = (double)npb * (double)I.npk;")
    E("I.rnpk = 1.0 / I.npk;")
    E("I.pend = npb * I.npk;")
    E("if (A.q_prange) I.pbeg = A.q_prange[qi].x, I.pend = A.q_prange[qi].y;")
    if mode == 'eri':
        E("I.pbeg <<= A.erfc, I.pend <<= A.erfc;")
    if mode == 'eri':
        E.block("if (S > 1)")
        E("const int b = I.pbeg, n = I.pend - b, k = tid % S;")
        E("I.pbeg = b + (int)((long long)n * k / S), I.pend = b + (int)((long long)n * (k + 1) / S);")
        E.end()
    if mode == 'fock':
        E("I.lnprec = A.q_lnprec[qi];")
        E("I.qprec = A.method == L2G_SCREEN_ORIGINAL || A.method == L2G_SCREEN_CONSERVATIVE ? exp(I.lnprec) : 0.0;")
    E.end()
    E("items[tid] = I;")
    E.end()
    E(f"rys_sync<{NW}>();")
    E("int len = 0;")
    E(f"for (int q = 0; q < {Q}; ++q) len = max(len, items[q].pend - items[q].pbeg);")
    E("len = __builtin_amdgcn_readfirstlane(len);")
    # product-stage role
    E(f"const int mq = min(tid / {NL}, {Q - 1}), mt = tid % {NL};")
    E(f"const bool mlive = tid < {Q * NL};")
    E(f"const unsigned tofs = {name}_tab[2 * mt], tinf = {name}_tab[2 * mt + 1];")
    E(f"const double* const gq = sm + {g0} + mq * {p.ng * 3 * p.gb};")
    E("const double* const rA = gq + (tofs & 255u);")
    E("const double* const rB = gq + ((tofs >> 8) & 255u);")
    E("const double* const rC = gq + ((tofs >> 16) & 255u);")
    if p.te == 2:
        E("const double* const rD = gq + (tofs >> 24);")
    for t in range(p.te):
        for k in range(len(p.inner)):
            E(f"double a{t}_{k} = 0.0;")
    E(f"const double* __restrict__ tab = A.rys + {rys_table.offset(NR)};")
    if mode == 'eri':
        E("if (A.gpart_mode == 2) len = 0;  // the contracted values come from the pieces")
    E.block(f"for (int p0 = 0; p0 < len; p0 += {NB})")
    E(f"const int nbat = min({NB}, len - p0);")

    def lanes(n, per):  # a lane per item of the batch
        if NB * per > NT:
            E.block(f"for (int it = tid; it < {n}; it += {NT})")
        else:
            E("const int it = tid;")
            E.block(f"if (it < {n})")
    # primitive stage
    E.block("")
    lanes(f"nbat * {Q}", Q)
    E(f"const int b = it / {Q}, q = it - b * {Q};")
    E(f"rys_prim(A, items[q], items[q].pbeg + p0 + b, sm + {rec} + it * {REC});")
    E.end()
    E.end()
    E(f"rys_sync<{NW}>();")
    # root stage
    E.block("")
    lanes(f"nbat * {Q * NR}", Q * NR)
    E(f"const int bq = it / {NR}, r = it - bq * {NR};")
    E(f"const double* const rc = sm + {rec} + bq * {REC};")
    E("double u, w;")
    E(f"rys_root<{NR}>(rc[13], tab, r, u, w);")
    E(f"sm[{uw} + it * 2] = u, sm[{uw} + it * 2 + 1] = w * rc[14];")
    E.end()
    E.end()
    E(f"rys_sync<{NW}>();")
    E("#pragma unroll 1")
    E.block("for (int b = 0; b < nbat; ++b)")
    # 2D stage
    if p.rl:
        for t in range(p.te):
            E("double " + ', '.join(f"t{t}_{k} = 0.0" for k in range(len(p.inner))) + ";")
        E("#pragma unroll 1")
        E.block(f"for (int r = 0; r < {NR}; ++r)")
    n2 = Q * p.ng * 3
    rounds = -(-n2 // NT)
    if rounds > 1:
        E.block(f"for (int it = tid; it < {n2}; it += {NT})")
    else:
        E("const int it = tid;")
        E.block(f"if (it < {n2})")
    E("const int qr = it / 3, ax = it - qr * 3;")
    if p.rl:
        E(f"const int q = qr, node = (b * {Q} + q) * {NR} + r;")
    else:
        E(f"const int q = qr / {NR}, node = b * {Q * NR} + qr;")
    E(f"const double* const rc = sm + {rec} + (b * {Q} + q) * {REC};")
    E(f"const double u = sm[{uw} + node * 2], w = sm[{uw} + node * 2 + 1];")
    E("const double ug = u * rc[9], up = u * rc[10], PQ = rc[ax * 3 + 2];")
    E("const double C00 = fma(-ug, PQ, rc[ax * 3]), D00 = fma(up, PQ, rc[ax * 3 + 1]);")
    E("const double B00 = up * rc[11], B10 = fma(-ug, rc[11], rc[11]), B01 = fma(-up, rc[12], rc[12]);")
    E("(void)C00; (void)D00; (void)B00; (void)B10; (void)B01;")
    E(f"double* const g = sm + {g0} + it * {p.gb};")
    E("const double g_0_0 = ax == 2 ? w : 1.0;")
    for k in range(2, p.na + 1 if p.na > 1 else 1):
        if k < p.na:
            E(f"const double B10_{k} = {k}.0 * B10;")
    for k in range(2, p.nc):
        E(f"const double B01_{k} = {k}.0 * B01;")
    for k in range(2, p.na + 1):
        E(f"const double B00_{k} = {k}.0 * B00;")

    def m(nm, k):
        return nm if k == 1 else f"{nm}_{k}"
    for i in range(p.na):
        s = f"C00 * g_{i}_0"
        if i > 0:
            s = f"fma(C00, g_{i}_0, {m('B10', i)} * g_{i - 1}_0)"
        E(f"const double g_{i + 1}_0 = {s};")
    for j in range(p.nc):
        for i in range(p.na + 1):
            s = f"D00 * g_{i}_{j}"
            if j > 0:
                s = f"fma({m('B01', j)}, g_{i}_{j - 1}, {s})"
            if i > 0:
                s = f"fma({m('B00', i)}, g_{i - 1}_{j}, {s})"
            E(f"const double g_{i}_{j + 1} = {s};")
    for i in range(p.na + 1):
        for j in range(p.nc + 1):
            o, n = (i, j) if p.side == 'bra' else (j, i)
            E(f"g[{o * ni1 + n}] = g_{i}_{j};")
    E.end()
    E(f"rys_sync<{NW}>();")
    # product stage
    E.block(f"if (mlive)") if Q * NL < NT and NW > 1 else E.block("")
    for k, part in enumerate(p.parts):
        if k:  # rows are read again: kept over the parts they would not fit the registers
            E('asm volatile("" ::: "memory");')
        E.block("")
        if not p.rl:
            for t in range(p.te):
                E("double " + ', '.join(f"t{t}_{k}" for k in part) + ";")
        rows_abc = p.rows_of(part)
        for r in range(p.ng):
            o = r * 3 * p.gb
            E.block("")
            for nm, ks in zip("ABC", rows_abc):
                for k in ks:
                    E(f"const double {nm}{k} = r{nm}[{o + k}];")
                    if nm == 'C' and p.te == 2:
                        E(f"const double D{k} = rD[{o + k}];")
            for fa, fb in sorted({p.inner[i][:2] for i in part}):
                E.block("")
                E(f"const double xy = A{fa} * B{fb};")
                for k in part:
                    f = p.inner[k]
                    if f[:2] == (fa, fb):
                        for t, nm in zip(range(p.te), "CD"):
                            E(f"t{t}_{k} = " + (f"xy * {nm}{f[2]};" if r == 0 and not p.rl else f"fma(xy, {nm}{f[2]}, t{t}_{k});"))
                E.end()
            E.end()
        if not p.rl:
            for t in range(p.te):
                for k in part:
                    E(f"a{t}_{k} += t{t}_{k};")
        E.end()
    E.end()
    E(f"rys_sync<{NW}>();")
    if p.rl:
        E.end()  # r
        for t in range(p.te):
            for k in range(len(p.inner)):
                E(f"a{t}_{k} += t{t}_{k};")
    E.end()  # b
    E.end()  # p0
    # component indices of the lane's targets
    E("const int c0 = tinf & 255, c1 = (tinf >> 8) & 255, cax = tinf >> 16;")
    E("(void)c1; (void)cax;")

    def inner_index(k):
        """physical index of the inner component whose (A, B, C) powers are inner[k], by C axis"""
        idx = {}
        for ax in (2, 1, 0):
            t = [0, 0, 0]
            for s, a in zip(p.inner[k], order[ax]):
                t[a] = s
            idx[ax] = p.inner.index(tuple(t))
        if p.te == 1 or idx[0] == idx[1] == idx[2]:
            return str(idx[2])
        return f"(cax == 2 ? {idx[2]} : cax == 1 ? {idx[1]} : {idx[0]})"

    def store_targets(base, estr, op='='):
        for t in range(p.te):
            # a tile of one component holds it twice
            single = t == 1 and op == '+=' and any(i == j for _, i, j in p.tiles)
            if single:
                E.block("if (c1 != c0)")
            for k in range(len(p.inner)):
                i = inner_index(k)
                at = f"c{t} * {estr} + {i}" if p.side == 'bra' else f"{i} * {estr} + c{t}"
                E(f"{base}[{at}] {op} a{t}_{k};")
            if single:
                E.end()
    if mode == 'eri':
        E.block("if (A.gpart_mode == 1)")
        E("// a piece: its contracted values and survivor flag, summed per quartet by the finish launch")
        E.block("if (mlive && items[mq].qi >= 0)")
        E("double* const gp = A.gpart + (long long)items[mq].qi * A.gpart_stride;")
        store_targets("gp", p.nf)
        E.end()
        E(f"if (tid < {Q} && items[tid].qi >= 0) "
          f"A.gpart[(long long)items[tid].qi * A.gpart_stride + {p.ne * p.nf}] = items[tid].nsurv;")
        E("return;")
        E.end()
    if mode == 'eri':
        E.block("if (S > 1)")
        E("// the items in front of the slots' array")
        E(f"rys_sync<{NW}>();")
        E("RysItem I;")
        E.block("if (tid < NI)")
        E("I = items[tid * S];")
        E("for (int k = 1; k < S; ++k) I.nsurv |= items[tid * S + k].nsurv;")
        E.end()
        E(f"rys_sync<{NW}>();")
        E("if (tid < NI) items[tid] = I;")
        E(f"rys_sync<{NW}>();")
        E.end()
    E("const int mi = mq / S, msub = mq - mi * S;")
    E("(void)msub;")
    E("// quartets per pass, LDS doubles of each, and their largest number of ket functions")
    E("int ncol = 0, cart = 0;")
    E.block("for (int q = 0; q < NI; ++q)")
    E("if (items[q].qi < 0) continue;")
    E("const int mt_ = items[q].meta;")
    E(f"ncol = max(ncol, ((mt_ >> 5) & 1 ? {2 * lc + 1} : {ge.ncart(lc)}) * ((mt_ >> 6) & 1 ? {2 * ld + 1} : {ge.ncart(ld)}));")
    d = [k for k in range(4) if p.l[k] >= 2]
    mask = sum(1 << (3 + k) for k in d)
    E(f"cart |= (mt_ & {mask}) != {mask};")
    E.end()
    E("ncol = __builtin_amdgcn_readfirstlane(ncol), cart = __builtin_amdgcn_readfirstlane(cart);")
    for nm, x in (("QP", qps), ("region", regs_), ("vofs", vofs)):
        E(f"const int {nm} = " + (f"{x[True]};" if x[True] == x[False] else f"cart ? {x[False]} : {x[True]};"))
    E("(void)cart;")
    E("#pragma unroll 1")
    E.block("for (int qlo = 0; qlo < NI; qlo += QP)")
    E("const int qn = min(QP, NI - qlo);")
    E(f"rys_sync<{NW}>();")
    if mode == 'eri':
        E.block("if (A.gpart_mode == 2)")
        E.block(f"for (int it = tid; it < qn * {p.ne * p.nf}; it += {NT})")
        E(f"const int qp = it / {p.ne * p.nf}, k = it - qp * {p.ne * p.nf};")
        E("const int qi = items[qlo + qp].qi;")
        E("const int x0 = qi >= 0 ? A.gpart_first[qi] : 0, x1 = qi >= 0 ? A.gpart_first[qi + 1] : 0;")
        E("const double s = rys_piece_sum(A.gpart + x0 * A.gpart_stride + k, A.gpart_stride, x1 - x0);")
        E(f"sm[qp * region + (k / {p.nf}) * {p.rstr} + k % {p.nf}] = s;")
        E.end()
        E.block("if (tid < qn && items[qlo + tid].qi >= 0)")
        E("const int qi = items[qlo + tid].qi;")
        E("const int x0 = A.gpart_first[qi], x1 = A.gpart_first[qi + 1];")
        E(f"const double s = rys_piece_sum(A.gpart + x0 * A.gpart_stride + {p.ne * p.nf}, A.gpart_stride, x1 - x0);")
        E("items[qlo + tid].nsurv = s > 0.0;")
        E.end()
        E.end()
    E("const bool mine = mlive && mi >= qlo && mi < qlo + qn" + (" && A.gpart_mode != 2;" if mode == 'eri' else ";"))
    E("double* const eb = sm + (mi - qlo) * region;")
    E.block("if (mine && msub == 0)")
    store_targets("eb", p.rstr)
    E.end()
    if mode == 'eri':
        E.block("for (int k = 1; k < S; ++k)")
        E(f"rys_sync<{NW}>();")
        E.block("if (mine && msub == k)")
        store_targets("eb", p.rstr, "+=")
        E.end()
        E.end()
    if mode == 'fock':
        E(f"if (tid < qn && items[qlo + tid].nsurv) rys_digest_setup(A, items[qlo + tid], {la}, {lb}, {lc}, {ld}, dig[tid]);")
    E(f"rys_sync<{NW}>();")
    # ket recurrence and transform: a lane per bra component
    E("#pragma unroll 1")
    E.block(f"for (int it = tid; it < qn * {p.ne}; it += {NT})")
    E(f"const int qp = it / {p.ne}, e = it - qp * {p.ne};")
    E("const int kp = items[qlo + qp].kp, meta = items[qlo + qp].meta;")
    E("const double CDx = A.pair_AB[3 * kp], CDy = A.pair_AB[3 * kp + 1], CDz = A.pair_AB[3 * kp + 2];")
    E("(void)CDx; (void)CDy; (void)CDz;")
    E(f"double* const row = sm + qp * region + e * {p.rstr};")
    for j in range(p.nf):
        E(f"const double x{j} = row[{j}];")
    vals = ge.emit_hrr(E, lc, ld, {p.fcs[j]: f"x{j}" for j in range(p.nf)}, "h", "CD")
    E.block("switch ((meta >> 5) & 3)")
    for pc, pd in ge.pure_variants(lc, ld):
        E.block(f"case {pc | (pd << 1)}:")
        _, _, v = ge.emit_sph_2(E, lc, ld, pc, pd, vals, "k")
        for col, x in enumerate(v):
            E(f"row[{col}] = {x};")
        E("break;")
        E.end()
    E("default: break;")
    E.end()
    E.end()
    E(f"rys_sync<{NW}>();")
    # bra recurrence and transform: a lane per ket function.  Where the block
    # goes over the rows, every lane reads its columns first
    ncols = {x: p.dims(x)[2] * p.dims(x)[3] for x in lay}
    rounds = max([-(-qps[x] * ncols[x] // NT) for x in lay if vofs[x] == 0], default=0)
    behind = {x for x in lay if vofs[x]}

    def columns(rd):
        if rd is None:
            E("#pragma unroll 1")
            E.block(f"for (int it = tid; it < qn * ncol; it += {NT})")
        else:
            E.block("")
            E(f"const int it = tid + {rd * NT};")
        E("const int qp = it / ncol, col = it - qp * ncol;")

    def finish(rd):
        columns(rd)
        E("const int qi = qp < qn ? items[qlo + qp].qi : -1;")
        E.block("if (qi >= 0)")
        E("const int bp = items[qlo + qp].bp, meta = items[qlo + qp].meta;")
        E(f"const int n3 = (meta >> 5) & 1 ? {2 * lc + 1} : {ge.ncart(lc)}, n4 = (meta >> 6) & 1 ? {2 * ld + 1} : {ge.ncart(ld)};")
        E.block("if (col < n3 * n4)")
        E("const double ABx = A.pair_AB[3 * bp], ABy = A.pair_AB[3 * bp + 1], ABz = A.pair_AB[3 * bp + 2];")
        E("(void)ABx; (void)ABy; (void)ABz;")
        if rd is None:
            for e in range(p.ne):
                E(f"const double y{rd}_{e} = sm[qp * region + {e * p.rstr} + col];")
        inp = {c: f"y{rd}_{e}" for e, c in enumerate(p.ecs)}
        vals = ge.emit_hrr(E, la, lb, inp, "g", "AB")
        E("const int ic = col / n4, id = col - ic * n4;")
        if mode == 'eri':
            E(f"const L2gStore st = make_store(meta, A, qi, {la}, {lb}, {lc}, {ld});")
            E("const int colofs = st.pos3(ic) * st.s3 + st.pos4(id) * st.s4;")
            E("const double colscale = st.uniform ? (st.p3 ? 1.0 : l2g_uniform_scale[st.l3][ic]) * "
              "(st.p4 ? 1.0 : l2g_uniform_scale[st.l4][id]) : 1.0;")
            E("(void)colscale;")
            E(f"[[maybe_unused]] const bool fits = vofs || rys_size(meta, {la}, {lb}, {lc}, {ld}) <= region;")
        E("double* const vb = sm + qp * region + vofs;")
        E("(void)vb;")
        E.block("switch ((meta >> 3) & 3)")
        for pa, pb in ge.pure_variants(la, lb):
            E.block(f"case {pa | (pb << 1)}:")
            d1, d2, v = ge.emit_sph_2(E, la, lb, pa, pb, vals, "b")
            if mode == 'fock':
                for i in range(d1 * d2):
                    E(f"vb[{i} * n3 * n4 + col] = {v[i]};")
            else:
                for k, (d, pk) in enumerate(((d1, pa), (d2, pb))):
                    for i in range(d):
                        E(f"const int o{k}_{i} = st.pos(st.l{k + 1}, {pk}, {i}) * st.s{k + 1};")
                        if not pk and p.l[k] >= 2:
                            E(f"const double u{k}_{i} = st.uniform ? l2g_uniform_scale[{p.l[k]}][{i}] : 1.0;")

                def val(i1, i2):
                    x = v[i1 * d2 + i2]
                    if not pa and la >= 2:
                        x += f" * u0_{i1}"
                    if not pb and lb >= 2:
                        x += f" * u1_{i2}"
                    if not (pa and pb) or max(lc, ld) >= 2:
                        x += " * colscale"
                    return x
                at = [(f"o0_{i1} + o1_{i2}", val(i1, i2)) for i1 in range(d1) for i2 in range(d2)]
                direct = rd is not None and d1 * d2 * ge.ncart(lc) * ge.ncart(ld) > min(regs_[x] for x in lay if not vofs[x])
                if direct:
                    E.block("if (!fits)")
                    E("double* const o = A.out + st.base + colofs;")
                    E.block("if (A.store_sub)")
                    for ad, x in at:
                        E(f"o[{ad}] -= {x};")
                    E.end()
                    E.block("else")
                    for ad, x in at:
                        E(f"o[{ad}] = {x};")
                    E.end()
                    E("break;")
                    E.end()
                E("double* const o = vb + colofs;")
                for ad, x in at:
                    E(f"o[{ad}] = {x};")
            E("break;")
            E.end()
        E("default: break;")
        E.end()
        E.end()
        E.end()
        E.end()

    # the copies of the code round alike: every fused operation is written out, and contraction is off
    if rounds:
        if behind:
            E.block("if (vofs == 0)")
        for rd in range(rounds):
            for e in range(p.ne):
                E(f"double y{rd}_{e} = 0.0;")
        for rd in range(rounds):
            columns(rd)
            E.block("if (qp < qn)")
            for e in range(p.ne):
                E(f"y{rd}_{e} = sm[qp * region + {e * p.rstr} + col];")
            E.end()
            E.end()
        E(f"rys_sync<{NW}>();")
        for rd in range(rounds):
            finish(rd)
        if behind:
            E.end()
    if behind:
        if rounds:
            E.block("else")
        finish(None)
        if rounds:
            E.end()
    if mode == 'eri':
        E(f"rys_sync<{NW}>();")
        E.block("for (int qp = 0; qp < qn; ++qp)")
        E("const int qi = items[qlo + qp].qi, meta = items[qlo + qp].meta;")
        E("if (qi < 0) break;")
        E(f"const int n = rys_size(meta, {la}, {lb}, {lc}, {ld});")
        E("if (!vofs && n > region) continue;  // stored directly")
        E("double* const dst = A.out + A.out_off[qi];")
        E("const double* const vb = sm + qp * region + vofs;")
        E.block("if (A.store_sub)")
        E(f"for (int k = tid; k < n; k += {NT}) dst[k] -= vb[k];")
        E.end()
        E.block("else")
        E(f"for (int k = tid; k < n; k += {NT}) dst[k] = vb[k];")
        E.end()
        E.end()
    n = p.dims(False)
    ncomb = sum(n[i] * n[j] for i in range(4) for j in range(i + 1, 4))
    if mode == 'fock':
        pure = ', '.join(map(str, p.dims(True)))
        call = f"rys_digest_pure<{NT}, {NW}, {pure}>(A, items + qlo, dig, qn, sm + vofs, region);"
        if not mask:
            E(call)
        else:
            E.block("if (!cart)")
            E(call)
            E.end()
            E.block("else")
            for what in (f"sm[qp * region + vofs + dig[qp].nv + o] = rys_density(A, dig[qp], o);",
                         f"rys_digest(A, dig[qp], o, sm + qp * region + vofs, sm + qp * region + vofs + dig[qp].nv);"):
                E("#pragma unroll 1")
                E.block(f"for (int it = tid; it < qn * {ncomb}; it += {NT})")
                E(f"const int qp = it / {ncomb}, o = it - qp * {ncomb};")
                E(f"if (items[qlo + qp].nsurv && o < dig[qp].off[6]) {what}")
                E.end()
                E(f"rys_sync<{NW}>();")
            E.end()
    E.end()  # passes
    if mode == 'eri':
        E(f"rys_sync<{NW}>();")
        E(f"if (A.nz && tid < NI && items[tid].qi >= 0) A.nz[A.qidx[items[tid].qi]] = items[tid].nsurv ? 1 : 0;")
    E.ind -= 1
    E("}")
    E(f"void {name}_launch(const L2gEriArgs& A, int, int, hipStream_t s) {{")
    E(f"  hipLaunchKernelGGL({name}, dim3(RysTier<{Q}>::blocks(A)), dim3({NT}), 0, s, A);")
    E("}")
    ge._FUSED = False
    return name, E.text()


def use(la, lb, lc, ld):
    """Whether a class has a Rys kernel: every class does."""
    return True


# Classes whose ERI batches have a per-lane kernel (gen_eri.py) besides their Rys kernel (launch_rules.h, LaneCost):
# nanoseconds per quartet and per primitive quartet on the per-lane kernel, the same on the Rys kernel (150,000 quartets
# of 1 and of 256 primitive quartets on one MI355X), and by how many microseconds a launch of few quartets takes longer
# on the per-lane kernel, of 1 and of many primitive quartets (300 quartets).  The tiles of a Rys kernel spend more on
# prologue, 2D integrals and epilogue than on the products in these classes: 150,000 (ps|ps) quartets of 256 primitive
# quartets took 0.55 ms a lane per quartet, take 1.11 on tiles and 0.35 on the per-lane kernel; of 20,000 quartets with
# K <= 6 820, 137 and 61 us.  The classes left out are slower there at 1 to 256 primitive quartets, or by less than a
# tenth faster.
LANE_COST = {
    '0000': (0.027, 0.0045, 0.035, 0.0103, -14, -30),
    '0010': (0.033, 0.0065, 0.126, 0.0145, -5, -7),
    '0011': (0.075, 0.0075, 0.214, 0.0216, -3, -2),
    '0020': (0.044, 0.0076, 0.202, 0.0209, -3, -1),
    '0021': (0.124, 0.0113, 0.346, 0.0274, 0, 5),
    '0022': (0.145, 0.0178, 0.463, 0.0403, 2, 13),
    '0030': (0.054, 0.0104, 0.188, 0.0249, -21, -53),
    '0031': (0.155, 0.0179, 0.415, 0.0415, 2, 11),
    '0032': (0.553, 0.0246, 0.482, 0.0462, -26, -69),
    '0033': (0.789, 0.0401, 3.812, 0.0934, 20, 68),
    '1010': (0.068, 0.0082, 0.144, 0.0275, -5, -15),
    '1011': (0.307, 0.0162, 0.181, 0.0381, -3, -11),
    '1020': (0.113, 0.0132, 0.181, 0.0370, -7, -14),
    '1021': (0.588, 0.0282, 0.230, 0.0541, 9, -1),  # through 16 and 256
    '1022': (1.053, 0.0471, 0.428, 0.0877, 19, 24),
    '1030': (0.124, 0.0251, 0.188, 0.0629, -5, -22),
    '1031': (0.842, 0.0487, 0.329, 0.0800, 14, 17),
    '1033': (3.344, 0.2538, 4.991, 0.1776, 96, 440),
    '1111': (0.833, 0.0282, 0.364, 0.0564, 16, 54),
    '1120': (0.445, 0.0286, 0.294, 0.0601, 10, 30),
    '1130': (0.607, 0.0612, 0.395, 0.0718, 18, 100),
    '2011': (0.497, 0.0245, 0.303, 0.0586, 11, 11),
    '2020': (0.147, 0.0233, 0.275, 0.0589, -2, 20),
    '2021': (0.943, 0.0567, 0.377, 0.0853, 22, 71),
    '2030': (0.404, 0.0527, 0.361, 0.0721, 11, 69),
    '2033': (6.405, 0.4845, 10.957, 0.3229, 164, 1014),
    '3021': (1.517, 0.1116, 0.558, 0.1339, 46, 192),
    '3030': (0.550, 0.1090, 0.522, 0.1882, 20, 142),
}


def lane_cost(la, lb, lc, ld):
    return LANE_COST.get(f"{la}{lb}{lc}{ld}")


def generate(classes, mode):
    """[(plan, kernel name, source)] of the classes."""
    return [(p, *emit(p, mode)) for p in (plan(*c) for c in classes)]


def files(kernels, n):
    """The sources in n files of about equal length."""
    out, load = [[] for _ in range(n)], [0] * n
    for _, _, src in sorted(kernels, key=lambda k: -len(k[2])):
        j = load.index(min(load))
        out[j].append(src)
        load[j] += len(src)
    return out


if __name__ == '__main__':
    for c in ge.canonical_classes(3):
        if use(*c):
            p = plan(*c)
            print(c, 'lanes on', p.side, 'tile', p.te, 'parts', len(p.parts), 'waves', p.nw, 'quartets', p.q, 'batch', p.nb,
                  'node by node' if p.rl else '', 'LDS a wave', p.lds_bytes('fock') // p.nw, 'registers', p.regs(),
                  'waves per SIMD', p.occupancy(), 'cost %.0f' % p.cost())
