"""Split columns of any circuit as subdomains with one exchange a step.

The staged factor of a split column (solver_plan.py) meets at a column barrier
after every stage above the lowest ones. Here the faces are cut by recursive
bisection into ``parts`` interiors that never touch and a set of separator faces
G between them. With K ordered [interiors, G], block elimination solves K x = b as

    b_G' = b_G - sum_p E_p b_p,        E_p = K_Gp K_pp^-1,
    x_G  = S^-1 b_G',                  S = K_GG - sum_p E_p K_pG,
    x_p  = K_pp^-1 b_p - E_p^T x_G,

so each workgroup forms its contribution to b_G' from its own faces, the workgroups
exchange those contributions once, and each computes the rows of x_G that border its
interior and then its interior alone. An interior is eliminated the same way one
level down: cells whose inverses are dense, and the separators between them. All
operators are dense blocks, kept as rows of (value, index) records that the kernel's
wave programs stream (the record format of the staged factor), in two phases before
the exchange and three after it.

Every junction belongs to one workgroup: the one whose interior it touches (two
interiors have no junction in common), or for a junction between separator faces one
that borders them. Every row's sum runs in an order fixed by the row alone, so x_G
has the same bits in all workgroups. K is symmetric positive definite, its
diagonal blocks and Schur complements too, so no pivoting is needed and the solve
is as exact as the factor's.
"""
from __future__ import annotations

import numpy as np
import scipy.sparse

from . import _native
from .solver_plan import WAVE

BLOCK = 512                 # threads of a workgroup
MAX_PAIRS = 4 * BLOCK       # junction pairs of one workgroup
MAX_FACES = 4 * BLOCK       # faces of one workgroup, its separator faces included
MAX_GAMMA = 4096            # separator faces
FACE_CODES = 8              # junctions of a face
LDS_DOUBLES = 163840 // 8 - 32
CELLS = (1, 2, 4, 8, 16, 32)
# jja_slice
RECORD = np.dtype([("base", "<i8"), ("ibase", "<i8"), ("rowbase", "<i4"), ("r0", "<i4"), ("n_iter", "<i4"), ("flags", "<i4")])


def bisect(faces, xy, touched, levels):
    """``faces`` cut into 2^levels parts and the separators between them: halves by
    the longer side's coordinate, the faces of the second half that the first half
    touches (``touched``: index array -> mask over all faces) taken out."""
    none = np.zeros(0, dtype=np.int64)
    if levels == 0:
        return [faces], none
    if len(faces) == 0:
        return [none] * (1 << levels), none
    p = xy[faces]
    axis = int(np.argmax(np.ptp(p, axis=0)))
    order = faces[np.argsort(p[:, axis], kind="stable")]
    half = (len(order) + 1) // 2
    a, b = order[:half], order[half:]
    cut = touched(a)[b]
    pa, sa = bisect(a, xy, touched, levels - 1)
    pb, sb = bisect(b[~cut], xy, touched, levels - 1)
    return pa + pb, np.concatenate((b[cut], sa, sb))


def spd_inverse(M):
    """Inverse of a symmetric positive definite matrix; LinAlgError when it is not
    (every pivot block of the elimination passes here, so this refuses exactly the
    matrices a Cholesky factorisation refuses)."""
    Li = np.linalg.inv(np.linalg.cholesky(M))
    inv = Li.T @ Li
    if not np.isfinite(inv).all():
        raise np.linalg.LinAlgError("not finite")
    return inv


def _phase(rows, blocks, kind):
    """A phase of a program: row i sums dense blocks (row numbers, column addresses,
    matrix) in turn."""
    n = len(rows)
    who = np.concatenate([np.repeat(r, len(c)) for r, c, _ in blocks])
    order = np.argsort(who, kind="stable")
    idx = np.concatenate([np.tile(c, len(r)) for r, c, _ in blocks])[order]
    val = np.concatenate([M.ravel() for _, _, M in blocks])[order]
    lens = np.bincount(who, minlength=n)
    return np.asarray(rows, dtype=np.int32), lens, idx, val, kind


class DomainPlan:
    """Subdomains of the face system ``K`` (faces at ``xy``) for ``parts`` workgroups
    and the junction incidence ``junc_code`` (circuit face order: 2*face + sign, -1
    empty, two per junction). ``ok`` is False where the circuit does not fit."""

    def __init__(self, K, xy, junc_code, parts):
        self.parts = parts
        self.ok = False
        self._desc = None
        K = scipy.sparse.csr_matrix(K)
        Nf, Nj = K.shape[0], len(junc_code) // 2
        self.Nf, self.Nj = Nf, Nj

        def touched(a):
            mask = np.zeros(Nf, dtype=bool)
            mask[K[a].indices] = True
            return mask
        interiors, gamma = bisect(np.arange(Nf), xy, touched, parts.bit_length() - 1)
        if min(len(i) for i in interiors) < 1 or len(gamma) > MAX_GAMMA or len(gamma) == 0:
            return
        gamma = np.sort(gamma)
        self.gamma = gamma
        part_of = -np.ones(Nf, dtype=np.int64)
        for p, f in enumerate(interiors):
            part_of[f] = p
        jc = np.asarray(junc_code, dtype=np.int64).reshape(Nj, 2)
        face = np.where(jc >= 0, jc >> 1, -1)
        fp = np.where(face >= 0, part_of[np.maximum(face, 0)], -1)
        owner = fp.max(axis=1)             # the interior it touches, or -1
        clash = (fp >= 0).all(axis=1) & (fp[:, 0] != fp[:, 1])
        if clash.any():
            return                         # interiors joined by a junction of weight zero in K
        # separator faces that border each interior, then those of the junctions it is given
        border = [set(gamma[touched(f)[gamma]].tolist()) for f in interiors]
        load = np.bincount(owner[owner >= 0], minlength=parts)
        beside = {int(g): {p for p in range(parts) if int(g) in border[p]} for g in gamma}   # the parts that border it
        for j in np.flatnonzero(owner < 0):
            mine = [int(f) for f in face[j] if f >= 0]
            held = [beside[f] for f in mine]
            # a part that borders all of them, else any of them, else any part; the
            # least loaded, the first among equals
            fits = (set.intersection(*held) or set.union(*held)) if held else set()
            p = min(sorted(fits) or range(parts), key=lambda q: load[q])
            owner[j] = p
            load[p] += 1
            border[p].update(mine)
            for f in mine:
                beside[f].add(p)
        # a separator face that no part borders would never be published
        for f in gamma:
            if not any(f in b for b in border):
                border[0].add(int(f))
        self.border = [np.array(sorted(b), dtype=np.int64) for b in border]
        self.interiors, self.owner = interiors, owner
        n_loc = max(len(i) + len(b) for i, b in zip(interiors, self.border))
        if n_loc > MAX_FACES:
            return
        self.n_local = n_loc
        try:
            if not self._choose_cells(K, xy):
                return
        except np.linalg.LinAlgError:
            return                         # not positive definite: left to the factor to refuse
        if not self._incidence(jc, face):
            return
        self._programs()
        self.ok = 2 * n_loc + len(gamma) + 2 * self.pairs + 2 <= LDS_DOUBLES

    # ------------------------------------------------------------- elimination
    def _eliminate(self, K, cells, seps, border):
        """Dense operators of one interior from its dense matrix K (local indices):
        per cell (faces, inverse, border rows, E); the separators' Schur inverse and
        E onto the border; the border's update."""
        rows = np.concatenate((seps, border))
        ns = len(seps)
        Krr = np.zeros((len(rows), len(rows)))   # minus what the cells add
        ops = []
        for c in cells:
            inv = spd_inverse(K[np.ix_(c, c)])
            Krc = K[np.ix_(rows, c)]
            hit = np.flatnonzero(np.abs(Krc).sum(axis=1))
            E = Krc[hit] @ inv
            Krr[np.ix_(hit, hit)] -= E @ Krc[hit].T
            ops.append((c, inv, hit, E))
        Sl = Eb = None
        up = Krr[ns:, ns:].copy()
        if ns:
            Sl = spd_inverse(K[np.ix_(seps, seps)] + Krr[:ns, :ns])
            Kbs = K[np.ix_(border, seps)] + Krr[ns:, :ns]
            Eb = Kbs @ Sl
            up -= Eb @ Kbs.T
        return ops, Sl, Eb, up

    def _choose_cells(self, K, xy):
        """Cells per interior: the count whose operators have the fewest entries,
        each phase counted as the entries a workgroup streams meanwhile. Then every
        part's operators and the separators' Schur inverse."""
        def local(p):
            f = np.concatenate((self.interiors[p], self.border[p]))
            return f, K[f][:, f].toarray(), len(self.interiors[p])

        def cut(D, at, n, levels):
            near = D[:n, :n] != 0
            return bisect(np.arange(n), at, lambda a: near[a].any(axis=0), levels)
        best = None
        f, D, n = local(int(np.argmax([len(i) for i in self.interiors])))
        for count in CELLS:
            if n < 4 * count:
                break
            cells, seps = cut(D, xy[f], n, count.bit_length() - 1)
            if min(len(c) for c in cells) < 1:
                break
            rows = np.concatenate((seps, np.arange(n, len(f))))
            work = sum(len(c) * (len(c) + 2 * int((D[np.ix_(rows, c)] != 0).any(axis=1).sum())) for c in cells)
            ns = len(seps)
            work += ns * (ns + 2 * (len(f) - n)) + (2 * 3000 if ns else 0)
            if best is None or work < best[0]:
                best = (work, count)
        if best is None:
            return False
        self.cells = best[1]
        gpos = -np.ones(self.Nf, dtype=np.int64)
        gpos[self.gamma] = np.arange(len(self.gamma))
        S = K[self.gamma][:, self.gamma].toarray()
        self.local = []
        for p in range(self.parts):
            f, D, n = local(p)
            count = self.cells
            while True:
                cells, seps = cut(D, xy[f], n, count.bit_length() - 1)
                if count == 1 or min(len(c) for c in cells) >= 1:
                    break
                count //= 2
            ops, Sl, Eb, up = self._eliminate(D, cells, seps, np.arange(n, len(f)))
            g = gpos[self.border[p]]
            S[np.ix_(g, g)] += up
            self.local.append(([(f[c], inv, hit, E) for c, inv, hit, E in ops], f[seps], Sl, Eb))
        self.gpos = gpos
        self.Sinv = spd_inverse(S)
        return True

    # --------------------------------------------------------------- incidence
    def _incidence(self, jc, face):
        """Per-part tables: junction pairs, their codes into the solution, and the
        faces' codes into the junction values."""
        parts, n_loc = self.parts, self.n_local
        pair_of = np.arange(self.Nj) >> 1
        lists = [np.unique(pair_of[self.owner == p]) for p in range(parts)]
        self.pairs = max(len(q) for q in lists)
        if self.pairs > MAX_PAIRS or 2 * max(self.pairs, n_loc) >= 0x7fff:
            return False
        self.pair = -np.ones((parts, self.pairs), dtype=np.int32)
        self.pair_code = np.full((parts, self.pairs, 2, 2), 0xffff, dtype=np.uint16)
        self.face_code = np.full((parts, n_loc, FACE_CODES), 0xffff, dtype=np.uint16)
        self.face_used = np.zeros((parts, n_loc), dtype=np.int32)
        self.face_id = -np.ones((parts, n_loc), dtype=np.int32)
        first = {}                       # the part that adds a separator face's flux
        for p, b in enumerate(self.border):
            for g in b.tolist():
                first.setdefault(g, p)
        self.addr = []
        for p in range(parts):
            ops, seps = self.local[p][0], self.local[p][1]
            order = np.concatenate([c for c, _, _, _ in ops] + [seps, self.border[p]])
            at = -np.ones(self.Nf, dtype=np.int64)
            at[order] = np.arange(len(order))
            self.addr.append((order, at))
            q = lists[p]
            slot = -np.ones((self.Nj + 1) // 2, dtype=np.int64)
            slot[q] = np.arange(len(q))
            js = np.flatnonzero(self.owner == p)
            flags = np.zeros(len(q), dtype=np.int64)
            np.add.at(flags, slot[js >> 1], (1 << (js & 1)) * 5)       # present and owned
            self.pair[p, :len(q)] = q * 16 + flags
            counts = np.zeros(len(order), dtype=np.int64)
            for i in range(2):
                has = js[jc[js, i] >= 0]
                a = at[face[has, i]]
                if (a < 0).any():
                    return False
                self.pair_code[p, slot[has >> 1], has & 1, i] = (2 * a + (jc[has, i] & 1)).astype(np.uint16)
            has = np.concatenate([np.stack((js, np.full_like(js, i)), 1) for i in range(2)])
            has = has[jc[has[:, 0], has[:, 1]] >= 0]
            code = jc[has[:, 0], has[:, 1]]
            a = at[code >> 1]
            o = np.lexsort((has[:, 0], a))
            a, j, sign = a[o], has[o, 0], code[o] & 1
            start = np.searchsorted(a, np.arange(len(order)))
            k = np.arange(len(a)) - start[a]
            if len(k) and k.max() >= FACE_CODES:
                return False
            self.face_code[p, a, k] = (2 * (2 * slot[j >> 1] + (j & 1)) + sign).astype(np.uint16)
            self.face_used[p, :len(order)] = 1
            inner = self.gpos[order] < 0
            mine = np.array([inner[i] or first[int(f)] == p for i, f in enumerate(order)])
            self.face_id[p, :len(order)] = np.where(mine, order, -1)
        return True

    # ---------------------------------------------------------------- programs
    def _phases(self, p):
        """The five phases of part p; addresses: b at 0.., x at n_local.., b_G' at
        2 n_local.. (in doubles)."""
        ops, seps, Sl, Eb = self.local[p]
        order, at = self.addr[p]
        b, n = self.border[p], self.n_local
        rows = np.concatenate((seps, b))
        before = [_phase(at[rows], [(hit, at[c], E) for c, _, hit, E in ops], 0)]
        if len(seps):
            before.append(_phase(at[b], [(np.arange(len(b)), at[seps], Eb)], 0))
        B = _native.SLICE_BLOCK
        after = [_phase(n + at[b], [(np.arange(len(b)), 2 * n + np.arange(len(self.gamma)), self.Sinv[self.gpos[b]])], B)]
        if len(seps):
            i = np.arange(len(seps))
            after.append(_phase(n + at[seps], [(i, at[seps], Sl), (i, n + at[b], -Eb.T)], B))
        cell_rows, row0, blocks = np.concatenate([c for c, _, _, _ in ops]), 0, []
        for c, inv, hit, E in ops:
            i = row0 + np.arange(len(c))
            blocks += [(i, at[c], inv), (i, n + at[rows[hit]], -E.T)]
            row0 += len(c)
        after.append(_phase(n + at[cell_rows], blocks, B))
        return before, after

    def _programs(self):
        programs = [half for p in range(self.parts) for half in self._phases(p)]
        phases = [ph for half in programs for ph in half]
        self.entries = sum(len(ph[2]) for ph in phases)
        ends = lambda counts, t: np.concatenate(([0], np.cumsum(counts))).astype(t)
        given = [ends([len(half) for half in programs], np.int32), ends([len(ph[0]) for ph in phases], np.int64),
                 np.array([ph[4] for ph in phases], dtype=np.int32), np.concatenate([ph[0] for ph in phases]),
                 ends(np.concatenate([ph[1] for ph in phases]), np.int64),
                 np.concatenate([ph[2] for ph in phases]).astype(np.int32), np.concatenate([ph[3] for ph in phases])]
        sizes = np.zeros(3, dtype=np.int64)
        waves = BLOCK // WAVE

        def build(*made):
            args = [a.ctypes.data for a in given] + [sizes.ctypes.data] + [a.ctypes.data if a is not None else None for a in made]
            rc = _native.lib().jja_domain_programs(len(programs), waves, *args)
            if rc != _native.JJA_OK:
                raise _native.NativeError(f"jja_domain_programs: libjja error {rc}")
        build(None, None, None, None, None)
        self.records = np.empty(sizes[0], dtype=RECORD)
        self.wave_ptr = np.empty(len(programs) * (waves + 1), dtype=np.int32)
        self.ent_val, self.ent_off = np.empty(sizes[1]), np.empty(sizes[1], dtype=np.uint16)
        self.slice_rows = np.empty(sizes[2], dtype=np.int32)
        build(self.records, self.wave_ptr, self.ent_val, self.ent_off, self.slice_rows)
        # published contributions: part by part, the border in order; their sources
        # per separator face
        self.pub_ptr = np.concatenate(([0], np.cumsum([len(b) for b in self.border]))).astype(np.int32)
        self.pub_at = np.concatenate([self.addr[p][1][b] for p, b in enumerate(self.border)]).astype(np.int32)
        lists = [[] for _ in self.gamma]
        for p, b in enumerate(self.border):
            for i, f in enumerate(b):
                lists[self.gpos[f]].append(int(self.pub_ptr[p]) + i)
        self.sources = max(len(s) for s in lists)
        self.source = -np.ones((len(self.gamma), self.sources), dtype=np.int32)
        for g, s in enumerate(lists):
            self.source[g, :len(s)] = s

    def desc(self):
        """ctypes jja_domains pointing at this object's arrays (keep it alive); the same
        one on every call, since problem descriptors hold its address."""
        if self._desc is not None:
            return self._desc
        d = _native.Domains()
        d.parts, d.pairs, d.faces, d.n_gamma = self.parts, self.pairs, self.n_local, len(self.gamma)
        d.sources, d.n_published, d.n_records = self.sources, int(self.pub_ptr[-1]), len(self.records)
        for name in ("records", "pair", "pair_code", "face_code", "face_id", "face_used", "pub_ptr", "pub_at", "source", "wave_ptr",
                     "slice_rows", "ent_val", "ent_off"):
            a = np.ascontiguousarray(getattr(self, name))
            setattr(self, name, a)
            setattr(d, name, a.ctypes.data)
        d.n_slice_rows, d.n_entries, d.n_index = len(self.slice_rows), len(self.ent_val), len(self.ent_off)
        self._desc = d
        return d

    def __getstate__(self):
        # pointers to this object's arrays: made again on the other side
        return dict(self.__dict__, _desc=None)

    # ----------------------------------------------------------- host emulation
    def emulate(self, b):
        """K^-1 b for b (Nf,) by the kernel's steps, from the phases' rows."""
        n, G = self.n_local, len(self.gamma)
        mem = np.zeros((self.parts, 2 * n + G))
        phases = [self._phases(p) for p in range(self.parts)]

        def run(m, ph):
            rows, lens, idx, val, kind = ph
            ptr = np.concatenate(([0], np.cumsum(lens)))
            sums = np.array([np.dot(val[ptr[i]:ptr[i + 1]], m[idx[ptr[i]:ptr[i + 1]]]) for i in range(len(rows))])
            m[rows] = sums if kind else m[rows] - sums
        pub = np.zeros(int(self.pub_ptr[-1]))
        for p in range(self.parts):
            order, _ = self.addr[p]
            mem[p, :len(order)] = np.where(self.face_id[p, :len(order)] >= 0, b[order], 0.0)
            for ph in phases[p][0]:
                run(mem[p], ph)
            s = slice(int(self.pub_ptr[p]), int(self.pub_ptr[p + 1]))
            pub[s] = mem[p, self.pub_at[s]]
        rhs = np.where(self.source >= 0, pub[np.maximum(self.source, 0)], 0.0).sum(axis=1)
        x = np.zeros(self.Nf)
        for p in range(self.parts):
            mem[p, 2 * n:] = rhs
            for ph in phases[p][1]:
                run(mem[p], ph)
            order, _ = self.addr[p]
            x[order] = mem[p, n:n + len(order)]
        return x
