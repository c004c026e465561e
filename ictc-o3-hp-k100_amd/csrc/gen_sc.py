"""Emit ``generated/ictc_sc.h``: straight-line symmetric-contraction polynomials.

The correlation-nu symmetric contraction of the reference
(ictc_o3/ops/_mace_symmetric_contraction.py:298-355, U from _mace_cg.py:118-190
with the ICTC bridge folded in, symmetric_contraction.py:50-96) is, per node n,
channel c and output component (L, m),

    out[L, m] = sum_nu sum_p W_nu^L[s_n, p, c] * sum_{i1..inu} U_nu^L[m, i1..inu, p] x_i1 ... x_inu .

Only the symmetric part of U in (i1..inu) contributes, so each (L, m) output
is a sparse polynomial in the NX = (LI+1)^2 input components whose
coefficients are linear in the per-species weights.  For every supported
(LI, LT, CORR) this script emits ``Sc<LI, LT, CORR>`` with device functions
working on per-lane registers (one lane = one channel):

  fwd     o[k]   = sum_mono mono(x) * (sum_{nu,p} coef * W)
  dx      d[i]   = d/dx_i of sum_k go[k] o[k]
  dw      dw[q]  = sum_k go[k] * d o[k] / d W_q           (q enumerates (L, nu, p))
  jvp     t[k]   = sum_i h_i d o[k] / d x_i
  hvp     d[i]   = sum_j h_j d^2 (go . o) / dx_i dx_j
  dwjvp   dw[q]  = sum_k go[k] * sum_i h_i d^2 o[k] / dW_q dx_i

Weights are read through a ``ScWeights`` table (one [S, P, C] array per (L, nu)).
"""
from __future__ import annotations

import itertools
import os
import sys

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(_HERE))

from ictc_o3.basis import e3nn_basis  # noqa: E402

ZERO = 1e-11
# (LI, LT) pairs compiled; every correlation 1..3.
CONFIGS = [(li, lt) for li in range(3) for lt in range(li + 1)] + [(3, 0), (3, 1), (3, 2)]


def f(v):
    return repr(float(v)) + "f"


def polynomial(li, lt, corr):
    """terms[k][mono] = [(L, nu, p, coef)] with k the packed output index, mono a sorted tuple."""
    nx = (li + 1) ** 2
    outs = []
    for L in range(lt + 1):
        for m in range(2 * L + 1):
            outs.append((L, m))
    terms = [dict() for _ in outs]
    counts = {}
    for L in range(lt + 1):
        for nu in range(1, corr + 1):
            U = e3nn_basis.mace_u_ictc(li, L, nu)
            if L == 0:
                U = U[None]
            P = U.shape[-1]
            counts[(L, nu)] = P
            for p in range(P):
                for m in range(2 * L + 1):
                    T = U[m, ..., p]
                    acc = {}
                    for idx in itertools.product(range(nx), repeat=nu):
                        v = T[idx]
                        if abs(v) > 1e-14:
                            key = tuple(sorted(idx))
                            acc[key] = acc.get(key, 0.0) + v
                    k = outs.index((L, m))
                    for key, v in acc.items():
                        if abs(v) > ZERO:
                            terms[k].setdefault(key, []).append((L, nu, p, v))
    return outs, terms, counts


def _weight_names(counts):
    q = []
    for (L, nu), P in sorted(counts.items()):
        for p in range(P):
            q.append((L, nu, p))
    return q


def _combo(entries):
    return " + ".join(f"{f(v)} * w{L}_{nu}_{p}" for L, nu, p, v in entries)


def _mono_expr(key):
    return " * ".join(f"x[{i}]" for i in key) if key else "1.f"


def _deriv(key):
    """[(i, multiplicity, remaining key)] of d/dx_i of the monomial."""
    out = []
    for i in sorted(set(key)):
        rest = list(key)
        rest.remove(i)
        out.append((i, key.count(i), tuple(rest)))
    return out


DW_BLOCK = 32   # weights per weight-gradient wave (kDwBlock in sc_kernels.h)


def sc_struct(li, lt, corr):
    outs, terms, counts = polynomial(li, lt, corr)
    nx, no = (li + 1) ** 2, len(outs)
    wq = _weight_names(counts)
    nq = len(wq)
    qindex = {w: i for i, w in enumerate(wq)}
    L = [f"template <> struct Sc<{li}, {lt}, {corr}> {{",
         f"  static constexpr int NX = {nx}, NO = {no}, NW = {nq};"]
    # weight counts table
    rows = []
    for Lo in range(4):
        rows.append("{" + ", ".join(str(counts.get((Lo, nu), 0)) for nu in (1, 2, 3)) + "}")
    L.append(f"  static constexpr int P[4][3] = {{{', '.join(rows)}}};")
    nterms = sum(len(e) for t in terms for e in t.values())
    L.append(f"  static constexpr int TERMS = {nterms};")

    def load_weights():
        # species row of each weight block (wave-uniform) + the lane's byte offset: SGPR-base loads
        s = ["    const int64_t sb = s;", "    const uint32_t off = sc_lane_offset(c);"]
        for (Lo, nu) in sorted({(Lo, nu) for (Lo, nu, p) in wq}):
            P = counts[(Lo, nu)]
            s.append(f"    const float* __restrict__ wb{Lo}_{nu} = t.w[{Lo}][{nu - 1}] + sb * {P} * C;")
        for (Lo, nu, p) in wq:
            s.append(f"    const float w{Lo}_{nu}_{p} = sc_load(wb{Lo}_{nu} + {p} * C, off);")
        return s

    # forward
    L.append("  __device__ __forceinline__ static void fwd(const float* __restrict__ x, const ScWeights& t, int s,"
             " int C, int c, float* __restrict__ o) {")
    L += load_weights()
    for k in range(no):
        expr = " + ".join(f"({_mono_expr(key)}) * ({_combo(e)})" for key, e in terms[k].items()) or "0.f"
        L.append(f"    o[{k}] = {expr};")
    L.append("  }")
    # dx: gradient of sum_k go[k] o[k]
    L.append("  __device__ __forceinline__ static void dx(const float* __restrict__ x, const ScWeights& t, int s,"
             " int C, int c, const float* __restrict__ go, float* __restrict__ d) {")
    L += load_weights()
    L.append(f"    float a[{nx}];")
    L.append(f"    for (int i = 0; i < {nx}; ++i) a[i] = 0.f;")
    mono_all = {}
    for k in range(no):
        for key, e in terms[k].items():
            mono_all.setdefault(key, []).append((k, e))
    for key, lst in mono_all.items():
        if not key:
            continue
        g = " + ".join(f"go[{k}] * ({_combo(e)})" for k, e in lst)
        L.append(f"    {{ const float g = {g};")
        for i, mult, rest in _deriv(key):
            L.append(f"      a[{i}] = fmaf(g, {float(mult)}f * ({_mono_expr(rest)}), a[{i}]);")
        L.append("    }")
    L.append(f"    for (int i = 0; i < {nx}; ++i) d[i] = a[i];")
    L.append("  }")
    # dw: per weight q, sum_k go[k] * coef * mono; emitted in blocks of DW_BLOCK weights
    # (dwb<B> accumulates weights B*DW_BLOCK ...) so one wave holds one block's accumulators.
    per_q = {q: [] for q in range(nq)}
    for k in range(no):
        for key, e in terms[k].items():
            for (Lo, nu, p, v) in e:
                per_q[qindex[(Lo, nu, p)]].append((k, key, v))
    nb = max(1, (nq + DW_BLOCK - 1) // DW_BLOCK)

    def by_monomial(b):
        """{mono key: {local q: [(k, coef)]}} for the weights of block b, in first-use order."""
        groups = {}
        for q in range(b * DW_BLOCK, min(nq, (b + 1) * DW_BLOCK)):
            for k, key, v in per_q[q]:
                groups.setdefault(key, {}).setdefault(q - b * DW_BLOCK, []).append((k, v))
        return groups

    def go_combo(lst):
        return " + ".join(f"{f(v)} * go[{k}]" for k, v in lst)

    # Each monomial is formed once and consumed at once (short live ranges).
    L.append(f"  static constexpr int NB = {nb};")
    L.append("  template <int B>")
    L.append("  __device__ __forceinline__ static void dwb(const float* __restrict__ x, const float* __restrict__ go,"
             " float* __restrict__ acc) {")
    for b in range(nb):
        L.append(f"    {'if' if b == 0 else 'else if'} constexpr (B == {b}) {{")
        for key, qs in by_monomial(b).items():
            L.append(f"      {{ const float m = {_mono_expr(key)};")
            for ql, lst in qs.items():
                L.append(f"        acc[{ql}] = fmaf(m, {go_combo(lst)}, acc[{ql}]);")
            L.append("      }")
        L.append("    }")
    L.append("  }")
    # jvp: directional derivative of o along h
    L.append("  __device__ __forceinline__ static void jvp(const float* __restrict__ x, const ScWeights& t, int s,"
             " int C, int c, const float* __restrict__ h, float* __restrict__ o) {")
    L += load_weights()
    for k in range(no):
        parts = []
        for key, e in terms[k].items():
            dparts = [f"{float(mult)}f * ({_mono_expr(rest)}) * h[{i}]" for i, mult, rest in _deriv(key)]
            if dparts:
                parts.append(f"({' + '.join(dparts)}) * ({_combo(e)})")
        L.append(f"    o[{k}] = {' + '.join(parts) or '0.f'};")
    L.append("  }")
    # hvp: d[i] = sum_j h_j d2(go.o)/dx_i dx_j
    L.append("  __device__ __forceinline__ static void hvp(const float* __restrict__ x, const ScWeights& t, int s,"
             " int C, int c, const float* __restrict__ go, const float* __restrict__ h, float* __restrict__ d) {")
    L += load_weights()
    L.append(f"    float a[{nx}];")
    L.append(f"    for (int i = 0; i < {nx}; ++i) a[i] = 0.f;")
    for key, lst in mono_all.items():
        if len(key) < 2:
            continue
        g = " + ".join(f"go[{k}] * ({_combo(e)})" for k, e in lst)
        L.append(f"    {{ const float g = {g};")
        for i, mi, rest in _deriv(key):
            # d/dx_i of mono = mi * rest ; then directional derivative of rest along h
            inner = [f"{float(mj)}f * ({_mono_expr(r2)}) * h[{j}]" for j, mj, r2 in _deriv(rest)]
            L.append(f"      a[{i}] = fmaf(g, {float(mi)}f * ({' + '.join(inner)}), a[{i}]);")
        L.append("    }")
    L.append(f"    for (int i = 0; i < {nx}; ++i) d[i] = a[i];")
    L.append("  }")
    # dwjvp: dw[q] = sum_k go[k] coef * (d mono . h), in the same weight blocks as dwb
    L.append("  template <int B>")
    L.append("  __device__ __forceinline__ static void dwjvpb(const float* __restrict__ x, const float* __restrict__ go,"
             " const float* __restrict__ h, float* __restrict__ acc) {")
    for b in range(nb):
        L.append(f"    {'if' if b == 0 else 'else if'} constexpr (B == {b}) {{")
        for key, qs in by_monomial(b).items():
            dparts = [f"{float(mult)}f * ({_mono_expr(rest)}) * h[{i}]" for i, mult, rest in _deriv(key)]
            if not dparts:
                continue
            L.append(f"      {{ const float m = {' + '.join(dparts)};")
            for ql, lst in qs.items():
                L.append(f"        acc[{ql}] = fmaf(m, {go_combo(lst)}, acc[{ql}]);")
            L.append("      }")
        L.append("    }")
    L.append("  }")
    # weight slot table: q -> (L, nu-1, p)
    L.append(f"  static constexpr int WQ[{max(nq, 1)}][3] = {{"
             + ", ".join(f"{{{Lo}, {nu - 1}, {p}}}" for Lo, nu, p in wq) + ("" if nq else "{0, 0, 0}") + "};")
    L.append("};")
    return "\n".join(L)


# (LI, LT) at correlation 3 that also get ScTab: the shapes whose terms (monomial x weight) outnumber their
# pairs (output x monomial) 3.8 to 7 times, so that forming the weight combination of each pair once per
# species instead of once per node removes most of the arithmetic.  (3, 0), whose 150 pairs have 509 terms, was
# faster per node (19 against 28 us over 8,191 nodes of 128 channels).
TABLE_CONFIGS = [(2, 2), (3, 1), (3, 2)]
ROW_GROUP = 16    # table rows loaded ahead, one group while the previous is used
PAIR_BLOCK = 64   # pairs per weight-gradient wave (kPairBlock in sc_table.h)


def tab_struct(li, lt, corr):
    """``ScTab<LI, LT, CORR>``: the same polynomials over the coefficients of (output, monomial) pairs.

    Pair r = (k, mono) has the coefficient coef_r[s, c] = sum_q VALUE * W_q[s, c] (terms TERM_PTR[r] ..
    TERM_PTR[r+1], weight TERM_Q, factor TERM_V), formed once per call into a table; the device functions read
    one 64-channel table row per pair (rows 64 floats apart) and work on B nodes of one species per lane.
    Pairs are numbered in the order the functions use them."""
    outs, terms, counts = polynomial(li, lt, corr)
    no = len(outs)
    wq = _weight_names(counts)
    qindex = {w: i for i, w in enumerate(wq)}
    mono_all = {}
    for k in range(no):
        for key, e in terms[k].items():
            mono_all.setdefault(key, []).append((k, e))
    # blocks: (i,) holds the degree-1 monomial x_i; (i, j) holds p_ij = x_i x_j, its degree-2 monomial p_ij and
    # the degree-3 monomials p_ij x_k.  Each p_ij is formed and used in its block only (kept across blocks the
    # products would take more registers than there are).
    blocks = sorted({m[:2] for m in mono_all}, key=lambda g: (g[0], len(g), g))
    third = {g: [m for m in sorted(mono_all) if len(m) == 3 and m[:2] == g] for g in blocks}
    pairs, first = [], {}
    for g in blocks:
        for m in ([g] if g in mono_all else []) + third[g]:
            first[m] = len(pairs)
            pairs += [(k, m, e) for k, e in mono_all[m]]
    R = len(pairs)
    L = [f"template <> struct ScTab<{li}, {lt}, {corr}> {{", f"  static constexpr int PAIRS = {R};"]

    def array(name, kind, values, fmt=str):
        L.append(f"  static constexpr {kind} {name}[{len(values)}] = {{{', '.join(map(fmt, values))}}};")
    ptr, tq, tv = [0], [], []
    for k, m, e in pairs:
        for (Lo, nu, p, v) in e:
            tq.append(qindex[(Lo, nu, p)])
            tv.append(v)
        ptr.append(len(tq))
    array("TERM_PTR", "int32_t", ptr)
    array("TERM_Q", "int16_t", tq)
    array("TERM_V", "float", tv, f)
    # the same terms by weight: WEIGHT_PTR[q] .. of (pair, factor)
    byq = [[] for _ in wq]
    for r, (k, m, e) in enumerate(pairs):
        for (Lo, nu, p, v) in e:
            byq[qindex[(Lo, nu, p)]].append((r, v))
    ptr = [0]
    for b in byq:
        ptr.append(ptr[-1] + len(b))
    array("WEIGHT_PTR", "int32_t", ptr)
    array("WEIGHT_R", "int16_t", [r for b in byq for r, _ in b])
    array("WEIGHT_V", "float", [v for b in byq for _, v in b], f)
    head = "  template <int B>\n  __device__ __forceinline__ static void "
    each = "SC_EACH(b) "
    nx = (li + 1) ** 2

    group = [None]

    def begin():
        group[0] = -2
        L.append(f"    float wa[{ROW_GROUP}], wb[{ROW_GROUP}];")

    def use(r, body):
        """body with w = the coefficient of pair r (the pairs come in order).  Rows are loaded a group ahead; the
        scheduling barrier keeps the loads before the group's arithmetic (left to the scheduler they sank to
        their uses in some of these bodies, each waiting for its row)."""
        n, i = divmod(r, ROW_GROUP)
        if n != group[0]:
            if n != group[0] + 1:   # a group was skipped (no pair of it is used): load this one now
                L.append(f"    SC_ROWS({'wb' if n % 2 else 'wa'}, {n});")
            group[0] = n
            if (n + 1) * ROW_GROUP < R:
                L.append(f"    SC_ROWS({'wa' if n % 2 else 'wb'}, {n + 1}); SC_AHEAD;")
        L.append(f"        {{ const float w = {'wb' if n % 2 else 'wa'}[{i}]; {body} }}")

    def product(g, tangent):
        """p = x_i x_j of block (i, j) (and dp, its derivative along h)."""
        i, j = g
        out = [f"      float p[B]; {each}p[b] = x[b][{i}] * x[b][{j}];"]
        if tangent:
            out.append(f"      float dp[B]; {each}dp[b] = fmaf(h[b][{i}], x[b][{j}], x[b][{i}] * h[b][{j}]);")
        return out

    # fwd / jvp: o[k] += coef * m (m the monomial, or its derivative along h)
    for name, tangent in (("fwd", False), ("jvp", True)):
        args = f"const float (&x)[B][{nx}], " + (f"const float (&h)[B][{nx}], " if tangent else "")
        L.append(head + f"{name}({args}const float* __restrict__ t, uint32_t off, float (&o)[B][{no}]) {{")

        def add(m, value):
            for n, (k, _) in enumerate(mono_all[m]):
                use(first[m] + n, f"{each}o[b][{k}] = fmaf(w, {value}, o[b][{k}]);")
        begin()
        for g in blocks:
            L.append("    {")
            if len(g) == 1:
                add(g, f"{'h' if tangent else 'x'}[b][{g[0]}]")
            else:
                L += product(g, tangent)
                if g in mono_all:
                    add(g, "dp[b]" if tangent else "p[b]")
                for m in third[g]:
                    c = m[-1]
                    e = f"fmaf(dp[b], x[b][{c}], p[b] * h[b][{c}])" if tangent else f"p[b] * x[b][{c}]"
                    L.append(f"      {{ float m[B]; {each}m[b] = {e};")
                    add(m, "m[b]")
                    L.append("      }")
            L.append("    }")
        L.append("  }")
    # dx / hvp: per monomial g = sum_k go[k] coef; in block (i, j), s = g_ij + sum_k g_ijk x_k and
    # d[k] += g_ijk p_ij, then d[i] += s x_j and d[j] += s x_i (hvp: the derivative of these along h)
    for name, tangent in (("dx", False), ("hvp", True)):
        args = f"const float (&x)[B][{nx}], " + (f"const float (&h)[B][{nx}], " if tangent else "")
        L.append(head + f"{name}({args}const float (&go)[B][{no}], const float* __restrict__ t, uint32_t off, "
                 f"float (&d)[B][{nx}]) {{")

        def combine(m, target):
            for n, (k, _) in enumerate(mono_all[m]):
                e = f"fmaf(w, go[b][{k}], {target}[b])" if n else f"w * go[b][{k}]"
                use(first[m] + n, f"{each}{target}[b] = {e};")
        begin()
        for g in blocks:
            if len(g) == 1 and tangent:
                continue   # degree 1: no second derivative
            L.append("    {")
            if len(g) == 1:
                L.append("      float g[B];")
                combine(g, "g")
                L.append(f"      {each}d[b][{g[0]}] += g[b];")
            else:
                i, j = g
                L += product(g, tangent)
                L.append(f"      float s[B]; {each}s[b] = 0.f;")
                if g in mono_all:
                    combine(g, "s")
                if tangent:
                    L.append(f"      float ds[B]; {each}ds[b] = 0.f;")
                for m in third[g]:
                    c = m[-1]
                    L.append("      { float g[B];")
                    combine(m, "g")
                    if tangent:
                        L.append(f"        {each}{{ d[b][{c}] = fmaf(g[b], dp[b], d[b][{c}]); "
                                 f"s[b] = fmaf(g[b], x[b][{c}], s[b]); ds[b] = fmaf(g[b], h[b][{c}], ds[b]); }}")
                    else:
                        L.append(f"        {each}{{ d[b][{c}] = fmaf(g[b], p[b], d[b][{c}]); "
                                 f"s[b] = fmaf(g[b], x[b][{c}], s[b]); }}")
                    L.append("      }")
                if tangent:
                    L.append(f"      {each}{{ d[b][{i}] = fmaf(ds[b], x[b][{j}], fmaf(s[b], h[b][{j}], d[b][{i}]));"
                             f" d[b][{j}] = fmaf(ds[b], x[b][{i}], fmaf(s[b], h[b][{i}], d[b][{j}])); }}")
                else:
                    L.append(f"      {each}{{ d[b][{i}] = fmaf(s[b], x[b][{j}], d[b][{i}]);"
                             f" d[b][{j}] = fmaf(s[b], x[b][{i}], d[b][{j}]); }}")
            L.append("    }")
        L.append("  }")
    # dw: acc[r - Q * PAIR_BLOCK] += go[k] m (m its derivative along h for the jvp form), pairs of block Q
    nb = (R + PAIR_BLOCK - 1) // PAIR_BLOCK
    L.append(f"  static constexpr int NB = {nb};")
    for name, tangent in (("dw", False), ("dwjvp", True)):
        hargs = "const float* __restrict__ h, " if tangent else ""
        L.append(f"  template <int Q>\n  __device__ __forceinline__ static void {name}(const float* __restrict__ x, {hargs}"
                 "const float* __restrict__ go, float* __restrict__ acc) {")
        for q in range(nb):
            L.append(f"    {'if' if q == 0 else 'else if'} constexpr (Q == {q}) {{")
            lo, hi = q * PAIR_BLOCK, min(R, (q + 1) * PAIR_BLOCK)

            def add(m, value):
                for n, (k, _) in enumerate(mono_all[m]):
                    r = first[m] + n
                    if lo <= r < hi:
                        L.append(f"          acc[{r - lo}] = fmaf({value}, go[{k}], acc[{r - lo}]);")
            for g in blocks:
                ms = [m for m in ([g] if g in mono_all else []) + third[g]
                      if first[m] < hi and first[m] + len(mono_all[m]) > lo]
                if not ms:
                    continue
                L.append("      {")
                if len(g) == 1:
                    add(g, f"{'h' if tangent else 'x'}[{g[0]}]")
                else:
                    i, j = g
                    L.append(f"        const float p = x[{i}] * x[{j}];"
                             + (f" const float dp = fmaf(h[{i}], x[{j}], x[{i}] * h[{j}]);" if tangent else ""))
                    for m in ms:
                        if len(m) == 2:
                            add(m, "dp" if tangent else "p")
                            continue
                        c = m[-1]
                        e = f"fmaf(dp, x[{c}], p * h[{c}])" if tangent else f"p * x[{c}]"
                        L.append(f"        {{ const float m = {e};")
                        add(m, "m")
                        L.append("        }")
                L.append("      }")
            L.append("    }")
        L.append("  }")
    L.append("};")
    return "\n".join(L)


def generate(path):
    parts = ["// Generated by csrc/gen_sc.py from the frozen ICTC basis and the e3nn/MACE coupling. Do not edit.",
             "#pragma once", "#include <stdint.h>", "namespace ictc {",
             "struct ScWeights { const float* w[4][3]; };",
             "// Lane byte offset kept opaque so that its zero extension stays next to each load.",
             "__device__ __forceinline__ uint32_t sc_lane_offset(int c) {",
             "  uint32_t off = (uint32_t)c * 4u;",
             "  asm volatile(\"\" : \"+v\"(off));",
             "  return off;",
             "}",
             "__device__ __forceinline__ float sc_load(const float* __restrict__ row, uint32_t off) {",
             "  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(row) + off);",
             "}",
             "// Coefficient of pair r for the lane's channel: row r of the 64-channel table block t.",
             "__device__ __forceinline__ float sc_tab(const float* __restrict__ t, int r, uint32_t off) {",
             "  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(t + r * 64) + off);",
             "}",
             f"#define SC_ROWS(w, n) _Pragma(\"unroll\") for (int q = 0; q < {ROW_GROUP}; ++q) "
             f"if ((n) * {ROW_GROUP} + q < PAIRS) w[q] = sc_tab(t, (n) * {ROW_GROUP} + q, off)",
             "#define SC_AHEAD __builtin_amdgcn_sched_barrier(0)",
             "#define SC_EACH(b) _Pragma(\"unroll\") for (int b = 0; b < B; ++b)",
             "template <int LI, int LT, int CORR> struct Sc;", "template <int LI, int LT, int CORR> struct ScTab;"]
    cfgs = []
    for li, lt in CONFIGS:
        for corr in (1, 2, 3):
            parts.append(sc_struct(li, lt, corr))
            cfgs.append((li, lt, corr))
    for li, lt in TABLE_CONFIGS:
        parts.append(tab_struct(li, lt, 3))
    parts.append("}  // namespace ictc")
    parts.append("#define ICTC_FOR_EACH_SC_TAB(X) " + " ".join(f"X({a},{b},3)" for a, b in TABLE_CONFIGS))
    parts.append("#define ICTC_FOR_EACH_SC(X) " + " ".join(f"X({a},{b},{c})" for a, b, c in cfgs))
    text = "\n".join(parts) + "\n"
    os.makedirs(os.path.dirname(path), exist_ok=True)
    old = open(path).read() if os.path.exists(path) else None
    if old != text:
        with open(path, "w") as fh:
            fh.write(text)
    return cfgs


if __name__ == "__main__":
    out = sys.argv[1] if len(sys.argv) > 1 else os.path.join(_HERE, "generated", "ictc_sc.h")
    print(len(generate(out)), "SC configurations ->", out)
