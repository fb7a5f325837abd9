"""Compile-time reaction records for the mechanisms shipped with the package.

    python -m xfluids_amd.gen_mech        (also run by xfluids_amd.build)

Writes csrc/gen/xf_mech_gen.h.  For every mechanism directory under
data/runtime.dat/Reaction it emits the per-reaction records the device rate
evaluation reads (A, B, Ea*4.184/Ru, masks and packed coefficients, exactly as
xf_set_mechanism builds them, see csrc/xf_api.hip) and the third-body table, as
constexpr functions.  The chemistry kernels instantiate one rate evaluation per
record set with these values known at compile time: the mask tests, scalar
loads and coefficient decoding of the generic loop fold away, and terms with a
zero factor are left out.  rxn_fast in csrc/xf_chem_kernels.h computes the values
of the generic loop's rxn_step in its order, so results are bit-identical; waves
whose temperatures or rates are out of its range take rxn_step itself.

A context uses a specialisation only when the records it was given compare
equal field by field (xf_mech_spec_find); any other mechanism runs the generic
loop.  Parsing follows the host reader (host/xf_setup.cpp read_reactions):
whitespace tokens, sections *forward_reaction, *backward_reaction,
*third_body, *Arrhenius, numbers by correctly rounded decimal conversion.
"""
import os
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
REACTION_DIR = os.path.join(PKG, "data", "runtime.dat", "Reaction")
OUT = os.path.join(PKG, "csrc", "gen", "xf_mech_gen.h")

RU = 6.02214076e26 * 1.380649e-23 * 1.0E-3   # Ru of csrc/xf_internal.h, same products


def read_mechanism(d):
    names = open(os.path.join(d, "species_list.dat")).read().split()
    ns = 0
    for w in names:
        try:
            float(w)
            break
        except ValueError:
            ns += 1
    sec = {}
    cur = None
    for w in open(os.path.join(d, "reaction_list.dat")).read().split():
        if w.startswith("*"):
            cur = sec.setdefault(w, []) if w in ("*forward_reaction", "*backward_reaction", "*third_body",
                                                  "*Arrhenius") else None
        elif cur is not None:
            try:
                cur.append(float(w))
            except ValueError:
                cur = None  # text after a section's numbers (a comment) ends it

    fw, bw, tb, ar = (sec.get(k, []) for k in ("*forward_reaction", "*backward_reaction", "*third_body",
                                               "*Arrhenius"))
    if ns == 0 or len(fw) % ns:
        raise ValueError("malformed mechanism in %s" % d)
    nr = len(fw) // ns
    if len(bw) < len(fw) or len(tb) < len(fw) or len(ar) < 3 * nr:
        raise ValueError("incomplete mechanism in %s" % d)
    return ns, nr, [int(v) for v in fw[:ns * nr]], [int(v) for v in bw[:ns * nr]], tb[:ns * nr], ar[:3 * nr]


def records(ns, nr, nu_f, nu_b, third, ar):
    """The DevRxn fields of xf_set_mechanism, reaction by reaction."""
    out = []
    for r in range(nr):
        md = mt = mf = mb = pd = pf = pb = 0
        tsum = 0.0
        for j in range(ns):
            tsum += third[r * ns + j]
        for j in range(ns):
            nf, nb = nu_f[r * ns + j], nu_b[r * ns + j]
            nd = nb - nf
            if not (0 <= nf <= 15 and 0 <= nb <= 15 and -8 <= nd <= 7):
                raise ValueError("coefficient out of range in reaction %d" % r)
            if nd:
                md |= 1 << j
                pd |= (nd + 8) << (4 * j)
            if third[r * ns + j] != 0.0:
                mt |= 1 << j
            if nf:
                mf |= 1 << j
                pf |= nf << (4 * j)
            if nb:
                mb |= 1 << j
                pb |= nb << (4 * j)
        A, B, E = ar[3 * r], ar[3 * r + 1], ar[3 * r + 2]
        out.append((A, B, E * 4.184 / RU, md, mt, mf, mb, pd, pf, pb, 1 if tsum > 0.0 else 0))
    return out


def hexd(x):
    return float(x).hex()


def emit(specs):
    L = ["// Generated by xfluids_amd/gen_mech.py from data/runtime.dat/Reaction; rebuilt on",
         "// every build.  Records of the shipped mechanisms as compile-time constants.",
         "#pragma once", "#include \"../xf_internal.h\"", "", "namespace xf {", "",
         "constexpr int XF_NMECH_SPEC = %d;" % len(specs), "",
         "template <int K> struct MechSpec;", ""]
    for k, (name, ns, nr, rec, third) in enumerate(specs):
        L.append("// %s: %d species, %d reactions" % (name, ns, nr))
        L.append("template <> struct MechSpec<%d> {" % k)
        L.append("    static constexpr int NS = %d, NR = %d;" % (ns, nr))
        L.append("    static constexpr DevRxn rx(int r)")
        L.append("    {")
        L.append("        switch (r) {")
        for r, (A, B, EaR, md, mt, mf, mb, pd, pf, pb, ti) in enumerate(rec):
            L.append("        case %d: return DevRxn{%s, %s, %s, 0x%xu, 0x%xu, 0x%xu, 0x%xu, 0x%xull, 0x%xull, 0x%xull, %d, 0};"
                     % (r, hexd(A), hexd(B), hexd(EaR), md, mt, mf, mb, pd, pf, pb, ti))
        L.append("        default: return DevRxn{};")
        L.append("        }")
        L.append("    }")
        L.append("    // third-body efficiency of species s in reaction r, third[r * NS + s]")
        L.append("    static constexpr double eff(int r, int s)")
        L.append("    {")
        L.append("        switch (r * NS + s) {")
        for i, v in enumerate(third):
            if v != 0.0:
                L.append("        case %d: return %s;" % (i, hexd(v)))
        L.append("        default: return 0.0;")
        L.append("        }")
        L.append("    }")
        L.append("};")
        L.append("")
    # host-side matching against the records a context was given
    L.append("template <int K> inline bool mech_spec_equal(int NS, int NR, const DevRxn *rx, const double *third)")
    L.append("{")
    L.append("    using S = MechSpec<K>;")
    L.append("    if (NS != S::NS || NR != S::NR) return false;")
    L.append("    for (int r = 0; r < NR; r++) {")
    L.append("        const DevRxn a = S::rx(r), &b = rx[r];")
    L.append("        if (a.A != b.A || a.B != b.B || a.EaR != b.EaR || a.md != b.md || a.mt != b.mt || a.mf != b.mf ||")
    L.append("            a.mb != b.mb || a.pd != b.pd || a.pf != b.pf || a.pb != b.pb || a.third_ind != b.third_ind)")
    L.append("            return false;")
    L.append("        for (int s = 0; s < NS; s++)")
    L.append("            if (S::eff(r, s) != third[r * NS + s]) return false;")
    L.append("    }")
    L.append("    return true;")
    L.append("}")
    L.append("")
    L.append("// index of the compiled specialisation with these records, or -1")
    L.append("inline int mech_spec_find(int NS, int NR, const DevRxn *rx, const double *third)")
    L.append("{")
    for k in range(len(specs)):
        L.append("    if (mech_spec_equal<%d>(NS, NR, rx, third)) return %d;" % (k, k))
    L.append("    (void)NS, (void)NR, (void)rx, (void)third;")
    L.append("    return -1;")
    L.append("}")
    L.append("")
    L.append("// species count of specialisation K (0 when K is not one)")
    L.append("template <int K> constexpr int mech_spec_ns()")
    L.append("{")
    L.append("    if constexpr (K >= 0 && K < XF_NMECH_SPEC) return MechSpec<K>::NS;")
    L.append("    else return 0;")
    L.append("}")
    L.append("")
    L.append("} // namespace xf")
    return "\n".join(L) + "\n"


def generate(out=OUT):
    specs = []
    if os.path.isdir(REACTION_DIR):
        for name in sorted(os.listdir(REACTION_DIR)):
            d = os.path.join(REACTION_DIR, name)
            if not os.path.isfile(os.path.join(d, "reaction_list.dat")):
                continue
            ns, nr, nu_f, nu_b, third, ar = read_mechanism(d)
            specs.append((name, ns, nr, records(ns, nr, nu_f, nu_b, third, ar), third))
    text = emit(specs)
    os.makedirs(os.path.dirname(out), exist_ok=True)
    if not os.path.exists(out) or open(out).read() != text:
        with open(out, "w") as f:
            f.write(text)
    return out, [s[0] for s in specs]


if __name__ == "__main__":
    path, names = generate()
    print(path, names)
    sys.exit(0)
