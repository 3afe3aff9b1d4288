"""Emit the device code for each robot from its model table (build step).

    python -m prrtc_amd.robots.gen_headers   ->  prrtc_amd/csrc/robots/<robot>.gen.h

For each robot the generated header defines

    template <class Ctx> __device__ void check_<robot>(const float *q, Ctx &ctx)

which computes the joint frames (T_j = T_parent * F_j * Rz(q_j) or Tz(q_j)),
with every constant of F_j folded in (zeros dropped, +-1 turned into signs),
then runs the robot's collision checks in the reference's order
(src/planning/utils.cuh:336-33131): link gate sphere -> leaf spheres for the
environment, gate pair -> sphere pairs for self-collision.  Sphere centres are
formed only where a check needs them (t_f + R_f * local, constants folded).

The checks talk to the caller through ``Ctx``:

    bool live()                      this lane still needs an answer
    void env_gates<N>(x, y, z, r, hit)  N gate spheres vs. the obstacles
    bool env_any<N, EARLY>(x, y, z, r, on)  whether one of N leaf spheres hits
                                     an obstacle (env_any_bounded: with a ball
                                     that holds them); whole-wave calls.  EARLY:
                                     leave once every lane has a hit
    bool self(ax, ay, az, bx, by, bz, rsum)   sphere pair (true = hit)
    bool near_point(ax, ay, az, bx, by, bz, d2)  within sqrt(d2) (NaN: yes)
    void hit()                       this lane's pose collides
    void share_gates(uint64_t &)     gate bits after the gate pass (ORed
                                     across waves that split the obstacles)
    bool stop()                      wave-uniform: no lane needs more work

``stop()`` is called after every check group, which is where a wavefront
leaves early once its answer is decided; ``share_gates`` is called exactly
once per check, before the first ``stop()``.

Also emitted: ``fk_spheres_<robot>(q, out)`` that writes every sphere centre
(for FK parity dumps), and the joint limits.
"""
from __future__ import annotations

import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(os.path.dirname(HERE), "csrc", "robots")

sys.path.insert(0, os.path.abspath(os.path.join(HERE, "..", "..")))
from prrtc_amd.robots import load_model  # noqa: E402


def flit(v: float) -> str:
    v = float(np.float32(v))
    r = repr(v)
    if "e" not in r and "." not in r:
        r += ".0"
    return r + "f"


def half_up(v: float) -> int:
    """Bits of the smallest binary16 at or above v (v > 0)."""
    h = np.float16(v)
    if float(h) < v:
        h = np.nextafter(h, np.float16(np.inf))
    return int(h.view(np.uint16))


class Lin:
    """A linear form sum(c_i * var_i) + const, with constant folding."""

    def __init__(self, terms=None, const=0.0):
        self.terms = [(c, v) for c, v in (terms or []) if c != 0.0]
        self.const = const

    @staticmethod
    def var(name):
        return Lin([(1.0, name)], 0.0)

    def code(self) -> str:
        # fmaf-friendly chain: const + c1*v1 + c2*v2 ...
        expr = None
        if self.const != 0.0 or not self.terms:
            expr = flit(self.const)
        for c, v in self.terms:
            if c == 1.0:
                term = v
            elif c == -1.0:
                term = None
            else:
                term = f"{flit(c)} * {v}"
            if expr is None:
                expr = term if term is not None else f"-{v}"
            elif term is None:
                expr = f"{expr} - {v}"
            else:
                expr = f"{expr} + {term}"
        return expr


def gen_robot(name: str) -> str:
    return gen_robot_from(load_model(name))


def gen_robot_from(m: dict) -> str:
    """Device code of one model table (robots/<name>.json, or a table the
    robot-model compiler produced)."""
    name = m["name"]
    dof = m["dof"]
    joints = m["joints"]
    sph = m["spheres"]
    L = []
    w = L.append
    w(f"// Generated by prrtc_amd/robots/gen_headers.py from {name}.json -- do not edit.")
    w("#pragma once")
    w("")
    w(f"namespace prrtc::gen::{name} {{")
    w(f"constexpr int DOF = {dof};")
    w(f"constexpr int NSPHERES = {len(sph)};")
    w(f"constexpr int SELF_GROUPS = {sum(kind == 'self' for kind, _ in m['order'])};")
    w("__device__ __host__ constexpr float lower(int i) { constexpr float v[] = {" +
      ", ".join(flit(x) for x in m["lower"]) + "}; return v[i]; }")
    w("__device__ __host__ constexpr float span(int i) { constexpr float v[] = {" +
      ", ".join(flit(x) for x in m["range"]) + "}; return v[i]; }")
    w("")

    # ---------------- FK ------------------------------------------------
    # Every frame entry is either a folded constant (float) or the name of an
    # emitted value; Rsym/tsym keep that symbolic state per joint.
    Rsym = {-1: [[1.0 if r == c else 0.0 for c in range(3)] for r in range(3)]}
    tsym = {-1: [0.0, 0.0, 0.0]}

    def as_lin(v):
        return Lin(const=v) if isinstance(v, float) else Lin.var(v)

    def emit(lines, name, lin):
        """Emit `name = lin` unless it folds to a constant; return symbol."""
        if not lin.terms:
            return float(lin.const)
        if lin.const == 0.0 and len(lin.terms) == 1 and lin.terms[0][0] == 1.0:
            return lin.terms[0][1]
        lines.append(f"    const float {name} = {lin.code()}; \\")
        return name

    def scaled(sc, v):
        """(scalar name) * v as a list of (sign, text) parts, v constant or name"""
        if isinstance(v, float):
            if v == 0.0:
                return []
            return [("+" if v > 0 else "-", sc if abs(v) == 1.0 else f"{flit(abs(v))} * {sc}")]
        return [("+", f"{sc} * {v}")]

    def join(parts):
        if not parts:
            return None
        out = ("-" if parts[0][0] == "-" else "") + parts[0][1]
        for sgn, t in parts[1:]:
            out += f" {sgn} {t}"
        return out

    fk = ["#define PRRTC_FK_BODY \\"]
    for j, jt in enumerate(joints):
        p = jt["parent"]
        F = jt["rot"]
        Ft = jt["trans"]
        fk.append(f"    /* joint {j} ({jt['type']}, parent {p}) */ \\")
        M = [[None] * 3 for _ in range(3)]
        for r in range(3):
            for c in range(3):
                terms, const = [], 0.0
                for k in range(3):
                    f = float(F[k][c])
                    if f == 0.0:
                        continue
                    e = as_lin(Rsym[p][r][k])
                    const += e.const * f
                    terms += [(cc * f, v) for cc, v in e.terms]
                M[r][c] = emit(fk, f"M{j}_{r}{c}", Lin(terms, const))
        tt = []
        for r in range(3):
            base = as_lin(tsym[p][r]) if not isinstance(tsym[p][r], Lin) else tsym[p][r]
            terms, const = list(base.terms), base.const
            for k in range(3):
                f = float(Ft[k])
                if f == 0.0:
                    continue
                e = as_lin(Rsym[p][r][k])
                const += e.const * f
                terms += [(cc * f, v) for cc, v in e.terms]
            tt.append(Lin(terms, const))
        R = [[None] * 3 for _ in range(3)]
        if jt["type"] == "revolute":
            fk.append(f"    float s{j}, c{j}; sincosf(q[{j}], &s{j}, &c{j}); \\")
            for r in range(3):
                m0, m1 = M[r][0], M[r][1]
                e0 = join(scaled(f"c{j}", m0) + scaled(f"s{j}", m1))
                neg0 = -m0 if isinstance(m0, float) else None
                e1_parts = scaled(f"c{j}", m1)
                if neg0 is not None:
                    e1_parts += scaled(f"s{j}", neg0)
                else:
                    e1_parts += [("-", f"s{j} * {m0}")]
                e1 = join(e1_parts)
                for c, e in ((0, e0), (1, e1)):
                    if e is None:
                        R[r][c] = 0.0
                    else:
                        fk.append(f"    const float R{j}_{r}{c} = {e}; \\")
                        R[r][c] = f"R{j}_{r}{c}"
                R[r][2] = M[r][2]
            tvals = []
            for r in range(3):
                tvals.append(emit(fk, f"t{j}_{r}", tt[r]))
        else:
            for r in range(3):
                for c in range(3):
                    R[r][c] = M[r][c]
            tvals = []
            for r in range(3):
                lin = tt[r]
                m2 = M[r][2]
                extra = scaled(f"q[{j}]", m2)
                if extra:
                    base = lin.code() if (lin.terms or lin.const != 0.0) else None
                    e = join(extra)
                    code = e if base is None else f"{base} + ({e})"
                    fk.append(f"    const float t{j}_{r} = {code}; \\")
                    tvals.append(f"t{j}_{r}")
                else:
                    tvals.append(emit(fk, f"t{j}_{r}", lin))
        Rsym[j] = R
        tsym[j] = tvals
    fk.append("    /* end FK */")

    def centre(i):
        sp = sph[i]
        f = sp["frame"]
        loc = [float(np.float32(x)) for x in sp["local"]]
        if f < 0:
            return [flit(loc[0]), flit(loc[1]), flit(loc[2])]
        out = []
        for r in range(3):
            terms, const = [], 0.0
            for k in range(3):
                if loc[k] == 0.0:
                    continue
                e = as_lin(Rsym[f][r][k])
                const += e.const * loc[k]
                terms += [(cc * loc[k], v) for cc, v in e.terms]
            tb = as_lin(tsym[f][r])
            out.append(Lin(terms + tb.terms, const + tb.const).code())
        return out

    L.extend(fk)
    w("")

    # ---------------- FK dump -------------------------------------------
    w("__device__ __forceinline__ void fk_spheres(const float *q, float *out) {")
    w("    PRRTC_FK_BODY")
    for i in range(len(sph)):
        c = centre(i)
        w(f"    out[{3 * i}] = {c[0]}; out[{3 * i + 1}] = {c[1]}; out[{3 * i + 2}] = {c[2]};")
    w("}")
    w("__host__ __device__ constexpr float radius(int i) { constexpr float v[] = {" +
      ", ".join(flit(s["r"]) for s in sph) + "}; return v[i]; }")
    w("")

    # ---------------- checks --------------------------------------------
    # Environment first: every gate sphere (and every direct single-sphere
    # check) against the obstacle tables in passes of up to GATE_CHUNK spheres,
    # giving a per-lane bit per env check; then, link by link in the
    # reference's order, the leaf spheres of the links whose gate hit; then
    # the self-collision gate pairs and their sphere pairs.  The verdict is
    # the same OR of gated terms the reference evaluates (utils.cuh:336-5270).
    GATE_CHUNK = 12
    def pair_reach(chk):
        """Distance beyond which a self group's gates cannot touch: the sum of
        their radii, padded by 2^-16 relative and 1 mm absolute."""
        a, b = chk["gate"]
        return (float(sph[a]["r"]) + float(sph[b]["r"])) * (1.0 + 2.0 ** -16) + 1e-3

    # Panda's forearm-hand group (216 pairs) and its like were 2,000 of the
    # 4,900 VALU instructions of a free pass: 1M edges 7.9 -> 6.7 ms, 64 edges
    # 24.9 -> 21.6 us, one solve 204 -> 195 us.  Splitting smaller groups too
    # left Panda as it was and cost Fetch's edge kernel 4% (72 -> 75 us).
    SPLIT_MIN_PAIRS = 48

    def split_pairs(chk):
        """(outer spheres, inner spheres, inner gate, radius R) of a self group
        whose pairs are all of outer x inner, with the inner spheres in the
        ball of radius R about their gate; None where a group's pairs are
        cheaper tested outright.  An outer sphere's test against the ball
        costs about 10 instructions with its branch, a pair 8.  Of the two
        links the one expected to cost less is the outer: with the gates in
        touch, an outer sphere is taken to be within reach of the ball with
        the ratio of the two reaches' volumes."""
        best = None
        if len(chk["pairs"]) < SPLIT_MIN_PAIRS:
            return None
        for side in (0, 1):
            outer, inner = [], []
            for p in chk["pairs"]:
                if p[side] not in outer:
                    outer.append(p[side])
                if p[1 - side] not in inner:
                    inner.append(p[1 - side])
            gate = chk["gate"][1 - side]
            n = len(outer) * len(inner)
            if n != len(chk["pairs"]) or len(inner) < 5 or any(sph[x]["frame"] != sph[gate]["frame"] for x in inner):
                continue
            R = ball_of(gate, inner)
            gates = sum(float(sph[x]["r"]) for x in chk["gate"])
            near = sum(min(1.0, ((R + float(sph[x]["r"])) / gates) ** 3) for x in outer) / len(outer)
            cost = 10 * len(outer) + 8 * n * near
            if cost < 8 * n and (best is None or cost < best[0]):
                best = (cost, (outer, inner, gate, R))
        return best and best[1]

    w("template <class Ctx>")
    w("__device__ __forceinline__ void check(const float *q, Ctx &ctx) {")
    w("    PRRTC_FK_BODY")

    def self_call(a, b):
        ca, cb = centre(a), centre(b)
        rs = flit(np.float32(sph[a]["r"]) + np.float32(sph[b]["r"]))
        return f"ctx.self({ca[0]}, {ca[1]}, {ca[2]}, {cb[0]}, {cb[1]}, {cb[2]}, {rs})"

    def env_group(spheres_idx, call, indent):
        """The centres and radii of some spheres in arrays ex, ey, ez, er of
        `n`, and the lines `call` over them."""
        n = len(spheres_idx)
        cs = [centre(i) for i in spheres_idx]
        w(f"{indent}{{")
        w(f"{indent}    const float ex[{n}] = {{" + ", ".join(c[0] for c in cs) + "};")
        w(f"{indent}    const float ey[{n}] = {{" + ", ".join(c[1] for c in cs) + "};")
        w(f"{indent}    const float ez[{n}] = {{" + ", ".join(c[2] for c in cs) + "};")
        w(f"{indent}    const float er[{n}] = {{" + ", ".join(flit(sph[i]['r']) for i in spheres_idx) + "};")
        for line in call:
            w(f"{indent}    {line}")
        w(f"{indent}}}")

    def ball_of(gate, spheres):
        """Radius of the ball about a gate's centre that holds spheres riding
        on its frame: max |local - local_gate| + r, padded by 2^-16 relative
        and 1 mm absolute, rounded up to float32."""
        R = max(float(np.linalg.norm(np.array(sph[x]["local"], dtype=np.float64) -
                                     np.array(sph[gate]["local"], dtype=np.float64))) + float(sph[x]["r"])
                for x in spheres)
        return float(np.nextafter(np.float32(R * (1.0 + 2.0 ** -16) + 1e-3), np.float32(np.inf)))

    GROUP_MIN_LEAVES = 6

    def group_bound(chk):
        """Ball about the gate centre (ball_of) that holds every leaf sphere
        of the check, when the leaves ride on the gate's frame (rigidly).
        None when a leaf is on another frame, or when the check has fewer than
        GROUP_MIN_LEAVES leaves."""
        g = sph[chk["gate"]]
        # one extra test per obstacle pays for itself only over enough leaves
        if len(chk["leaves"]) < GROUP_MIN_LEAVES or any(sph[l]["frame"] != g["frame"] for l in chk["leaves"]):
            return None
        return centre(chk["gate"]), ball_of(chk["gate"], chk["leaves"])

    env = m["env_checks"]
    w("    uint64_t gate = 0;  /* bit k: env check k's gate sphere hit */")
    w("    if (ctx.any(ctx.live())) {")
    for c0 in range(0, len(env), GATE_CHUNK):
        ks = list(range(c0, min(len(env), c0 + GATE_CHUNK)))
        bits = " | ".join(f"((uint64_t)eh[{j}] << {k})" for j, k in enumerate(ks))
        env_group([env[k]["gate"] for k in ks],
                  [f"bool eh[{len(ks)}];", f"ctx.template env_gates<{len(ks)}>({c0}, ex, ey, ez, er, eh);",
                   f"gate |= {bits};"], "        ")
    w("    }")
    # the one point where waves that split the obstacles exchange gate bits:
    # before any early return, so every wave reaches it once per call
    w("    ctx.share_gates(gate);")
    direct_mask = sum(1 << k for k, c in enumerate(env) if c["direct"])
    if direct_mask:
        w(f"    if (ctx.live() && (gate & {direct_mask}ull)) ctx.hit();")
    w("    if (ctx.stop()) return;")
    for kind, k in m["order"]:
        if kind != "env":
            continue
        chk = env[k]
        if chk["direct"]:
            continue
        w(f"    /* env leaves: {chk['label']} */")
        w(f"    if (ctx.any(ctx.live() && (gate >> {k} & 1))) {{")
        n, bound = len(chk["leaves"]), group_bound(chk)
        if bound is None:
            call = f"ctx.template env_any<{n}, true>(ex, ey, ez, er, on)"
        else:
            gc, gr = bound
            call = f"ctx.template env_any_bounded<{n}, true>(ex, ey, ez, er, on, {gc[0]}, {gc[1]}, {gc[2]}, {flit(gr)})"
        w(f"        const bool on = ctx.live() && (gate >> {k} & 1);")
        env_group(chk["leaves"], [f"const bool eh = {call};", "if (on && eh) ctx.hit();"], "        ")
        w("        if (ctx.stop()) return;")
        w("    }")
    # Self groups are numbered in emission order; ctx.mine(j) lets a context
    # whose waves share a pose set give each group to one wave, and rules out
    # the groups whose gates stay apart over the whole wave (by the balls of
    # the gate pass, where every moving gate of the self groups took part in
    # it: forming a ball costs about as much as a group's own gate test).
    selfs = [m["self_checks"][k] for kind, k in m["order"] if kind == "self"]
    number = {c["gate"]: k for k, c in enumerate(env)}
    extra = [g for g in sorted({g for c in selfs for g in c["gate"]}) if g not in number]
    by_balls = bool(selfs) and all(sph[g]["frame"] < 0 for g in extra) and len(env) + len(extra) <= 64
    if by_balls:
        for g in extra:
            number[g] = len(number)
            c = centre(g)
            w(f"    ctx.fixed_gate({number[g]}, {c[0]}, {c[1]}, {c[2]});")
        w(f"    ctx.template self_near<{len(selfs)}>(self_gates);")
        words = [number[c["gate"][0]] | number[c["gate"][1]] << 8 | half_up(pair_reach(c)) << 16 for c in selfs]
        at = next(i for i, line in enumerate(L) if line == "template <class Ctx>")
        L[at:at] = ["// self groups: the two gates' numbers and, rounded up to binary16, their reach",
                    f"__device__ const uint32_t self_gates[{len(words)}] = {{" +
                    ", ".join(f"{x:#x}u" for x in words) + "};", ""]
    elif selfs:
        w(f"    ctx.template self_own<{len(selfs)}>();")
    BLOCK = 16   # groups passed over together where there are many (blocks do not cross a 64-group word)
    for j, chk in enumerate(selfs):
        if len(selfs) > 64 and j % BLOCK == 0:
            if j:
                w("    }")
            w(f"    if (ctx.mine_any({j}, {min(BLOCK, len(selfs) - j)})) {{")
        ga, gb = chk["gate"]
        w(f"    /* self: {chk['label']} */")
        w(f"    if (ctx.mine({j})) {{")
        w(f"        const bool g = ctx.live() && {self_call(ga, gb)};")
        w("        if (ctx.any(g)) {")
        if chk["direct"]:
            w("            if (g) ctx.hit();")
        else:
            sides = split_pairs(chk)
            ind = "            "
            if sides is None:
                w("            if (g) {")
                ind += "    "
            used = []
            for a, b in chk["pairs"]:
                for x in (a, b):
                    if x not in used:
                        used.append(x)
            for x in used:
                c = centre(x)
                w(f"{ind}const float s{x}x = {c[0]}, s{x}y = {c[1]}, s{x}z = {c[2]};")
            w(f"{ind}bool h = false;")

            def pair(a, b, indent):
                rs = flit(np.float32(sph[a]["r"]) + np.float32(sph[b]["r"]))
                w(f"{indent}h |= ctx.self(s{a}x, s{a}y, s{a}z, s{b}x, s{b}y, s{b}z, {rs});")

            if sides is None:
                for a, b in chk["pairs"]:
                    pair(a, b, ind)
                w(f"{ind}if (h) ctx.hit();")
                w("            }")
            else:
                # the spheres of one link one by one against the ball of the
                # other link's: most are out of its reach on every lane
                outer, inner, gate, R = sides
                c = centre(gate)
                w(f"{ind}const float cx = {c[0]}, cy = {c[1]}, cz = {c[2]};")
                for x in outer:
                    reach2 = np.nextafter(np.float32((R + float(sph[x]["r"])) ** 2), np.float32(np.inf))
                    w(f"{ind}if (ctx.any(g && ctx.near_point(s{x}x, s{x}y, s{x}z, cx, cy, cz, {flit(reach2)}))) {{")
                    for a, b in chk["pairs"]:
                        if x in (a, b):
                            pair(a, b, ind + "    ")
                    w(f"{ind}}}")
                w(f"{ind}if (g && h) ctx.hit();")
        w("            if (ctx.stop()) return;")
        w("        }")
        w("    }")
    if len(selfs) > 64:
        w("    }")
    w("}")
    w("#undef PRRTC_FK_BODY")
    w("")
    w(f"}}  // namespace prrtc::gen::{name}")
    return "\n".join(L) + "\n"


def main():
    os.makedirs(OUT, exist_ok=True)
    for name in ("panda", "fetch", "baxter", "ur5"):
        text = gen_robot(name)
        path = os.path.join(OUT, name + ".gen.h")
        old = open(path).read() if os.path.exists(path) else None
        if old != text:
            with open(path, "w") as fh:
                fh.write(text)


if __name__ == "__main__":
    main()
