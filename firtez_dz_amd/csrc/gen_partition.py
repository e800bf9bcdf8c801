"""Generate fz_partition_gen.h: the partition-function programs of
fz_atomdata.h (PARTITION_FUNCTION, atom_database.f90:121-1036, one stack
program per element) turned into straight-line device code: one out-of-line
function per element, dispatched by a switch on the (wave-uniform) element
index.  The operations and their order are those of the programs, FP
contraction is off, and conditional assignments stay selects, so the results
are those of the stack-program interpreter bit for bit where PF_DIV and PF_EXP
are the plain division and exponential (as they are unless the includer
defines them); what goes away is the interpreter's per-opcode dispatch and its
register-indexed stack.  Each element has a second function without the
derivatives.

  python firtez_dz_amd/csrc/gen_partition.py     (rewrites fz_partition_gen.h)
"""
from __future__ import annotations

import os
import re

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "fz_atomdata.h")
OUT = os.path.join(HERE, "fz_partition_gen.h")

OPS = ["END", "CONST", "VAR", "ADD", "SUB", "MUL", "DIV", "NEG", "EXP", "MAX", "AMAX1",
       "STORE", "GT", "LT", "LE", "GE", "NE", "EQ", "SEL", "AND"]
VARS = ["vT", "vX", "vY", "vDX", "vUI", "vUII", "vUIII", "vDUI", "vDUII", "vDUIII"]


def array(text, name, conv):
    m = re.search(r"%s\[[^\]]*\]\s*=\s*\{(.*?)\};" % re.escape(name), text, re.S)
    return [conv(x) for x in m.group(1).replace("\n", " ").split(",") if x.strip()]


def lit(x: float) -> str:
    r = repr(float(x))
    if "e" not in r and "." not in r and "inf" not in r:
        r += ".0"
    return r


def element_code(ops, args, consts):
    lines, stack, n = [], [], [0]

    def tmp(expr):
        name = "t%d" % n[0]
        n[0] += 1
        lines.append("const double %s = %s;" % (name, expr))
        return name

    for op, a in zip(ops, args):
        name = OPS[op]
        if name == "END":
            continue
        if name == "CONST":
            stack.append(lit(consts[a]))
        elif name == "VAR":
            stack.append(VARS[a])
        elif name == "STORE":
            lines.append("%s = %s;" % (VARS[a], stack.pop()))
        elif name == "NEG":
            stack.append(tmp("-%s" % stack.pop()))
        elif name == "EXP":
            stack.append(tmp("PF_EXP(%s)" % stack.pop()))
        elif name == "SEL":
            c, old, nw = stack.pop(), stack.pop(), stack.pop()
            stack.append(tmp("(%s != 0.0) ? %s : %s" % (c, nw, old)))
        else:
            y, x = stack.pop(), stack.pop()
            expr = {
                "ADD": "%s + %s", "SUB": "%s - %s", "MUL": "%s * %s", "DIV": "PF_DIV(%s, %s)",
                "MAX": "(%s > %s) ? {x} : {y}", "AMAX1": "pf_amax1(%s, %s)",
                "GT": "(%s > %s) ? 1.0 : 0.0", "LT": "(%s < %s) ? 1.0 : 0.0", "LE": "(%s <= %s) ? 1.0 : 0.0",
                "GE": "(%s >= %s) ? 1.0 : 0.0", "NE": "(%s != %s) ? 1.0 : 0.0", "EQ": "(%s == %s) ? 1.0 : 0.0",
                "AND": "(%s != 0.0 && %s != 0.0) ? 1.0 : 0.0",
            }[name]
            if name == "MAX":
                expr = ("(%s > %s) ? %s : %s" % (x, y, x, y))
            else:
                expr = expr % (x, y)
            stack.append(tmp(expr))
    assert not stack, stack
    return lines


def without_derivatives(lines):
    """The lines that the partition functions themselves need."""
    need, out = {"vUI", "vUII", "vUIII"}, []
    for ln in reversed(lines):
        name, expr = re.match(r"(?:const double )?(\w+) = (.*);$", ln).groups()
        if name in need:
            out.append(ln)
            need.update(re.findall(r"\b(?:v[A-Z]+|t\d+)\b", expr))
    return out[::-1]


def main():
    text = open(SRC).read()
    nelem = int(re.search(r"#define FZ_NELEM (\d+)", text).group(1))
    start = array(text, "fz_pf_start", int)
    ops = array(text, "fz_pf_op", int)
    args = array(text, "fz_pf_arg", int)
    consts = array(text, "fz_pf_const", float)
    out = ["/* Generated by gen_partition.py from fz_atomdata.h (the partition-function",
           " * programs of atom_database.f90:121-1036).  Do not edit by hand. */",
           "#pragma once", "",
           "namespace fz {", "",
           "// REAL(4) AMAX1 of two values, as the programs' AMAX1 opcode",
           "__device__ __forceinline__ double pf_amax1(double x, double y) {",
           "  const float fx = (float)x, fy = (float)y;",
           "  return (double)(fx > fy ? fx : fy);",
           "}", "",
           "#ifndef PF_DIV",
           "#define PF_DIV(x, y) ((x) / (y))",
           "#define PF_EXP(x) exp(x)",
           "#endif", "",
           "// One function per element (kept out of line: inlined into one switch the",
           "// 92 bodies are scheduled together and the register demand explodes).",
           "struct PfOut { double u[3], du[3]; };",
           "struct PfVal { double u[3]; };"]
    for e in range(nelem):
        body = element_code(ops[start[e]:start[e + 1]], args[start[e]:start[e + 1]], consts)
        out += ["__device__ __noinline__ PfOut pf_elem_%d(double vT, double vX, double vY, double vDX) {" % e,
                "#pragma clang fp contract(off)",
                "  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;",
                "  (void)vT; (void)vX; (void)vY; (void)vDX;"]
        out += ["  " + ln for ln in body]
        out += ["  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};", "}", ""]
        out += ["__device__ __noinline__ PfVal pf_value_%d(double vT, double vX, double vY) {" % e,
                "#pragma clang fp contract(off)",
                "  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;",
                "  (void)vT; (void)vX; (void)vY;"]
        out += ["  " + ln for ln in without_derivatives(body)]
        out += ["  return PfVal{{vUI, vUII, vUIII}};", "}", ""]
    out += ["// The same without derivatives, vX = log(5040 / T) and vY = 1e-3 T given",
            "__device__ __forceinline__ void partition_values(int elem, double vT, double vX, double vY, double u[3]) {",
            "  PfVal r = {{0.0, 0.0, 0.0}};",
            "  switch (elem) {"]
    for e in range(nelem):
        out.append("    case %d: r = pf_value_%d(vT, vX, vY); break;" % (e, e))
    out += ["    default: break;", "  }",
            "  u[0] = r.u[0]; u[1] = r.u[1]; u[2] = r.u[2];",
            "}", ""]
    out += ["// U_I, U_II, U_III and their d ln U / dT at T for element elem (0-based)",
            "__device__ __forceinline__ void partition_at(int elem, double vT, double vX, double vY, double vDX, double u[3],",
            "                                             double du[3]) {",
            "  PfOut r = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};",
            "  switch (elem) {"]
    for e in range(nelem):
        out.append("    case %d: r = pf_elem_%d(vT, vX, vY, vDX); break;" % (e, e))
    out += ["    default: break;", "  }",
            "  u[0] = r.u[0]; u[1] = r.u[1]; u[2] = r.u[2];",
            "  du[0] = r.du[0]; du[1] = r.du[1]; du[2] = r.du[2];",
            "}", "",
            "__device__ __forceinline__ void partition_gen(int elem, double T, double u[3], double du[3]) {",
            "  partition_at(elem, T, log(5040.0 / T), 1.0e-3 * T, -1.0 / T, u, du);",
            "}", "", "}  // namespace fz", ""]
    with open(OUT, "w") as fh:
        fh.write("\n".join(out))


if __name__ == "__main__":
    main()
