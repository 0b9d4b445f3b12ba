"""Build libqfe.so (HIP kernels for gfx950 + host engine + C ABI) in-tree.

    python qdk-chemistry_amd/build.py [-j N]

Steps: Rys table (generated once, cached in qdk_chemistry_amd/lib/), one
translation unit per ERI class (csrc/gen/, keeps compile times bounded and
parallel), then hipcc compile + link into qdk_chemistry_amd/lib/libqfe.so.
Every step recompiles only what changed (mtime check), except with --force.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "qdk_chemistry_amd", "lib")
MAX_L = int(os.environ.get("QFE_MAX_L", "3"))
# generated sources and objects per compiled maximum l (the macro reaches every TU)
GEN = os.path.join(CSRC, "gen", f"l{MAX_L}")
OBJ = os.path.join(CSRC, "_build", f"l{MAX_L}")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HIP_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++20", "-fPIC", f"-DQFE_MAX_L={MAX_L}",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-result"]
CXX = os.environ.get("CXX", "g++")
CXX_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-fopenmp", f"-DQFE_MAX_L={MAX_L}", "-I/opt/rocm/include",
             "-D__HIP_PLATFORM_AMD__"]


def pair_classes(maxl):
    out = []
    for la in range(maxl + 1):
        for lb in range(la + 1):
            out.append((la, lb))
    return out


def _ncart(l):
    return (l + 1) * (l + 2) // 2


def _nsph(l):
    return 2 * l + 1 if l >= 2 else _ncart(l)


# Accumulators per thread of classes whose kernels spilled with the default
# (48 up to d shells; with an f shell 24): the class's generated sources define
# QFE_JK_ACC_F, which JKChunks (csrc/eri_class.hpp) then uses.
JK_ACC_F = {(2, 1, 1, 1): 40}


def jk_acc(la, lb, lc, ld):
    if (la, lb, lc, ld) in JK_ACC_F:
        return JK_ACC_F[(la, lb, lc, ld)]
    return 48 if max(la, lb, lc, ld) <= 2 else 24


def jk_chunks(la, lb, lc, ld):
    """(bra function x ket cartesian) chunks of ClassOps (JKChunks in csrc/eri_class.hpp)."""
    rows_max = 6
    acc = jk_acc(la, lb, lc, ld)
    nsa, nsb = _nsph(la), _nsph(lb)
    nbra, nketc = nsa * nsb, _ncart(lc) * _ncart(ld)
    kch = min(nketc, acc)
    nkch = -(-nketc // kch)

    def rows(q0, q1):
        nma = (q1 - 1) // nsb - q0 // nsb + 1
        return nma + (nsb if nma > 1 else q1 - q0)

    bch_ = max(1, min(nbra, acc // kch))
    bch = bch_
    while bch > 1 and max(rows(q0, min(q0 + bch, nbra)) for q0 in range(0, nbra, bch)) > rows_max:
        bch -= 1
    nbu = -(-nbra // bch)
    wa = min(bch_ if bch_ < nsb else nsb, rows_max - 1)
    mp = -(-nsb // wa)
    return min(nsa * mp, nbu) * nkch


def jk_segment(la, lb, lc, ld):
    """Whether a class has segment kernels (csrc/eri_class.hpp).  Every chunk of
    a class is a launch that repeats its integrals; from eight chunks on, the
    f-shell classes are faster in the cooperative kernel (csrc/eri_jk_coop.hpp)
    at every size measured: (ff|ff) in 343 chunks 9.4 ms against 36 us for 167
    quartets, (fd|dp) 35 chunks 2.5 against 1.8 ms for 114,826."""
    return max(la, lb, lc, ld) <= 2 or jk_chunks(la, lb, lc, ld) <= 7


def jk_coop_tasks(la, lb, lc, ld):
    """Quartets up to which a class with segment kernels runs in the cooperative
    kernel.  A segment kernel takes 0.1-1 ms however few quartets there are (a
    thread's chain of primitive quartets, once per chunk); the cooperative one
    takes 3-15 ns a quartet, more than a full segment kernel."""
    return (50000 if jk_chunks(la, lb, lc, ld) >= 3 or (la, lb, lc, ld) == (1, 1, 1, 1)
            else 25000 if la + lb + lc + ld <= 1 else 15000)


# highest l of the gradient kernels
GRAD_MAX_L = 3


def grad_coop_tasks(ltot):
    """Quartets up to which a class without f shells runs in the cooperative
    gradient kernel (csrc/eri_grad_coop.hpp, a block per quartet) instead of
    the chunk kernels of csrc/eri_grad.hpp (a thread per quartet and chunk).
    With few quartets a thread's chain of primitive quartets is the time, and
    every chunk repeats it: (dp|pp) at 14,376 quartets 4.2 ms in 18 chunks
    against 0.32 ms.  With many the chunk kernels win, as they read no LDS
    tables: (dp|pp) at 808,005 quartets 8.1 against 11.1 ms.  The two meet at
    60-150 thousand quartets up to L = 3 and from L = 6 ((pp|ss) at 135,741:
    0.56 and 0.54 ms; (dd|dd) at 34,133: 2.3 and 2.6 ms) and near 200-400
    thousand between ((ds|pp) at 417,355: 3.4 and 3.3 ms)."""
    return 200000 if 4 <= ltot <= 5 else (100000 if ltot < 4 else 60000)


def grad_chunks(la, lb, lc, ld):
    """(bra x ket) cartesian chunks of GradOps (GradChunks in csrc/eri_grad.hpp)."""
    weights = 12
    nbc, nketc = _ncart(la) * _ncart(lb), _ncart(lc) * _ncart(ld)
    kch = min(nketc, weights)
    nkch = -(-nketc // kch)
    bch = max(1, min(nbc, weights // kch))
    return -(-nbc // bch) * nkch


def _parts(nch, kernels_per_chunk, ltot, budget=90.0):
    """Split chunks [0, nch) into ranges whose estimated compile time (seconds,
    measured: ~1.7 s per kernel at L = 8, x1.75 per unit of L) fits the budget."""
    per_chunk = kernels_per_chunk * 1.7 * 1.75 ** (ltot - 8)
    nparts = max(1, min(nch, int(-(-nch * per_chunk // budget))))
    step = -(-nch // nparts)
    return [(c0, min(nch, c0 + step)) for c0 in range(0, nch, step)]


def gen_sources():
    os.makedirs(GEN, exist_ok=True)
    pcs = pair_classes(MAX_L)
    files = []
    decls, jk_cases, jc_cases, sw_cases, gr_cases, dn_cases = [], [], [], [], [], []
    head = ["// generated by build.py", '#include "../../eri_grad.hpp"', "namespace qfe {"]
    for b, (la, lb) in enumerate(pcs):
        for k, (lc, ld) in enumerate(pcs[: b + 1]):
            tag = f"{la}{lb}{lc}{ld}"
            ops = f"ClassOps<{la}, {lb}, {lc}, {ld}, true>"
            fcls = max(la, lb, lc, ld) >= 3
            ltot = la + lb + lc + ld
            nch = jk_chunks(la, lb, lc, ld)
            # ERI J/K (+ Schwarz on the diagonal): kernels per chunk
            seg = jk_segment(la, lb, lc, ld)
            kpc = (1 if fcls else 4) + (1 if b == k else 0)  # segment kernels (+ Schwarz)
            jk_calls, sw_calls = [], []
            parts = _parts(nch, kpc, ltot) if seg else []
            for i, (c0, c1) in enumerate(parts):
                last = "true" if c1 == nch else "false"
                sfx = f"_p{i}" if len(parts) > 1 else ""
                fn = "jk_seg_only_range" if fcls else "jk_range"
                acc_def = [f"#define QFE_JK_ACC_F {JK_ACC_F[(la, lb, lc, ld)]}"] if (la, lb, lc, ld) in JK_ACC_F else []
                body = head[:1] + acc_def + head[1:] + [f"void jk_cls_{tag}{sfx}(const JKLaunch& a, hipStream_t s) {{ "
                               f"{ops}::{fn}<{c0}, {c1}, {last}>(a, s); }}"]
                decls.append(f"void jk_cls_{tag}{sfx}(const JKLaunch& a, hipStream_t s);")
                jk_calls.append(f"jk_cls_{tag}{sfx}(a, s);")
                if b == k and not fcls:
                    body.append(f"void schwarz_cls_{tag}{sfx}(const SchwarzLaunch& a, hipStream_t s) {{ "
                                f"{ops}::schwarz_range<{c0}, {c1}, {last}>(a, s); }}")
                    decls.append(f"void schwarz_cls_{tag}{sfx}(const SchwarzLaunch& a, hipStream_t s);")
                    sw_calls.append(f"schwarz_cls_{tag}{sfx}(a, s);")
                path = os.path.join(GEN, f"cls_{tag}{sfx}.hip")
                _write_if_changed(path, "\n".join(body + ["}  // namespace qfe"]) + "\n")
                files.append(path)
            # the cooperative J/K kernel (a block per quartet), and the
            # Schwarz kernel of the f-shell classes
            body = ["// generated by build.py", '#include "../../eri_jk_coop.hpp"', "namespace qfe {",
                    f"void jkc_cls_{tag}(const JKLaunch& a, hipStream_t s) {{ "
                    f"jk_coop<{la}, {lb}, {lc}, {ld}>(a, s); }}"]
            decls.append(f"void jkc_cls_{tag}(const JKLaunch& a, hipStream_t s);")
            if b == k and fcls:
                body.append(f"void schwarz_cls_{tag}(const SchwarzLaunch& a, hipStream_t s) {{ "
                            f"schwarz_coop<{la}, {lb}>(a, s); }}")
                decls.append(f"void schwarz_cls_{tag}(const SchwarzLaunch& a, hipStream_t s);")
                sw_calls.append(f"schwarz_cls_{tag}(a, s);")
            path = os.path.join(GEN, f"jkc_{tag}.hip")
            _write_if_changed(path, "\n".join(body + ["}  // namespace qfe"]) + "\n")
            files.append(path)
            if not fcls:  # the class of the dense AO tensor (MO transforms, shells up to d)
                dn = ["// generated by build.py", '#include "../../eri_dense_coop.hpp"', "namespace qfe {",
                      f"void dense_cls_{tag}(const DenseLaunch& a, const RysArgs& ra, hipStream_t s) {{ "
                      f"dense_coop<{la}, {lb}, {lc}, {ld}>(a, ra, s); }}", "}  // namespace qfe"]
                decls.append(f"void dense_cls_{tag}(const DenseLaunch& a, const RysArgs& ra, hipStream_t s);")
                dn_cases.append(f"  if (cb == {b} && ck == {k}) {{ dense_cls_{tag}(a, ra, s); return; }}")
                path = os.path.join(GEN, f"dense_{tag}.hip")
                _write_if_changed(path, "\n".join(dn) + "\n")
                files.append(path)
            few = f"coop && ntask <= {jk_coop_tasks(la, lb, lc, ld)}" if seg else "true"
            jc_cases.append(f"  if (cb == {b} && ck == {k}) return {few};")
            jk_cases.append(f"  if (cb == {b} && ck == {k}{' && few' if seg else ''}) {{ jkc_cls_{tag}(a, s); return; }}")
            if seg:
                jk_cases.append(f"  if (cb == {b} && ck == {k}) {{ {' '.join(jk_calls)} return; }}")
            if b == k:
                sw_cases.append(f"  if (c == {b}) {{ {' '.join(sw_calls)} return; }}")
            # cooperative gradient kernel (a block per quartet): every class with
            # an f shell, the others up to grad_coop_tasks quartets
            body = ["// generated by build.py", '#include "../../eri_grad_coop.hpp"', "namespace qfe {",
                    f"void gradc_cls_{tag}(const GradLaunch& a, hipStream_t s) {{ "
                    f"grad_coop<{la}, {lb}, {lc}, {ld}>(a, s); }}", "}  // namespace qfe"]
            decls.append(f"void gradc_cls_{tag}(const GradLaunch& a, hipStream_t s);")
            path = os.path.join(GEN, f"gradc_{tag}.hip")
            _write_if_changed(path, "\n".join(body) + "\n")
            files.append(path)
            few = "" if fcls else f" && a.coop && a.ntask <= {grad_coop_tasks(ltot)}"
            gr_cases.append(f"  if (cb == {b} && ck == {k}{few}) {{ gradc_cls_{tag}(a, s); return; }}")
            if fcls:
                continue
            gops = f"GradOps<{la}, {lb}, {lc}, {ld}, true>"
            gnch = grad_chunks(la, lb, lc, ld)
            gparts = _parts(gnch, 1, ltot + 1)
            gcalls = []
            for i, (c0, c1) in enumerate(gparts):
                last = "true" if c1 == gnch else "false"
                sfx = f"_p{i}" if len(gparts) > 1 else ""
                body = head + [f"void grad_cls_{tag}{sfx}(const GradLaunch& a, hipStream_t s) {{ "
                               f"{gops}::run_range<{c0}, {c1}, {last}>(a, s); }}", "}  // namespace qfe"]
                decls.append(f"void grad_cls_{tag}{sfx}(const GradLaunch& a, hipStream_t s);")
                gcalls.append(f"grad_cls_{tag}{sfx}(a, s);")
                path = os.path.join(GEN, f"grad_{tag}{sfx}.hip")
                _write_if_changed(path, "\n".join(body) + "\n")
                files.append(path)
            gr_cases.append(f"  if (cb == {b} && ck == {k}) {{ {' '.join(gcalls)} return; }}")
    disp = ["// generated by build.py -- class dispatch", '#include "../../kernels.hpp"',
            '#include "../../eri_dense.hpp"', "#include <stdexcept>",
            "namespace qfe {"] + decls + [
        "bool jk_cooperative(int cb, int ck, long long ntask, bool coop) {"] + jc_cases + ["  return false;", "}",
        "void launch_jk(int cb, int ck, bool pure, const JKLaunch& a, hipStream_t s) {",
        '  if (!pure) throw std::runtime_error("cartesian bases are not compiled");',
        "  const bool few = jk_cooperative(cb, ck, a.ntask, a.coop != 0);"] + jk_cases + [
        '  throw std::runtime_error("ERI class not compiled");', "}",
        "void launch_schwarz(int c, bool pure, const SchwarzLaunch& a, hipStream_t s) {",
        '  if (!pure) throw std::runtime_error("cartesian bases are not compiled");'] + sw_cases + [
        '  throw std::runtime_error("Schwarz class not compiled");', "}",
        "void launch_grad(int cb, int ck, bool pure, const GradLaunch& a, hipStream_t s) {",
        '  if (!pure) throw std::runtime_error("cartesian bases are not compiled");'] + gr_cases + [
        '  throw std::runtime_error("gradient class not compiled");', "}",
        "void launch_dense(int cb, int ck, const DenseLaunch& a, const RysArgs& ra, hipStream_t s) {"] + dn_cases + [
        '  throw std::runtime_error("dense class not compiled");', "}",
        f"int grad_max_l() {{ return {min(MAX_L, GRAD_MAX_L)}; }}", "}  // namespace qfe"]
    path = os.path.join(GEN, "dispatch.hip")
    _write_if_changed(path, "\n".join(disp) + "\n")
    files.append(path)
    # the chunk geometry of every class, read from the C++ (JKChunks), for
    # the FLOP model: qfe_class_chunks.  Classes compiled with their own
    # QFE_JK_ACC_F get a translation unit of their own with that definition.
    def _table_tu(acc_def, fname, classes, extern):
        t = ["// generated by build.py -- chunk geometry of the J/K class kernels"] + acc_def + [
             '#include "../../eri_class.hpp"', "namespace qfe {", "template <class Ops>",
             "static int chunk_table(int cap, int* out) {",
             "  using K = typename Ops::K;",
             "  hsfor<K::NCH>([&](auto c) {",
             "    using A = typename K::template At<c>;",
             "    if ((int)c < cap) {",
             "      out[4 * c + 0] = A::Q0; out[4 * c + 1] = A::Q1; out[4 * c + 2] = A::K0; out[4 * c + 3] = A::K1;",
             "    }", "  });", "  return K::NCH;", "}", "}  // namespace qfe",
             f'{extern}int {fname}(int la, int lb, int lc, int ld, int cap, int* out) {{']
        for (la, lb, lc, ld) in classes:
            if not jk_segment(la, lb, lc, ld):  # one cooperative kernel for the whole quartet
                t.append(f"  if (la == {la} && lb == {lb} && lc == {lc} && ld == {ld}) {{ if (cap > 0) {{ out[0] = "
                         f"out[2] = 0; out[1] = {_nsph(la) * _nsph(lb)}; out[3] = {_ncart(lc) * _ncart(ld)}; }} "
                         f"return 1; }}")
                continue
            t.append(f"  if (la == {la} && lb == {lb} && lc == {lc} && ld == {ld}) "
                     f"return qfe::chunk_table<qfe::ClassOps<{la}, {lb}, {lc}, {ld}, true>>(cap, out);")
        return t + ["  return -1;", "}"]

    all_cls = [(la, lb, lc, ld) for b, (la, lb) in enumerate(pcs) for (lc, ld) in pcs[: b + 1]]
    ch = []
    for acc in sorted(set(JK_ACC_F.values())):
        cl = [c for c in all_cls if JK_ACC_F.get(c) == acc]
        tu = _table_tu([f"#define QFE_JK_ACC_F {acc}"], f"qfe_class_chunks_acc{acc}", cl, "")
        path = os.path.join(GEN, f"chunks_acc{acc}.hip")
        _write_if_changed(path, "\n".join(tu) + "\n")
        files.append(path)
        ch.append(f"int qfe_class_chunks_acc{acc}(int la, int lb, int lc, int ld, int cap, int* out);")
    ch = _table_tu([], "qfe_class_chunks_default", [c for c in all_cls if c not in JK_ACC_F], "static ") + ch
    ch.append('extern "C" int qfe_class_chunks(int la, int lb, int lc, int ld, int cap, int* out) {')
    for c, acc in sorted(JK_ACC_F.items()):
        ch.append(f"  if (la == {c[0]} && lb == {c[1]} && lc == {c[2]} && ld == {c[3]}) "
                  f"return qfe_class_chunks_acc{acc}(la, lb, lc, ld, cap, out);")
    ch += ["  return qfe_class_chunks_default(la, lb, lc, ld, cap, out);", "}"]
    path = os.path.join(GEN, "chunks.hip")
    _write_if_changed(path, "\n".join(ch) + "\n")
    files.append(path)
    # heaviest first, so the longest compiles start early
    def _cost(f):
        n = os.path.basename(f)
        digits = [c for c in n if c.isdigit()][:4]
        return -sum(int(c) for c in digits) if len(digits) == 4 else 0
    return sorted(files, key=_cost)


def _write_if_changed(path, text):
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, "w") as f:
        f.write(text)


QFE_H = os.path.join(HERE, "..", "include", "qfe.h")


def _deps(src):
    """Headers each translation unit includes (build.py changes need --force)."""
    name = os.path.basename(src)
    core = ["eri_core.hpp", "sph_coef.inc", "kernels.hpp"]
    if name == "dispatch.hip":
        hs = core + ["dfj.hpp", "eri_dense.hpp"]
    elif name.startswith("chunks"):
        hs = core + ["eri_class.hpp"]
    elif name.startswith("dense_"):
        hs = core + ["fixed_point.hpp", "eri_class.hpp", "eri_coop.hpp", "eri_jk_coop.hpp", "dfj.hpp", "eri_dense.hpp",
                     "eri_dense_coop.hpp"]
    elif name.startswith("jkc_"):
        hs = core + ["fixed_point.hpp", "eri_class.hpp", "eri_coop.hpp", "eri_jk_coop.hpp"]
    elif name.startswith("gradc_"):
        hs = core + ["eri_class.hpp", "eri_grad.hpp", "eri_coop.hpp", "eri_grad_coop.hpp"]
    elif name.startswith("grad_") or name.startswith("cls_"):
        hs = core + ["eri_class.hpp", "eri_grad.hpp"]
    elif name == "kernels.hip":
        hs = core + ["screen.hpp"]
    elif name == "engine.cpp":
        hs = core + ["screen.hpp", "host_common.hpp", "onebody_gpu.hpp", "dfj.hpp", "eri_dense.hpp"]
    elif name == "onebody_gpu.hip":
        hs = core + ["onebody_gpu.hpp"]
    elif name == "dfj.hip":
        hs = core + ["dfj.hpp"]
    elif name == "eri_dense.hip":
        hs = core + ["dfj.hpp", "eri_dense.hpp"]
    else:  # onebody.cpp
        hs = ["host_common.hpp", "sph_coef.inc"]
    out = [os.path.join(CSRC, h) for h in hs]
    if name in ("engine.cpp", "onebody.cpp"):
        out.append(QFE_H)
    return out


def _stale(obj, src, force):
    if force or not os.path.exists(obj):
        return True
    t = os.path.getmtime(obj)
    return any(os.path.getmtime(d) >= t for d in [src] + _deps(src) if os.path.exists(d))


def _spills(stderr):
    """Kernels with VGPR spills, from the kernel-resource-usage remarks."""
    out, name = [], None
    for line in stderr.splitlines():
        if "remark: Function Name:" in line:
            name = line.split("Function Name:", 1)[1].split("[-Rpass")[0].strip()
        elif "remark:" in line and "VGPRs Spill:" in line:
            n = int(line.split("VGPRs Spill:", 1)[1].split()[0])
            if n > 0:
                out.append((name, n))
    return out


def _compile(src, obj, force):
    """Compile one TU.  Every HIP kernel must be free of VGPR spills: spilling
    instances of the ERI kernels have produced wrong results on gfx950, so a
    spill fails the build (the chunk sizes in csrc keep every class below)."""
    if not _stale(obj, src, force):
        return obj, 0.0, ""
    import time
    t0 = time.time()
    hip = src.endswith(".hip")
    if hip or src.endswith("engine.cpp"):
        cmd = [HIPCC] + HIP_FLAGS + (["-Rpass-analysis=kernel-resource-usage"] if hip else []) + \
            ["-x", "hip", "-c", src, "-o", obj]
    else:
        cmd = [CXX] + CXX_FLAGS + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stderr[-4000:]}")
    sp = _spills(r.stderr) if hip else []
    if sp:
        if os.path.exists(obj):
            os.remove(obj)
        listing = "\n".join(f"  {n} VGPRs spilled: {k}" for k, n in sp[:20])
        raise RuntimeError(f"kernels with register spills in {os.path.basename(src)}:\n{listing}")
    return obj, time.time() - t0, ""


def ensure_rys_table(force=False):
    path = os.path.join(LIB, "rys_table.bin")
    if os.path.exists(path) and not force:
        return path
    os.makedirs(LIB, exist_ok=True)
    subprocess.run([sys.executable, os.path.join(CSRC, "gen_rys_table.py"), path], check=True)
    return path


def build(jobs=None, force=False, verbose=False):
    jobs = jobs or min(8, os.cpu_count() or 4)
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIB, exist_ok=True)
    ensure_rys_table()
    srcs = [os.path.join(CSRC, f) for f in ("kernels.hip", "engine.cpp", "onebody.cpp", "onebody_gpu.hip", "dfj.hip",
                                             "eri_dense.hip")] + gen_sources()
    objs = []
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        futs = []
        for s in srcs:
            o = os.path.join(OBJ, os.path.basename(s).replace(".", "_") + ".o")
            objs.append(o)
            futs.append(ex.submit(_compile, s, o, force))
        errors = []
        for f in futs:
            try:
                o, dt, err = f.result()
            except RuntimeError as e:  # compile every TU, then report all failures
                errors.append(str(e))
                continue
            if verbose and dt > 0:
                print(f"  compiled {os.path.basename(o)} in {dt:.1f}s", flush=True)
    if errors:
        raise RuntimeError("\n".join(errors))
    out = os.path.join(LIB, "libqfe.so")
    if force or not os.path.exists(out) or any(os.path.getmtime(o) > os.path.getmtime(out) for o in objs):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out + ".tmp"] + objs + ["-lgomp", "-L/opt/rocm/lib", "-lrocsolver", "-lrocblas"]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stderr[-4000:]}")
        os.replace(out + ".tmp", out)
    return out


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=None)
    ap.add_argument("--force", action="store_true")
    a = ap.parse_args()
    print(build(a.j, a.force, verbose=True))
