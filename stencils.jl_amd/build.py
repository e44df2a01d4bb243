"""Build libstencils_hip.so for gfx950.

Generates one translation unit per build-time stencil shape (the offset
table is emitted as constants, so the compiler specialises the gather on it)
and one per element type for the runtime-offset kernels, compiles them in
parallel with hipcc and links the shared library into ``lib/``.

    python stencils.jl_amd/build.py [--jobs N] [--incremental]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
REPO = HERE.parent
sys.path.insert(0, str(HERE))

from stencils_hip import stencil as S  # noqa: E402

CSRC = HERE / "csrc"
GEN = HERE / "_build" / "gen"
OBJ = HERE / "_build" / "obj"
LIB = HERE / "lib" / "libstencils_hip.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

CXXFLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # Julia never contracts a + b * c; keep every product and sum rounded.
    "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt",
    # Packed FP32 instructions stay off (plain float code only).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{REPO / 'include'}", f"-I{CSRC}",
]

# Storage types: C++ type name, sth_dtype code name.
FLOAT_TYPES = [("float", "STH_F32"), ("double", "STH_F64"),
               ("bf16_t", "STH_BF16"), ("f16_t", "STH_F16")]
INT_TYPES = [("bool", "STH_BOOL"), ("uint8_t", "STH_U8"), ("int8_t", "STH_I8"),
             ("uint16_t", "STH_U16"), ("int16_t", "STH_I16"), ("uint32_t", "STH_U32"),
             ("int32_t", "STH_I32"), ("uint64_t", "STH_U64"), ("int64_t", "STH_I64")]

FOLD_OPS = ["OP_SUM", "OP_MEAN", "OP_MIN", "OP_MAX", "OP_KP"]

# Build-time catalogue: (stencil, ops) for float storage types.  Shapes outside
# it, and every integer type, use the runtime-offset kernels.
CATALOG = [
    (S.Window(1), FOLD_OPS), (S.Window(2), FOLD_OPS), (S.Window(3), FOLD_OPS),
    (S.Moore(1), FOLD_OPS), (S.Moore(2), FOLD_OPS),
    (S.VonNeumann(1), FOLD_OPS + ["OP_LAP"]), (S.VonNeumann(2), FOLD_OPS),
    (S.VonNeumann(3), FOLD_OPS),
    (S.Circle(1), FOLD_OPS), (S.Circle(2), FOLD_OPS), (S.Circle(3), FOLD_OPS),
    (S.VonNeumann(1, 3), FOLD_OPS + ["OP_LAP"]), (S.Moore(1, 3), FOLD_OPS),
]


def shape_name(st) -> str:
    return f"{type(st).__name__.lower()}_r{st.R}_n{st.N}"


ESIZE = {"float": 4, "double": 8, "bf16_t": 2, "f16_t": 2}


def stream_variants(ctype: str, st) -> list[tuple[int, int]]:
    """(V, KY) variants of the streaming kernel compiled for a shape: V cells
    per lane along dim 1 (16 bytes, or 8 for 16-bit types at radius >= 2 to
    bound the register box), KY rows per wave; the autotuner picks one."""
    r = max(abs(c) for o in st.offsets() for c in o)
    v = 16 // ESIZE[ctype]
    if ESIZE[ctype] == 2 and (r >= 2 or st.N == 3):
        v = 4
    # the first variant is the default (and the batched kernels' choice):
    # ordered by what tuned fastest on large arrays
    if st.N == 3:
        kys = (4, 2)
    elif r <= 1:
        kys = (4, 8)
    elif r == 2:
        kys = (4, 2)
    else:
        kys = (2, 1)
    if ESIZE[ctype] <= 4 and r == 3 and st.N == 2:
        # four rows per lane, fewer loads (and conversions) per result: 13%
        # faster on the 16384^2 7x7 Gaussian in f32 and in bf16 storage
        kys = (4, 2, 1)
    return [(v, ky) for ky in kys]


def zmarch1_variants(ctype: str) -> list[tuple[int, int, int, int]]:
    """(V, R, D, NT) variants of the z-marching one-step kernel (3-D, reach
    1): V cells per lane along dim 1 (two for 16-bit types, so a lane's access
    is 32 bits), R output rows per wave, D planes in the register queue, NT
    non-temporal stores (name suffix `nt`, else `c`).  The first is the default (fastest measured on
    512^3); the autotuner may pick another."""
    if ESIZE[ctype] == 2:
        return [(2, 8, 4, 1), (4, 8, 4, 1), (2, 8, 4, 0)]
    if ESIZE[ctype] == 8:
        return [(1, 4, 6, 1), (1, 8, 4, 1), (1, 4, 6, 0)]
    return [(2, 8, 4, 1), (1, 16, 4, 1), (1, 16, 4, 0)]


def gen_static_tu(st, ops, ctype: str, code: str) -> str:
    offs = st.offsets()
    L = len(offs)
    o3 = [tuple(o) + (0,) * (3 - len(o)) for o in offs]
    rx = max(abs(o[0]) for o in o3)
    ry = max(abs(o[1]) for o in o3)
    rz = max(abs(o[2]) for o in o3)
    name = shape_name(st)
    cfg, (tx, ty, tz) = ("CFG_STATIC3D", (32, 8, 8)) if st.N == 3 else ("CFG_STATIC2D", (64, 32, 1))
    table = ", ".join("{%d, %d, %d}" % o for o in o3)
    lines = [
        f"// Generated by stencils.jl_amd/build.py: {type(st).__name__}{{{st.R},{st.N}}} over {ctype}, "
        f"offsets in fold order.",
        '#include "registry.hpp"',
        '#include "tile_kernel.hpp"',
        '#include "stream_kernel.hpp"',
        '#include "zmarch2_kernel.hpp"',
        '#include "zmarch1_kernel.hpp"',
        '#include "ymarch_kernel.hpp"',
        '#include "zmarch_kernel.hpp"',
        "namespace sth {",
        "namespace {",
        f"struct Shape_{name} {{",
        "  static constexpr bool kStatic = true;",
        f"  static constexpr int L = {L}, RX = {rx}, RY = {ry}, RZ = {rz};",
        f"  static constexpr int8_t off[{L}][3] = {{{table}}};",
        "};",
    ]
    i = 0
    for op in ops:
        # streaming variants first: the first registered entry is the default
        if st.N == 3 and max(rx, ry, rz) <= 1:
            # one step per launch, marching along z (every plane loaded once
            # per wave): registered first, the default where it applies
            for v, rows, depth, nt in zmarch1_variants(ctype):
                fn = f"&launch_zmarch1<{ctype}, {op}, Shape_{name}, {v}, {rows}, {depth}, {nt}>"
                lines.append(
                    f"Registrar reg{i}(KernelEntry{{{code}, {op}, CFG_ZMARCH1, {L}, {st.N}, "
                    f"&Shape_{name}::off[0][0], {fn}, \"{name}_{ctype}_{op}/zm1v{v}r{rows}d{depth}"
                    f"{'nt' if nt else 'c'}\", {v}, {rows}}});")
                i += 1
        for v, ky in stream_variants(ctype, st):
            fn = f"&launch_stream<{ctype}, {op}, Shape_{name}, {v}, {ky}>"
            lines.append(
                f"Registrar reg{i}(KernelEntry{{{code}, {op}, CFG_STREAM, {L}, {st.N}, "
                f"&Shape_{name}::off[0][0], {fn}, \"{name}_{ctype}_{op}/stream{v}x{ky}\", {v}, {ky}}});")
            i += 1
        fn = f"&launch_tile<{ctype}, {op}, Shape_{name}, {tx}, {ty}, {tz}>"
        lines.append(
            f"Registrar reg{i}(KernelEntry{{{code}, {op}, {cfg}, {L}, {st.N}, "
            f"&Shape_{name}::off[0][0], {fn}, \"{name}_{ctype}_{op}/lds\"}});")
        i += 1
        if st.N == 3 and max(rx, ry, rz) <= 1:
            if all(sum(map(abs, o)) <= 1 for o in o3) and ESIZE[ctype] <= 4:
                # up to four steps per launch (star stencils, 4-byte values)
                lines.append(
                    f"Registrar reg{i}(Fused2Entry{{{code}, {op}, {L}, {st.N}, "
                    f"&Shape_{name}::off[0][0], &launch_zmarch<{ctype}, {op}, Shape_{name}>, kZmGens, 1, "
                    f"\"zmarch/4\"}});")
                i += 1
            # two steps per launch for iterations (3-D: march along z)
            lines.append(
                f"Registrar reg{i}(Fused2Entry{{{code}, {op}, {L}, {st.N}, "
                f"&Shape_{name}::off[0][0], &launch_zmarch2<{ctype}, {op}, Shape_{name}>, "
                f"zmarch2_rows<Staged<{ctype}>::type>(), 0, \"zmarch2/2\"}});")
            i += 1
        if st.N == 2 and max(rx, ry) <= 1:
            # several steps per launch for iterations (2-D: march along y)
            for gens in (f"ymarch_gens<Elem<{ctype}>::raw>({L})", "kYmShortGens"):
                lines.append(
                    f"Registrar reg{i}(Fused2Entry{{{code}, {op}, {L}, {st.N}, "
                    f"&Shape_{name}::off[0][0], &launch_ymarch<{ctype}, {op}, Shape_{name}, {gens}>, {gens}, 1, "
                    f"ymarch_name({gens})}});")
                i += 1
    lines += ["}  // namespace", "}  // namespace sth", ""]
    return "\n".join(lines)


# Batched launches: every build-time shape with the four folds (and the
# Laplacian where the catalogue has it), in the storage types batches accept.
BATCH_OPS = ["OP_SUM", "OP_MEAN", "OP_MIN", "OP_MAX"]
BATCH_TYPES = [("float", "STH_F32"), ("double", "STH_F64"), ("bf16_t", "STH_BF16")]


def shape_struct(st) -> tuple[str, int, tuple[int, int, int]]:
    offs = st.offsets()
    o3 = [tuple(o) + (0,) * (3 - len(o)) for o in offs]
    r = tuple(max(abs(o[d]) for o in o3) for d in range(3))
    name = shape_name(st)
    table = ", ".join("{%d, %d, %d}" % o for o in o3)
    text = "\n".join([
        f"struct Shape_{name} {{",
        "  static constexpr bool kStatic = true;",
        f"  static constexpr int L = {len(offs)}, RX = {r[0]}, RY = {r[1]}, RZ = {r[2]};",
        f"  static constexpr int8_t off[{len(offs)}][3] = {{{table}}};",
        "};",
    ])
    return text, len(offs), r


# Every (shape, op) of the catalogue gets its own batched kernel: one op's
# streaming body per kernel keeps the code small (instruction cache) and the
# register count that of that body; a batch of one 2-D variant, and 3-D ones,
# launch it.  Batch translation units are grouped per shape.
BATCH_SHAPES = [shape_name(st) for st, _ in CATALOG]


def batch_ops(ops) -> list[str]:
    return BATCH_OPS + (["OP_LAP"] if "OP_LAP" in ops else [])


def gen_batch_tu(ctype: str, code: str, shape: str) -> str:
    lines = [
        f"// Generated by stencils.jl_amd/build.py: batched kernels for {ctype}, shape {shape}.",
        '#include "batch_kernel.hpp"',
        "namespace sth {",
        "namespace {",
    ]
    regs = []
    for idx, (st, ops) in enumerate(CATALOG):
        if shape_name(st) != shape:
            continue
        text, L, r = shape_struct(st)
        lines.append(text)
        sv, sky = stream_variants(ctype, st)[0]
        for k, op in enumerate(batch_ops(ops)):
            v = 100 * (idx + 1) + k  # variant id, unique per (shape, op)
            disp = f"Dispatch_{ctype}_{shape}_{op}"
            lines += [f"struct {disp} {{",
                      "  __device__ static __forceinline__ void run(const BatchJob& j, int bx, int by, int bz, "
                      "int lane, int wave) {",
                      f"    stream_body<{ctype}, {op}, Shape_{shape}, {sv}, {sky}>(j, bx, by, bz, lane, wave);",
                      "  }", "};"]
            regs.append(f"  batch_variants().push_back(BatchVariant{{{code}, {op}, {L}, {st.N}, "
                        f"&Shape_{shape}::off[0][0], {v}, {sv}, {sky}, {v}}});")
            regs.append(f"  batch_kernels().push_back(BatchKernelEntry{{{code}, {v}, "
                        f"&launch_batch<{ctype}, {disp}>, {st.N}}});")
    lines += ["struct Init {", "  Init() {", *regs, "  }", "} init;",
              "}  // namespace", "}  // namespace sth", ""]
    return "\n".join(lines)


def gen_batch_all_tu(ctype: str, code: str) -> str:
    """One kernel that runs any 2-D variant of the catalogue, chosen per job:
    a batch of several variants is one launch."""
    lines = [
        f"// Generated by stencils.jl_amd/build.py: the batched kernel of every 2-D variant for {ctype}.",
        '#include "batch_kernel.hpp"',
        "namespace sth {",
        "namespace {",
    ]
    cases = []
    for idx, (st, ops) in enumerate(CATALOG):
        if st.N != 2:
            continue
        text, _, _ = shape_struct(st)
        lines.append(text)
        sv, sky = stream_variants(ctype, st)[0]
        for k, op in enumerate(batch_ops(ops)):
            cases.append(f"      case {100 * (idx + 1) + k}: stream_body<{ctype}, {op}, Shape_{shape_name(st)}, {sv}, "
                         f"{sky}>(j, bx, by, bz, lane, wave); break;")
    lines += [f"struct Dispatch_{ctype}_all {{",
              "  __device__ static __forceinline__ void run(const BatchJob& j, int bx, int by, int bz, int lane, "
              "int wave) {",
              "    switch (j.variant) {", *cases, "      default: break;", "    }", "  }", "};",
              "struct Init {", "  Init() {",
              f"    batch_kernels().push_back(BatchKernelEntry{{{code}, kBatchAll, "
              f"&launch_batch_all<{ctype}, Dispatch_{ctype}_all>, 2}});",
              "  }", "} init;",
              "}  // namespace", "}  // namespace sth", ""]
    return "\n".join(lines)


# Element types of the multi-array gather (one kernel per tile shape each).
MULTI_TYPES = ["float", "double", "uint8_t", "int32_t", "int64_t"]


def gen_runtime_tu(ctype: str) -> str:
    qual = f"sth::{ctype}" if ctype in ("bf16_t", "f16_t") else ctype
    multi = f" sth::register_multi_type<{qual}>();" if ctype in MULTI_TYPES else ""
    return "\n".join([
        f"// Generated by stencils.jl_amd/build.py: runtime-offset kernels for {ctype}.",
        '#include "runtime_kernels.hpp"',
        '#include "multi_kernel.hpp"',
        "namespace {",
        "struct Init {",
        f"  Init() {{ sth::register_runtime_type<{qual}>(\"rt_{ctype}\");{multi} }}",
        "} init;",
        "}  // namespace",
        "",
    ])


# Headers the runtime compiler (hipRTC) builds stream-kernel specialisations
# from, embedded in the library as text, and the device options it uses: the
# library's own, minus host-only and include flags.
JIT_HEADERS = [("stencils_hip.h", REPO / "include" / "stencils_hip.h"), ("common.hpp", CSRC / "common.hpp"),
               ("tile_kernel.hpp", CSRC / "tile_kernel.hpp"), ("stream_kernel.hpp", CSRC / "stream_kernel.hpp"),
               ("zmarch2_kernel.hpp", CSRC / "zmarch2_kernel.hpp"), ("march_tiles.hpp", CSRC / "march_tiles.hpp"),
               ("ymarch_kernel.hpp", CSRC / "ymarch_kernel.hpp"),
               ("scatter_kernel.hpp", CSRC / "scatter_kernel.hpp"), ("bytes_kernel.hpp", CSRC / "bytes_kernel.hpp")]
JIT_OPTIONS = [f for f in CXXFLAGS if f not in ("-fPIC", "-Wno-unused-command-line-argument") and not f.startswith("-I")]


def gen_jit_tu() -> str:
    def lit(text: str) -> str:
        delim = "sthjit"
        assert f"){delim}\"" not in text
        return f'R"{delim}({text}){delim}"'
    names = ", ".join(f'"{n}"' for n, _ in JIT_HEADERS)
    texts = ",\n    ".join(lit(p.read_text()) for _, p in JIT_HEADERS)
    opts = ", ".join(f'"{o}"' for o in JIT_OPTIONS)
    return (f"// Generated by stencils.jl_amd/build.py: the kernel headers and device options\n"
            f"// the runtime compiler builds stream-kernel specialisations from (jit.hpp).\n"
            f"namespace sth {{\n"
            f"extern const int kJitHeaderCount = {len(JIT_HEADERS)};\n"
            f"extern const char* const kJitHeaderNames[] = {{{names}}};\n"
            f"extern const char* const kJitHeaderTexts[] = {{\n    {texts}}};\n"
            f"extern const int kJitOptionCount = {len(JIT_OPTIONS)};\n"
            f"extern const char* const kJitOptions[] = {{{opts}}};\n"
            f"}}  // namespace sth\n")


def write_if_changed(path: Path, text: str):
    if path.exists() and path.read_text() == text:
        return
    path.write_text(text)


def sources():
    GEN.mkdir(parents=True, exist_ok=True)
    srcs = [CSRC / "api.hip", CSRC / "life_packed.hip"]
    for st, ops in CATALOG:
        for ctype, code in FLOAT_TYPES:
            p = GEN / f"static_{shape_name(st)}_{ctype}.hip"
            write_if_changed(p, gen_static_tu(st, ops, ctype, code))
            srcs.append(p)
    for ctype, _ in FLOAT_TYPES + INT_TYPES:
        p = GEN / f"runtime_{ctype}.hip"
        write_if_changed(p, gen_runtime_tu(ctype))
        srcs.append(p)
    for ctype, code in BATCH_TYPES:
        for shape in BATCH_SHAPES:
            p = GEN / f"batch_{ctype}_{shape}.hip"
            write_if_changed(p, gen_batch_tu(ctype, code, shape))
            srcs.append(p)
        p = GEN / f"batch_{ctype}_all.hip"
        write_if_changed(p, gen_batch_all_tu(ctype, code))
        srcs.insert(0, p)  # the longest to compile
    p = GEN / "jit_sources.hip"
    write_if_changed(p, gen_jit_tu())
    srcs.append(p)
    return srcs


def compile_one(src: Path, incremental: bool) -> Path:
    obj = OBJ / (src.stem + ".o")
    if incremental and obj.exists():
        deps = [src] + list(CSRC.glob("*.hpp")) + [REPO / "include" / "stencils_hip.h"]
        if all(obj.stat().st_mtime >= d.stat().st_mtime for d in deps):
            return obj
    cmd = [HIPCC, *CXXFLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src.name}\n{r.stderr[-6000:]}")
    return obj


def build(jobs: int | None = None, incremental: bool = False, verbose: bool = True) -> Path:
    OBJ.mkdir(parents=True, exist_ok=True)
    LIB.parent.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(16, os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda s: compile_one(s, incremental), srcs))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs), "-lhiprtc"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed\n{r.stderr[-6000:]}")
    shutil.move(str(tmp), str(LIB))
    if verbose:
        print(f"built {LIB} from {len(objs)} translation units")
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("--incremental", action="store_true")
    a = ap.parse_args()
    build(a.jobs, a.incremental)
