"""The runtime compiler's self-test compiles a source of every generator, and
each boundary's multi-step kernel."""
import re

from conftest import REPO

CSRC = REPO / "stencils.jl_amd" / "csrc"


def test_every_generator_is_in_the_self_test():
    generators = set(re.findall(r"inline bool (jit_\w+_source)\(", (CSRC / "jit.hpp").read_text()))
    body = (CSRC / "api.hip").read_text().split("int sth_jit_selftest(", 1)[1].split("STH_GUARD_END", 1)[0]
    assert {"jit_stream_source", "jit_bytes_source", "jit_fused_source", "jit_multi_source"} <= generators
    assert not [g for g in sorted(generators) if g + "(" not in body]
    # kernels are loaded from a generator's source only
    loads = re.findall(r"return jit_load\((\w+), (\w+),", (CSRC / "jit.hpp").read_text())
    assert loads and all(l == ("src", "expr") for l in loads)
    for bc in ("STH_WRAP", "STH_REMOVE", "STH_REFLECT"):
        for dims in (2, 3):
            assert re.search(rf"\{{STH_\w+, STH_OP_\w+, {dims}, {bc}, \d\}}", body), (bc, dims)
