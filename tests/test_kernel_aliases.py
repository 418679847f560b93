"""No launch passes one array to two pointers that its kernel declares __restrict__.

The qualifier tells the compiler that the two never overlap, so code that works today
may not with another schedule, which no run shows reliably.  This reads the kernels'
signatures and their launches in the sources: pointers that a launch writes as the same
expression must not both be restrict-qualified (two that are only read are allowed to
overlap)."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tealeaf.jl_amd", "csrc")


def _split(text):
    """Top-level comma-separated parts."""
    out, depth, cur = [], 0, ""
    for ch in text:
        depth += ch in "([{"
        depth -= ch in ")]}"
        if ch == "," and depth == 0:
            out.append(cur.strip())
            cur = ""
        else:
            cur += ch
    return out + [cur.strip()]


def _group(text, start):
    """The parenthesised text that opens at `start`."""
    depth = 0
    for i in range(start, len(text)):
        depth += text[i] == "("
        depth -= text[i] == ")"
        if depth == 0:
            return text[start + 1:i]
    raise AssertionError("unbalanced")


def test_no_restrict_pointers_alias():
    text = "\n".join(re.sub(r"//[^\n]*", "", open(f).read()) for f in sorted(glob.glob(os.path.join(CSRC, "*.hip"))))
    kernels = {}
    for m in re.finditer(r"__global__[^;{]*?\b(k_\w+)\s*\(", text):
        kernels[m.group(1)] = _split(_group(text, m.end() - 1))
    assert len(kernels) > 40
    seen = 0
    for m in re.finditer(r"\b(k_\w+)\s*(?:<[^;{}]*?>)?\s*<<<.*?>>>\s*\(", text, re.S):
        params = kernels[m.group(1)]
        args = _split(_group(text, m.end() - 1))
        assert len(params) == len(args) or "TL_CGP_ARGS" in params[0], (m.group(1), params, args)
        if len(params) != len(args):
            continue
        seen += 1
        ptr = [(a, p) for a, p in zip(args, params) if "__restrict__" in p and a not in ("nullptr", "0")]
        for i, (a, p) in enumerate(ptr):
            for b, q in ptr[i + 1:]:
                assert a != b or (p.startswith("const") and q.startswith("const")), (m.group(1), a, p, q)
    assert seen > 60, seen


def test_sum_sets_of_consecutive_register_launches_differ():
    """k_cgr is launched through an argument array: it reads the sums of iteration t0 - 1
    and writes those of t0 - 1 + CGR_BATCH, in sets that alternate with the iteration."""
    text = open(os.path.join(CSRC, "tl_internal.hpp")).read()
    assert int(re.search(r"CGR_BATCH\s*=\s*(\d+)", text).group(1)) % 2 == 1
