"""Kernels that record a stop in the launch whose entry they test decide that entry
once per block.

Block 0 of such a launch may write Ctrl::stop_iter while other blocks are starting.
A wave that tested it for itself could leave while the other waves of its block go
on into block-wide sums.  That is a race, so no run shows it reliably: this reads
the kernels' source.  Every kernel of several waves that records a stop, itself or
through the functions it calls, takes its entry decision from past_stop (one read
and a barrier) or has none."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tealeaf.jl_amd", "csrc",
                   "tl_kernels.hip")
# one block each, whose thread 0 writes the stop behind a barrier that every wave has passed after its test;
# the p update records a stop at its own iteration t, which t > stop_iter lets run
SINGLE = {"k_fin", "k_jacobi_end", "k_init_ctrl", "k_set_mode", "k_cg_p"}


def _bodies():
    """Function name -> body, of every function defined at the start of a line."""
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    out = {}
    for m in re.finditer(r"\b(\w+)\((?:[^(){};]|\([^()]*\))*\)\s*\n\{", text):
        end = text.index("\n}", m.end())
        out[m.group(1)] = (text[max(0, text.rfind("\n\n", 0, m.start())):m.start()], text[m.end():end])
    return out


def test_entry_is_decided_once_per_block():
    bodies = _bodies()
    assert {"k_cgs", "k_cgr", "k_cgg", "k_cgf", "k_steps", "k_cg_ur", "cgp_sweep", "past_stop"} <= set(bodies)
    writers = {n for n, (_, b) in bodies.items() if re.search(r"stop_iter\s*=[^=]", b)}
    assert "record_stop" in writers and "cg_alpha" in writers
    while True:
        more = {n for n, (_, b) in bodies.items() if any(re.search(rf"\b{w}\b\s*(<[^;]*?>)?\(", b) for w in writers)}
        if more <= writers:
            break
        writers |= more
    kernels = {n for n in writers if n.startswith("k_") and n not in SINGLE}
    assert {"k_cgs", "k_cgr", "k_cgg", "k_cgf", "k_steps", "k_cg_ur", "k_cgp", "k_ppcg_ur_sd"} <= kernels
    for n in sorted(kernels | {"cgp_sweep"}):
        assert not re.search(r"t0?\s*>\s*ctrl->stop_iter", bodies[n][1]), n
        if n not in ("k_cgp", "k_cgp_cached"):  # cgp_sweep's body
            assert re.search(r"if \(past_stop\(ctrl, t0?\)\) return;", bodies[n][1]), n
