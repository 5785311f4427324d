"""Where the kernels read the abort word (CPU, over the sources).

The word may be set while a block's waves read it.  A kernel whose waves form global addresses from
LDS words that other waves wrote takes one reading for the whole block; a kernel that lets each wave
go by its own has to be one whose addresses do not depend on such words."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "momij_amd", "csrc")

# Kernels of several waves with LDS in which a wave that leaves alone takes only values with it:
# every address the others use comes from the block's index, their thread and global memory.
VALUES_ONLY = {
    "k_lm_head", "k_lm_head_q4",          # strips and rows by block and wave; LDS: rows, partials
    "k_rmsnorm_qx", "k_attn_front",       # a row a block; LDS: four partial sums
    "k_route_logits",                     # a row and eight experts a block; LDS: the normed row
    "k_route_topk",                       # a row a wave, with LDS of its own
    "k_gather",                           # tiles by block and wave; LDS: act values
    "k_row_max", "k_row_prep",            # a slice a block; ids clamped to it
    "k_resid_walk", "k_nucleus_pick",     # the walk's block and chunk are wave 0's alone
    "k_nucleus_round",                    # ids and bins by thread; LDS: counts and masses
    "k_attn_combine",                     # appends: two rows a block, by thread, no LDS
}
# The block takes one reading in a form of its own.
OWN_FORM = {"k_attn_chunk": "*s_abort", "k_gather5": None, "k_moe_fused": None,
            "k_head_final_accept": "ab != 0"}


def _functions():
    """(kernel?, name, threads, body) of every function of the HIP sources."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        src = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"(__global__|__device__)[^;{}]*?(\w+)\(([^;{}]*?)\)\s*\{", src):
            depth, i = 1, m.end()
            while depth:
                depth += {"{": 1, "}": -1}.get(src[i], 0)
                i += 1
            bounds = re.search(r"__launch_bounds__\(([^()]*(?:\([^()]*\))?[^()]*)\)", m.group(0))
            name = [n for n in re.findall(r"\b(k_\w+|g5_body|bucket_pairs|walk_write|nuc_scan)\s*\(",
                                          m.group(0))]
            if name:
                yield (m.group(1) == "__global__", name[0], bounds.group(1) if bounds else "",
                       src[m.end():i])


def test_every_kernel_is_classed():
    seen = set()
    for kernel, name, threads, body in _functions():
        if not kernel:
            continue
        seen.add(name)
        waves_share = "__shared__" in body or "extern" in body or re.search(
            r"\b(g5_body|bucket_pairs|walk_write|nuc_scan|rmsnorm_qx_row)\s*(<|\()", body)
        if threads.strip() == "64" or not waves_share or name in OWN_FORM:
            continue
        if re.search(r"(?<!block_)\baborted\(", body):
            assert name in VALUES_ONLY, (
                f"{name}: its waves share LDS and each goes by its own reading of the abort word")
    assert VALUES_ONLY | set(OWN_FORM) <= seen, (VALUES_ONLY | set(OWN_FORM)) - seen


def test_blocks_that_index_with_shared_words_decide_once():
    fns = {n: b for _, n, _, b in _functions()}
    for name in ("k_wide_slots", "k_bucket_inds", "k_topk_bucket", "k_nucleus_sums",
                 "k_sample_decide", "k_kv_commit"):
        body = fns[name]
        assert "block_aborted(" in body, name
        assert not re.search(r"(?<!block_)\baborted\(", body), name
    for name, form in OWN_FORM.items():
        if form:
            assert form in fns[name], name
    # the tile gather: no wave returns by its own reading
    assert not re.search(r"if \((?:[^()]*\|\| )?aborted\([^()]*\)[^;{]*\)\s*(return|break)",
                         fns["g5_body"])
