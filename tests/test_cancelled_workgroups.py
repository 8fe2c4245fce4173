"""Kernels whose threads take indices that other waves have left in LDS.  Each wave looks at a run's abort word by itself, so a cancel that comes while a workgroup starts may be seen by some of its waves only: those leave, and what they
would have written is not there.  Values may then be anything (a cancelled run's results are dropped), but not indices: such a kernel decides for the whole workgroup, or looks only once the indices are there.  Read from the sources; on
the device the moment cannot be met on purpose."""
import glob
import os
import re

import pytest

KERNELS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pipeinfer_amd", "csrc", "kernels")
# the look behind the barrier that follows the last write of an index: nobody who stays lacks one
LOOKS_BEHIND = {"k_linear_attention", "k_channel_recurrence", "k_channel_pieces", "k_channel_walk", "k_attention_tiles"}
# what is in LDS only narrows a range that the arguments bound (k_latent_scores), says whether cells that the arguments bound are looked at again (k_prompt_attention) or is a result (k_topk1)
BOUNDED = {"k_latent_scores", "k_prompt_attention", "k_topk1"}


def kernels_with_indices_in_lds():
    found = {}
    for path in glob.glob(os.path.join(KERNELS, "*.hip")):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for part in text.split("__global__")[1:]:
            name = re.search(r"\b(k_\w+)\s*\(", part).group(1)
            body = part[:part.index("\n}\n") if "\n}\n" in part else len(part)]
            if re.search(r"__shared__[^;(]*\bint(32_t)?\b", body):
                found[name] = body
    return found


def test_a_cancel_leaves_no_workgroup_without_its_indices():
    found = kernels_with_indices_in_lds()
    assert LOOKS_BEHIND | BOUNDED <= set(found) and len(found) > 15
    for name, body in found.items():
        together = "pi_aborted_together(" in body
        assert together != (name in LOOKS_BEHIND | BOUNDED), name
        if together:
            assert not re.search(r"\bpi_aborted\(|\bpi_abort_late\(", body), name


@pytest.mark.parametrize("name,last", [("k_linear_attention", "la_find_piece("), ("k_channel_recurrence", "seg[0] = "), ("k_channel_pieces", "seg[0] = "), ("k_channel_walk", "cr_runs("), ("k_attention_tiles", "range[0] = 0; range[1] = words")])
def test_kernels_that_look_behind_their_indices(name, last):
    body = kernels_with_indices_in_lds()[name]
    written, barrier = body.rindex(last), body.rindex("__syncthreads()", 0, max(body.find("pi_abort_late("), body.find("aborted & 1"))) if name != "k_channel_walk" else body.rindex(last)
    assert written <= barrier < max(body.find("pi_abort_late("), body.find("aborted & 1"))
