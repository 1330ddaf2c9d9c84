"""Host-side check of the sources: partial results reach the work-group that arrives last through one helper, which holds both forms of the hand-over and refuses other targets."""
import glob
import os

from helpers.device import ROOT


def test_arrivals_are_counted_in_one_place():
    found = {}
    for path in glob.glob(os.path.join(ROOT, "neural-api_amd", "csrc", "*.h*p")):
        with open(path) as f:
            for line in f:
                if "atomic_inc32(" in line:
                    found.setdefault(os.path.basename(path), []).append(line.strip())
    # the two forms of arrives_last, and the flag of host_signal, behind which no work-group reads
    assert {k: len(v) for k, v in found.items()} == {"cai_internal.hpp": 3}, found
