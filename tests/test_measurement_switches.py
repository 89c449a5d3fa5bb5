"""Switches that leave parts of the kernels out stand in one header, which refuses them in a product build."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turboquant_plus_amd", "csrc")


def test_conditional_code_is_named_in_one_header():
    header = open(os.path.join(CSRC, "tq_measure.h")).read()
    layout = {"TQ_ROWS_PER_BLOCK", "TQ_KIND_K_VALUE"}      # constants that the host build of the layout header brings along
    for path in glob.glob(os.path.join(CSRC, "*.h*")):
        for line in re.findall(r"^\s*#\s*(?:if|ifdef|ifndef|elif)\b(.*)$", open(path).read(), flags=re.M):
            for name in re.findall(r"\bTQ_\w+", line):
                assert name in header or name in layout or name == os.path.basename(path).upper().replace(".", "_"), (path, name)
