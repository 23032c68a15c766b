"""Launch classes of the benchmark by kernel name, as a kernel trace prints them."""
import re

import pytest

from bench import CLASSES, KERNEL_NAMES, TRACE_PATTERNS

NAMES = [
    ("k_phase<float, 3, 0, false, 1, false>", "metropolis"),
    ("k_phase<float, 2, 1, true, 2, true>", "overrelaxation_with_plaquette"),
    ("k_pair<float, 0, 1, false, false, 1>", "metropolis_pair"),
    ("k_pair<float, 1, 2, true, false, 0>", "overrelaxation_pair_with_plaquette"),
    ("k_pair_packed<float, 0, false>", "metropolis_pair"),
    ("k_pair_packed<float, 1, true>", "overrelaxation_pair_with_plaquette"),
    ("k_walk<float, 0, 0, true, false>", "metropolis_pair"),
    ("k_walk<float, 1, 0, false, true>", "overrelaxation_pair"),
    ("k_walk<float, 1, 1, false, false>", "overrelaxation_pair_with_plaquette"),
    ("k_chain<float, 1, 2, false>", "overrelaxation_pass"),
    ("k_walk<double, 1, 0, false, false>", None),
]


@pytest.mark.parametrize("kernel,cls", NAMES)
def test_trace_names(kernel, cls):
    name = f"void u1d::(anonymous namespace)::{kernel}(float*, unsigned int)"
    assert [c for c, p in zip(CLASSES, TRACE_PATTERNS) if re.search(p, name)] == ([cls] if cls else [])


def test_class_labels_name_their_kernels():
    for cls, label in zip(CLASSES, KERNEL_NAMES):
        for kernel in re.findall(r"k_\w+", " ".join(k for k, c in NAMES if c == cls)):
            assert kernel.replace("_packed", "") in label, (cls, kernel)
