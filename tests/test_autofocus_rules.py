"""What the host decides about the resident autofocus from sizes alone (csrc/autofocus_rules.hpp), compiled
and run on the CPU."""
from __future__ import annotations

import subprocess

import pytest

from isar_imaging_cuda_amd import build as B


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """rules(expression): the value of a C++ expression of the header's functions, as printed."""
    d = tmp_path_factory.mktemp("rules")

    def value(*expressions: str) -> list[str]:
        src, exe = d / "main.cpp", d / "main"
        body = "".join(f"std::cout << ({e}) << '\\n';" for e in expressions)
        src.write_text('#include <iostream>\n#include "autofocus_rules.hpp"\nusing namespace isar;\n'
                       f"int main() {{ {body} }}\n")
        B._run([B.GXX, "-std=c++20", "-O1", "-Wall", "-I", str(B.CSRC), str(src), "-o", str(exe)])
        return subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()

    return value


def test_wait_bound_of_the_default_form_goes_with_the_iterations(rules):
    """A wait in the default form may last as long as the frames ahead run, which is proportional to the
    iterations (at most 22 us each, a poll takes 0.25), and should give up after few times that."""
    its = [0, 1, 120, 140, 9000, 1 << 20, (1 << 31) - 1]
    polls = [int(v) for v in rules(*(f"af_guarded_polls({i})" for i in its))]
    for i, p in zip(its, polls):
        assert p > 0
        assert p >= min(4 * 2 * 22 * i, (1 << 31) - 1), (i, p)
        assert p <= 4 * 4 * 22 * i + 32768, (i, p)
