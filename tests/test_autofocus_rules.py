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


# pulses: columns of a sub-chunk, LDS bytes of a workgroup, workgroups that fit a CU
SHAPES = {64: (16, 9220, 16), 128: (16, 18436, 8), 192: (16, 28164, 4), 256: (16, 36868, 4), 384: (16, 55428, 1),
          512: (16, 73860, 2), 1024: (8, 77892, 2)}


def test_placing_of_resident_workgroups(rules):
    """Every frame is taken by exactly one launch, whatever its number of bins; a batch whose frames are
    alike runs in no more rounds than with the LDS that its workgroups need; and one with up to 64 bins
    is not packed closer than a third more places than its workgroups call for, where it fits at all."""
    cases = [(m, k) for m in SHAPES for k in (1, 2, 3, 7, 8, 9, 13, 16, 24, 32, 33, 40, 49, 64, 96, 100, 127, 128)]
    exprs = []
    for m, k in cases:
        sub, need, fit = SHAPES[m]
        r = f"af_resident_shapes({k}, {sub}, {need}, {fit})"
        exprs += [f"{r}.n"] + [f"{r}.shape[{i}].{f}" for i in (0, 1) for f in ("lds", "places", "sub_chunks")]
    out = [int(v) for v in rules(*exprs)]
    for i, (m, k) in enumerate(cases):
        sub, need, fit = SHAPES[m]
        n, *rest = out[7 * i:7 * i + 7]
        shapes = [rest[:3], rest[3:]][:n]
        assert shapes[-1][2] == 512 // sub and all(a[2] < b[2] for a, b in zip(shapes, shapes[1:])), (m, k, shapes)
        for lds, places, _ in shapes:
            granules = -(-lds // 1280) * 1280
            assert lds >= need and places == 256 * min(fit, 160 * 1024 // granules), (m, k, lds, places)
        for log2_bins in range(1, 10):
            groups = -(-(1 << log2_bins) // sub)
            lds, places, _ = next(s for s in shapes if groups <= s[2])
            assert -(-k * groups // places) <= -(-k * groups // (256 * fit)), (m, k, groups, shapes)
        if shapes[0][1] < 256 * fit:
            assert shapes[0][1] >= k * (64 // sub) * 4 / 3
            assert shapes[0][1] <= 256 or shapes[0][1] - 256 < k * (64 // sub) * 4 / 3
