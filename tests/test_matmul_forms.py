"""Which form of the batched kernel a launch takes (no GPU: the host code on
the stand-in runtime, 256 CUs), on both sides of each line of its rule."""
import json

import pytest

import fake_hip
import test_gpu_matmul_units as units
import test_gpu_matmul_wide as wide

SPLIT, SHARED, WIDE, TWO, WIDE_TWO = (4, 1, 4), (4, 1, 1), (8, 1, 1), (4, 2, 1), (8, 2, 1)


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("hip"))


def forms(runtime, cases):
    got = json.loads(fake_hip.run(runtime, "matmul_forms_check.py", stdin=json.dumps(cases)))
    return [(tuple(f), g) for f, g in got]


def test_lines_of_the_rule(runtime):
    lines = [   # tiles, K, B: form
        (1, 128, 1, SPLIT), (383, 512, 64, SPLIT), (384, 512, 64, SHARED),
        (383, 2048, 8, SPLIT), (384, 2048, 8, SHARED), (384, 2176, 8, SPLIT),
        (383, 12288, 33, SPLIT), (384, 12288, 33, SHARED),
        (767, 4096, 32, SPLIT), (768, 4096, 8, SHARED), (768, 6016, 8, SHARED),
        # tiles of 48 groups and more
        (1023, 6144, 8, SPLIT), (1024, 6144, 8, SHARED),
        (768, 6144, 16, SPLIT), (769, 6144, 16, SHARED),
        (512, 6144, 17, SPLIT), (513, 6144, 32, SHARED), (513, 6016, 32, SPLIT),
        # more than a unit of four tiles per CU, more than 8 tiles per CU
        (1024, 12288, 64, SHARED), (1025, 12288, 8, WIDE), (2048, 128, 64, WIDE),
        (2049, 128, 64, TWO), (3686, 128, 8, TWO), (3686, 128, 9, TWO), (3687, 128, 9, WIDE_TWO),
        (3687, 128, 8, TWO),
    ]
    for plan in (False, True):
        got = forms(runtime, [([16 * t], K, B, plan) for t, K, B, _ in lines])
        for (t, K, B, want), (f, grid) in zip(lines, got):
            assert f == (want[0], want[1], (B + 15) // 16, want[2],
                         int(want == SPLIT and B <= 8), int(plan)), (t, K, B)
            units = -(-t // (want[1] * want[0] // want[2]))
            assert grid == min(units, 256 if want[0] == 8 else 512), (t, K, B)
    # units are of one matrix: 1024 tiles of three matrices may be 257
    # units of four; and it is a tile's groups on average that count
    assert forms(runtime, [([16 * 1019, 32, 48], 128, 16, False)])[0] == ((8, 1, 1, 1, 0, 0), 130)
    assert forms(runtime, [([16 * 700, 16 * 100], [1024, 12288], 8, True)])[0][0] == \
        (4, 1, 1, 1, 0, 1)


def test_gpu_cases_cover_every_instance(runtime):
    # the GPU tests' cases take the form they are listed under, and together
    # every instance that a launch can take
    listed = [(form, list(c)) for m in (units, wide) for form, cs in m.CASES.items() for c in cs]
    listed += [(SPLIT, list(c)) for c in units.MIXED]
    got = forms(runtime, [c + [plan] for _, c in listed for plan in (False, True)])
    seen = set()
    for i, (f, grid) in enumerate(got):
        form, (rows, K, B) = listed[i // 2]
        assert (f[0], f[1], f[3]) == form, (rows, K, B)
        if (rows, K, B) in units.MIXED:      # ... and a workgroup has several units
            assert sum(-(-n // 16) for n in rows) > grid
        seen.add(f)
    every = {(4, 1, ct, 4, h, p) for ct in (1, 2, 3, 4) for h in ((0, 1) if ct == 1 else (0,))
             for p in (0, 1)}
    every |= {(nw, tm, ct, 1, 0, p) for nw in (4, 8) for tm in (1, 2) for ct in (1, 2, 3, 4)
              for p in (0, 1)}
    assert seen == every, (every - seen, seen - every)
