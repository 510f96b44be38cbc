"""The launch rule for the parts of blocks against measured stage launches: for
a number of workgroups' blocks (groups), the microseconds of a launch with
whole blocks, halves, quarters, ... down to one plane per part (one MI355X,
the least of three).  The rule's choice is never slower than whole blocks by
more than 2 % (repeated launches differ by about as much) and at most a tenth
behind the best shape; the workgroups that a compute unit holds follow from
the kernel's LDS."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "batsrus_amd", "csrc")
CODE = """
#include "launch_shape.hpp"
extern "C" int split(int g, int nb, int per, int w) {
  return bats::auto_split(g, nb, per, w);
}
extern "C" int per_cu(int nb, int es, int w, int b) {
  return bats::stage_per_cu(nb, es, w, b);
}
"""
# block size, bytes of a real, 8-wave source, body (with B0): groups:times
MEASURED = {
    (8, 8, False, False): """
        1:74,42,26,18 16:76,43,26,19 54:77,44,28,27 64:75,44,28,28
        96:77,45,37,46 136:80,57,59,61 200:81,62,67,82 256:81,64,71,87
        264:100,96,89,98 343:105,106,101,120 396:106,113,119,143
        448:105,115,127,151 520:167,144,146,176 640:179,163,171,209
        900:201,213,237,286 1200:284,280,312,373""",
    (16, 8, False, False): """
        1:132,72,40,24,16 16:135,72,40,26,19 54:140,74,43,34,40
        64:135,73,43,35,43 96:134,74,55,59,69 136:135,89,86,78,85
        200:141,97,100,104,126 256:135,95,105,118,140 264:168,157,133,129,156
        343:172,174,146,162,192 396:176,176,177,194,237
        448:175,181,189,210,250 520:298,245,225,246,299
        640:343,275,257,285,341 900:366,369,390,431,509
        1200:528,470,501,551,659""",
    (8, 8, True, False): """
        1:87,49,29,21 16:91,51,30,21 54:93,53,34,31 64:91,53,35,33
        96:94,56,44,53 136:96,67,73,74 200:101,73,80,97 256:107,77,84,101
        264:121,121,111,124 343:124,133,122,146 396:129,137,152,182
        448:130,138,152,187 520:213,184,184,223 640:237,201,223,275
        900:257,275,304,369 1200:385,363,398,481""",
    (8, 8, True, True): """
        1:112,64,38,26 16:117,66,39,26 54:127,71,44,55 64:125,71,44,56
        96:127,74,83,83 136:130,141,123,134 200:132,143,163,183
        256:133,148,172,217 264:250,209,206,236 343:250,212,244,293
        396:257,281,284,340 448:259,280,291,373 520:384,358,367,446
        640:425,395,445,556 900:577,620,653,791 1200:729,786,844,1052""",
    (16, 8, True, True): """
        1:217,116,64,38,25 16:223,120,66,41,32 54:248,132,81,62,77
        64:244,132,83,64,80 96:243,142,102,106,117 136:244,172,167,152,170
        200:276,186,196,211,242 256:295,208,224,255,324
        264:352,332,284,288,339 343:386,364,338,378,452
        396:397,410,411,433,523 448:406,420,446,472,587
        520:669,574,536,570,680""",
    (8, 4, False, False): """
        1:62,36,22,15 16:63,36,21,15 54:64,36,23,19 64:62,36,23,19
        96:63,37,27,23 136:66,43,32,37 200:66,46,49,59 256:66,46,50,61
        264:77,54,58,68 343:78,56,60,72 396:80,77,70,78 448:80,78,71,86
        520:95,87,86,99 640:98,90,98,119 900:141,129,132,157
        1200:161,160,176,213""",
    (8, 4, True, False): """
        1:43,25,16,13 16:45,27,17,13 54:47,28,19,17 64:47,29,20,18
        96:48,30,24,23 136:49,36,29,34 200:50,37,42,54 256:51,39,44,55
        264:61,45,49,61 343:63,47,52,64 396:64,65,63,75 448:64,66,64,80
        520:74,74,75,91 640:77,76,86,109 900:113,109,118,147
        1200:131,137,156,197""",
    (16, 4, True, False): """
        1:75,41,24,15,10 16:79,43,25,16,12 54:83,45,26,21,24 64:80,44,26,21,26
        96:83,46,32,25,31 136:83,55,38,43,52 200:84,57,57,52,58
        256:82,57,61,71,85 264:100,66,63,63,74 343:104,70,73,81,97
        396:105,100,86,86,106 448:104,99,85,91,112 520:120,111,102,114,136
        640:127,116,124,136,168 900:184,166,161,180,223
        1200:227,224,236,264,322""",
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "r.cpp").write_text(CODE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC,
                    "-o", str(d / "r.so"), str(d / "r.cpp")], check=True)
    return ctypes.CDLL(str(d / "r.so"))


@pytest.mark.parametrize("variant", list(MEASURED))
def test_no_grid_is_slower_than_whole_blocks(rule, variant):
    nb, es, wave8, body = variant
    per = rule.per_cu(nb, es, wave8, body)
    for item in MEASURED[variant].split():
        group, times = item.split(":")
        us = [float(t) for t in times.split(",")]
        s = rule.split(int(group), nb, per, wave8)
        assert us[s] <= 1.02 * us[0], (group, s)
        assert us[s] <= 1.10 * min(us), (group, s)


def test_workgroups_per_compute_unit(rule):
    for nb in (8, 16):
        for wave8 in (0, 1):
            assert rule.per_cu(nb, 8, wave8, 0) == 2
            assert rule.per_cu(nb, 4, wave8, 0) == 3
    assert rule.per_cu(8, 8, 1, 1) == 1
    assert rule.per_cu(16, 8, 1, 1) == rule.per_cu(8, 8, 0, 1) == 2


def test_small_grids_end_in_planes(rule):
    """Few blocks take one plane per part, very many stay whole."""
    for per in (1, 2, 3):
        for wave8 in (0, 1):
            assert rule.split(1, 8, per, wave8) == 3
            assert rule.split(1, 16, per, wave8) == 4
            assert rule.split(1 << 20, 8, per, wave8) == 0
            assert rule.split(1 << 20, 16, per, wave8) == 0
