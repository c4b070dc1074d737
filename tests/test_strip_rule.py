"""Which lattices take 8 steps per launch in strips (chemsim_amd/csrc/strip_rule.hpp):
the rule's answers for lattices whose two routes were both timed.  Host
arithmetic, compiled here without a GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(os.path.dirname(HERE), "chemsim_amd", "csrc", "strip_rule.hpp")
STORAGE = {"f32": 0, "f64": 1, "bf16": 2, "f16": 3, "f32dev": 4}
# geometry: half-way mode, zero edge, inlet/outlet, reference mask
GEOMETRY = {"periodic": (0, 0, 0, 0), "cavity": (1, 1, 0, 0), "channel": (1, 1, 1, 0), "porous": (1, 0, 0, 0),
            "mask": (0, 0, 0, 1), "mask, zero edge": (0, 1, 0, 1)}
MAIN = """
#include <cstdio>
#include "%s"
int main()
{
    cs::StripCase c;
    int half, zero, io, mask, sr;
    while (std::scanf("%%d %%d %%d %%d %%d %%d %%d %%d", &c.w, &c.h, &c.storage, &half, &zero, &io, &mask, &sr) == 8) {
        c.half = half;
        c.zero_edge = zero;
        c.io = io;
        c.mask = mask;
        c.stochastic = sr;
        std::printf("%%d %%d\\n", (int)cs::ts_takes(c), (int)cs::ts_takes_remainder(c));
    }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    src, exe = str(d / "rule.cpp"), str(d / "rule")
    with open(src, "w") as f:
        f.write(MAIN % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, src], check=True, timeout=120)

    def ask(storage, geometry, w, h, stochastic=False):
        half, zero, io, mask = GEOMETRY[geometry]
        r = subprocess.run([exe], input=f"{w} {h} {STORAGE[storage]} {half} {zero} {io} {mask} {int(stochastic)}",
                           capture_output=True, text=True, timeout=20, check=True)
        return [int(x) for x in r.stdout.split()]
    return ask


# us per 8 steps in regions / in strips
@pytest.mark.parametrize("geometry,w,h", [
    ("channel", 1800, 1700),   # 175 / 235
    ("channel", 1950, 2047),   # 207 / 224
    ("channel", 2048, 2048),   # 220 / 231
    ("channel", 2003, 2300),   # 237 / 240
    ("channel", 517, 9100),    # 258 / 272
    ("channel", 250, 15000),   # 237 / 287
    ("channel", 150, 20000),   # 247 / 287
    ("channel", 60, 60000),    # 362 / 415
    ("channel", 1260, 3561),   # 236 / 247
    ("channel", 3361, 3100),   # 540 / 563, one column in the last strip
    ("channel", 1572, 3361),   # 281 / 354, four
    ("cavity", 1800, 1700),    # 175 / 192, eight
    ("cavity", 1353, 2300),    # 173 / 193, nine
    ("cavity", 1459, 2302),    # 177 / 217, three
    ("cavity", 1793, 2600),    # 255 / 264, one
    ("cavity", 250, 15000),    # 245 / 243, TRT 300 / 316
    ("cavity", 229500, 48),    # 607 / 638
    ("periodic", 229500, 48),  # 366 / 455
    ("periodic", 229500, 144),  # 1085 / 1217
    ("periodic", 1024, 1024),
    ("periodic", 1536, 1536),
])
@pytest.mark.parametrize("storage", ["f32", "f32dev"])
def test_fp32_keeps_regions_where_they_are_faster(rule, storage, geometry, w, h):
    assert rule(storage, geometry, w, h)[0] == 0


@pytest.mark.parametrize("geometry,w,h", [
    ("channel", 3000, 3000),   # 463 / 406
    ("channel", 9100, 517),    # 259 / 227
    ("channel", 101, 30011),   # 287 / 258
    ("channel", 3369, 3100),   # 540 / 455, nine columns in the last strip
    ("cavity", 2360, 3000),    # 365 / 338, eight
    ("cavity", 1721, 1542),    # 153 / 148
    ("cavity", 1700, 2100),    # 198 / 170
    ("cavity", 2001, 1499),
    ("cavity", 2048, 2048),    # 227 / 183
    ("cavity", 517, 9100),     # 262 / 228
    ("cavity", 150, 20000),    # 268 / 243
    ("cavity", 49, 60000),     # 407 / 327
    ("porous", 1800, 1700),    # 242 / 192
    ("mask", 2500, 2000),      # 200 / 200
    ("mask", 3000, 3000),      # 347 / 296
    ("periodic", 2003, 2300),  # 161 / 148
    ("periodic", 57400, 96),   # 197 / 179
    ("periodic", 250000, 24),  # 381 / 268
    ("periodic", 4096, 4096),
])
@pytest.mark.parametrize("storage", ["f32", "f32dev"])
def test_fp32_takes_strips_where_they_are_faster(rule, storage, geometry, w, h):
    assert rule(storage, geometry, w, h)[0] == 1


# us per 8 steps in one-step launches / in strips
@pytest.mark.parametrize("storage,stochastic,geometry,w,h", [
    ("bf16", True, "mask", 2048, 2048),      # 271 / 294 with six obstacles, 272 / 306 with 2% solid
    ("bf16", True, "mask", 2500, 2000),      # 319 / 338, 321 / 346
    ("bf16", True, "mask", 1800, 1700),      # 223 / 245, 224 / 256
    ("bf16", False, "mask", 1500, 1500),     # 173 / 178, 170 / 182
    ("bf16", False, "mask", 250, 15000),     # 265 / 280 with 2% solid
    ("f16", True, "mask", 57400, 144),       # 489 / 569
    ("f16", True, "channel", 2048, 2048),    # 330 / 363
    ("bf16", True, "channel", 2048, 2048),   # 329 / 379
    ("bf16", True, "channel", 3000, 3000),   # 627 / 659
    ("bf16", True, "channel", 2671, 3271),   # 608 / 645
    ("bf16", True, "channel", 3710, 3135),   # 780 / 819
    ("bf16", True, "cavity", 2353, 3000),    # 539 / 577, one column in the last strip
    ("f16", True, "cavity", 2353, 3000),     # 540 / 555
    ("bf16", True, "cavity", 3361, 3100),    # 737 / 779
    ("f16", True, "cavity", 57400, 288),     # 1107 / 1157
    ("bf16", True, "cavity", 400000, 17),    # 540 / 612
    ("f16", True, "cavity", 400000, 17),     # 540 / 570
    ("bf16", False, "cavity", 250000, 32),   # 569 / 723
    ("bf16", False, "periodic", 250000, 32),  # 473 / 528
    ("bf16", True, "periodic", 229500, 96),  # 1271 / 1515
    ("f16", True, "periodic", 57400, 288),   # 907 / 1032
    ("f16", True, "periodic", 60001, 120),   # 434 / 475
    ("f16", True, "periodic", 2048, 2048),
])
def test_16bit_keeps_single_steps_where_they_are_faster(rule, storage, stochastic, geometry, w, h):
    assert rule(storage, geometry, w, h, stochastic)[0] == 0


@pytest.mark.parametrize("storage,stochastic,geometry,w,h", [
    ("bf16", True, "mask", 3000, 3000),      # 536 / 520 with 2% solid
    ("bf16", True, "mask", 9100, 817),       # 464 / 433, 469 / 465
    ("bf16", False, "mask", 2048, 2048),     # 275 / 262 with 2% solid
    ("bf16", False, "mask", 101, 30011),     # 273 / 223
    ("f16", False, "mask", 1800, 1700),      # 214 / 173
    ("f16", True, "mask", 4096, 4096),       # 1001 / 906
    ("f16", True, "channel", 4096, 4096),    # 1131 / 1073
    ("f16", True, "channel", 101, 30011),    # 417 / 367
    ("bf16", True, "channel", 517, 9100),    # 440 / 411
    ("bf16", False, "channel", 2048, 2048),  # 334 / 330
    ("f16", False, "channel", 2048, 2048),   # 320 / 256
    ("f16", True, "cavity", 2048, 2048),     # 347 / 324
    ("bf16", False, "cavity", 57400, 144),   # 582 / 548
    ("f16", True, "porous", 1950, 2047),     # 422 / 336
    ("f16", False, "periodic", 229500, 96),  # 1262 / 975
    ("bf16", True, "periodic", 1800, 1700),  # 220 / 199
    ("f16", True, "periodic", 4096, 4096),   # 892 / 837
    ("f16", True, "periodic", 21280, 800),
    ("bf16", False, "periodic", 70, 90011),  # 624 / 383
])
def test_16bit_takes_strips_where_they_are_faster(rule, storage, stochastic, geometry, w, h):
    assert rule(storage, geometry, w, h, stochastic)[0] == 1


# us per 4 steps in regions / in strips, of lattices that take strips for 8
@pytest.mark.parametrize("geometry,w,h,strips", [
    ("cavity", 49, 60000, 0),       # 148 / 164
    ("cavity", 150, 20000, 0),      # 123 / 118; channel 126 / 140
    ("cavity", 2048, 2048, 1),      # 140 / 101
    ("cavity", 517, 9100, 1),       # 157 / 134
    ("channel", 3000, 3000, 1),     # 308 / 220
    ("periodic", 2893, 1432, 0),    # 91 / 95
    ("periodic", 1100, 4003, 0),    # 91 / 92
    ("periodic", 1794, 3541, 1),    # 130 / 126
    ("periodic", 4096, 4096, 1),    # 337 / 309
    ("periodic", 101, 30011, 1),    # 83 / 79
    ("mask", 1848, 2434, 0),        # 99 / 105
    ("mask", 1780, 2635, 0),        # 102 / 108
    ("mask", 1491, 3577, 0),        # 116 / 122
    ("mask", 3202, 1526, 0),        # 114 / 118
    ("mask", 3000, 3000, 1),        # 202 / 190
])
def test_remainder_takes_the_faster_of_both(rule, geometry, w, h, strips):
    assert rule("f32", geometry, w, h) == [1, strips]


@pytest.mark.parametrize("storage,stochastic,geometry,w,h", [
    *[("f32", False, g, 2003, 2300) for g in ("periodic", "mask", "mask, zero edge", "porous", "cavity")],
    *[("f32", False, g, 101, 30011) for g in ("mask, zero edge", "cavity")],
    *[("f32", False, g, 24641, 163) for g in ("mask, zero edge", "cavity")],
    ("f32", False, "cavity", 2001, 1499), ("f32", False, "channel", 4100, 3001), ("f32", False, "channel", 3001, 1802),
    *[(s, r, g, 3001, 3003) for s in ("bf16", "f16") for r in (False, True) for g in ("periodic", "mask", "cavity")],
    *[(s, r, "channel", 101, 30011) for s in ("bf16", "f16") for r in (False, True)],
    ("f64", False, "cavity", 1100, 1001), ("f64", False, "channel", 2100, 512),
])
def test_lattices_of_the_streaming_tests_take_strips(rule, storage, stochastic, geometry, w, h):
    """The GPU tests compare the streaming kernel only where a lattice takes it."""
    assert rule(storage, geometry, w, h, stochastic)[0] == 1
