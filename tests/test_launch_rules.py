"""Where launches change kernel by size (cubek_amd/csrc/cq_launch_rules.hpp), compiled for the host: on each size below the
rule has to name the kernel that was the fastest there, or one within 5 % of it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def answer(tmp_path_factory):
    """Evaluates C++ expressions over the rules, each to a whole number."""
    where = tmp_path_factory.mktemp("rules")

    def evaluate(expressions):
        body = "".join(f'    std::printf("%d\\n", static_cast<int>({e}));\n' for e in expressions)
        (where / "rules.cpp").write_text('#include <cstdio>\n#include "cq_launch_rules.hpp"\nusing namespace cq;\nint main() {\n' + body + "}\n")
        build = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", f"-I{os.path.join(ROOT, 'cubek_amd', 'csrc')}",
                                str(where / "rules.cpp"), "-o", str(where / "rules")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert build.returncode == 0, build.stdout
        run = subprocess.run([str(where / "rules")], stdout=subprocess.PIPE, text=True)
        assert run.returncode == 0
        return [int(line) for line in run.stdout.split()]

    return evaluate


REGISTERS, STEP, WHOLE = 0, 1, 2


def transposed_tile(bits, float_bytes, given, rows, cols, block=32):
    row_tiles = -(-rows // (256 // float_bytes))
    step_cols = 128 if block == 128 and not given else 64
    whole, steps = row_tiles * -(-cols // (1024 // bits)), row_tiles * -(-cols // step_cols)
    return f"transposed_tile({bits}, {float_bytes}, {str(given).lower()}, {rows}, {whole}, {steps}, {step_cols})"


# (bits, bytes of a float, given scales, rows, columns, block): the kernels that are within 5 % of the fastest
TRANSPOSED = {
    (2, 2, False, 14336, 4096, 32): {WHOLE}, (2, 2, False, 31072, 1408, 32): {WHOLE}, (2, 2, False, 14336, 2048, 32): {WHOLE},
    (2, 2, False, 16384, 1024, 32): {WHOLE, REGISTERS}, (2, 2, False, 4096, 4096, 32): {STEP}, (2, 2, False, 2048, 2048, 64): {STEP},
    (4, 2, False, 8192, 2048, 32): {WHOLE}, (4, 2, False, 12288, 2048, 32): {WHOLE}, (4, 2, False, 6144, 4096, 64): {WHOLE},
    (4, 2, False, 14336, 1024, 32): {WHOLE}, (2, 2, False, 14336, 1024, 32): {STEP}, (4, 2, False, 11008, 1024, 64): {STEP},
    (4, 2, False, 1024, 28672, 32): {STEP}, (4, 2, False, 2048, 8192, 32): {WHOLE, STEP}, (4, 2, False, 2048, 4096, 32): {STEP}, (4, 2, False, 1056, 16384, 128): {STEP}, (8, 2, False, 24576, 512, 32): {WHOLE},
    (2, 4, False, 12288, 2048, 32): {WHOLE}, (2, 4, False, 4096, 2048, 32): {STEP},
    (2, 2, True, 14336, 4096, 32): {REGISTERS}, (2, 2, True, 10240, 4096, 64): {REGISTERS}, (2, 2, True, 8192, 2048, 32): {REGISTERS},
    (2, 2, True, 4096, 4096, 32): {STEP}, (2, 2, True, 14336, 1024, 32): {STEP}, (2, 2, True, 512, 1024, 64): {STEP}, (4, 2, True, 12288, 2048, 32): {REGISTERS, WHOLE},
    (4, 2, True, 8192, 2048, 32): {REGISTERS}, (4, 2, True, 2048, 4096, 32): {STEP}, (8, 2, True, 6144, 2048, 32): {WHOLE},
    (4, 4, True, 12288, 1024, 32): {WHOLE}, (2, 4, True, 8192, 3072, 32): {WHOLE}, (2, 4, True, 8192, 1536, 32): {REGISTERS},
    (4, 2, False, 28672, 8192, 32): {WHOLE}, (8, 2, True, 28672, 8192, 64): {WHOLE},
}


def test_transposed_quantize_takes_the_fastest_of_its_kernels(answer):
    got = answer([transposed_tile(*case) for case in TRANSPOSED])
    wrong = {case: g for (case, good), g in zip(TRANSPOSED.items(), got) if g not in good}
    assert not wrong


# (rows, columns of a 16-bit type, bits, block): whether the codes of whole tiles should stay in the caches
STAY = {
    (4096, 4096, 4, 32): False, (4096, 5120, 4, 32): True, (4096, 4096, 8, 32): False,
    (1056, 16384, 8, 32): True, (65536, 256, 8, 128): False, (4096, 5120, 8, 32): True, (8192, 4096, 4, 32): True,
    (14336, 4096, 4, 32): True, (16384, 8192, 4, 64): True, (11264, 4096, 8, 32): True, (14336, 4160, 4, 32): True,
    (16384, 8192, 8, 32): True, (28672, 8192, 4, 32): True, (28672, 8192, 8, 64): True, (28672, 8192, 8, 128): True,
    (24576, 8192, 8, 32): False, (28672, 8192, 8, 32): False, (8192, 28672, 8, 32): False, (28672, 12288, 4, 32): False,
    (28672, 16384, 2, 32): False, (28672, 16384, 4, 32): False, (28672, 16384, 8, 64): False,
}


def test_transposed_codes_stay_in_the_caches_where_they_fit(answer):
    got = answer([f"transposed_codes_stay({rows * cols * 2}ull, {rows * cols * bits // 8}ull, {rows * cols // block * 4}ull, {block})" for rows, cols, bits, block in STAY])
    assert got == [int(stay) for stay in STAY.values()], dict(zip(STAY, got))


# (bytes of the output, rows on whole lines): whether a re-pack's output should leave through plain stores
REPACK = {
    (8 << 20, True): False, (28 << 20, True): False, (64 << 20, True): True, (80 << 20, True): True, (112 << 20, True): False,
    (224 << 20, True): False, (15 << 20, False): True, (112 << 20, False): True,
}


def test_repacked_words_stay_in_the_caches_where_lines_are_shared_or_both_launches_fit(answer):
    got = answer([f"repack_stays({n}ull, {str(lines).lower()})" for n, lines in REPACK])
    assert got == [int(stay) for stay in REPACK.values()], dict(zip(REPACK, got))


ONE, PLAN, OUTPUTS = "kOneLaunch", "kPlan", "kPerOutput"


def reduce_way(outer, length, inner, elem_bytes, ragged, tiles, wanted, room, long_axis=True):
    """`tiles`: of the plan (0: a lane per chunk of columns); slices that the plan wants and that the workspace has room for;
    `long_axis`: whether it would want any, were their partials no bytes."""
    return (f"[] {{ ReduceColumns c{{}}; c.outer = {outer}, c.len = {length}, c.inner = {inner}, c.per_chunk = {16 // elem_bytes}, c.ragged = {str(ragged).lower()}, "
            f"c.tiles = {tiles}, c.wanted = {wanted}, c.slices = {room}, c.long_axis = {str(long_axis).lower()}; return reduce_way(c); }}()")


# the arguments of reduce_way(): the way that was the faster one, or within 5 % of it
REDUCE = {
    # no workspace, or too little
    (1, 43625, 2348, 2, True, 0, 681, 1): ONE, (1, 20000, 4097, 2, True, 0, 312, 1): ONE, (1, 2000, 301, 2, True, 1, 31, 1): ONE,
    (16, 3000, 77, 2, True, 16, 46, 1): ONE, (1, 4096, 4096, 2, False, 0, 64, 1): ONE, (1, 5000, 801, 2, True, 2, 78, 30): ONE,
    (1, 5000, 801, 2, True, 2, 78, 40): PLAN, (2, 155, 128, 2, False, 2, 2, 1): PLAN,
    # a workspace
    (1, 1041, 9088, 2, False, 0, 16, 16): ONE, (1, 250, 32000, 4, False, 0, 7, 7): ONE, (1, 20000, 4097, 2, True, 0, 312, 312): PLAN,
    (1, 2443, 4469, 2, True, 0, 38, 38): PLAN, (1, 5, 25600, 2, False, 0, 1, 1, False): PLAN,
    # axes too short for slices
    (1, 15, 832, 2, False, 2, 1, 1, False): PLAN, (1, 20, 1640, 2, False, 4, 1, 1, False): PLAN, (1, 8, 24256, 2, False, 0, 1, 1, False): PLAN,
    (3, 89, 64, 2, False, 3, 1, 1, False): PLAN, (212, 14, 799, 2, True, 424, 1, 1, False): PLAN, (5, 12, 10885, 4, True, 0, 1, 1, False): PLAN,
    (1, 15, 11951, 4, True, 0, 1, 1, False): ONE, (3905, 8, 431, 2, True, 3905, 1, 1, False): PLAN, (4485, 225, 11, 2, True, 4485, 1, 1, False): PLAN,
    (34978, 9, 23, 2, True, 34978, 1, 1, False): OUTPUTS, (13557, 2, 125, 2, True, 13557, 1, 1, False): OUTPUTS,
    (10812, 76, 11, 2, True, 10812, 1, 1, False): OUTPUTS, (1248, 17, 89, 2, True, 1248, 1, 1, False): OUTPUTS, (8141, 1, 29, 2, True, 8141, 1, 1, False): OUTPUTS,
    (7362, 85, 9, 4, True, 7362, 1, 1, False): PLAN, (6, 13, 2901, 2, True, 0, 1, 1, False): ONE, (155, 2, 949, 2, True, 310, 1, 1, False): OUTPUTS, (620, 12, 11, 2, True, 620, 1, 1, False): OUTPUTS, (200000, 3, 5, 4, True, 0, 1, 1, False): OUTPUTS,
    (3038, 1, 365, 4, True, 0, 1, 1, False): PLAN, (166490, 1, 11, 4, True, 0, 1, 1, False): PLAN,
    # rows of whole lines: the longest axes of one launch by the number of its tiles, 104, 128, 160, 172, 224, 256, 274, then of 16 columns
    (1, 1600, 6656, 2, False, 0, 20, 20): ONE, (1, 3000, 6656, 2, False, 0, 40, 40): PLAN, (1, 4096, 6656, 2, False, 0, 64, 64): PLAN,
    (1, 2048, 3328, 4, False, 0, 64, 64): PLAN, (1, 2048, 8192, 2, False, 0, 32, 32): ONE, (1, 3726, 8192, 2, False, 0, 58, 58): PLAN,
    (1, 2048, 4096, 4, False, 0, 64, 64): ONE, (1, 3726, 4096, 4, False, 0, 116, 116): PLAN, (1, 2048, 10240, 2, False, 0, 32, 32): ONE,
    (1, 3000, 10240, 2, False, 0, 46, 46): PLAN, (1, 4093, 11008, 2, False, 0, 63, 63): ONE, (1, 4093, 5504, 4, False, 0, 127, 127): ONE,
    (1, 4093, 14336, 2, False, 0, 63, 63): ONE, (1, 4093, 16384, 2, False, 0, 63, 63): ONE, (1, 1281, 17536, 2, False, 0, 20, 20): ONE,
    (1, 2048, 17536, 2, False, 0, 32, 32): PLAN, (1, 2048, 32768, 2, False, 0, 32, 32): ONE, (1, 500, 34816, 2, False, 0, 7, 7): ONE,
    (1, 1281, 34816, 2, False, 0, 20, 20): PLAN, (1, 900, 49152, 2, False, 0, 14, 14): ONE, (1, 900, 65536, 2, False, 0, 14, 14): ONE,
    # ragged rows, few columns
    (1, 1283, 115, 4, True, 1, 11, 11): ONE, (1, 1748, 5, 4, True, 1, 2, 2): ONE, (1, 2213, 61, 4, True, 1, 9, 9): ONE, (1, 1557, 1751, 2, True, 4, 24, 24): ONE,
    (1, 2160, 73, 2, True, 1, 17, 17): PLAN, (1, 2442, 501, 4, True, 2, 76, 76): PLAN, (1, 1900, 4469, 2, True, 0, 29, 29): PLAN, (1, 1800, 1752, 2, False, 4, 28, 28): PLAN,
    # few outputs
    (1, 631, 47, 2, True, 1, 9, 9): OUTPUTS, (1, 325, 11, 2, True, 1, 1, 1, False): OUTPUTS, (1, 901, 423, 2, True, 1, 14, 14): ONE, (1, 452, 47, 4, True, 1, 7, 7): ONE,
}


def test_reductions_along_an_outer_axis_take_the_faster_way(answer):
    got = answer([f"{reduce_way(*case)} == ReduceWay::{way}" for case, way in REDUCE.items()])
    wrong = [case for case, right in zip(REDUCE, got) if not right]
    assert not wrong


# (outer, length, inner, bytes of an element, ragged): whether loading ahead was the faster way in one launch, or within 3 % of it
LOADS_AHEAD = {
    (1, 1041, 9088, 2, False): True, (1, 600, 8448, 2, False): True, (1, 752, 19680, 2, False): True, (1, 457, 21968, 2, False): True, (1, 250, 19368, 2, False): True,
    (1, 1005, 3968, 4, False): True, (2, 405, 5760, 2, False): True, (5, 446, 7552, 4, False): True, (1, 602, 32768, 2, False): True,
    (1, 602, 32896, 2, False): False, (2, 655, 17728, 2, False): False,
    (1, 558, 9249, 2, True): False, (5, 738, 3761, 2, True): False, (1, 509, 10464, 2, False): False, (1, 1116, 2307, 2, True): False, (1, 1134, 115, 4, True): False,
    (1, 1154, 512, 2, False): False, (1, 1134, 16384, 2, False): False, (1, 1082, 11776, 2, False): False, (5, 138, 25216, 2, False): False, (1, 250, 9728, 2, False): False,
    (1, 4093, 11008, 2, False): False, (1, 3726, 16384, 2, False): False,
}


def test_the_one_launch_of_a_reduction_loads_ahead_where_that_is_faster(answer):
    got = answer([f"[] {{ ReduceColumns c{{}}; c.outer = {outer}, c.len = {length}, c.inner = {inner}, c.per_chunk = {16 // size}, c.ragged = {str(ragged).lower()}; "
                  f"return reduce_loads_ahead(c, reduce_tile(c)); }}()" for outer, length, inner, size, ragged in LOADS_AHEAD])
    assert got == [int(ahead) for ahead in LOADS_AHEAD.values()], dict(zip(LOADS_AHEAD, got))


MIB = 1 << 16  # chunks
# (chunks, bits, bytes of a float, captured): whether one read of the tensor is the faster way
ONE_READ = {
    (4, 8, 2, False): True, (16 * MIB, 8, 2, False): True, (16 * MIB + 4, 8, 2, False): False, (48 * MIB - 4, 8, 2, False): False,
    (48 * MIB, 8, 2, False): True, (384 * MIB, 8, 2, False): True, (400 * MIB, 8, 2, False): False, (4096 * MIB, 8, 2, False): False,
    (48 * MIB, 4, 2, False): False, (56 * MIB - 4, 4, 2, False): False, (56 * MIB, 4, 2, False): True, (640 * MIB, 4, 2, False): True, (1024 * MIB, 4, 2, False): False,
    (16 * MIB, 2, 2, False): True, (56 * MIB, 2, 2, False): False, (80 * MIB, 2, 2, False): False, (128 * MIB, 2, 2, False): True, (56 * MIB, 2, 4, False): True,
    (48 * MIB, 8, 4, False): True, (640 * MIB, 8, 4, False): True, (2048 * MIB, 8, 4, False): False,
    (4, 8, 2, True): False, (16 * MIB, 8, 2, True): False, (64 * MIB, 8, 2, True): False, (72 * MIB, 8, 2, True): True, (60 * MIB - 4, 8, 4, True): False,
    (60 * MIB, 8, 4, True): True, (440 * MIB, 8, 2, True): True, (512 * MIB, 8, 2, True): False, (100 * MIB, 4, 2, True): False, (120 * MIB, 4, 2, True): True,
    (200 * MIB, 2, 2, True): False, (96 * MIB - 4, 4, 4, True): False, (96 * MIB, 4, 4, True): True, (96 * MIB, 2, 4, True): True, (2048 * MIB, 2, 4, True): False,
}


def test_one_scale_is_read_once_where_that_is_faster(answer):
    got = answer([f"quantize_stays_resident({chunks}ull, {bits}, {size}, {str(captured).lower()})" for chunks, bits, size, captured in ONE_READ])
    assert got == [int(once) for once in ONE_READ.values()], dict(zip(ONE_READ, got))


# (row groups, columns, vectors, values in 16 bytes of codes, e4m3 or e5m2): the shape that was the fastest, or within 5 % of it
GEMV = {
    # up to four stages of 8 x 16 bytes of codes are one round of four waves
    (148, 320, 5, 32, False): "k1x4", (160, 512, 5, 32, False): "k1x4", (175, 576, 7, 32, False): "k1x4", (226, 512, 12, 16, False): "k1x4",
    (171, 384, 16, 16, True): "k1x4", (252, 960, 7, 32, False): "k1x4", (64, 512, 3, 32, False): "k1x8",
    # five to eight are two rounds of four waves and one of eight
    (115, 1440, 5, 32, False): "k1x8", (163, 1728, 5, 32, False): "k1x8", (83, 800, 12, 16, False): "k1x8", (46, 1952, 7, 32, False): "k1x8",
    (117, 2912, 8, 32, False): "k1x4", (145, 3840, 6, 32, False): "k1x8", (112, 9088, 16, 16, True): "k1x8", (193, 12288, 12, 32, False): "k1x8",
    (896, 4096, 8, 32, False): "k2x4", (1792, 8192, 16, 32, False): "k4x2", (589, 8192, 3, 32, False): "k1x4", (990, 8192, 16, 32, False): "k4x2",
}


def test_products_with_several_vectors_take_the_fastest_shape(answer):
    def shape(groups, cols, vectors, per_unit, is_bytes):
        x = (vectors * 2 * 8 * per_unit + 1023) // 1024 * 1024
        return f"gemv_batch_shape({groups}, {x}, {16 * (x + 2560)}, {cols // per_unit}, {str(is_bytes).lower()})"

    got = answer([f"{shape(*case)} == GemvShape::{want}" for case, want in GEMV.items()])
    wrong = [case for case, right in zip(GEMV, got) if not right]
    assert not wrong


def test_products_with_several_vectors_stream_their_codes_where_that_is_faster(answer):
    # (whole lines, rows, bytes of a row, vectors): streaming was the faster way, or within 3 % of it
    cases = {(True, 28672, 4096, 16): True, (False, 3507, 10944, 16): True, (False, 3449, 16736, 16): True, (False, 3855, 14496, 14): True,
             (False, 2788, 2128, 5): False, (False, 3590, 7376, 16): False, (False, 20000, 6752, 8): False, (False, 2744, 12096, 16): False, (False, 3873, 14496, 5): False}
    got = answer([f"gemv_batch_streams({str(lines).lower()}, {-(-rows // 16)}, {row_bytes}, {vectors})" for lines, rows, row_bytes, vectors in cases])
    assert got == [int(streams) for streams in cases.values()], dict(zip(cases, got))


# (rows, columns, vectors, values in 16 bytes of codes, 4-bit fields, x in f16, e4m3 or e5m2): waves of the kernel of four rows a wave, 0 where
# another is faster, or within 5 % of it
QUADS = {
    (28672, 8192, 1, 32, True, False, False): 0, (4524, 16512, 1, 32, True, False, False): 16, (1024, 28672, 1, 32, True, False, False): 16,
    (6867, 3584, 1, 32, True, False, False): 0, (3011, 1408, 1, 32, True, False, False): 0, (25471, 2240, 1, 32, True, False, False): 16,
    (7455, 2240, 1, 32, True, True, False): 8, (18484, 6912, 1, 32, True, True, False): 16, (5888, 1664, 1, 16, False, False, True): 0,
    (9472, 18176, 1, 16, False, False, True): 16, (1163, 23392, 2, 16, False, False, False): 16, (1486, 4288, 2, 32, True, False, False): 8,
    (3454, 1920, 2, 32, True, False, False): 0, (16384, 5120, 4, 16, False, False, False): 0, (14336, 4096, 4, 16, False, False, True): 16,
    (14336, 4096, 2, 32, True, False, False): 0, (23373, 10080, 4, 32, True, False, False): 16, (1024, 28672, 4, 32, True, False, False): 0,
    (14336, 4096, 5, 32, True, True, False): 0, (9559, 1952, 3, 16, False, True, False): 0, (19328, 1280, 4, 16, False, False, True): 16,
    # several vectors, and waves without rows: two groups of four rows in three or four steps, five groups of short rows
    (1693, 1920, 2, 32, True, False, False): 0, (1362, 1920, 4, 32, True, True, False): 0, (1439, 1664, 4, 32, False, True, False): 0, (1085, 2080, 2, 32, True, False, False): 8,
    (1024, 2048, 4, 32, True, False, False): 8, (5120, 1024, 2, 16, False, False, False): 0, (5120, 1024, 4, 16, False, True, True): 0, (4608, 3456, 3, 16, False, False, True): 0,
    (5120, 3072, 4, 16, False, False, False): 16, (4736, 5504, 3, 16, False, False, True): 16,
    # ... rows of whole lines: short ones, long ones in three groups, groups that fill rounds of sixteen waves badly
    (5120, 2048, 3, 32, True, False, False): 0, (5120, 2080, 3, 32, True, False, False): 8, (2048, 4096, 4, 32, False, True, False): 0, (19754, 1024, 3, 32, True, False, False): 0,
    (2863, 14080, 4, 32, True, False, False): 0, (2863, 14112, 4, 32, True, False, False): 16, (9435, 5120, 3, 32, True, False, False): 0, (14336, 8192, 2, 32, True, False, False): 0,
    (14336, 8192, 2, 32, True, True, False): 16, (28672, 5120, 3, 32, True, False, False): 16, (2048, 4096, 2, 32, True, False, False): 8, (28672, 8192, 4, 32, True, False, False): 16,
    (11008, 11008, 2, 32, True, False, False): 16,
    # ... of bytes: near memory's rate
    (2048, 1024, 4, 16, False, True, True): 0, (28672, 2048, 3, 16, False, True, True): 0, (28672, 4096, 3, 16, False, True, True): 16, (14336, 14336, 4, 16, False, False, True): 0,
    (28672, 11008, 2, 16, False, False, True): 16, (25344, 1664, 4, 16, False, False, True): 0, (6784, 7040, 3, 16, False, False, True): 0,
    (9728, 23936, 2, 16, False, False, True): 16, (9216, 16128, 1, 16, False, False, True): 16, (11008, 14336, 1, 16, False, True, True): 16, (19712, 14336, 1, 16, False, False, True): 0,
    (9856, 1664, 1, 16, False, False, True): 0, (6144, 6144, 1, 16, False, False, True): 0, (11008, 4096, 1, 16, False, True, True): 16,
    # one vector: eight waves with five groups
    (4708, 1152, 1, 16, False, False, False): 0, (4959, 3072, 1, 32, True, False, False): 0, (1024, 2048, 1, 32, True, True, False): 0, (1024, 4096, 1, 32, True, True, False): 8,
    # one vector of 4 bits of f16 in the smallest launches
    (1514, 1280, 1, 32, True, True, False): 0, (1814, 1792, 1, 32, True, True, False): 0, (2347, 1408, 1, 32, True, True, False): 8, (3425, 1344, 1, 32, True, True, False): 8,
    # ... of bytes: few groups of four rows, shares 2^18 bytes apart, large weights
    (4096, 4096, 1, 16, False, False, True): 0, (4736, 4352, 1, 16, False, True, True): 0, (2048, 14336, 1, 16, False, False, True): 16, (8576, 3328, 1, 16, False, False, True): 16,
    (8192, 8192, 1, 16, False, False, True): 0, (16384, 4096, 1, 16, False, True, True): 0, (8192, 11008, 1, 16, False, False, True): 16, (24576, 8192, 1, 16, False, False, True): 0,
    (14336, 11008, 1, 16, False, True, True): 0, (28672, 10624, 1, 16, False, False, True): 0, (5120, 28672, 1, 16, False, False, True): 16, (6144, 24576, 1, 16, False, True, True): 16,
    # ... of 8 bits and e2m1 bytes in short launches
    (2774, 2432, 1, 16, False, False, False): 0, (2583, 3360, 1, 16, False, False, False): 0, (4120, 4320, 1, 32, False, False, False): 0, (1024, 8192, 1, 16, False, True, False): 8,
    (2614, 5440, 1, 16, False, False, False): 16,
}


def quads_split(rows, cols, vectors, per_unit, *flags):
    return f"quads_split({rows}u, {cols // per_unit}u, {per_unit}, {vectors}, {', '.join(str(flag).lower() for flag in flags)})"


def test_products_take_four_rows_a_wave_where_that_is_faster(answer):
    got = answer([f"{quads_split(*case)}.waves" for case in QUADS])
    assert got == list(QUADS.values()), dict(zip(QUADS, got))


def gemv_route(case, vectors, native):
    """The kernel of a product that the other tests list: x in 16 bits, fields of 4 or 8 bits, whole units and blocks of a power of two of them."""
    value, rows, cols = case[1].name, case[4], case[5]
    per_unit = 16 if value in ("Q8S", "Q8F", "E4M3", "E5M2") else 32
    return f"{quads_split(rows, cols, vectors, per_unit, per_unit == 32 and not native, case[0].name == 'F16', native and value in ('E4M3', 'E5M2'))}.grid != 0"


def test_listed_products_reach_the_kernels_they_are_listed_for(answer):
    from test_gpu_gemv import CASES, NATIVE_CASES, NOT_QUADS, QUADS_CASES, STREAM_CASES

    got = answer([gemv_route(case, case[7], case[8]) for case in QUADS_CASES])
    assert [(case[4], case[5], case[7]) for case, quads in zip(QUADS_CASES, got) if not quads] == NOT_QUADS
    contiguous = [case for case in STREAM_CASES if case[6] is None]
    assert answer([gemv_route(case, 1, case[8]) for case in contiguous]) == [0] * len(contiguous)
    # the products with odd scales: every kind of codes, one vector and three
    odd = [quads_split(70, 16416, vectors, per_unit, *flags) for vectors in (1, 3) for f16 in (False, True)
           for per_unit, *flags in ((32, True, f16, False), (16, False, f16, False), (16, False, f16, True), (32, False, f16, False))]
    assert answer([f"{q}.grid != 0" for q in odd]) == [1] * len(odd)
    # among the others both kernels occur, with either type of x
    for listed, native in ((CASES, False), (NATIVE_CASES, True)):
        listed = [case for case in listed if case[0].name != "F32" and not case[1].name.startswith("Q2") and case[5] % 32 == 0 and (case[2] is None or case[2][-1] % 16 == 0)]
        routes = {(case[0].name, quads) for case, quads in zip(listed, answer([gemv_route(case, 1, native) for case in listed]))}
        assert routes >= {("F16", 0), ("BF16", 0)} and (native or routes >= {("F16", 1), ("BF16", 1)})


def test_four_rows_a_wave_fit_what_the_kernel_keeps(answer):
    """Quads per workgroup in 8 bits, what is left over in 24, x and the sums in the shared memory of a compute unit, workgroups no more than quads."""
    cases = [(rows, cols, vectors, 32, True, True, False) for rows in (1, 4, 5, 1023, 65536, 65541, 1 << 22, (1 << 31) - 1)
             for cols in (32, 544, 19424, 38880) for vectors in (1, 2, 3, 4)]
    got = answer([f"[] {{ const QuadsSplit q = {quads_split(*case)}; const uint32_t quads = ({case[0]}u + 3) / 4; return q.grid == 0 ? 2 : q.grid <= quads && "
                  f"(quads + q.grid - 1) / q.grid <= 64 && quads % q.grid < (1u << 24) && (1u << q.shares_log2) <= q.waves && q.lds <= 160 * 1024; }}()" for case in cases])
    assert 0 not in got and got.count(1) > 40, dict(zip(cases, got))


# (bytes of a float, rows and columns of a block, rows and columns): chunks per lane of the tile kernel, 0 where another is faster or it cannot
BLOCK_TILES = {
    (2, 128, 128, 14336, 4096): 8, (2, 64, 64, 14336, 4096): 4, (2, 32, 32, 2048, 4096): 2, (2, 32, 32, 128, 512): 2, (4, 64, 64, 14336, 4096): 4,
    (2, 64, 64, 65536, 512): 4, (2, 32, 32, 65536, 288): 2, (2, 24, 32, 2400, 4096): 0, (2, 32, 48, 2048, 4800): 0, (2, 32, 32, 128, 96): 0,
    # blocks of a few rows: one chunk, wider tiles from 10 MiB on, the general kernel where there is no room for those
    (2, 8, 128, 744, 1792): 1, (2, 16, 64, 1104, 1408): 1, (2, 8, 128, 5840, 10112): 2, (2, 16, 64, 8512, 1472): 4, (4, 16, 16, 310176, 80): 0,
    (2, 8, 32, 8880, 4800): 2, (4, 8, 64, 17392, 1728): 2, (2, 8, 32, 103208, 320): 0, (2, 4, 128, 5840, 1024): 1, (2, 4, 128, 44832, 768): 0,
    (4, 4, 128, 30360, 256): 1, (4, 4, 128, 26088, 4096): 0,
}


def test_blocks_over_two_dimensions_take_the_faster_kernel(answer):
    got = answer([f"block_tiles_of({str(size == 4).lower()}, {br}, {bc * size // 16}, {rows}, {cols * size // 16}).per_lane" for size, br, bc, rows, cols in BLOCK_TILES])
    assert got == list(BLOCK_TILES.values()), dict(zip(BLOCK_TILES, got))


def test_lanes_of_one_chunk_where_they_are_faster(answer):
    """(chunks, lanes per block if no power of two)"""
    cases = {(512000, 0): True, (640000, 0): True, (776192, 0): True, (819200, 0): False, (314880, 3): True, (393216, 3): True, (479232, 6): False,
             (565248, 12): False, (639744, 3): False}
    got = answer([f"{chunks} < small_lane_chunks({group})" for chunks, group in cases])
    assert got == [int(one) for one in cases.values()], dict(zip(cases, got))
    scales = {409600: True, 502000: True, 598016: False, 778240: False}
    assert answer([f"{chunks} < kSmallLaneScaleChunks" for chunks in scales]) == [int(one) for one in scales.values()]
