"""The launch rules of the distance-driven kernels, evaluated from the library's own header,
against the times that they were drawn from (MLEM iterations, MI355X): for every measured
launch the rule takes the faster side, or one within 4% of it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "iterative_tomographic_reconstruction_algorithms_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def evaluate(tmp_path, expressions):
    """The values of integer C++ expressions over csrc/itomo_internal.h."""
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text("#include \"itomo_internal.h\"\n#include <cstdio>\nusing namespace itomo;\n"
                   "int main()\n{\n%s\n}\n"
                   % "\n".join('    std::printf("%%d\\n", (int)(%s));' % e for e in expressions))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True).stdout
    return [int(v) for v in out.split()]


# npix, slices: us with 64^2, 32^2 and 16^2 tiles
BACK = {(512, 1): (400, 243, 194), (363, 2): (295, 185, 156), (448, 2): (403, 268, 265),
        (363, 3): (328, 216, 218), (384, 3): (348, 228, 230), (480, 2): (435, 290, 297),
        (672, 1): (566, 366, 387), (192, 13): (195, 131, 138), (704, 1): (608, 395, 417),
        (320, 5): (311, 209, 218), (512, 2): (457, 300, 329), (363, 4): (344, 245, 251),
        (724, 4): (1271, 1196, 1398), (512, 11): (1132, 1161, 1374)}

# npix, views, slices: us with views of 4 to 6 candidates along diagonals and staged
FORWARD = {(64, 45, 200): (78, 90), (64, 45, 400): (117, 131), (130, 100, 133): (392, 417),
           (256, 180, 14): (242, 257), (256, 180, 111): (1259, 1347), (363, 251, 53): (1710, 1750),
           (512, 360, 6): (690, 709), (512, 360, 27): (2412, 2494), (640, 450, 2): (521, 517),
           (640, 450, 4): (886, 851), (724, 512, 3): (974, 963), (800, 560, 1): (523, 560),
           (800, 560, 2): (822, 815), (900, 700, 1): (767, 764), (1024, 500, 1): (648, 641),
           (1024, 656, 1): (807, 828), (1024, 720, 1): (890, 897), (1024, 900, 1): (1143, 1088),
           (1100, 500, 1): (720, 744), (1100, 800, 1): (1200, 1092), (1200, 400, 1): (761, 723),
           (1448, 200, 1): (668, 600), (1448, 900, 1): (2246, 2026), (2048, 100, 1): (746, 692),
           (2048, 180, 1): (991, 861), (2048, 328, 1): (1380, 1419)}


def test_back_tile(tmp_path):
    got = evaluate(tmp_path, ["back_variant_for(dd_back_blocks(%d, 64) * %d, dd_back_blocks(%d, 32) * %d)"
                              % (n, z, n, z) for n, z in BACK])
    for (case, us), v in zip(BACK.items(), got):
        assert us[{0: 0, 1: 1, 3: 2}[v]] <= 1.04 * min(us), (case, us, v)


def test_forward_path(tmp_path):
    got = evaluate(tmp_path, ["fwd_path(%d, %d) == kFwdLarge" % (n, (n + 63) // 64 * v * z)
                              for n, v, z in FORWARD])
    for (case, us), staged in zip(FORWARD.items(), got):
        assert us[staged] <= 1.04 * min(us), (case, us, staged)
