"""The marches (k_march) that the library holds are those its dispatch can pick:
x and y together for one and two fluids, z for up to three, y alone for three on
unequal widths in FP64; FP32 on unequal widths only; built-in equal-width
coefficients in the contracted form only; with the primitive field in the plain
form's x and y march only."""
import re
import subprocess

from microfc_amd import rhs as R


def test_marches_in_the_library():
    names = subprocess.run(["nm", "-C", "--defined-only", R.LIB_PATH], capture_output=True, text=True, check=True).stdout
    got = set(re.findall(r"mfc::(\w+)::k_march<(\d+), (\d+), (\d+), (\w+), (\w+), (\d+), (\w+)>", names))
    want = set()
    for form, real, kinds in (("ieee", "double", "01"), ("f64fast", "double", "012"), ("f32", "float", "0")):
        for kind in kinds:
            for nf in "12":
                for D in "23":
                    want.add((form, nf, D, "1", real, "true", kind, "false"))
                    if form == "ieee":
                        want.add((form, nf, D, "1", real, "true", kind, "true"))
            for nf in "123":
                want.add((form, nf, "3", "2", real, "false", kind, "false"))
        if real == "double":
            want.add((form, "3", "3", "1", real, "false", "0", "false"))
    assert got == want, (sorted(got - want), sorted(want - got))
