"""The FP64 pair energies of energy steps (blade_amd/csrc/energy64.h),
compiled for the CPU and compared with long double: no larger an error than
with IEEE square root and division and a library's erfc."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_errors_against_long_double(tmp_path):
    exe = str(tmp_path / "energy64_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "energy64_check.cpp")],
                   check=True)
    lines = [w.split() for w in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    print()
    for w in lines:
        print(*w)
    # erfc: half an ulp (1.1e-16) each from the last sum and the row's first
    # coefficient; the other terms, at most 0.38 of it, a rounding more
    err, rms, lib, librms = map(float, lines[0][1:])
    edge, far = float(lines[1][1]), float(lines[1][3])
    assert err < 2.7e-16 and edge < 2.7e-16 and rms < librms
    assert far < 2.2e-17 * 1e-6
    # sqrt within 0.51 ulp; 1/sqrt as a division by the rounded root
    s, sl, si, sil = (float(lines[2][k]) for k in (1, 2, 4, 5))
    assert s < 1.02 * sl and si < 1.02 * sil
    # energies: the rounding of r and 1/r, common to both, dominates
    assert len(lines) == 3 + 6
    for w in lines[3:]:
        q, qp, qmax, qpmax, lj, ljp, ljmax, ljpmax = map(float, w[4:])
        assert q < 1.02 * qp and lj < 1.02 * ljp
        assert qmax < 1.2 * qpmax and ljmax < 1.2 * ljpmax
