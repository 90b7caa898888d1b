"""The rules that choose a kernel or a launch shape by size, compiled from their header and asked
about measured points: the dense-product kernel of the collapsed shapes against the kernel it
replaces (1.5 times apart or more), and the wide launch of the hex Helmholtz kernels.  The rule
takes the faster one."""
import math
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ithaca-sem_amd", "csrc")
MAIN = """
#include "mf_routes.hpp"
#include <cstdio>
int main() {
    int s, h, f, p, c; long M, Q, n;
    while (std::scanf("%d %d %d %d %d %ld %ld %ld", &s, &h, &f, &p, &c, &M, &Q, &n) == 8)
        if (s < 0)  // hex Helmholtz: points, FP64, deformed, elements
            std::printf("%d\\n", imf::helm_wide_from(h, f, p) > 0 && n >= imf::helm_wide_from(h, f, p));
        else
            std::printf("%d\\n", imf::dense_pays({s, h != 0, f != 0, p != 0, c != 0, M, Q, n}));
}
"""
SHAPES = ["tri", "tet", "prism", "pyr"]
# shape, operator, Jacobian per point, pencil kernel is the alternative, nm, nq, elements,
# dense us, alternative us (MI355X)
MEASURED = [
    ("tri", "BwdTrans", 0, 0, 2, 10, 3000, 7.43, 4.7), ("tri", "BwdTrans", 0, 0, 2, 2, 10000, 3.98, 6.84),
    ("tri", "Helmholtz", 0, 0, 2, 2, 1, 3.69, 8.35), ("tri", "Helmholtz", 0, 0, 6, 6, 30000, 8.67, 129.77),
    ("tri", "IProduct", 0, 0, 2, 4, 1, 3.14, 5.48), ("tri", "IProduct", 1, 0, 8, 8, 10000, 7.57, 37.48),
    ("tet", "BwdTrans", 0, 0, 7, 7, 1000, 14.68, 9.21), ("tet", "BwdTrans", 0, 0, 4, 12, 1000, 10.2, 16.17),
    ("tet", "BwdTrans", 0, 1, 7, 9, 20833, 82.82, 52.48), ("tet", "Helmholtz", 0, 0, 8, 8, 1000, 69.28, 36.97),
    ("tet", "Helmholtz", 0, 0, 3, 3, 256, 4.72, 12.5), ("tet", "Helmholtz", 0, 1, 8, 9, 3000, 69.66, 38.87),
    ("tet", "Helmholtz", 0, 1, 3, 5, 1, 4.04, 6.96), ("tet", "IProduct", 0, 0, 8, 12, 256, 142.5, 14.2),
    ("tet", "IProduct", 0, 0, 8, 8, 3000, 44.95, 29.44), ("tet", "IProduct", 0, 0, 4, 12, 8264, 66.92, 159.49),
    ("tet", "IProduct", 0, 1, 6, 7, 3000, 18.18, 9.95), ("tet", "IProduct", 0, 1, 4, 6, 10000, 9.32, 14.99),
    ("tet", "IProduct", 1, 0, 3, 11, 3000, 72.59, 41.95), ("tet", "IProduct", 1, 0, 7, 7, 30000, 51.86, 123.56),
    ("tet", "IProduct", 1, 1, 6, 7, 3000, 26.18, 10.1), ("tet", "IProduct", 1, 1, 6, 8, 30000, 61.5, 100.23),
    ("prism", "BwdTrans", 0, 0, 8, 8, 3000, 35.14, 23.17), ("prism", "BwdTrans", 0, 0, 5, 13, 1000, 17.91, 31.59),
    ("prism", "BwdTrans", 0, 1, 4, 5, 120000, 58.57, 37.39), ("prism", "Helmholtz", 0, 0, 6, 6, 3000, 74.39, 40.67),
    ("prism", "Helmholtz", 0, 0, 2, 10, 256, 4.04, 22.33), ("prism", "Helmholtz", 0, 1, 6, 7, 40816, 220.11, 104.43),
    ("prism", "Helmholtz", 0, 1, 2, 4, 10000, 4.23, 6.66), ("prism", "IProduct", 0, 0, 6, 10, 16, 87.7, 8.3),
    ("prism", "IProduct", 0, 0, 3, 11, 3000, 54.73, 34.65), ("prism", "IProduct", 0, 0, 2, 6, 3000, 7.64, 13.65),
    ("prism", "IProduct", 0, 1, 6, 7, 40816, 100.21, 59.21), ("prism", "IProduct", 0, 1, 2, 4, 120000, 14.13, 22.51),
    ("prism", "IProduct", 1, 0, 6, 14, 100, 329.9, 13.0), ("prism", "IProduct", 1, 1, 6, 7, 30000, 74.39, 46.75),
    ("pyr", "BwdTrans", 0, 0, 7, 7, 1000, 18.61, 11.57), ("pyr", "BwdTrans", 0, 0, 5, 13, 1000, 14.44, 37.28),
    ("pyr", "BwdTrans", 0, 1, 6, 7, 40816, 80.96, 45.79), ("pyr", "Helmholtz", 0, 0, 6, 6, 1000, 42.84, 25.97),
    ("pyr", "Helmholtz", 0, 0, 5, 5, 10000, 20.97, 83.41), ("pyr", "Helmholtz", 0, 1, 5, 6, 3000, 19.97, 10.49),
    ("pyr", "Helmholtz", 0, 1, 3, 5, 3000, 4.91, 8.1), ("pyr", "IProduct", 0, 0, 2, 10, 1000, 27.27, 9.39),
    ("pyr", "IProduct", 0, 0, 5, 13, 5917, 132.93, 298.82), ("pyr", "IProduct", 0, 1, 6, 7, 10000, 30.73, 18.35),
    ("pyr", "IProduct", 0, 1, 3, 5, 30000, 8.7, 13.89), ("pyr", "IProduct", 1, 0, 3, 11, 3000, 79.52, 40.31),
    ("pyr", "IProduct", 1, 1, 8, 9, 18518, 231.73, 120.01),
]


def _sizes(shape, m, q):
    return {"tri": (m * (m + 1) // 2, q * (q - 1)), "tet": (m * (m + 1) * (m + 2) // 6, q * (q - 1) ** 2),
            "prism": (m * m * (m + 1) // 2, q * q * (q - 1)),
            "pyr": (m * (m + 1) * (2 * m + 1) // 6, q * q * (q - 1))}[shape]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{SRC}", "-o", str(d / "routes"), str(d / "main.cpp")],
                   check=True)

    def run(cases):
        text = "".join(" ".join(str(int(x)) for x in c) + "\n" for c in cases)
        out = subprocess.run([str(d / "routes")], input=text, capture_output=True, text=True, check=True).stdout
        return [bool(int(x)) for x in out.split()]
    return run


def _case(shape, op, point, pencil, nm, nq, n):
    M, Q = _sizes(shape, nm, nq)
    return SHAPES.index(shape), op == "Helmholtz", op != "IProduct", point, pencil, M, Q, n


def test_the_faster_kernel_is_taken(ask):
    got = ask([_case(*m[:7]) for m in MEASURED])
    assert len(got) == len(MEASURED)
    for m, dense in zip(MEASURED, got):
        assert dense == (m[7] < m[8]), m


def test_the_choice_changes_once_with_the_number_of_elements(ask):
    ns = [1 + int(math.exp(0.2 * i)) for i in range(60)]
    keys = [(shape, op, point, pencil, nm, nm + extra) for shape in SHAPES
            for op in ("Helmholtz", "BwdTrans", "IProduct") for point in (0, 1) for pencil in (0, 1)
            for nm in range(2, 9) for extra in (0, 1, 2, 4, 8)]
    got = ask([_case(*k, n) for k in keys for n in ns])
    for i, k in enumerate(keys):
        one = got[i * len(ns):(i + 1) * len(ns)]
        assert one == sorted(one), k


@pytest.mark.parametrize("nq,fp64,deformed,n,narrow,wide", [
    (6, 1, 1, 16, 5.9, 7.6), (6, 1, 1, 1000, 8.0, 8.8), (6, 1, 1, 6000, 22.1, 20.1), (6, 1, 0, 400, 6.0, 7.1),
    (6, 1, 0, 6000, 14.5, 12.8), (6, 0, 0, 2000, 6.7, 7.3), (6, 0, 0, 6000, 10.9, 9.9), (9, 1, 1, 256, 11.5, 13.6),
    (9, 1, 1, 1500, 28.8, 20.4), (9, 0, 0, 1000, 9.2, 10.1), (9, 0, 0, 1500, 12.5, 10.5), (9, 0, 1, 100, 7.5, 9.2),
    (9, 0, 1, 3000, 23.6, 21.7), (7, 0, 0, 3000, 9.3, 9.8), (7, 0, 0, 16000, 26.6, 24.4), (7, 1, 1, 35000, 133, 150),
    (6, 0, 1, 55000, 74, 79)])
def test_hex_helmholtz_launch(ask, nq, fp64, deformed, n, narrow, wide):
    assert ask([(-1, nq, fp64, deformed, 0, 0, 0, n)]) == [wide < narrow]
