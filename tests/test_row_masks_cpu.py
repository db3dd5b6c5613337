"""Masks that the product rows take their created pairs and signs from, on the CPU: those of the sphere
(dh_row_masks of dh_sphere_row.h, compiled for the host) and the mirrored words of the momentum lattice
(lattice_mirror and lattice_row_free of dh_lattice.hip, their arithmetic restated here)."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_sphere_masks_and_signs(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "row_masks_selftest")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    "-I" + os.path.join(ROOT, "diagham_amd", "csrc"),
                    os.path.join(ROOT, "tests", "row_masks_selftest.cc"), "-o", exe], check=True)
    checks, wrong = map(int, subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True).stdout.split())
    assert checks > 1000000 and wrong == 0


def popc(v):
    return bin(v).count("1")


def mirror(word, n, ny, rot, ay, stay, wrap):
    """bit m of the result: bit P(m) of the word, P(m) the partner of m"""
    full = (1 << n) - 1
    rev = int(format(word, "0%db" % n)[::-1], 2)
    g = ((rev >> rot) | (rev << (n - rot))) & full if rot else rev
    return ((g >> ay) & stay) | ((g << (ny - ay)) & wrap)


@pytest.mark.parametrize("nx,ny", [(3, 3), (4, 2), (2, 5), (1, 9), (5, 2)])
def test_lattice_mirror_and_signs(nx, ny):
    n = nx * ny
    full = (1 << n) - 1
    for jx, jy in itertools.product(range(nx), range(ny)):
        partner = [((jx - m // ny) % nx) * ny + (jy - m % ny) % ny for m in range(n)]
        rot, ay = (nx - 1 - jx) % nx * ny, (ny - 1 - jy) % ny
        stay = sum(1 << m for m in range(n) if m % ny + ay < ny)
        small = sum(1 << m for m in range(n) if m < partner[m])
        for s in range(0, 1 << n, 3 if n > 8 else 1):
            f = ~s & full
            mirrored = mirror(f, n, ny, rot, ay, stay, full & ~stay)
            assert mirrored == sum(1 << m for m in range(n) if (f >> partner[m]) & 1)
            pm = f & mirrored & small  # bit m1: the pair (m1, P(m1)) is free in s
            par = sum(1 << m for m in range(n) if popc(s & ((1 << m) - 1)) & 1)
            for n1 in range(n):
                n2 = partner[n1]
                if n1 >= n2 or not (s >> n1) & 1 or not (s >> n2) & 1:
                    continue
                t = s ^ (1 << n1) ^ (1 << n2)
                pt = par ^ (((2 << n2) - 1) & ~((2 << n1) - 1))  # prefix parities of t
                q = pt ^ mirror(pt, n, ny, rot, ay, stay, full & ~stay)
                q = q if (q >> n1) & 1 else ~q
                annihilated = popc(s >> n2) + popc((s ^ (1 << n2)) >> n1)
                for m1 in range(n):
                    m2 = partner[m1]
                    if m1 >= m2 or (t >> m1) & 1 or (t >> m2) & 1:
                        continue
                    sign = (annihilated + popc(t >> m2) + popc((t | (1 << m2)) >> m1)) & 1
                    if m1 == n1:  # the diagonal term, -conj(F)
                        assert sign == 1
                    else:
                        assert (pm >> m1) & 1 and sign == (q >> m1) & 1, (jx, jy, s, n1, m1)
