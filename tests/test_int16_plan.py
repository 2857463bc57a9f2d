"""When float32 activations of a 16-bit multiplication are quantized by a launch of their own: the library's rule (a host
function) against the times kept in profiles/int16_forms.txt."""
import os

from conftest import ROOT, load


def measured():
    """(M, K, N, us of the one launch in the form that is taken, us of the two launches, the decision the table shows)"""
    rows = []
    for line in open(os.path.join(ROOT, "profiles", "int16_forms.txt")):
        parts = [p.split() for p in line.split("|")]
        if len(parts) == 4 and parts[0][0].isdigit():
            forms = dict(zip(("16x16", "16x32", "32x32", "64x64", "128x128"), parts[2]))
            rows.append((*map(int, parts[0]), float(forms[parts[2][5]]), float(parts[3][1]), parts[3][2]))
    return rows


def test_quantizing_first_where_it_pays():
    lib = load("_lib").lib()
    rows = measured()
    assert len(rows) == 99
    behind = []
    for M, K, N, one, both, shown in rows:
        scratch = lib.marian_hip_int16_scratch_bytes(M, K, N)
        assert scratch in (0, 2 * M * K + 4) and (scratch > 0) == (shown == "q"), (M, K, N)
        taken = both if scratch else one
        if taken > 1.035 * min(one, both):
            behind.append((M, K, N, taken, min(one, both)))
    assert len(behind) <= 2 and all(t < 1.2 * b for *_, t, b in behind), behind
