"""The rows kernel's loop over K waits for the oldest of its loads only, in the builds whose last unit is short as in those where it is
whole (compiled to assembly here; a wait for every load in flight costs such a product 5 to 14 %)."""
import os
import re
import subprocess

import pytest

from mlx_eagle_spec_decoding_tree_amd import build

FORMS = [(1, 1, 1, 1), (2, 1, 1, 2), (3, 3, 1, 1), (2, 2, 2, 1), (3, 2, 2, 2)]       # tiles, tiles, tiles of x, K parts


def least_waits(path):
    """{(tiles, tiles, tiles of x, K parts, chunks of the last unit): the least vmcnt of each loop that requests weights}"""
    out = {}
    with open(path) as f:
        text = f.read()
    for m in re.finditer(r"^(_Z\S*qmm_rows_kernel\S*):.*?\.Lfunc_end", text, re.S | re.M):
        rt, rt2, mt, kp, _, _, rem = (int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1)))
        blocks = re.split(r"^(\.LBB\S+):", m.group(0), flags=re.M)
        for label, body in zip(blocks[1::2], blocks[2::2]):
            if label in re.findall(r"s_cbranch\S+ (\.LBB\S+)", body) and "v_mfma" in body and body.count("buffer_load") >= 4:
                waits = [int(v) for v in re.findall(r"vmcnt\((\d+)\)", body)]
                out.setdefault((rt, rt2, mt, kp, rem), []).append(min(waits))
    return out


def test_short_last_units_leave_the_loads_in_flight(tmp_path):
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src, asm = tmp_path / "forms.hip", tmp_path / "forms.s"
    calls = "".join(f"  rc |= rows_launch<{a}, {b}, {mt}, {kp}, 4, false, {rem}>(a, 1, s);\n" for a, b, mt, kp in FORMS for rem in (2, 4))
    src.write_text(f'#include "rows.h"\nusing namespace eagle_rows;\nint forms(const RowsArgs& a, hipStream_t s) {{\n  int rc = 0;\n{calls}  return rc;\n}}\n')
    flags = [f for f in build.FLAGS if f not in ("-shared", "-Rpass-analysis=kernel-resource-usage")]
    subprocess.run([cc, *flags, f"-I{build.CSRC}", "-S", "--cuda-device-only", str(src), "-o", str(asm)], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    waits = least_waits(asm)
    assert len(waits) == 2 * len(FORMS) and os.path.getsize(asm)
    for a, b, mt, kp in FORMS:
        whole, short = waits[a, b, mt, kp, 4], waits[a, b, mt, kp, 2]
        assert len(whole) == len(short) == (1 if a == b else 2)
        assert min(whole) > 0 and short == whole, (a, b, mt, kp, short, whole)


def test_the_sources_of_forms_share_one_definition_of_their_types():
    """The launches that rows.hip calls take an argument type of all sources, not one of each source's unnamed namespace."""
    objects = [os.path.join(build.HERE, "build", f"rows_{i}.hip.o") for i in range(1, 5)]
    if not all(os.path.exists(o) for o in objects):
        pytest.skip("no objects of a build here")
    for obj in objects:
        names = subprocess.run(["nm", "-C", obj], check=True, stdout=subprocess.PIPE).stdout.decode()
        launches = [line for line in names.splitlines() if "::rows_launch<" in line]
        assert launches and all("(eagle_rows::RowsArgs const&" in line for line in launches), launches[:1]
