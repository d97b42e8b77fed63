"""The narrow training step's weight gradients are accumulated by inline assembly
(train_fused.hip's fused_dw), for whose products the compiler inserts no wait
states.  What makes that sound is a property of the generated code, checked here
on the device assembly of every instantiation: inside the tile loop nothing but
those products touches their accumulators, and the first access after them has
the two s_nop 15 of fused_dw_done before it (32 wait states; the compiler puts 12
after such a product of its own)."""
import os
import re
import subprocess

import pytest

from rdv_project_amd import build as B

PRODUCT = re.compile(r"\s*v_mfma_f32_32x32x16_f16 a\[(\d+):(\d+)\],")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(B._hipcc()):
        pytest.skip("needs hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "train_fused.s")
    src = "train_fused.hip"
    subprocess.run([B._hipcc(), *B.COMMON_FLAGS, *B.SOURCE_FLAGS[src], "-S", "--cuda-device-only",
                    os.path.join(B.CSRC, src), "-o", out], check=True, capture_output=True)
    with open(out) as f:
        text = f.read()
    found = re.findall(r"^(_Z\S*train_fused_kernelILi(\d+)ELi(\d+)ELi(\d+)E\S*):.*?$(.*?)^\.Lfunc_end", text, re.S | re.M)
    return {tuple(map(int, k[1:4])): k[4].split("\n") for k in found}


def _accumulators(line):
    regs = {int(r) for r in re.findall(r"\ba(\d+)\b", line)}
    for lo, hi in re.findall(r"\ba\[(\d+):(\d+)\]", line):
        regs |= set(range(int(lo), int(hi) + 1))
    return regs


def test_every_shape_is_built(kernels):
    assert set(kernels) == {(1, d, i) for d in range(1, 6) for i in (1, 2)} | {(2, d, i) for d in range(1, 5) for i in (1, 2)}


@pytest.mark.parametrize("shape", [(1, d, i) for d in range(1, 6) for i in (1, 2)] +
                         [(2, d, i) for d in range(1, 5) for i in (1, 2)])
def test_accumulators_are_left_alone_until_the_wait(kernels, shape):
    lines = kernels[shape]
    products = [i for i, l in enumerate(lines) if PRODUCT.match(l)]
    dw = set().union(*(set(range(int(m[1]), int(m[2]) + 1)) for m in map(PRODUCT.match, (lines[i] for i in products))))
    label = {l.split(":")[0]: i for i, l in enumerate(lines) if re.match(r"\.LBB\S+:", l)}
    loops = [(label[m[1]], i) for i, l in enumerate(lines)
             if (m := re.search(r"s_c?branch\S*\s+(\.LBB\S+)", l)) and label.get(m[1], i) < i]
    begin, end = min(((a, b) for a, b in loops if a <= products[0] and b >= products[-1]), key=lambda r: r[1] - r[0])
    inside = [l.strip() for l in lines[begin:end] if not PRODUCT.match(l) and _accumulators(l) & dw]
    assert not inside, f"{len(inside)} other accesses in the tile loop, the first: {inside[0]}"
    after = lines[products[-1] + 1:]
    first = next(i for i, l in enumerate(after) if _accumulators(l) & dw)
    assert sum(l.split() == ["s_nop", "15"] for l in after[:first]) >= 2, f"no wait before {after[first].strip()}"
