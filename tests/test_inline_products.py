"""The matrix kernels whose products are inline assembly (csrc/matrix_async.h): the compiler does not know these instructions for products and
keeps no distance from them by itself.  Their assembly, made here from the sources, is read for two distances on every path: from a product
to whatever else touches its sum, and from a vector instruction to a product that reads what it wrote."""
import os
import re
import subprocess

import pytest

FILES = {"gemm_tiles_bf16.hip": 13, "gemm_groups_bf16.hip": 8, "gemm_f32.hip": 4}      # kernels with such products
# Instructions in between, an s_nop counted as what it waits: a product of the longest kind has its sum written after 18, and a vector
# instruction's result may be read by a product after 2 (ma_wait_products waits 32, ma_wait_written 4).
SUM, OPERAND = 18, 2
REGISTER = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+))")


def registers(text):
    return {f"{m[1]}{i}" for m in REGISTER.finditer(text) for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)}


def kernels(text):
    """(name, instructions, label -> place) of every function; an instruction is (text, whether inline assembly)."""
    for name, body in re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.M | re.S):
        code, labels, inline = [], {}, False
        for line in body.split("\n"):
            line = line.strip()
            if line.startswith(";;#ASM"):
                inline = line.startswith(";;#ASMSTART")
            line = line.split(";")[0].strip()
            label = re.match(r"(\.L\w+):", line)
            if label:
                labels[label[1]] = len(code)
            elif line and not line.startswith("."):
                code.append((line, inline))
        yield name, code, labels


def behind(at, code, labels, most):
    """Every instruction that fewer than ``most`` wait states separate from the one at ``at`` on some path."""
    def after(i):
        branch = re.match(r"s_(c?)branch\w* (\S+)", code[i][0])
        if branch:
            return ([i + 1] if branch[1] else []) + [labels[branch[2]]]
        return [] if code[i][0].startswith("s_endpgm") else [i + 1]
    least, todo = {}, [(i, 0) for i in after(at)]
    while todo:
        i, states = todo.pop()
        if states < most and states < least.get(i, most):
            least[i] = states
            wait = re.match(r"s_nop (\d+)", code[i][0])
            todo += [(j, states + (int(wait[1]) + 1 if wait else 1)) for j in after(i)]
    return [code[i][0] for i in least]


def too_near(code, labels):
    found = []
    for at, (op, inline) in enumerate(code):
        written = registers(op.split(",")[0])
        if op.startswith("v_mfma") and inline:
            for other in behind(at, code, labels, SUM):
                if other.startswith("v_mfma"):               # (products add to one sum one after another; none reads a sum as an operand)
                    parts = other.split(",")
                    near = registers(",".join(parts[1:3])) & written or (registers(parts[0]) & written and registers(parts[0]) != written)
                else:
                    near = registers(other) & written
                if near:
                    found.append((op, other))
        elif op.startswith("v_") and written:
            found += [(op, other) for other in behind(at, code, labels, OPERAND) if other.startswith("v_mfma") and registers(other) & written]
    return found


@pytest.mark.parametrize("name", list(FILES))
def test_nothing_comes_too_near_to_an_inline_product(name, tmp_path):
    from rust_inference_amd.errors import KernelError
    from rust_inference_amd.kernels import build
    try:
        hipcc = build._hipcc()
    except KernelError as e:
        pytest.skip(str(e))
    out = str(tmp_path / "kernels.s")
    subprocess.run([hipcc, *build.HIPCC_FLAGS, *build.FILE_FLAGS.get(name, []), "--cuda-device-only", "-S", os.path.join(build.CSRC, name), "-o", out],
                   check=True, env=dict(os.environ, HOME=os.environ.get("HOME", str(tmp_path))), capture_output=True)
    with open(out) as f:
        text = f.read()
    with_products = [k for k in kernels(text) if any(op.startswith("v_mfma") and inline for op, inline in k[1])]
    assert len(with_products) == FILES[name]
    for kernel, code, labels in with_products:
        assert not too_near(code, labels), kernel
    # the reading itself: a move of a sum behind its product, a move into an operand before one
    _, code, labels = with_products[0]
    at = next(i for i, (op, inline) in enumerate(code) if op.startswith("v_mfma") and inline)
    sums, operand = (re.match(r"v_mfma\S+ a\[(\d+):\d+\], v\[(\d+):\d+\]", code[at][0])[i] for i in (1, 2))
    for place, move in ((at + 1, f"v_accvgpr_read_b32 v0, a{sums}"), (at - 1, f"v_mov_b32_e32 v{operand}, v0")):
        assert too_near(code[:place] + [(move, False)] + code[place + 1:], labels), move
