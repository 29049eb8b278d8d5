"""Matrix instructions of the built library and the first instruction that
touches their result: on every path at least as many wait states lie between
them as the compiler keeps on straight code (8 after a 16x16x32 or 16x16x16
product, 10 after a 16x16x4 fp32 one; the hardware does not wait by itself).

The compiler counts them too, but not along every path: where a short side
branch joins the code that reads a result, it counted the branch's own
instructions for the path without the branch as well (5 states instead of 8:
row tiles of gemm_few_kernel came out wrong), so code with such a join has to
be written another way.
"""
import os
import re
import shutil
import subprocess

import pytest

from llambda_amd import build

OBJDUMP = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(build.HIPCC))),
                       "llvm", "bin", "llvm-objdump")
STATES = {"v_mfma_f32_16x16x4_f32": 10}  # the others: 8


def _registers(text):
    out = set()
    for kind, first, last, one_kind, one in re.findall(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        out |= ({(kind, i) for i in range(int(first), int(last) + 1)} if kind
                else {(one_kind, int(one))})
    return out


def _parse(listing):
    """{kernel: [(address, opcode, operands, target address or None)]}"""
    kernels, code, base = {}, None, 0
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(\S+)>:", line)
        if head:
            base, code = int(head.group(1), 16), kernels.setdefault(head.group(2), [])
            continue
        item = re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)", line)
        if code is None or not item:
            continue
        opcode, operands, at, rest = item.groups()
        target = re.search(r"<[^>+]+(?:\+0x([0-9a-f]+))?>", rest)
        code.append((int(at, 16), opcode, operands,
                     base + int(target.group(1) or "0", 16) if target else None))
    return kernels


def _short_waits(code):
    """Sites with too few wait states: (states, product, instruction)."""
    index = {at: i for i, (at, *_) in enumerate(code)}
    found = []
    for i, (_, product, operands, _) in enumerate(code):
        if not product.startswith("v_mfma"):
            continue
        need = STATES.get(product, 8)
        result = _registers(operands.split(",")[0])
        paths, least = [(i + 1, 0)], {}
        while paths:
            p, states = paths.pop()
            while p < len(code) and states < need and least.get(p, need) > states:
                least[p] = states
                _, opcode, args, target = code[p]
                if opcode.startswith("s_cbranch") or opcode == "s_branch":
                    if target in index:
                        paths.append((index[target], states + 1))
                    if opcode == "s_branch":
                        break
                elif opcode == "s_endpgm":
                    break
                elif opcode == "s_nop":
                    states += int(args, 0)
                elif opcode.startswith("v_mfma"):  # waits for an earlier product's result by itself
                    if _registers(args.split(",")[0]) & result:
                        break
                elif opcode.startswith(("v_", "ds_", "global_", "buffer_", "scratch_", "flat_")):
                    if _registers(args) & result:
                        found.append((states, f"{product} {operands}", f"{opcode} {args}"))
                        break
                states += 1
                p += 1
    return found


def test_join_of_two_paths_is_seen():
    lines = ["v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[8:11], v[0:3]", "s_cbranch_vccnz 6", "s_nop 3",
             "v_fma_f32 v20, v21, v0, v20", "s_endpgm", "v_mov_b32_e32 v30, 0", "v_mov_b32_e32 v31, 0",
             "s_branch 65531"]
    targets = {1: " <k+0x14>", 7: " <k+0x8>"}
    listing = "0000000000000000 <k>:\n" + "".join(
        f"\t{text} // {4 * i:012X}: 00000000{targets.get(i, '')}\n" for i, text in enumerate(lines))
    assert [s for s, *_ in _short_waits(_parse(listing)["k"])] == [5]
    assert not _short_waits(_parse(listing.replace("s_nop 3", "s_nop 6"))["k"])


def test_built_kernels(tmp_path):
    if not os.path.exists(build.LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("no built library or no llvm-objdump here")
    lib = shutil.copy(build.LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    products, bad = 0, []
    for name in sorted(os.listdir(tmp_path)):
        if build.ARCH not in name:
            continue
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=tmp_path, check=True,
                                 stdout=subprocess.PIPE, text=True).stdout
        for kernel, code in _parse(listing).items():
            products += sum(c[1].startswith("v_mfma") for c in code)
            bad += [(kernel, *site) for site in _short_waits(code)]
    assert products > 1000
    assert not bad, bad[:8]
