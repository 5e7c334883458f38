"""The lanes of a wave hand each other keys through LDS in attn_flash_kernel without a workgroup
barrier. The compiler reasons per lane, so only a fence keeps a lane's read behind the other lanes'
writes (and the next writes behind the reads): in the kernel's intermediate code, as compiled for
gfx950, no LDS store may meet an LDS load with no fence between them."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fusor-ai_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("ir") / "qwen2.ll"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-w", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", "-emit-llvm", "--cuda-device-only",
                    os.path.join(CSRC, "qwen2.hip"), "-o", str(out)], check=True)
    return out.read_text()


def blocks_of(body):
    """The function's basic blocks: name -> (its fences and LDS accesses in order, its successors)."""
    blocks, name = {}, "entry"
    blocks[name] = ([], [])
    for line in body.splitlines()[1:]:
        label = re.match(r"(\d+):", line)
        if label:
            name = label.group(1)
            blocks[name] = ([], [])
        elif re.match(r"\s*fence ", line):
            blocks[name][0].append("fence")
        elif re.match(r"\s*store .*addrspace\(3\)", line):
            blocks[name][0].append("store")
        elif re.search(r"= load .*addrspace\(3\)", line):
            blocks[name][0].append("load")
        elif re.match(r"\s*br ", line):
            blocks[name][1].extend(re.findall(r"label %(\d+)", line))
        else:
            assert not re.match(r"\s*(switch|indirectbr) ", line), line
    return blocks


@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_lds_stores_and_loads_are_fenced(code, head_dim):
    name = rf"attn_flash_kernelILi{head_dim}E"
    blocks = blocks_of(re.search(rf"^define [^\n]*{name}.*?^}}", code, re.M | re.S).group(0))
    assert sum(k == "store" for ops, _ in blocks.values() for k in ops) >= 4
    assert sum(k == "load" for ops, _ in blocks.values() for k in ops) >= 4
    # along every path: the kinds of LDS accesses since the last fence, at each block's entry
    since = {b: set() for b in blocks}
    todo = ["entry"] + list(blocks)
    while todo:
        b = todo.pop()
        live = set(since[b])
        for kind in blocks[b][0]:
            live = set() if kind == "fence" else live | {kind}
            assert len(live) < 2, f"block {b}: an LDS store and an LDS load with no fence between them"
        for n in blocks[b][1]:
            if not live <= since[n]:
                since[n] |= live
                todo.append(n)
