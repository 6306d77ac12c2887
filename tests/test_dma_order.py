"""The T64 GEMMs' counted waits, replayed on the host (tests/cpp/dma_order.cpp): no operand is read before the wait that
covers its load, from the first step of a tile to the last."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "inferd_amd", "csrc")
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


def _host_source(text):
    """The device part of a source file with its asm statements as host code: waits, accumulator reads, nothing."""
    text, *host = text.split("// ---- host side")
    text = re.sub(r'#include "host.h"\n', "", text)
    text = re.sub(r'asm volatile\("s_waitcnt vmcnt\(%0\)[^"]*" ::"n"\((.*)\) : "memory"\);', r"emu::wait(\1);", text)
    text = re.sub(r'asm volatile\("s_waitcnt vmcnt\((\d+)\)[^;]*;', r"emu::wait(\1);", text)
    text = re.sub(r'asm volatile\("v_accvgpr_read_b32 %0, %1" : "=v"\((.*?)\) : "a"\((.*?)\)\);', r"\1 = \2;", text)
    text = re.sub(r'asm volatile\("(s_nop|s_waitcnt lgkmcnt|")[^;]*;', ";", text)
    assert "asm volatile" not in text
    return text + "}  // namespace ifd\n" if host else text


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    d = tmp_path_factory.mktemp("dma_order")
    for name in ("gemm_n.hip", "gemm_w.hip", "dma.h"):
        with open(os.path.join(CSRC, name)) as f:
            (d / name).write_text(_host_source(f.read()))
    exe = str(d / "dma_order")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-w", "-I", str(d), "-I", os.path.join(HERE, "cpp", "host_hip"), "-I", CSRC,
                    os.path.join(HERE, "cpp", "dma_order.cpp"), "-o", exe], check=True)
    return lambda kernel: subprocess.run([exe, kernel], check=True, capture_output=True, text=True).stdout.splitlines()


@pytest.mark.parametrize("kernel,cases", [("n", 8 * 9), ("w", 5 * 9)])
def test_operands_have_landed(replay, kernel, cases):
    lines = replay(kernel)
    assert len(lines) == cases
    assert not [x for x in lines if not x.endswith(": 0 operands, 0 scales")]
