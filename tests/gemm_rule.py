"""The share GEMM's dispatch rule (csrc/gemm_rule.hpp), asked on the host: which
kernel a product takes, so that a test can say which one it means to reach."""
import functools
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def _exe():
    exe = os.path.join(tempfile.mkdtemp(prefix="gemm_rule"), "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "privacy-rag_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "gemm_rule_check.cpp"), "-o", exe], check=True)
    return exe


def choices(products):
    """products: (x, w, w_bits, m, k, n) with the operands' addresses; returns
    (kernel, k_split, splits, planes, adds) of each."""
    text = "".join(" ".join(str(int(v)) for v in p) + "\n" for p in products)
    r = subprocess.run([_exe()], input=text, capture_output=True, text=True)
    assert r.returncode == 0, f"rule ended with status {r.returncode}"
    rows = [line.split() for line in r.stdout.splitlines()]
    assert len(rows) == len(products)
    return [(k, int(a), int(b), int(c), d == "1") for k, a, b, c, d in rows]


W_BITS = {"i8": 8, "i32split": 24, "i32": 32}


def kernel(wdt, m, k, n, x=0, w=0):
    return choices([(x, w, W_BITS[wdt], m, k, n)])[0]
