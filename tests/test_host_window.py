"""When x that the host writes into device memory is there (no device needed): what window_written compiles to, and where the call on
host arrays has it."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llama2.rs_amd", "csrc")

PROBE = r"""
#include <string.h>
#include "host_window.h"
extern "C" void launch();
extern "C" void call(float *window, const float *x, size_t n, volatile uint32_t *flush) {
    memcpy(window, x, n);
    window_written(flush);
    launch();
}
"""


def test_the_writes_are_flushed_and_waited_for_before_the_launch(tmp_path):
    src, out = tmp_path / "probe.cpp", tmp_path / "probe.s"
    src.write_text(PROBE)
    subprocess.run(["g++", "-O3", "-std=c++17", "-I", CSRC, "-S", str(src), "-o", str(out)], check=True)
    body = out.read_text().split("\ncall:")[1].split(".cfi_endproc")[0]
    lines = [line.strip() for line in body.splitlines() if line.startswith("\t") and not line.strip().startswith(".")]
    at = [next(i for i, line in enumerate(lines) if re.search(pattern, line))
          for pattern in (r"memcpy", r"^sfence", r"^movl\s+\$1, \(%r", r"^movl\s+\(%r\w+\), %e", r"^mfence", r"\blaunch\b")]
    assert at == sorted(at), body


def test_the_call_on_host_arrays_waits_between_the_copy_and_its_first_kernel():
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "host.cpp")).read())
    call = text[text.index("static int matvec_host("):text.index('extern "C" int l2_qlinear_matvec(')]
    copies = [m.start() for m in re.finditer(r"memcpy\(x \+", call)]
    assert len(copies) == 1
    behind = call[copies[0]:]
    assert behind.index("if (window.x) window_written(window.flush);") < min(behind.index(k) for k in ("_launch(", "q4_one", "gemm_operator("))
