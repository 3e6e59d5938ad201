"""store_through in the AMD assembly of a probe built here (no GPU needed): the store goes past the L2, and the compiler knows
of it, so that it waits where the hardware does not."""
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "llama2.rs_amd"))

PROBE = r"""
#include "l2_internal.h"
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
// the data come straight out of a matrix instruction
__global__ void of_matrix(float4 *p, float a, float b) {
    const f4v v = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, f4v{}, 0, 0, 0);
    store_through(p + threadIdx.x, make_float4(v[0], v[1], v[2], v[3]));
}
// ... and their registers are written again right behind the store
__global__ void over_data(float4 *p, u4v *q) {
    u4v v = q[threadIdx.x];
    asm volatile("; data" : "+{v[8:11]}"(v));
    store_through(p + threadIdx.x, __builtin_bit_cast(float4, v));
    v = u4v{1, 2, 3, 4};
    asm volatile("; again" : "+{v[8:11]}"(v));
    q[threadIdx.x] = v;
}
"""


def _body(asm, name):
    lines = asm[asm.index(f"; @_Z{len(name)}{name}"):].split("s_endpgm")[0].splitlines()
    return [l.split(";")[0].strip() for l in lines if l.split(";")[0].strip()]


def _wait_states(lines):
    """What the instructions between two others let pass: one each, and what s_nop adds."""
    return sum(int(l.split()[1]) + 1 if l.startswith("s_nop") else 1 for l in lines)


def test_the_compiler_waits_around_the_store(tmp_path):
    import build as b  # llama2.rs_amd/build.py: the flags of the product build
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE)
    r = subprocess.run([b.hipcc(), *b.COMMON, *b.DEVICE_FLAGS, "-mllvm", "-amdgpu-mfma-vgpr-form=1", "-I", b.CSRC,
                        "--offload-device-only", "-S", str(src), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    asm = out.read_text()

    body = _body(asm, "of_matrix")
    at = next(i for i, l in enumerate(body) if l.startswith("v_mfma"))
    st = next(i for i, l in enumerate(body) if "store_dwordx4" in l)
    assert re.search(r"\bsc1\b", body[st]) and not re.search(r"\b(sc0|nt)\b", body[st]), body[st]
    # 16x16x4 fp32: 8 passes of 4 cycles; a store may read the result 10 wait states later
    assert at < st and _wait_states(body[at + 1:st]) >= 10, body

    body = _body(asm, "over_data")
    st = next(i for i, l in enumerate(body) if "store_dwordx4" in l)
    nxt = next(i for i in range(st + 1, len(body)) if re.match(r"v_mov_b\d+\S* v(\[)?(8|9|10|11)\b", body[i]))
    assert _wait_states(body[st + 1:nxt]) >= 2, body


def test_no_store_in_a_statement_of_assembly():
    import build as b
    for name in sorted(os.listdir(b.CSRC)):
        text = re.sub(r"//[^\n]*", "", open(os.path.join(b.CSRC, name)).read())
        for m in re.finditer(r"\basm\b[^;]*;", text):
            assert not re.search(r"(store_dword|store_b|ds_write|atomic)", m.group(0)), (name, m.group(0))
