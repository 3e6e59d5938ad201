"""How bench.py finds the HBM traffic of the q4 launches in a committed counter summary (no GPU needed)."""
import pytest

import bench

KERNELS = {"q4_qkv": "q4_stream_kernel<128, 2, 8, false, 3, 2, false>", "q4_wo": "q4_stream_kernel<128, 2, 8, false, 3, 2, false>",
           "q4_w13": "q4_stream_kernel<128, 2, 4, true, 0, 2, false>", "q4_w2": "q4_stream_kernel<128, 6, 2, false, 0, 3, false>"}
ROWS = """
{section}: plain device copy of 268435456 bytes (bench.py's copy leg, kernel __amd_rocclr_copyBuffer) reads 131092.4
  -> scale factor 2047.7 bytes per unit
  dispatches         mean          bytes  kernel
         576      24020.8      {0}  q4_stream_kernel<128, 2, 4, true, 0, 2, false>{parameters}
        1152       9146.5      {1}  q4_stream_kernel<128, 2, 8, false, 3, 2, false>{parameters}
         576      12108.8      {2}  q4_stream_kernel<128, 6, 2, false, 0, 3, false>{parameters}
          18     256168.6     524551411  dense_matvec_kernel<16, 2>(DenseArgs)
         576        235.8        482880  __amd_rocclr_copyBuffer
"""


@pytest.fixture
def summary(tmp_path, monkeypatch):
    digest = bench.q4_sources_digest()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    monkeypatch.setattr(bench, "q4_sources_digest", lambda: digest)
    (tmp_path / "profiles").mkdir()

    def write(name, parameters, digest=digest):
        text = f"a summary\nsources of the q4 kernels: {digest}\n"
        for section, scale in (("FETCH_SIZE", 1000), ("WRITE_SIZE", 1)):
            text += ROWS.format(40 * scale, 20 * scale, 30 * scale, section=section, parameters=parameters)
        (tmp_path / "profiles" / name).write_text(text)

    return write


# whatever the kernel's parameters are: the library names its kernels without them
@pytest.mark.parametrize("parameters", ["(Q4Launch)", "(float const*, float const*, int const*, int, int, int, StreamArgs)"])
def test_traffic_is_found_by_the_kernels_names(summary, parameters):
    summary("q4_matvec_7B_decode_hbm_counters.txt", parameters)
    assert bench.measured_traffic("7B", KERNELS) == (round(1001 * (20 + 20 + 40 + 30) / 4), "profiles/q4_matvec_7B_decode_hbm_counters.txt")
    table, _ = bench.counter_summary("q4_matvec_7B_decode_hbm_counters.txt")
    assert set(table["FETCH_SIZE"]) == set(KERNELS.values()) | {"dense_matvec_kernel<16, 2>", "__amd_rocclr_copyBuffer"}


def test_other_kernels_are_refused(summary):
    value, note = bench.measured_traffic("7B", KERNELS)
    assert value is None and "no counter summary" in note
    summary("q4_matvec_7B_decode_hbm_counters.txt", "(StreamArgs)", digest="0" * 16)  # of the same names
    value, note = bench.measured_traffic("7B", KERNELS)
    assert value is None and "other kernels" in note
    summary("q4_matvec_7B_decode_hbm_counters.txt", "(StreamArgs)")
    value, note = bench.measured_traffic("7B", {**KERNELS, "q4_w2": "q4_stream_kernel<128, 6, 2, false, 0, 4, false>"})
    assert value is None and "0, 4, false" in note


def test_digest_is_of_the_code_alone(tmp_path, monkeypatch):
    where = tmp_path / "llama2.rs_amd" / "csrc"
    where.mkdir(parents=True)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))

    def digest(text):
        for name in bench.Q4_SOURCES:
            (where / name).write_text(text)
        return bench.q4_sources_digest()

    assert digest("int a; // one\n/* two\n */ int b;") == digest("int a;\n\n int b; // other")
    assert digest("int a;") != digest("int b;")
