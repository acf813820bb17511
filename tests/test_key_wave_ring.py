"""The pipelined kernel's waves that split the keys refill a ring of their own: in the compiled code every read of LDS has been waited
for when a fill of LDS is requested (no barrier stands between the two).  Compiles the kernel's variants to assembly, on the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-attention_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _reads_in_flight_at_a_fill(lines):
    """(fills, line numbers of fills that follow an LDS read not waited for), in the order of the code; the loop over the steps ends
    with the wait, so that its backward branch needs no look of its own"""
    reading, fills, bad = False, 0, []
    for n, line in enumerate(lines, 1):
        code = line.split(";")[0].strip()
        if code.startswith("ds_read"):
            reading = True
        elif code.startswith("s_waitcnt") and "lgkmcnt(0)" in code:
            reading = False
        elif code.startswith("global_load_lds"):
            fills += 1
            if reading:
                bad.append(n)
    return fills, bad


def test_the_check_sees_a_read_in_flight():
    assert _reads_in_flight_at_a_fill(["ds_read_b128 v[0:3], v4", "s_waitcnt lgkmcnt(1)", "global_load_lds_dwordx4 v1, s[0:1]"]) == (1, [3])
    assert _reads_in_flight_at_a_fill(["ds_read_b128 v[0:3], v4", "s_waitcnt vmcnt(0) lgkmcnt(0)", "global_load_lds_dwordx4 v1, s[0:1]"]) == (1, [])


@pytest.mark.parametrize("key_waves", [4, 2])
@pytest.mark.parametrize("d,dv,bn", [(64, 64, 64), (64, 32, 64), (128, 128, 32), (128, 96, 32)])
def test_no_refill_while_a_read_is_in_flight(tmp_path, d, dv, bn, key_waves):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    source = tmp_path / "variant.hip"
    source.write_text('#include "fa_prefill_il.h"\n' + "".join(
        "template __global__ void fa::prefill_il_kernel<__bf16, fa::ILCfg<__bf16, %d, %d, %d, %d>, false, %s, false>(const fa::KParams);\n"
        % (d, bn, dv, key_waves, rot) for rot in ("false", "true")))
    out = tmp_path / "variant.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w",
                    "-I" + CSRC, "-I" + os.path.join(os.path.dirname(os.path.dirname(CSRC)), "include"), "--cuda-device-only", "-S", str(source), "-o", str(out)], check=True)
    text = out.read_text()
    fills, bad = _reads_in_flight_at_a_fill(text.splitlines())
    assert text.count("ds_read") > 50 and fills > 50 and not bad, bad
    # stated by the kernel, not left to where the compiler waits: after the first product and at the end of every step
    assert text.count("own ring") >= 4
