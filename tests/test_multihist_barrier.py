"""The barrier between a run's workgroups in the compiled multihistogram
kernels: the block sums are stored past the L2 (agent scope), every wave waits
for its own before the workgroup's barrier that precedes the arrival (that
barrier waits for LDS only, and the arrival's release covers the stores of its
own wave only), and the arrival is a release."""
import os
import re
import subprocess

import pytest

from conftest import PKG_DIR


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    import build

    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("asm") / "mh.s"
    subprocess.run([build.HIPCC, *build.CFLAGS, "-S", "--cuda-device-only", str(PKG_DIR / "csrc" / "ptmc_multihist.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    body, name = {}, None
    for line in out.read_text().splitlines():
        m = re.match(r"(_Z\w*mh_iterate_kernel\w*):", line)
        if m:
            name = m.group(1)
            body[name] = []
        elif ".end_amdhsa_kernel" in line or "s_endpgm" in line:
            name = None
        elif name:
            code = line.split(";")[0].strip()
            if code and not code.startswith("."):
                body[name].append(code)
    return body


def test_stores_are_complete_before_the_arrival(kernels):
    assert len(kernels) == 2
    for name, code in kernels.items():
        arrivals = [i for i, c in enumerate(code) if c.startswith("global_atomic_add")]
        assert arrivals, name
        for i in arrivals:
            b = max(k for k in range(i) if code[k].startswith("s_barrier"))
            before, release = code[max(0, b - 40):b], code[b:i]
            wait = max((k for k, c in enumerate(before) if c.startswith("s_waitcnt") and "vmcnt(0)" in c), default=-1)
            stores = [k for k, c in enumerate(before) if c.startswith(("global_store", "flat_store"))]
            assert wait >= 0 and all(k < wait for k in stores), (name, before)
            assert any(c.startswith("buffer_wbl2") and "sc1" in c for c in release), (name, release)
        # the sums' stores: one agent-scope store of a double per kernel
        sums = [c for c in code if c.startswith("global_store_dwordx2") and c.endswith("sc1")]
        assert sums, name
