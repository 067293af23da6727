"""The gfx950 code of the row movers (csrc/rows.hip, compiled to assembly): what
their copy loops rely on and the source alone does not show."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instructions of each kernel of rows.hip, by a part of its name."""
    if shutil.which(HIPCC) is None:
        pytest.skip("hipcc is not available")
    import importlib.util

    spec = importlib.util.spec_from_file_location("_kvx_build", os.path.join(ROOT, "kv_offload_proto_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    out = tmp_path_factory.mktemp("rows") / "rows.s"
    subprocess.run([HIPCC] + build.HIP_FLAGS + ["--cuda-device-only", "-S", "-I", build.INCLUDE, "-I", build.CSRC, "-o", str(out),
                                                os.path.join(build.CSRC, "rows.hip")],
                   check=True, capture_output=True, timeout=300)
    found, name = {}, None
    for line in out.read_text().splitlines():
        m = re.match(r"_Z\w*?(kvx_(?:gather|export|stream)_\w+?)E\w*:", line)
        if m:
            name = m.group(1)
            found[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name is not None and line.startswith("\t") and not line.lstrip().startswith((".", ";")):
            found[name].append(line.split(";")[0].strip())
    return found


THROUGH = ["kvx_gather_one", "kvx_export_alllayer", "kvx_export_rows_copy", "kvx_export_rows_small"]


def _kernel(kernels, name):
    (found,) = [code for k, code in kernels.items() if k.startswith(name)]
    return found


@pytest.mark.parametrize("name", THROUGH)
def test_stores_through_the_caches_keep_their_wait_states(kernels, name):
    """A 16-byte store's data registers must stay for two wait states
    (gfx950); the compiler does not see the store in the asm."""
    code = _kernel(kernels, name)
    stores = [i for i, op in enumerate(code) if re.match(r"global_store_dwordx4 .* sc0 sc1 nt", op)]
    assert stores
    for i in stores:
        assert code[i + 1] == "s_nop 1", code[i:i + 3]


@pytest.mark.parametrize("name", THROUGH)
def test_copy_loops_keep_their_chunks_in_flight(kernels, name):
    """A copy loop that stores through the caches issues its loads, waits once, and issues its stores: no wait
    for memory from a loop's first load to its last, nor from its first store
    to its last."""
    code = _kernel(kernels, name)
    unroll = 4 if name == "kvx_export_rows_small" else 8
    for kind in ("load", "store"):
        at = [i for i, op in enumerate(code) if op.startswith("global_{}_dwordx4".format(kind))]
        assert len(at) == unroll
        assert not [op for op in code[at[0]:at[-1]] if "vmcnt" in op]
