"""Cache policies of the compiled kernels' loads and stores, read from this
build's own gfx950 code: a buffer access streams past the caches (nt), is
written through the L2 (sc1) or has the default policy (neither)."""
import re
import subprocess

import pytest

from fufft_amd import isa_report as R

pytestmark = pytest.mark.skipif(not R.tools_available() or not list(R.OBJ.glob("*.o")),
                                reason="needs this build's objects and the ROCm LLVM tools")


def policies(obj, workdir):
    """kernel name -> list of (opcode, policy) of its buffer accesses, in order"""
    text = subprocess.run([str(R.LLVM / "llvm-objdump"), "-d", "--no-show-raw-insn", str(R.code_object(obj, workdir))],
                          check=True, capture_output=True, text=True).stdout
    out, name = {}, None
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if m:
            name = m.group(1)
            out[name] = []
            continue
        m = re.search(r"\b(buffer_(?:load|store)_\w+) ([^/]*)", line)
        if m and name:
            mods = set(m.group(2).split()) & {"nt", "sc1"}
            out[name].append((m.group(1), "+".join(sorted(mods)) or "default"))
    return out


@pytest.fixture(scope="module")
def conv1d(tmp_path_factory):
    return policies(R.OBJ / "conv1d.o", tmp_path_factory.mktemp("co1"))


def kernel(n, v, kind, mid=0, layout=2):
    return f"_ZN5fufft13conv1d_kernelILi{n}ELi{v}ELi{layout}ELi{kind}ELi{mid}EEEvNS_12Conv1dParamsE"


def stores(accesses, width="dword"):
    return {p for op, p in accesses if op.startswith("buffer_store_" + width)}


@pytest.mark.parametrize("n,v,policy", [(256, 16, "default"), (512, 16, "nt"), (512, 8, "nt"), (4096, 16, "nt")])
def test_real_conv_streams_whole_lines_only(conv1d, n, v, policy):
    """At N = 256 sixteen lanes store 64 bytes of a real result at a time: half a
    line, which a streamed store sends out by itself."""
    assert stores(conv1d[kernel(n, v, 1)]) == {policy}


@pytest.mark.parametrize("n,v", [(256, 16), (512, 8), (1024, 16), (4096, 8), (4096, 16), (16384, 16)])
def test_c2c_results(conv1d, n, v):
    """Written through for the launch that reads them next, with kernels that
    stream for results the last-level cache cannot hold."""
    for kind, far in ((6, 17), (7, 18)):
        assert stores(conv1d[kernel(n, v, kind, mid=2)]) == {"sc1"}
        assert stores(conv1d[kernel(n, v, far, mid=2)]) == {"nt"}


def test_n16384_conv_results(conv1d):
    """As the C2C's; the signals are streamed in both."""
    for kind, policy in ((0, "nt"), (14, "sc1")):
        got = conv1d[kernel(16384, 16, kind)]
        assert stores(got) == {policy}
        assert sum(p == "nt" for op, p in got if op == "buffer_load_dwordx2") == 16


@pytest.mark.parametrize("n,v", [(256, 16), (512, 8), (1024, 16), (4096, 16), (4096, 8), (8192, 8), (16384, 16)])
def test_phase_timer_has_the_policies_of_the_conv(conv1d, n, v):
    """The timed kernel holds the loads and stores of both convs of the plan, the one
    for batches that the caches keep (K_CONV_NEAR) and the one for the others."""
    layout = 1 if (n, v) == (8192, 8) else 2
    conv, near, timed = (conv1d[kernel(n, v, k, layout=layout)] for k in (0, 14, 9))
    assert stores(timed, "dwordx2") == stores(conv, "dwordx2") | stores(near, "dwordx2")
    plain = sum(p == "default" for op, p in conv if op == "buffer_load_dwordx2")       # the twiddles
    for policy in ("nt", "default"):
        of = [sum(p == policy for op, p in k if op == "buffer_load_dwordx2") for k in (conv, near, timed)]
        assert of[2] == max(of[:2]), policy
    assert {sum(p == "default" for op, p in k if op == "buffer_load_dwordx2") for k in (conv, near)} == \
        ({plain} if n == 16384 else {plain, plain + v})


@pytest.mark.parametrize("h,w,policy", [(8, 64, "default"), (16, 64, "default"), (32, 64, "nt"), (64, 64, "nt"),
                                        (8, 32, "nt"), (8, 128, "nt"), (512, 16, "nt")])
def test_small_images_of_half_line_stores(tmp_path, h, w, policy):
    """Rows of 64 points are stored half a line at a time; images of few such rows
    leave the halves to the L2 to put together."""
    got = policies(R.OBJ / "conv2d.o", tmp_path)
    for mid in (0, 1, 2):
        name = f"_ZN5fufft14small2d_kernelILi{h}ELi{w}ELi{mid}EEEvNS_13Small2dParamsE"
        assert stores(got[name]) == {policy}
