"""The build refuses kernels that count their vector-memory waits by hand and keep registers in scratch memory: which kernels those are is
read from the sources here, and the check itself from remarks made up for it."""
import glob
import importlib.util
import os
import re

import pytest

ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vla.cpp_amd")
spec = importlib.util.spec_from_file_location("vla_build", os.path.join(ROOT, "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)


def device_functions(path):
    """(is a kernel, name, text) of every function of a source that runs on the device."""
    with open(path) as f:
        text = f.read()
    heads = list(re.finditer(r"^(__global__|__device__)[^\n]*?(\w+)\((?:[^()]|\([^()]*\))*\)\s*\{", text, re.M))
    for h, after in zip(heads, heads[1:] + [None]):
        yield h.group(1) == "__global__", h.group(2), text[h.end():after.start() if after else len(text)]


def counts_its_waits(body):
    return bool(re.search(r"wait_(vmcnt|vm_mem|tiles)<", body) and re.search(r"load_to_lds16|dma16\(|tern_aload_lds\(|tern_wload", body))


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(ROOT, "csrc", "*.hip"))), ids=os.path.basename)
def test_kernels_with_counted_waits_are_listed(path):
    listed = build.NO_SPILL_KERNELS.get(os.path.basename(path), {})
    functions = list(device_functions(path))
    helpers = {name for kernel, name, body in functions if not kernel and counts_its_waits(body)}
    for kernel, name, body in functions:
        if kernel and (counts_its_waits(body) or any(h + "(" in body or h + "<" in body for h in helpers)):
            assert name in listed, name


def test_the_sources_are_read():
    found = {name for _, name, body in device_functions(os.path.join(ROOT, "csrc", "attention.hip")) if counts_its_waits(body)}
    assert {"attn_kernel", "attn_stream_kernel", "attn_tiles_kernel", "attn_rows_kernel", "attn_wide_kernel"} <= found


def remarks(*kernels):
    return "".join("x.hip:1:1: remark: Function Name: %s [-R]\nx.hip:1:1: remark:     ScratchSize [bytes/lane]: %d [-R]\n" % k for k in kernels)


def test_direct_to_lds_attention_may_not_spill():
    others = [(k, 0) for k in build.NO_SPILL_KERNELS["attention.hip"] if k != "attn_kernel"]
    staged, ring = "_ZN1_11attn_kernelItLi64ELi1ELb1ELi0ELi0ELi1EEEvNS_8AttnArgsE", "_ZN1_11attn_kernelItLi128ELi4ELb0ELi0ELi1ELi2EEEvNS_8AttnArgsE"
    build._check_no_spill("attention.hip", remarks((staged, 140), (ring, 0), *others))
    with pytest.raises(RuntimeError, match="spills 12 bytes"):
        build._check_no_spill("attention.hip", remarks((staged, 140), (ring, 12), *others))
    with pytest.raises(RuntimeError, match="no resource remarks for attn_kernel"):
        build._check_no_spill("attention.hip", remarks((staged, 140), *others))
