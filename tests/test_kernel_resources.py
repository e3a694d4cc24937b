"""The search kernel's memory, from the code that hipcc makes of its source
for gfx950 (CPU only: hipcc cross-compiles).  ft_search_noalloc launches it
and allocates nothing, so no instantiation that is launched may need scratch
memory, which the runtime allocates for a launch that asks for more than it
holds."""

import os
import re
import shutil
import subprocess

import pytest
import yaml

import build as ftbuild  # flash-trie_amd/build.py


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(louds, streamed, lean): the instantiation's metadata}"""
    if not (os.path.exists(ftbuild.HIPCC) or shutil.which("hipcc")):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("kernel") / "k.s"
    subprocess.run([ftbuild.HIPCC] + ftbuild.HIP_FLAGS +
                   ["-x", "hip", "--offload-device-only", "-S", "-o", str(out),
                    os.path.join(ftbuild.CSRC, "tbs_kernel.hip")],
                   check=True, capture_output=True, text=True)
    text = out.read_text()
    meta = re.search(r"\.amdgpu_metadata\n(.*?)\n\s*\.end_amdgpu_metadata", text, re.S).group(1)
    found = {}
    for k in yaml.safe_load(meta)["amdhsa.kernels"]:
        m = re.search(r"10tbs_kernelILb(\d)ELb(\d)ELb(\d)E", k[".name"])
        if m:
            found[tuple(int(x) for x in m.groups())] = k
    return found


# (the LOUDS instantiation is never launched: ft_create refuses its index)
@pytest.mark.parametrize("streamed", [0, 1])
@pytest.mark.parametrize("lean", [0, 1])
def test_no_scratch(kernels, streamed, lean):
    k = kernels[0, streamed, lean]
    assert k[".private_segment_fixed_size"] == 0, k
    assert k[".vgpr_spill_count"] == 0, k
    assert not k.get(".uses_dynamic_stack", False), k


@pytest.mark.parametrize("streamed", [0, 1])
def test_general_holds_nothing_of_the_lean_one(kernels, streamed):
    """The row's token bits (4 KB) are the lean instantiation's alone."""
    general, lean = (kernels[0, streamed, x][".group_segment_fixed_size"] for x in (0, 1))
    assert general + 4096 <= lean <= 160 * 1024
