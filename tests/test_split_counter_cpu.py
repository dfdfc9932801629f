"""The counter of a tile whose windows share its finishing (wq_gemm_stream.hip): what the built kernels do to it."""
import os
import re
import subprocess

import pytest

from tests.test_lds_requests_cpu import CSRC, listing


def shared_split_kernels(name, tmp_path):
    """{kernel: its instructions} of the builds of an object that split K over workgroups on tiles of 128 columns and 64 rows or more."""
    if not os.path.exists(os.path.join(CSRC, name)):
        subprocess.run(["make", "-C", CSRC, name], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    kernels, here = {}, None
    for line in listing(os.path.join(CSRC, name), tmp_path):
        label = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if label:
            shape = re.search(r"wq_gemm_stream_kernelILi\dELi(\d)ELi(\d)ELi(\d)E(?:Li\d+E){5}Lb[01]ELi1ELb[01]E", label[1])
            shares = shape and int(shape[1]) >= 2 and int(shape[2]) * int(shape[3]) == 4
            here = kernels.setdefault(label[1], []) if shares else None
        elif here is not None:
            here.append(re.sub(r"\s*//.*", "", line).strip())
    return kernels


@pytest.mark.parametrize("name", ["wq_gemm_stream4.o", "wq_gemm_stream8.o"])
def test_every_access_to_the_counter_but_its_return_to_zero_is_an_add(name, tmp_path):
    """Arrive, look, resign and account are each an add that returns what was there, so that all of them are in one order.  (A look
    that adds a zero which the compiler sees becomes a load.)  The two stores: the counter's return to zero, and the host's mark."""
    kernels = shared_split_kernels(name, tmp_path)
    assert len(kernels) == 6, "two tiles: tile-major, scales in pieces, scales by macro step"
    for kernel, code in kernels.items():
        accesses = [i.split()[0] for i in code if re.match(r"(global|flat)_", i)]
        assert sorted(accesses) == ["global_atomic_add"] * 4 + ["global_store_dword"] * 2, (kernel, accesses)
        assert all("sc0" in i for i in code if i.startswith("global_atomic_add")), kernel
