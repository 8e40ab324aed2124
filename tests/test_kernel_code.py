"""What the compiler made of the kernels whose occupancy or ordering the results and timings rely on, from one
device-only compile to assembly of each source (no GPU needed): registers, scratch and the ordering points that stay
in the listing as comments."""
import os
import re
import subprocess
from collections import namedtuple

import pytest

from veymoe import build

Kernel = namedtuple("Kernel", "vgprs scratch sgpr_spills wave_barriers")
SOURCES = ("grouped.hip", "decode.hip", "glue.hip")
_COMPILED = {}


def _listing(proc, listing):
    """Kernel by mangled name of one finished compile."""
    _, err = proc.communicate()
    assert proc.returncode == 0, err[-2000:]
    text = listing.read_text()
    meta = {m.group(1): m.group(0) for m in re.finditer(r"\.amdhsa_kernel (\S+)\n.*?\.end_amdhsa_kernel", text, re.S)}
    spills = dict(re.findall(r"\.name: +(\S+)\n(?:    \..*\n)*?    \.sgpr_spill_count: (\d+)", text))
    found = {}
    for m in re.finditer(r"^(_Z\S+):.*?^\.Lfunc_end\d+:", text, re.M | re.S):
        name = m.group(1)
        if name not in meta:
            continue
        value = lambda key: int(re.search(rf"\.amdhsa_{key} (\d+)", meta[name]).group(1))
        found[name] = Kernel(value("next_free_vgpr"), value("private_segment_fixed_size"), int(spills[name]),
                             m.group(0).count("; wave barrier"))
    return found


def _kernels(source, tmp_path_factory):
    """Kernel by mangled name for one file of csrc; the files are compiled once, side by side."""
    if not _COMPILED:
        try:
            hipcc = build.hipcc()
        except RuntimeError:
            pytest.skip("hipcc is not installed")
        path = tmp_path_factory.mktemp("listings")
        jobs = {}
        for name in SOURCES:
            out = path / f"{name}.s"
            cmd = [hipcc, *build.HIP_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, name), "-o", str(out)]
            jobs[name] = subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True), out
        _COMPILED.update({name: _listing(*job) for name, job in jobs.items()})
    return _COMPILED[source]


def _instances(kernels, prefix):
    found = {name: k for name, k in kernels.items() if prefix in name}
    assert found, f"no kernel matching {prefix}"
    return found


def test_down_rows_keeps_the_order_of_its_strips(tmp_path_factory):
    """k_down_rows passes each column block's scales through one strip of LDS per wave: stores, then reads by other
    lanes, then the next block's stores.  Both orders are points the compiler may not move LDS accesses across: with
    SPB column blocks, 2 SPB - 1 of them in each of the three tile heights' code.  Two blocks of eight waves per CU
    (four waves per SIMD) take at most 128 registers."""
    kernels = _instances(_kernels("grouped.hip", tmp_path_factory), "k_down_rowsILi")
    for name, k in kernels.items():
        blocks = int(re.search(r"k_down_rowsILi\d+ELi8ELi(\d+)E", name).group(1))
        assert k.wave_barriers == 3 * (2 * blocks - 1), (name, k)
        assert k.vgprs <= 128 and k.scratch == 0, (name, k)


def test_decode_kernels_take_no_scratch(tmp_path_factory):
    """No decode GEMV has a scratch frame, whatever the compiler keeps in it."""
    kernels = _kernels("decode.hip", tmp_path_factory)
    for name, k in {**_instances(kernels, "k_gateupINS_"), **_instances(kernels, "k_downINS_")}.items():
        assert k.scratch == 0, (name, k)


def test_float32_gateup_keeps_its_scalars(tmp_path_factory):
    """The fp32 gate/up of several groups per lane, whose row index in a scalar had cost 180 spills to VGPR lanes."""
    found = {name: k for name, k in _instances(_kernels("decode.hip", tmp_path_factory), "k_gateupINS_6ActF32E").items()
             if "ELi64ELi2E" in name or "ELi64ELi4E" in name}
    assert found
    for name, k in found.items():
        assert k.sgpr_spills <= 40, (name, k)


def test_folded_down_runs_two_blocks_per_cu(tmp_path_factory):
    """The bf16 down kernel of rows a quarter over a power of two: two blocks of twelve waves per CU, six waves per
    SIMD, take at most 80 registers each."""
    for name, k in _instances(_kernels("decode.hip", tmp_path_factory), "k_downINS_7ActBF16E").items():
        if "ELb0ELi4ELi4E" in name:  # no injection, folded, four row groups
            assert k.vgprs <= 80, (name, k)


def test_hyper_connection_tiles_register_budgets(tmp_path_factory):
    """k_hc_low runs three blocks of four waves per CU (at most 168 registers), k_hc_mix four for up to four streams
    (128), else three; none spills."""
    kernels = _kernels("glue.hip", tmp_path_factory)
    for name, k in {**_instances(kernels, "k_hc_lowE"), **_instances(kernels, "k_hc_mixILb")}.items():
        limit = 128 if "k_hc_mixILb1ELi4E" in name else 168
        assert k.vgprs <= limit and k.scratch == 0, (name, k)
