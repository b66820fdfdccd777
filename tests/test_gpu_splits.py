"""Suggested split counts against what the built split kernels hold: a single
long head is cut into as many splits as stay resident on the GPU, from the
registers and LDS in the kernels' metadata."""
import re

import pytest

import kvexp_amd
from test_registers import code_objects, kernel_metadata

pytestmark = pytest.mark.gpu

LDS_PER_CU = 160 * 1024


def resident_per_cu():
    """(head_dim, query rows) -> resident XKV splits per CU (the fewer of the two orders')."""
    msgpack = pytest.importorskip("msgpack")
    with open(kvexp_amd.LIB_PATH, "rb") as f:
        data = f.read()
    out = {}
    for elf in code_objects(data):
        for k in kernel_metadata(elf, msgpack):
            m = re.search(r"attn_(team|wave)_kernelILi(\d+)ELi(\d+)ELb1ELi\dE", k[".name"])
            if m is None:
                continue
            rows, dim = int(m.group(2)), int(m.group(3))
            waves_per_wg = k[".max_flat_workgroup_size"] // 64
            splits_per_wg = waves_per_wg if m.group(1) == "wave" else 1
            waves = min(8, 512 // ((k[".vgpr_count"] + 7) // 8 * 8)) * 4
            wgs = min(waves // waves_per_wg, LDS_PER_CU // k[".group_segment_fixed_size"])
            out[dim, rows] = min(out.get((dim, rows), 1 << 30), wgs * splits_per_wg)
    return out


def test_suggested_splits_fill_one_round():
    import torch

    ctx = kvexp_amd.Context(0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = 8192  # more than any resident count
    resident = resident_per_cu()
    assert {d for d, _ in resident} == {32, 64, 80, 96, 112, 128, 160, 192, 224, 256}
    got = {key: ctx.suggest_splits(1, tiles * 128, 128, key[0], key[1]) for key in resident}
    assert got == {key: n * cus for key, n in resident.items()}
