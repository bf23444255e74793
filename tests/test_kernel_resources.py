"""What the compiler notes in the built hybrid library: no kernel of the prefill keeps registers in memory (a spilled accumulator costs more than what it was
spilled for), and none takes more LDS than a workgroup may have."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from conftest import ROOT

LIBRARY = ROOT / "qimeng-megakernel_amd" / "libqmk_hybrid.so"
DECODE = ROOT / "qimeng-megakernel_amd" / "libqmk_hip.so"
READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")


def device_code(data):
    """The gfx950 code objects among the bundles a library holds."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for found in re.finditer(re.escape(magic), data):
        at = found.start() + len(magic)
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24 : at + 24 + length]
            at += 24 + length
            if b"gfx950" in target and size:
                yield data[found.start() + offset : found.start() + offset + size]


def notes_of(library, tmp_path):
    if not library.is_file() or not READELF.is_file():
        pytest.skip("needs the built library and llvm-readelf")
    kernels = {}
    for i, code in enumerate(device_code(library.read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True, check=True).stdout
        for entry in notes.split(".agpr_count:")[1:]:
            field = dict(re.findall(r"\.(\w+):\s+(\S+)", entry))
            kernels[field["symbol"]] = field
    return kernels


def test_no_prefill_kernel_spills(tmp_path):
    kernels = notes_of(LIBRARY, tmp_path)
    assert any("gemm_direct" in name for name in kernels) and any("window_attention" in name for name in kernels) and any("attention_rows" in name for name in kernels)
    prefill = {name: k for name, k in kernels.items() if "decode_megakernel" not in name}
    spilled = {name: k["vgpr_spill_count"] for name, k in prefill.items() if int(k["vgpr_spill_count"])}
    assert not spilled, spilled
    assert all(int(k["group_segment_fixed_size"]) <= 160 * 1024 for k in prefill.values())


def test_tiles_engine_kernels(tmp_path):
    """Two and four tiles of keys ahead are kernels of their own for heads of 64 (one for both is slower in either), and none keeps registers in memory."""
    kernels = {name: k for name, k in notes_of(DECODE, tmp_path).items() if "decode_megakernel_batch" in name}
    found = sorted(re.search(r"batchINS_\d+(\w+?)ELi(\d)EE", name).groups() for name in kernels)
    assert found == [("Llama1B", "2"), ("Llama1B", "4"), ("Qwen3_1p7B", "4")]
    assert not any(int(k["vgpr_spill_count"]) for k in kernels.values())


def test_largest_heads_of_a_delta_rule(tmp_path):
    """Of the preparation of its chunks three workgroups of four waves share a CU: 512 registers a SIMD."""
    (kernel,) = [k for name, k in notes_of(LIBRARY, tmp_path).items() if "chunk_prepareILi1ELi4E" in name]
    assert int(kernel["vgpr_count"]) <= 168 and 3 * int(kernel["group_segment_fixed_size"]) <= 160 * 1024
