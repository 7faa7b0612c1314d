"""What the built kernels ask of the chip, read from the library's own code objects, on the CPU."""
import os
import re
import shutil
import subprocess

import pytest

from inferx_amd.csrc import build

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(tmp_path):
    """Name of every kernel of the library -> bytes of scratch memory a lane."""
    with open(build.find_built() or build.build(verbose=False), "rb") as f:
        data = f.read()
    scratch, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:  # (one bundle a source file: a number of entries, each offset, size and the length of its name)
        number, p = int.from_bytes(data[at + 24:at + 32], "little"), at + 32
        for _ in range(number):
            offset, size, length = (int.from_bytes(data[p + 8 * i:p + 8 * i + 8], "little") for i in range(3))
            name, p = data[p + 24:p + 24 + length], p + 24 + length
            if b"gfx950" in name and size:
                obj = tmp_path / "code"
                obj.write_bytes(data[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for block in notes.split("- .agpr_count")[1:]:
                    scratch[re.search(r"\.symbol: +'?(\S+)\.kd", block).group(1)] = int(
                        re.search(r"\.private_segment_fixed_size: (\d+)", block).group(1))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)
    return scratch


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_the_products_kernels_keep_everything_in_registers(tmp_path):
    scratch = kernels(tmp_path)
    of = {n: b for n, b in scratch.items() if re.search("linear_tiled|moe_grouped_tiled|moe_grouped_mfma|moe_grouped_dual|linear_skinny|qkv_rope_skinny|heads_product|moe_grouped_queue", n)}
    assert len(of) > 40
    assert not any(of.values()), {n: b for n, b in of.items() if b}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("names,count", [("attn_prefill_keys", 1), ("latent_whole", 1), ("latent_attn_few", 3), ("latent_merge_product", 1),
                                         ("latent_prepare_product", 2), ("delta_chunks_|general_chunks_", 18)])
def test_kernels_of_counted_registers_keep_everything_in_them(tmp_path, names, count):
    """Those whose waits are counted by hand, or whose launch bounds give a lane just the registers that it needs."""
    of = {n: b for n, b in kernels(tmp_path).items() if re.search(names, n)}
    assert len(of) == count and not any(of.values()), of
