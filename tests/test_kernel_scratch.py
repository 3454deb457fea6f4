"""Kernels whose time a spill to scratch multiplies keep everything in registers, as
the compiler reports it.

The gridding adjoint: a reference to a kernel argument handed to a called function
copies all of it to every lane's private memory (230 us against 100 us for 500k
15 x 15 rows on a 4096 x 4096 grid).  The runtime-length FFT: addresses that do not
change from stage to stage are hoisted out of the loop over the stages and spilled
(1020 against 133 us for 16 images of 500 x 720)."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'faceted-hypersara_amd')


@pytest.mark.parametrize('source,kernels,count', [('gmat', 'adjoint_tiled', 4), ('data', 'adjoint_tiled', 4),
                                                  ('nufft', '_rt', 12)])
def test_no_scratch(source, kernels, count, tmp_path):
    spec = importlib.util.spec_from_file_location('fhs_build', os.path.join(PKG, 'build.py'))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)):
        pytest.skip('no hipcc')
    out = tmp_path / 'k.s'
    subprocess.run([build.HIPCC] + build.CFLAGS + ['-S', '--cuda-device-only', os.path.join(build.CSRC, source + '.hip'),
                                                   '-o', str(out)], check=True, capture_output=True)
    sizes = re.findall(r'\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)', out.read_text())
    found = {name: int(size) for name, size in sizes if kernels in name}
    assert len(found) == count, sizes
    assert not any(found.values()), found
