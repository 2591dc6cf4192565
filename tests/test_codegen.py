"""What the compiler has to keep in the gfx950 code of the kernels, read from the assembly that the build's own flags give.
No GPU is needed."""
import os
import re
import subprocess

import pytest

from kerops_amd import build


@pytest.fixture(scope='module')
def stream_ops(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip('no hipcc')
    out = tmp_path_factory.mktemp('asm') / 'stream_ops.s'
    subprocess.run([build.HIPCC, *build.COMMON_FLAGS, '--offload-device-only', '-S',
                    os.path.join(build.CSRC, 'stream_ops.hip'), '-o', str(out)], check=True, capture_output=True)
    return out.read_text()


def longest_run_of_loads(body):
    """Most global loads that are issued with no store, wait or branch between them."""
    best = run = 0
    for line in body.splitlines():
        op = line.split()[0] if line.split() else ''
        if op.startswith('global_load'):
            run += 1
            best = max(best, run)
        elif op.startswith(('global_store', 's_cbranch')) or (op == 's_waitcnt' and 'vmcnt' in line):
            run = 0
    return best


def test_window_quantisers_issue_their_loads_together(stream_ops):
    # a streaming kernel of few wavefronts is as fast as the loads it has in flight: all U of a step, not one at a time
    names = re.findall(r'^(_ZN6kerops\d+(?:de)?quant_u8_kernelI\S*):', stream_ops, re.M)
    assert len(names) == 3 * 2 * 4 + 3 * 2 * 2  # type x unroll x (window form, store hint); the inverse has one form
    for name in names:
        unroll = int(re.search(r'Li(\d+)E', name).group(1))
        body = stream_ops[stream_ops.index(f'\n{name}:'):]
        assert longest_run_of_loads(body[:body.index('s_endpgm')]) >= unroll, name
