"""LDS that one wavefront's lanes write and others of it read: no instruction separates the two, so no run on the GPU can show
that the compiler was told to keep them in order. Read from the sources."""
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / 'fast_sp_gs_amd' / 'csrc'


@pytest.mark.parametrize('source,start,write,read', [
    ('block_lists.hpp', 'int build_block_lists(', 'fill[e + lane] =', 'if (on) lists['),
    ('block_lists.hpp', 'int build_block_lists(', 'if (on) lists[', 'return longest'),
    ('block_lists.hpp', 'int build_row_lists(', '((uint2*) lists)[lane] =', 'if (on) lists['),
    ('block_lists.hpp', 'int build_row_lists(', 'if (on) lists[', 'return longest'),
    ('gs3d_blend.hip', 'gs3d_backward_kernel(', 's_total[e][4 * h + c] =', 'float sum = s_total[e][c]'),
])
def test_lanes_exchange_in_order(source, start, write, read):
    text = (CSRC / source).read_text()
    body = text[text.index(start):]
    body = body[body.index(write):]
    between = body[:body.index(read)]
    assert 'wave_lds_sync();' in between
