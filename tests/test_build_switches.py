"""The kernels hold one variant of themselves: no macro that a build can set chooses batch lengths, lanes per list or paddings, which
other kernels rely on (a forward with other blocks than the backward reads would give wrong gradients without an error)."""
import re
from pathlib import Path

PKG = Path(__file__).resolve().parents[1] / 'fast_sp_gs_amd'


def test_no_macro_selects_a_variant():
    sources = [*PKG.glob('csrc/*.hip'), *PKG.glob('csrc/*.hpp'), *PKG.glob('csrc/host/*')]
    assert len(sources) > 30
    found = {p.name: re.findall(r'^\s*#\s*(?:ifn?def|if|elif)\b.*\bFSGS_\w+', p.read_text(), re.M) for p in sources}
    assert not {k: v for k, v in found.items() if v}
    assert 'DEFINES' not in (PKG / 'build.py').read_text()
