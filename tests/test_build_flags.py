"""The per-neutron build flags keep FP64 constants out of the sampling kernels'
registers and slow down the kernels that build tables with long FP64 loops: those
are in files without them."""
import re

from ncrystal_amd import build


def test_table_builders_without_per_neutron_flags():
    heavy = {"k_kb_bounds", "k_sab_analyse", "k_sab_derive", "k_vdos_fill"}
    where = {}
    for src in build.SOURCES:
        for k in re.findall(r"__global__[^;{]*?\b(k_\w+)\s*\(", (build.CSRC / src).read_text()):
            where[k] = src
    assert heavy <= set(where)
    assert not {k: where[k] for k in heavy if where[k] in build.PER_NEUTRON}
