"""Kernels that no launch can reach are not in the library."""
import re

from test_code_object import kernels  # noqa: F401  (fixture)

# lindblad_rk4_resident<NB, W, BPW, MINW, DENSE, REC, BRD, DB>
NAME = re.compile(r"lindblad_rk4_residentILi(\d)ELi(\d+)ELi(\d)ELi(\d)ELb(\d)ELb(\d)ELb(\d)ELb(\d)E")


def test_shapes_that_other_kernels_took_over_are_gone(kernels):  # noqa: F811
    found = [tuple(map(int, m.groups())) for m in (NAME.search(k[".name"]) for k in kernels) if m]
    assert found
    for nb, w, bpw, _, dense, rec, brd, db in found:
        assert not (dense and bpw == 1), "lindblad_rk4_resident_ops runs these"
        built_in = not dense and not brd and db and nb >= 2 and (bpw == 1 or nb == 5)
        # two tiles a wave without records: the odd lengths still run here
        assert not built_in or (bpw == 2 and not rec), (nb, w, bpw, rec)
