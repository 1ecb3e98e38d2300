"""Where fp32 rows are cut into parts of their keys, and where a workgroup of matrix instructions walks them."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S


class _Seg:
    def __init__(self, rows, before):
        self.row0_host, self.pos0_host = [0, rows], [before]


@pytest.mark.parametrize("rows,before,tiles,parts", [(128, 22, False, 2), (128, 22, True, 0), (127, 23, True, 2), (255, 1, True, 0),
                                                     (255, 2, True, 3), (128, 172, True, 3), (256, 600, False, 0), (100, 0, False, 0)])
def test_parts(rows, before, tiles, parts):
    got = S._rows_parts(_Seg(rows, before), rows, 16, 8, 128, torch.device("cpu"), tiles=tiles)
    assert got[0] == parts and all((t is None) == (parts == 0) for t in got[1:])
