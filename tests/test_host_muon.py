"""Muon's host-side rules: which calls share Gram matrices between iterations, and what they hold (no device work)."""
import pytest

from grokking_optimizers import _cabi


@pytest.mark.parametrize("count, m, n, ns", [
    (24, 1024, 1024, 5), (24, 1024, 1280, 5), (24, 768, 1152, 5), (48, 512, 1024, 5), (12, 1536, 1920, 5), (12, 1536, 2304, 5), (60, 400, 800, 5),
    (12, 1536, 2304, 3), (24, 256, 1024, 3), (6, 1024, 2048, 2), (2, 2048, 4096, 2), (6, 1024, 1536, 5), (2, 1024, 1536, 5), (1, 200, 800, 5)])
def test_one_gram_matrix_an_iteration_where_that_is_faster(count, m, n, ns):
    """Sets whose step took longer with shared Gram matrices (1 to 14 %) on the GPU."""
    assert _cabi.muon_stages_for([(m, n) if i % 2 == 0 else (n, m) for i in range(count)], ns) == ns


@pytest.mark.parametrize("count, m, n", [(24, 1024, 4096), (24, 1024, 2048), (12, 1536, 3072), (16, 512, 2048), (12, 300, 1200), (2, 1024, 4096), (1, 200, 4000)])
def test_shared_gram_matrices_where_that_is_faster(count, m, n):
    """... and shorter by 7 to 25 %."""
    assert _cabi.muon_stages_for([(m, n)] * count, 5) == 2


@pytest.mark.parametrize("count, m, n, squares", [(24, 1024, 1024, 2), (3, 512, 768, 2), (24, 1024, 4096, 5)])
def test_workspace_holds_what_the_call_can_use(count, m, n, squares):
    """Two iterates, and the m x m matrices: five where iterations can share a Gram matrix, two where none does."""
    shapes = [(m, n)] * count
    assert {_cabi.muon_stages_for(shapes, ns) < ns for ns in (3, 6, 9)} == {squares == 5}
    transposes = 2 if count == 3 else 0             # kept for the apply step on 64x64 tiles
    held = 2 * count * m * ((2 + transposes) * n + squares * m)
    assert held <= _cabi.muon_workspace_bytes(shapes) <= held + 65536 + count * m * n // 512


def test_sharing_is_likeliest_at_three_iterations():
    """The workspace is laid out by that, whatever ns_steps the call has."""
    for count, m, r in [(c, m, r) for c in (1, 3, 8, 24, 60) for m in (130, 260, 500, 1000, 2000) for r in (1, 1.3, 1.6, 2, 3, 5)]:
        shapes = [(m, int(m * r))] * count
        if _cabi.muon_stages_for(shapes, 3) == 3:
            assert all(_cabi.muon_stages_for(shapes, ns) == ns for ns in (1, 2, 4, 5, 6, 9, 12, 1000)), shapes
