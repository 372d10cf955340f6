"""CPU checks of bench.py's byte model for plans whose inner products take the
outputs' row passes with them, at the benchmark shape, term by term."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

N, L, K, ALPHA, NP, B = 1 << 16, 24, 6, 6, 4, 64
T = 8 * N                                   # one tower
KEY = 2 * NP / B                            # key rows of a row, per op
FUSED = ["tensor_ib", "modup", "ksi", "moddown", "ksi"]


def steps(kinds, **kw):
    return {s[0]: s[1] for s in bench.step_bytes(N, L, K, ALPHA, NP, kinds, B, **kw)}


def test_last_step_forms_the_tensor_products():
    """The benchmark's plan: per op, the tensor step reads c1 of both factors and
    writes t2's row pass, but for the dropped tower, whose products are all
    stored; the last step reads the four input towers, three transformed
    digits, both ModDown towers and the key, and writes both outputs."""
    s = steps(FUSED)
    assert list(s) == ["tensor_intt_rowpass", "modup_fused", "rowpass_inner_p_drop", "moddown_fused", "rowpass_inner_q_final"]
    assert s["tensor_intt_rowpass"] == T * (23 * (2 + 1) + 4 + 3 + 1)
    assert s["rowpass_inner_q_final"] == pytest.approx(T * 23 * (3 + KEY + 4 + 2 + 2))
    # 6 P rows of four digits and two outputs; the dropped row with t0 and t1 in
    assert s["rowpass_inner_p_drop"] == pytest.approx(T * (6 * (4 + KEY + 2) + (3 + 1) + KEY + 2 + 2))
    # counted by the hardware on this plan (FETCH_SIZE and WRITE_SIZE, 64 ops):
    # 2.615e9, 1.538e9 and 8.855e9 bytes
    for name, seen in (("tensor_intt_rowpass", 2.615e9), ("rowpass_inner_p_drop", 1.538e9), ("rowpass_inner_q_final", 8.855e9)):
        assert 0.9 * seen < s[name] * B < 1.01 * seen, name


@pytest.mark.parametrize("kinds,kw", [(FUSED, dict(ksi_tensor=False)),
                                      (["tensor", "ntt_inv_b", "modup", "ksi", "moddown", "ksi"], {})])
def test_last_step_reads_the_tensor_products(kinds, kw):
    """With ksi_tensor or tensor_ib off the tensor step stores all three
    products of every row, and the last step reads them and not the inputs."""
    s = steps(kinds, **kw)
    assert sum(s[k] for k in s if k in ("tensor", "intt_modup_rowpass", "tensor_intt_rowpass")) == T * 24 * (4 + 3 + 1)
    assert s["rowpass_inner_q_final"] == pytest.approx(T * 23 * (3 + 1 + KEY + 2 + 2 + 2))
