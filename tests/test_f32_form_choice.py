"""Which form an fp32 launch takes by itself: 128 rows per workgroup, or 32 rows whose wavefronts share the walk.  Each row is a launch
that was timed in both forms on the GPU (us, in the comments); the slower one must not be taken."""
import pytest

from simt import simt as S

FORWARD, BACKWARD, DENSE, RAGGED = 0, 1, 0, 1
# direction, d, causal, kind, B, longest N, H, H_kv -> 32 rows?                          128 rows   32 rows
TIMED = [
    (FORWARD, 64, True, DENSE, 2, 512, 8, 8, True),         # 38.7       14.8
    (FORWARD, 64, False, DENSE, 1, 2048, 16, 16, False),    # 139        176
    (FORWARD, 128, False, DENSE, 2, 512, 8, 8, True),       # 68.5       27.2
    (FORWARD, 64, True, DENSE, 6, 376, 24, 24, False),      # 47         65
    (FORWARD, 128, True, DENSE, 2, 1106, 32, 32, False),    # 224        277
    (FORWARD, 128, True, DENSE, 1, 16, 8, 8, False),        # 8.1        13.8
    (FORWARD, 64, True, RAGGED, 4, 48, 8, 8, False),        # 8.0        8.6
    (FORWARD, 64, False, DENSE, 1, 64, 8, 8, True),         # 8.3        7.5
    (BACKWARD, 128, False, DENSE, 4, 16, 8, 8, False),      # 40         51
    (BACKWARD, 128, False, DENSE, 4, 32, 8, 8, True),       # 41         37
    (BACKWARD, 64, True, DENSE, 1, 2048, 16, 16, True),     # 807        436
    (BACKWARD, 128, False, DENSE, 2, 2048, 16, 16, False),  # 2594       2813
    (BACKWARD, 64, False, DENSE, 1, 2048, 16, 4, True),     # 1817       738
    (FORWARD, 64, False, RAGGED, 1, 4096, 16, 16, False),   # 508        680
    (FORWARD, 64, False, RAGGED, 4, 1024, 16, 16, False),   # 134        175
    (FORWARD, 64, True, RAGGED, 4, 1024, 8, 8, True),       # 74         70
    (FORWARD, 128, False, RAGGED, 24, 240, 16, 16, False),  # 94         219
    (FORWARD, 128, True, RAGGED, 24, 240, 16, 16, False),   # 96         177
    (FORWARD, 128, True, RAGGED, 4, 512, 16, 16, False),    # 72         86
    (FORWARD, 128, True, RAGGED, 2, 2048, 8, 8, True),      # 261        190
    (BACKWARD, 128, False, RAGGED, 24, 240, 16, 16, False),  # 499        775
    (BACKWARD, 64, False, RAGGED, 12, 512, 16, 16, False),  # 561        656
    (BACKWARD, 64, True, RAGGED, 8, 904, 8, 8, True),       # 417        201
    (BACKWARD, 128, True, RAGGED, 4, 1024, 8, 2, True),     # 1885       574
    (BACKWARD, 128, False, RAGGED, 9, 1024, 16, 16, False),  # 3135       3536
    (BACKWARD, 128, True, RAGGED, 25, 512, 12, 12, False),  # 1327       1788
    (BACKWARD, 128, False, RAGGED, 11, 264, 24, 12, False),  # 482        628
]


@pytest.mark.parametrize("backward,d,causal,ragged,B,N,H,H_kv,rows_32", TIMED)
def test_the_faster_form_is_taken(backward, d, causal, ragged, B, N, H, H_kv, rows_32):
    assert bool(S.load().simt_f32_split(backward, d, int(causal), ragged, B, N, H, H_kv)) == rows_32
