"""LayerNorm-modulation at the widths and shift options whose kernels the
general test does not reach: each side of the 3072 and 4096 lines, ragged
last chunks."""
import pytest

import test_gpu_kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,shift", [(3072, False), (3080, True), (3064, True), (4096, True),
                                         (4088, False), (8, True), (4104, False)])
def test_layer_norm_mod_widths(gpu, qd, oracle, width, shift):
    K.test_layer_norm_mod(gpu, qd, oracle, width, shift)
