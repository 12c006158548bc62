"""The causal convolution over prompts at the sizes where its rows a thread change (4, 8, 12, 16, 32), with sequences shorter than the window and
portions that end inside a thread's rows; kept inputs are copied, so they are exact."""
import pytest
import torch

from msa_amd import seq_ops
from oracle import recurrent_layers as R
from seq_helpers import BF16, F32, F64, Rand, batch, close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,C,counts", [(5, 8, [4, 1, 5, 3, 9]), (2, 4096, [505, 7]), (4, 4096, [2, 515]), (5, 4096, [1000, 3, 25]), (3, 4096, [1, 1100]),
                                        (4, 4096, [4000, 90, 6]), (5, 8192, [3, 1, 2050]), (4, 8192, [4080, 21])])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_portions(dtype, K, C, counts):
    r = Rand(C + K)
    T, slots = sum(counts), [2 * i + 1 for i in range(len(counts))]
    (x, x_), (taps, taps_), (b, b_), (state, state_) = r(T, C + 16, dtype=dtype), r(C, K), r(C), r(2 * len(counts) + 1, K - 1, C)
    if dtype == BF16:                                        # kept inputs are inputs
        state_ = state_.to(BF16).to(F64)
        state.copy_(state_)
    got = seq_ops.conv_silu(x[:, 8:8 + C], taps, b, state, batch(counts, slots))
    at = 0
    for n, s in zip(counts, slots):
        seen = torch.cat([state_[s], x_[at:at + n, 8:8 + C]])
        close(got[at:at + n], R.silu(R.causal_conv(seen, taps_, b_))[K - 1:], dtype)
        state_[s] = seen[-(K - 1):]
        at += n
    assert torch.equal(state.cpu().to(F64), state_)
