"""Front end at every length it takes, 2 .. 2^18 and 2^22: each pair of row and column transforms, the one-row
form and the radix-2 one, with the bins that mirror themselves (0, N/2) and the rows around them.  White noise
has the same power in every bin, so a misplaced bin or sign stands out by its full size: each bin's error is at
most 2e-6 of the RMS (an FP32 transform of these lengths errs by 1.1 .. 1.7e-7 RMS, 5 sigma of it stay below 1e-6).
"""

import numpy as np
import pytest

from fdas_amd.io import FrontEnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2n", [*range(1, 19), 22])
def test_every_bin_of_every_length(log2n):
    torch = pytest.importorskip("torch")
    n = 1 << log2n
    s = torch.randn(2 * n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(log2n))
    out = torch.zeros(n, dtype=torch.complex64, device="cuda")
    with FrontEnd(n) as fe:
        torch.cuda.synchronize()
        fe.run(s, out=out)
        fe.run(s.cpu().numpy())  # host input and output of the same length
    ref = torch.fft.fft(s.double())[:n] / (2 * n)
    err = (out.to(torch.complex128) - ref).abs().cpu().numpy()
    rms = float(ref.abs().square().mean().sqrt())
    assert err.max() <= 2e-6 * rms, f"bin {int(np.argmax(err))}"
