"""A recurrence's step in the launch of the other branch's convolution: the same bits as two launches."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# heads of 64 and 128 and states of one and two registers' width share the launch; heads of 32, key heads of 192 and 32 bits take two
@pytest.mark.parametrize("n, dtype, hd, d, dv, taps", [(1, torch.bfloat16, 64, 64, 128, 4), (3, torch.bfloat16, 128, 64, 96, 4), (65, torch.bfloat16, 64, 128, 64, 2),
                                                       (2, torch.bfloat16, 128, 100, 130, 1), (3, torch.bfloat16, 32, 64, 64, 4),
                                                       (2, torch.bfloat16, 64, 192, 32, 3), (2, torch.float32, 64, 64, 64, 4)])
def test_both_branches_of_single_tokens_in_one_launch(n, dtype, hd, d, dv, taps):
    from kestrel_amd.ops import core

    gen = torch.Generator().manual_seed(n + hd + d)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    Hq, Hk, H, rank, page = 4, 2, 3, 40, 16
    C = (Hq + 2 * Hk) * hd
    width = H * (2 * d + 2 * dv) + rank
    projected = rnd(n, C + (-C) % 8 + width + (-width) % 8).to(dtype).to(DEV)
    u, row = projected[:, :C], projected[:, C + (-C) % 8:C + (-C) % 8 + width]
    offsets = (0, H * d, 2 * H * d, 2 * H * d + H * dv, 2 * H * (d + dv))
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)  # noqa: E731
    row_slot = ints([r + 1 if r != 1 else -1 for r in range(n)])
    places = (ints(range(n + 1)), row_slot, ints(range(n)), ints([5 + 3 * r for r in range(n)]), ints([page * (r + 1) + r % page if r != 1 else -1 for r in range(n)]))
    conv_taps, freqs = rnd(C, taps).to(DEV), (rnd(hd // 2).abs() * 0.1).to(DEV)
    a2, bias, gain = (rnd(H * d, rank) * 0.2).to(dtype).to(DEV), rnd(H * d).to(DEV), rnd(dv).to(DEV)
    conv_state, state = rnd(n + 2, taps - 1, C).to(DEV) if taps > 1 else None, rnd(n + 2, H * dv * d).to(DEV)

    def results(together):
        mine = conv_state.clone() if conv_state is not None else None
        S, q = state.clone(), torch.full((n, Hq * hd), 7.0, dtype=dtype, device=DEV)
        k, v = (torch.zeros(n + 2, Hk, *shape, dtype=dtype, device=DEV) for shape in ((page, hd), (hd, page)))
        out = torch.full((n, H * dv + 8), 7.0, dtype=dtype, device=DEV)[:, :H * dv]
        step = (row, offsets, a2, bias, gain, 16.0, d ** -0.5, 1e-5, S, row_slot, out, H, d, dv)
        job = core.gated_step(*step, later=True) if together else None
        core.conv_prepare(u, conv_taps, mine, *places, q, k, v, Hq, Hk, hd, Hk, hd, page, freqs, single_tokens=True, beside=job)
        if not together:
            assert core.gated_step(*step)
        return [t for t in (q, k, v, mine, S, out) if t is not None]

    for a, b in zip(results(True), results(False)):
        assert torch.equal(a, b)


def test_a_step_beside_it_is_of_the_same_tokens():
    from kestrel_amd.ops import core

    z = lambda *shape, dtype=torch.bfloat16: torch.zeros(*shape, dtype=dtype, device=DEV)  # noqa: E731
    f32, i32 = torch.float32, torch.int32
    job = core.gated_step(z(2, 400), (0, 64, 128, 192, 256), z(64, 16), z(64, dtype=f32), z(64, dtype=f32), 16.0, 1.0, 1e-5, z(3, 4096, dtype=f32),
                          z(2, dtype=i32), z(2, 64), 1, 64, 64, later=True)
    with pytest.raises(core.KernelError, match="same single tokens"):
        core.conv_prepare(z(1, 192), z(192, 1, dtype=f32), None, z(2, dtype=i32), z(1, dtype=i32), z(1, dtype=i32), z(1, dtype=i32), None, z(1, 64), None, None,
                          1, 1, 64, 1, 64, 16, single_tokens=True, beside=job)
