"""Recurrences over runs in chunks, several tiles of value columns a workgroup (so many heads that the columns are taken together): columns that end inside a tile,
tiles without columns, more than one workgroup a head."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,dk,dv,taps,ng", [(768, 1, 128, 33, 2, 1), (768, 2, 64, 48, 2, 1), (512, 1, 40, 65, 2, 2), (512, 2, 16, 100, 2, 1), (1200, 1, 100, 31, 2, 1)])
def test_any_cutting(H, G, dk, dv, taps, ng):
    import test_gpu_lelatar as lelatar

    for dtype in lelatar.DTYPES:
        lelatar.test_the_recurrence_carries_state_and_inputs_through_any_cutting(dtype, "ssd", H, G, dk, dv, taps, ng)


@pytest.mark.parametrize("lengths", [[1] * 31 + [130], [1, 70, 1, 1, 2, 130, 1, 64, 65, 1], [3, 1, 1, 66] + [1] * 300 + [2, 1, 90]])
@pytest.mark.parametrize("H", [3, 640])
def test_long_runs_among_single_tokens(H, lengths):
    """Runs of several tokens are taken ahead of those of one, wherever they stand, tokens of nobody between them; every run is taken once."""
    import torch

    import test_gpu_lelatar as lelatar

    if H > 3 and len(lengths) > 40:
        lengths = lengths[:40]
    for dtype in lelatar.DTYPES if H == 3 else [torch.bfloat16]:
        case = lelatar.Case("ssd", H, 1, 24, 40, 2, lengths, len(lengths) + H, dtype)
        state = case.state(len(lengths))
        rows, slots, positions, places = [], [], [], []
        for i, (n, seq) in enumerate(zip(lengths, case.seqs)):
            r = case.rows(seq)
            if i % 5 == 2:  # a token of nobody
                rows.append(r[:1]), slots.append(-1), positions.append(0)
            places.append(len(slots))
            rows.append(r)
            slots += [len(lengths) - 1 - i] * n
            positions += range(n)
        out = case.run(torch.cat(rows), slots, positions, state, len(lengths) + 4)
        want = [case.plain(seq) for seq in case.seqs]
        lelatar.check_rows(torch.cat([out[at:at + n] for at, n in zip(places, lengths)]), torch.cat([w for w, _ in want]), dtype)
        for i, (_, S) in enumerate(want):
            err = (case.matrices(state, len(lengths) - 1 - i).cpu().double() - S).abs().max() / S.abs().max().clamp(min=1e-3)
            assert float(err) < (1e-4 if dtype == torch.float32 else 1e-2), (i, float(err))
        assert all(float(out[t].abs().max()) == 0.0 for t, s in enumerate(slots) if s < 0)
