"""The decode reader cuts a batch into slots of about equal length: batches at
the edges of that rule (one slot each, two combine levels, more sequences than
a wave has lanes or than the GPU has compute units), small workspaces, and
workspaces that hold anything, against the float64 oracle (tolerance: close()
of test_gpu_decode)."""
import numpy as np
import pytest

import pbe_handoff as P
from tests.conftest import say
from tests.gpu_util import stream_ptr
from tests.test_gpu_decode import DecodeCase, close

pytestmark = pytest.mark.gpu


def _mixed(n, most, seed):
    r = np.random.default_rng(seed)
    lens = [int(x) for x in np.exp(r.uniform(0, np.log(most), n))]
    lens[0], lens[-1] = most, lens[-1] if n == 1 else 0
    return lens


BATCHES = {
    "one_slot_each": [16 * 16] * 3 + [1, 0],
    "second_slot_of_one_block": [16 * 16 + 1] * 2,
    "one_level": [16 * 16 * 32],          # 32 slots: the most that are combined in one go
    "two_levels": [16 * 16 * 32 + 1],     # 33
    "two_levels_mixed": [12000, 700, 0, 9001],
    "lanes": _mixed(64, 3000, 1),
    "lanes_and_one": _mixed(65, 3000, 2),
    "kept_lengths_and_one": _mixed(257, 700, 3),
    "round_and_a_half": [320] * 160,      # equal lengths, fewer than compute units
    "more_than_compute_units": _mixed(300, 900, 4),
    "empty": [0] * 70,
}


@pytest.mark.parametrize("name", list(BATCHES))
@pytest.mark.parametrize("fp8,H,D,kvm", [(True, 2, 128, 3), (False, 1, 64, 8), (True, 4, 64, 1), (False, 2, 128, 8)])
def test_slots(torch_cuda, name, fp8, H, D, kvm):
    say(f"decode slots {name} fp8={fp8} H{H} D{D} kvm{kvm}")
    case = DecodeCase(torch_cuda, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=BATCHES[name], seed=17)
    got = case.run()
    assert close(got, case.oracle()).all()


@pytest.mark.parametrize("splits", [1, 2, 3, 64])
@pytest.mark.parametrize("fill", [0x00, 0xFF, None])
def test_any_split_count_and_any_workspace_contents(torch_cuda, splits, fill):
    """Nothing is assumed of the workspace: zeros, all ones or random bytes,
    at an address that is a multiple of 4 only."""
    torch = torch_cuda
    say(f"decode splits {splits}, workspace {fill}")
    case = DecodeCase(torch, fp8=True, layers=1, H=2, D=128, kvm=6, seq_lens=[5000, 31, 2222], seed=18)
    n = P.decode_workspace_bytes(case.batch, case.H * case.kvm, case.D, splits)
    want, first = case.oracle(), None
    for rep in range(3):
        room = torch.randint(0, 256, (n + 16,), dtype=torch.uint8, device="cuda") if fill is None else \
            torch.full((n + 16,), fill, dtype=torch.uint8, device="cuda")
        got = case.run(splits=splits, ws=room[4:4 + n])
        assert close(got, want).all(), rep
        first = got if first is None else first
        assert np.array_equal(got, first), rep  # combined in slot order, whoever is last
        assert (room[:4] == room[0]).all() or fill is None
        assert fill is None or ((room[:4] == fill).all() and (room[n + 4:] == fill).all())


def test_replays_share_a_workspace_with_other_launches(torch_cuda):
    """A captured launch replays with the same ticket tag: with other launches'
    partials in its workspace between replays, and with other lengths."""
    torch = torch_cuda
    say("decode graph replays on a shared workspace")
    case = DecodeCase(torch, fp8=False, layers=1, H=2, D=128, kvm=6, seq_lens=[6000, 900, 40, 3333], seed=19)
    other = DecodeCase(torch, fp8=True, layers=1, H=3, D=64, kvm=5, seq_lens=[2000, 2500], seed=20)
    n = max(P.decode_workspace_bytes(4, 12, 128, 32), P.decode_workspace_bytes(2, 15, 64, 32))
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device="cuda")
    lens = case.s_dev.clone()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            P.paged_decode(case.view, P.PBE_KV_BF16, 0, 0, case.kv, case.layer, case.q.data_ptr(), case.out.data_ptr(),
                           case.batch, 12, case.t_dev.data_ptr(), lens.data_ptr(), case.max_blocks, 32, ws.data_ptr(),
                           ws.numel(), stream_ptr(torch))
    torch.cuda.synchronize()
    want_other = other.oracle()
    for rep, now in enumerate([[6000, 900, 40, 3333], [10, 900, 0, 3000], [5999, 1, 33, 16], [6000, 900, 40, 3333]]):
        lens.copy_(torch.tensor(now, dtype=torch.int32))
        case.out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = case.out.cpu().numpy().view(np.uint16)
        eager = torch.tensor(now, dtype=torch.int32, device="cuda")
        case.run(splits=32, seq_lens=eager)
        assert np.array_equal(got, case.out.cpu().numpy().view(np.uint16)), rep
        assert close(other.run(splits=32, ws=ws), want_other).all(), rep


@pytest.mark.parametrize("fp8", [True, False])
def test_a_workspace_in_pinned_host_memory_takes_no_atomics(torch_cuda, fp8):
    """Host memory is accepted as a workspace. Arrival tickets there would rest
    on atomics that the link may not carry (no output, or a wait without end),
    so nothing of it is touched by them: it keeps its bytes or gets partials."""
    torch = torch_cuda
    say(f"decode fp8={fp8}, pinned host workspace")
    case = DecodeCase(torch, fp8=fp8, layers=1, H=2, D=128, kvm=6, seq_lens=[5000, 31, 0, 2222], seed=22)
    n = P.decode_workspace_bytes(case.batch, 12, 128, 128)
    want = case.oracle()
    for splits in (0, 1, 64):
        ws = torch.zeros(n, dtype=torch.uint8, pin_memory=True)
        for _ in range(2):
            case.out.fill_(7)
            assert close(case.run(splits=splits, ws=ws), want).all(), splits


def test_a_batch_beyond_the_threads_of_one_launch(torch_cuda):
    """8.5 million sequences of one KV head: more workgroups than a launch
    takes. The same 128 sequences over and over, so every row is known."""
    torch = torch_cuda
    say("decode of 8.5 million sequences")
    H, D, n, times = 1, 64, 128, 66500
    small = DecodeCase(torch, fp8=True, layers=1, H=H, D=D, kvm=1, seq_lens=[1 + i % 40 for i in range(n)], seed=23)
    want = small.run(splits=1)
    assert close(want, small.oracle()).all()
    want = small.out.clone()
    batch = n * times
    q, tables, lens = (x.repeat(times, *([1] * (x.dim() - 1))) for x in (small.q, small.t_dev, small.s_dev))
    out = torch.zeros_like(q)
    ws = torch.empty(P.decode_workspace_bytes(batch, 1, D, 1), dtype=torch.uint8, device="cuda")
    P.paged_decode(small.view, P.PBE_KV_FP8_E4M3, small.scales.data_ptr(), small.scales.numel() * 4, small.kv, small.layer, q.data_ptr(),
                   out.data_ptr(), batch, 1, tables.data_ptr(), lens.data_ptr(), small.max_blocks, 1, ws.data_ptr(), ws.numel(),
                   stream_ptr(torch))
    torch.cuda.synchronize()
    assert bool((out.view(times, n, -1) == want.view(1, n, -1)).all())


@pytest.mark.parametrize("fp8,H,D,kvm,lens", [
    (False, 4, 128, 2, [300] * 5 + [2000, 8210, 0]),      # 514 table columns x 8 x 4: over 64 blocks of a head per workgroup
    (False, 4, 128, 7, [600] * 13 + [2500]),              # over 32, a batch of 12 or more
    (True, 8, 64, 1, [1300] * 9),                         # 8 heads, FP8: over 20
    (True, 2, 64, 7, [200] * 7 + [16600]),               # 64-byte rows: over 64
])
def test_small_batches_of_paired_heads(torch_cuda, fp8, H, D, kvm, lens):
    say(f"decode paired heads, a batch of {len(lens)}: fp8={fp8} H{H} D{D} kvm{kvm}")
    case = DecodeCase(torch_cuda, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=lens, seed=24)
    assert close(case.run(), case.oracle()).all()
