"""The decode reader cuts a batch into slots of about equal length, or into
equal splits where those are faster: batches at the edges of these rules (one
slot each, two combine levels, more sequences than a wave has lanes or than the
GPU has compute units, lengths that decide), small workspaces, and workspaces
that hold anything, against the float64 oracle (tolerance: close() of
test_gpu_decode). Each case checks on the CPU that it is at the edge it names."""
import numpy as np
import pytest

import pbe_handoff as P
from oracle import oracle as O
from tests.conftest import say
from tests.gpu_util import stream_ptr
from tests.test_decode_plan import EITHER, SPLITS, plan
from tests.test_gpu_decode import DecodeCase, bf16_to_f64, close

pytestmark = pytest.mark.gpu


def _mixed(n, most, seed):
    r = np.random.default_rng(seed)
    lens = [int(x) for x in np.exp(r.uniform(0, np.log(most), n))]
    lens[0], lens[-1] = most, lens[-1] if n == 1 else 0
    return lens


WHOLE, DIRECT = 24, 64  # blocks of a sequence that stays whole; slots that are combined in one go


def cut(case, splits=0):
    """The slots of every sequence, by the rule the kernel follows."""
    s = splits or P.decode_splits(case.batch, case.H, case.max_blocks, P.PBE_KV_FP8_E4M3 if case.fp8 else P.PBE_KV_BF16)
    got = plan((case.batch, case.H, case.kvm, case.D, case.fp8, case.max_blocks, s, 256, 1, 4096))[0]
    assert got["mode"] != SPLITS
    least = 8 if case.D * (1 if case.fp8 else 2) >= 256 else 16
    slots, one_round, batch = got["slots"], got["one_round"], case.batch
    n = [(x + 15) // 16 for x in case.seq_lens]
    if slots == batch:
        return [1] * batch, got
    of = lambda x, c: 1 if x <= WHOLE else -(-x // c)
    total, longest, many = sum(n), max(n), batch >= one_round
    for last in (False, True):
        T = slots if many or last else min(slots, one_round)
        extra, mean = T - batch, total // batch if many else 0
        if not many and total <= extra * least and longest <= 1024 * least:
            c = least
        else:
            lo = max(-(-total // T), -(-longest // 1024), mean + mean // 4, least)
            hi = max(lo, min(max(1, longest), -(-total // extra)))
            fits = [lo + w * (hi - lo) // 8 for w in range(8)]
            c = min([x for x in fits if sum(of(y, x) for y in n) <= T] + [hi])
        if many or slots <= one_round or c <= least or total * 4 >= c * one_round * 3:
            break
    return [of(x, max(1, -(-x // of(x, c)))) for x in n], got


def _mixed(n, most, seed):
    r = np.random.default_rng(seed)
    lens = [int(x) for x in np.exp(r.uniform(0, np.log(most), n))]
    lens[0], lens[-1] = most, lens[-1] if n == 1 else 0
    return lens


BATCHES = {
    "whole": [16 * WHOLE] * 3 + [1, 0],
    "whole_and_one_block_more": [16 * WHOLE + 1, 16 * WHOLE, 6400, 1, 400, 0],
    "one_long": [12000, 700, 0, 9001],
    "lanes": _mixed(64, 3000, 1),
    "lanes_and_one": _mixed(65, 3000, 2),
    "kept_lengths_and_one": _mixed(257, 700, 3),
    "more_than_compute_units": _mixed(300, 900, 4),
    "empty": [0] * 70,
}


@pytest.mark.parametrize("name", list(BATCHES))
@pytest.mark.parametrize("fp8,H,D,kvm", [(True, 2, 128, 3), (False, 1, 64, 8), (True, 4, 64, 1), (False, 2, 128, 8)])
def test_slots(torch_cuda, name, fp8, H, D, kvm):
    say(f"decode slots {name} fp8={fp8} H{H} D{D} kvm{kvm}")
    case = DecodeCase(torch_cuda, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=BATCHES[name], seed=17)
    k, _ = cut(case)
    if name == "whole" or name == "empty":
        assert max(k) == 1
    if name == "whole_and_one_block_more":
        assert k[0] > 1 and k[1] == 1
    got = case.run()
    assert close(got, case.oracle()).all()


@pytest.mark.parametrize("fp8,H,D,kvm,others", [
    (False, 2, 128, 6, 3), (True, 2, 128, 3, 3), (False, 2, 64, 7, 3), (True, 1, 64, 2, 3),
    (False, 2, 128, 8, 17), (True, 4, 64, 1, 8), (False, 2, 64, 7, 17),  # two KV heads per workgroup
])
@pytest.mark.parametrize("more", [0, 1])
def test_one_and_two_levels_of_combining(torch_cuda, fp8, H, D, kvm, others, more):
    """A sequence of exactly as many slots as are combined in one go, and of one more."""
    least = 8 if D * (1 if fp8 else 2) >= 256 else 16
    say(f"decode levels fp8={fp8} H{H} D{D} kvm{kvm} {DIRECT + more} slots")
    case = DecodeCase(torch_cuda, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=[5] * others + [16 * least * DIRECT + more], seed=25)
    k, got = cut(case)
    assert k[-1] == DIRECT + more and got["hshift"] == (others >= 8)
    assert close(case.run(), case.oracle()).all()


def test_a_second_round_of_slots(torch_cuda):
    """Equal FP8 sequences that would leave a quarter of one round idle."""
    say("decode slots, two rounds")
    case = DecodeCase(torch_cuda, fp8=True, layers=1, H=2, D=128, kvm=6, seq_lens=[500] * 160, seed=26)
    k, got = cut(case)
    assert got["one_round"] == 256 and got["slots"] == 320 and set(k) == {2}
    assert close(case.run(), case.oracle()).all()


@pytest.mark.parametrize("fp8", [True, False])
@pytest.mark.parametrize("batch", [3, 20])
def test_more_blocks_than_a_wave_holds_ids_of(torch_cuda, fp8, batch):
    """Unsplit contexts: a wave keeps the next 64 block ids, of every 8th block
    of the sequence, or of every 4th where two KV heads share the workgroup."""
    every = 4 if batch > 16 else 8
    edge = 16 * 64 * every
    say(f"decode unsplit, fp8={fp8} a batch of {batch}")
    case = DecodeCase(torch_cuda, fp8=fp8, layers=1, H=2, D=128, kvm=2, seq_lens=[edge, edge + 1, 20000] + [7] * (batch - 3), seed=27)
    k, got = cut(case, 1)
    assert max(k) == 1 and got["hshift"] == (batch > 16)
    assert close(case.run(1), case.oracle()).all()


EITHER_BATCHES = [  # fp8, H, D, kvm, sequences, blocks
    (False, 2, 128, 2, 130, 64), (True, 4, 128, 1, 65, 64), (False, 2, 64, 2, 130, 64), (False, 5, 64, 1, 32, 160), (True, 8, 128, 1, 30, 192),
]


@pytest.mark.parametrize("fp8,H,D,kvm,n,blocks", EITHER_BATCHES)
def test_lengths_choose_between_splits_and_slots(torch_cuda, fp8, H, D, kvm, n, blocks):
    """Batches for which the kernels look at the lengths: equal ones, down to 7/8
    of the longest, one block less (slots), an empty one, and a bad table."""
    torch = torch_cuda
    say(f"decode either fp8={fp8} H{H} D{D} kvm{kvm} {n} x {16 * blocks}")
    case = DecodeCase(torch, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=[16 * blocks] * n, seed=28)
    got = plan((n, H, kvm, D, fp8, blocks, P.decode_splits(n, H, blocks, P.PBE_KV_FP8_E4M3 if fp8 else P.PBE_KV_BF16), 256, 1, 4096))[0]
    assert got["mode"] == EITHER
    alike = -(-blocks * 7 // 8)  # the fewest blocks that are about equal
    for last in (16 * blocks, 16 * alike - 15, 16 * alike - 16, 1, 0):
        lens = [16 * blocks - 3 * (i % 11) for i in range(n - 1)] + [last]
        lens[0] = 16 * blocks
        out = case.run(seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
        want = O.paged_decode(case.host, fp8, case.host_scales, 1, H, D, case.layer, case.q_host, case.tables, lens)
        assert close(out, want).all(), last
    tables = case.tables.copy()
    tables[1, 5] = 1 << 30
    equal = case.oracle()
    for bad in ([1], [1, 2]):  # a bad id, in splits; a bad length too, which has no blocks: in slots
        lens = [16 * blocks] * n
        if 2 in bad:
            lens[2] += 1
        out = case.run(tables=torch.from_numpy(tables).cuda(), seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
        good = [b for b in range(n) if b not in bad]
        assert np.isnan(out[bad]).all() and close(out[good], equal[good]).all()


def test_a_replayed_choice_follows_the_lengths(torch_cuda):
    """One captured call, replayed over equal and over mixed lengths, with the
    eager call between the replays on the same workspace."""
    torch = torch_cuda
    say("decode either, graph replays")
    fp8, H, D, kvm, n, blocks = EITHER_BATCHES[0]
    case = DecodeCase(torch, fp8=fp8, layers=1, H=H, D=D, kvm=kvm, seq_lens=[16 * blocks] * n, seed=29)
    splits = P.decode_splits(n, H, blocks, P.PBE_KV_BF16)
    ws = torch.full((P.decode_workspace_bytes(n, H * kvm, D, splits),), 0xFF, dtype=torch.uint8, device="cuda")
    lens, side, graph = case.s_dev.clone(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            P.paged_decode(case.view, P.PBE_KV_BF16, 0, 0, case.kv, case.layer, case.q.data_ptr(), case.out.data_ptr(), n, H * kvm,
                           case.t_dev.data_ptr(), lens.data_ptr(), blocks, splits, ws.data_ptr(), ws.numel(), stream_ptr(torch))
    torch.cuda.synchronize()
    for now in ([16 * blocks] * n, [1 + 7 * i for i in range(n)], [16 * blocks - 5] * n, [16 * blocks] * 5 + [0] * (n - 5), [16 * blocks] * n):
        lens.copy_(torch.tensor(now, dtype=torch.int32))
        case.out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = case.out.cpu().numpy().view(np.uint16)
        case.run(splits=splits, seq_lens=lens, ws=ws)
        assert np.array_equal(got, case.out.cpu().numpy().view(np.uint16))
        assert close(bf16_to_f64(got), O.paged_decode(case.host, fp8, None, 1, H, D, case.layer, case.q_host, case.tables, now)).all()


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
        around = torch.cat([room[:4], room[n + 4:]]).clone()
        got = case.run(splits=splits, ws=room[4:4 + n])
        assert close(got, want).all(), rep
        first = got if first is None else first
        assert np.array_equal(got, first), rep  # combined in slot order, whoever is last
        assert torch.equal(torch.cat([room[:4], room[n + 4:]]), around)


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
