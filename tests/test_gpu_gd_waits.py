"""gate_up_down's single kernel beside its waits: a down unit that leaves its block to the unit that forms h gives the bits
of the launch whose units wait (tests/test_gd_schedule.py is the rule's model), and launches that overlap give theirs."""
import numpy as np
import pytest

from cases import Case, Dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import exl3c4
    exl3c4.lib()
    return torch


@pytest.mark.parametrize("n_tok,top_k,n_expert,geoms,bits,dn_bits,cb,drop", [
    (4, 10, 64, [(512, 256)], 4, 4, "mul1", 0.0),               # 40 rows: the fewest whose units go to all XCDs
    (8, 10, 128, [(512, 256), (256, 128)], 3, 6, "mul1", 0.05),  # a narrower class's blocks wait for nothing
    (7, 8, 20, [(256, 384)], 8, 8, "mcg", 0.1),                 # chunks of several rows
    (1, 41, 64, [(6144, 128)], 2, 2, "mul1", 0.0),              # 48 blocks: the most a row's counter has a bit for
    (1, 41, 64, [(6272, 128)], 2, 2, "3inst", 0.0),             # 49: a list an XCD, no unit leaves
    (3, 13, 48, [(512, 256)], 5, 5, "mul1", 0.0),               # 39 rows: a list an XCD
    (56, 1, 3, [(256, 1536)], 4, 4, "mul1", 0.0)])              # chunks of 16 rows, an h of twelve blocks: slow to form
def test_units_that_leave_give_the_bits_of_units_that_wait(torch_cuda, n_tok, top_k, n_expert, geoms, bits, dn_bits, cb,
                                                           drop):
    import exl3c4 as ex
    import oracle
    torch = torch_cuda
    case = Case(seed=900 + n_tok * top_k, n_tok=n_tok, top_k=top_k, n_expert=n_expert, geoms=geoms, bits=bits, cb=cb,
                dn_bits=dn_bits, drop=drop)
    dev = Dev(case)
    N = max(d["rows"] for d in dev.tabs["dn"])
    _, _, _, row_of = oracle.moe_scatter_full(case.ids, n_expert)
    w = torch.from_numpy(np.random.default_rng(9).random((n_tok, top_k)).astype(np.float32)).cuda()
    rt = torch.from_numpy(row_of).cuda()
    y0, out0 = dev.out(N, fill=0x1234), dev.out(N, fill=0x1234, rows=n_tok)
    o = dev.gd_op(y0)
    assert case.T >= ex.GD_FUSE_MIN_T and not ex.is_prefill(case.T, n_expert)
    assert ex.launch(o, dev.scratch(o)) == 0 and ex.moe_gather(y0, True, w, rt, out0) == 0
    ctr = dev.guard(ex.ctr_bytes(o), fill=0)
    for polls in (0, 1, 4, 128):
        y, out = dev.out(N, fill=0x1234), dev.out(N, fill=0x1234, rows=n_tok)
        o = dev.gd_op(y)
        print(f"T {case.T} {geoms} K {bits}/{dn_bits} {cb} polls {polls}", flush=True)
        assert ex.launch_leaving(o, dev.scratch(o), ctr.view, w, rt, out, polls) == 0
        torch.cuda.synchronize()
        assert torch.equal(y, y0) and torch.equal(out, out0)
        assert int(torch.count_nonzero(ctr.view)) == 0 and ctr.ok()
    assert ex.launch_leaving(o, dev.scratch(o), ctr.view, w, rt, out, 129) == -12
    dev.check_guards("launch_leaving")


def test_launches_on_two_streams_each_give_their_bits(torch_cuda):
    """Two streams, each with its own scratch, counter block and output, run launches of 320 rows over 512 experts at once
    (more waiting down units than the card has slots): every output the bits of the launch alone, both blocks zero."""
    import exl3c4 as ex
    torch = torch_cuda
    M, k, E, H, W, K = 32, 10, 512, 2048, 512, 4
    g = torch.Generator(device="cuda").manual_seed(17)

    keep = []                                                   # a class holds addresses

    def codes(nbytes):
        keep.append(torch.randint(0, 256, (E, nbytes), dtype=torch.uint8, device="cuda", generator=g))
        return keep[-1]

    def scales(n, mag):
        s = torch.randint(0, 2, (E, n), device="cuda", generator=g).float() * 2 - 1
        keep.append((s * (torch.rand((E, n), device="cuda", generator=g) + 0.5) * mag).half().view(torch.int16))
        return keep[-1]
    gu = [ex.make_class(2 * W, H, codes=codes(2 * W * H * K // 8), suh=scales(H, 1.0), suh1=scales(H, 1.0),
                        svh=scales(2 * W, H ** -0.5), dn_suh=scales(W, 1.0))]
    dn = [ex.make_class(H, W, codes=codes(H * W * K // 8), svh=scales(H, W ** -0.5))]
    x = torch.randn((M, H), device="cuda", generator=g).half().view(torch.int16)
    w, ids = torch.zeros((M, k), device="cuda"), torch.zeros((M, k), dtype=torch.int32, device="cuda")
    st, row_of = (torch.zeros(M * k, dtype=torch.int32, device="cuda") for _ in range(2))
    off = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
    logits = torch.randn((M, E), device="cuda", generator=g)
    assert ex.router_topk_scatter(logits, k, True, ids, w, st, off, None, row_of) == 0

    def launch(y, out, stream):
        o = ex.make_op(ex.GU_DN, K, "mul1", gu, x, st, off, y, M, k, dn=dn)
        scratch = ex.alloc_scratch(o)
        ctr = torch.zeros(ex.ctr_bytes(o), dtype=torch.uint8, device="cuda")
        keep.append(scratch)
        return lambda: ex.launch_gather(o, scratch, ctr, w, row_of, out, stream), ctr

    def bufs():
        return (torch.zeros((M * k, H), dtype=torch.int16, device="cuda"),
                torch.zeros((M, H), dtype=torch.int16, device="cuda"))
    y0, out0 = bufs()
    assert launch(y0, out0, torch.cuda.current_stream())[0]() == 0
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out0.view(torch.float16)).all()) and int(torch.count_nonzero(out0)) > 0
    sides = []
    for _ in range(2):
        y, out = bufs()
        sides.append((y, out, *launch(y, out, torch.cuda.Stream())))
    torch.cuda.synchronize()                                    # both sides' buffers are zero before either runs
    print("two streams, 20 launches each", flush=True)
    for _ in range(20):
        for side in sides:
            assert side[2]() == 0
    torch.cuda.synchronize()
    for y, out, _, ctr in sides:
        assert torch.equal(y, y0) and torch.equal(out, out0)
        assert int(torch.count_nonzero(ctr)) == 0
